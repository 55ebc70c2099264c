"""Adapter factors that start off a 16-byte boundary (parameters viewed out of one
flat buffer) against aligned copies of themselves."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _factors(dtype, h, d, r, off):
    g = torch.Generator(device="cuda").manual_seed(3)

    def t(*shape, std=0.02):
        v = (torch.randn(shape, device="cuda", generator=g) * std).to(dtype)
        if off:
            v = torch.empty(v.numel() + 1, dtype=dtype, device="cuda")[1:].view(shape).copy_(v)
        return v.requires_grad_()
    # gate, up (A [r, h], B [d, r]) and down (A [r, d], B [h, r])
    return [(t(r, i), t(o, r, std=0.05)) for o, i in ((d, h), (d, h), (h, d))]


def _run(function, dtype, n, mode, off):
    from compact_amd import flashffn as F
    h, d, r = 320, 704, 8
    g = torch.Generator(device="cuda").manual_seed(1)

    def rnd(*shape, std=1.0):
        return (torch.randn(shape, device="cuda", generator=g) * std).to(dtype)
    x, gy = rnd(n, h).requires_grad_(), rnd(n, h)
    wg, wu, wd = rnd(d, h, std=0.05), rnd(d, h, std=0.05), rnd(h, d, std=0.05)
    (ag, bg), (au, bu), (ad, bd) = f = _factors(dtype, h, d, r, off)
    tail = (2.0, 2.0, 2.0, mode, 64)
    if function == "v3":
        y = F.FlashFFNv3Function.apply(x, wg, ag, bg, wu, au, bu, wd, ad, bd, *tail)
    else:
        y = F.FlashFFNv3AdapterFunction.apply(x, wg, ag, bg, None, None, wu, au, bu, None, None, wd,
                                              ad, bd, None, None, *tail)
    grads = torch.autograd.grad(y, [x] + [t for pair in f for t in pair], gy)
    return [y.detach()] + list(grads)


@pytest.mark.parametrize("function", ["v3", "adapter"])
@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("n,mode", [(4, "int8"), (300, "int8"), (300, "recompute")])
def test_unaligned_factors_equal_aligned_copies(function, dt, n, mode):
    """The same products; the ones whose own operand is a factor may run on the
    general-layout kernel, another order of the same fp32 sums, so outputs agree to
    a few roundings of their 16-bit steps (2^-8 bf16, 2^-11 fp16, relative)."""
    got, ref = (_run(function, DT[dt], n, mode, off) for off in (True, False))
    bound = 4 * (2.0 ** -8 if dt == "bf16" else 2.0 ** -11)
    for i, (u, v) in enumerate(zip(got, ref)):
        assert u.shape == v.shape
        rel = ((u.double() - v.double()).norm() / v.double().norm()).item()
        assert rel < bound, (i, rel)

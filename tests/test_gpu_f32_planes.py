"""fp32 products on the bf16 MFMAs (three bf16 planes per operand) against
float64 and the general-layout kernel."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(*shape, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, device="cuda", generator=g)


def _operands(layout, m, n, k, seed=0):
    a = _rand(m, k, seed=seed) if layout[0] == "n" else _rand(k, m, seed=seed).t()
    b = _rand(n, k, seed=seed + 1).t() if layout[1] == "t" else _rand(k, n, seed=seed + 1)
    return a, b


def _errors(got, a, b):
    """(relative Frobenius error, largest error over |A| |B|) against float64."""
    ref = a.double() @ b.double()
    err = (got.double() - ref).abs()
    return ((err.norm() / ref.norm()).item(),
            (err / (a.double().abs() @ b.double().abs())).max().item())


@pytest.mark.parametrize("layout", ["nt", "nn", "tn", "tt"])
@pytest.mark.parametrize("m,n,k", [(8, 8, 64), (136, 264, 192), (1, 128, 2048), (520, 2048, 5632),
                                   (2048, 5632, 2048)])
def test_error_no_larger_than_the_fp32_instruction(layout, m, n, k):
    """Each product is off by at most 3 * 2^-24 (the terms left out) and the sum
    rounds once per 32 k: below the general-layout kernel's error, which rounds
    every 2, at every size but the few-k ones, where both are a few ulp."""
    from compact_amd import gemm as G
    if layout[0] == "t" and m % 8:
        m = 8
    a, b = _operands(layout, m, n, k)
    assert G.x3_fits(a, b)
    got = G.mm_x3(a, b, G.Planes())
    rel, worst = _errors(got, a, b)
    rel_any, worst_any = _errors(G.mm_any_kernel(a, b), a, b)
    assert rel <= max(rel_any, 2.0 ** -23) and worst <= max(worst_any, 2.0 ** -22)
    assert torch.equal(got, G.mm_x3(a, b, G.Planes()))


@pytest.mark.parametrize("k", [1, 63, 65, 200])
def test_partial_last_k_tile(k):
    from compact_amd import gemm as G
    a, b = _operands("tn", 136, 264, k)
    assert G.x3_fits(a, b)
    assert _errors(G.mm_x3(a, b, G.Planes()), a, b)[1] < 2.0 ** -22


@pytest.mark.parametrize("m", [72, 2048])
def test_two_pairs_and_alpha(m):
    from compact_amd import gemm as G
    a, b = _operands("nn", m, 264, 448)
    a2, b2 = _operands("nn", m, 264, 448, seed=5)
    P = G.Planes()
    got = G.mm_x3(a, b, P, a2, b2, alpha=0.5)
    ref = 0.5 * (a.double() @ b.double() + a2.double() @ b2.double())
    bound = 2.0 ** -22 * 0.5 * (a.double().abs() @ b.double().abs()
                                + a2.double().abs() @ b2.double().abs())
    assert bool(((got.double() - ref).abs() <= bound).all())
    # an operand read again (here as its transpose) is not split again
    n = len(P._made)
    G.mm_x3(a.t(), a2, P)
    assert len(P._made) == n


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 1e38, 1e17, 1e-31,
                                   1e-40])
@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("m", [64, 640])
def test_values_outside_the_planes_take_the_general_kernel(value, side, m):
    """One such value anywhere gives the general-layout kernel's result bit for
    bit (infinities, NaN, overflow and subnormals as fp32 has them)."""
    from compact_amd import gemm as G
    a, b = _operands("nn", m, 264, 1024)
    (a if side == 0 else b)[5, 7] = value
    got, ref = G.mm_x3(a, b, G.Planes(), alpha=0.5), G.mm_any_kernel(a, b, 0.5, G.ANY_SCALE)
    assert torch.equal(got.view(torch.int32), ref.view(torch.int32))
    got = G.mm_x3(a, b, G.Planes(), a, b)
    ref = G.mm_any_kernel(a, b, 1.0, G.ANY_ADD, out=G.mm_any_kernel(a, b))
    assert torch.equal(got.view(torch.int32), ref.view(torch.int32))


def test_zeros_and_range_edges_stay_on_the_planes():
    from compact_amd import gemm as G
    a, b = _operands("nn", 64, 128, 64)
    a[3, :] = 0.0
    a[4, 1], a[5, 2] = 2.0 ** 55, 2.0 ** -100
    P = G.Planes()
    got = G.mm_x3(a, b, P)
    assert not bool(P._flags.any()) and bool((got[3] == 0).all())
    assert _errors(got[4:], a[4:], b)[1] < 2.0 ** -22


def test_planes_sum_to_the_operand():
    from compact_amd import gemm as G
    x = _rand(33, 264) * torch.exp(8 * _rand(33, 264, seed=3))
    planes, flag = G.Planes().of(x)
    assert torch.equal(planes.double().sum(0).float(), x) and int(flag) == 0


@pytest.mark.parametrize("bad", [lambda t: t[:, 1:], lambda t: t[:, ::2], lambda t: t[:, :60]])
def test_other_views_keep_the_general_kernel(bad):
    from compact_amd import gemm as G
    a, b = _operands("nn", 64, 128, 129)
    v = bad(a)
    assert not G.x3_fits(v, b[:v.shape[1]])


@pytest.mark.parametrize("layout", ["nt", "nn", "tn", "tt"])
@pytest.mark.parametrize("m,n,k", [(8, 8, 64), (264, 200, 128), (520, 384, 448), (256, 1000, 1024)])
@pytest.mark.parametrize("ranges", [1, 2])
def test_192_column_tiles_equal_256(layout, m, n, k, ranges, monkeypatch):
    """The same plane products in the same order, whatever the width of a tile."""
    from compact_amd import gemm as G
    a, b = _operands(layout, m, n, k)
    a2, b2 = _operands(layout, m, n, k, seed=5)
    got = []
    for tiles in (192, 256):
        monkeypatch.setattr(G, "x3_plan", lambda *_: (tiles, ranges))
        got.append((G.mm_x3(a, b, G.Planes()), G.mm_x3(a, b, G.Planes(), a2, b2)))
    assert all(torch.equal(u, v) for u, v in zip(*got))
    assert _errors(got[0][0], a, b)[1] < 2.0 ** -22


@pytest.mark.parametrize("layout", ["nt", "nn", "tn", "tt"])
@pytest.mark.parametrize("m,n,k", [(1000, 776, 512), (264, 2056, 320), (2304, 8, 640)])
def test_panels_equal_the_whole_product(layout, m, n, k, monkeypatch):
    """A product run in panels (its planes over the bound) has the bits of the whole
    one where both take the same tiles, and a value outside the planes' range
    sends its panels to the general-layout kernel."""
    from compact_amd import gemm as G
    monkeypatch.setattr(G, "x3_plan", lambda *_: (256, 1))
    a, b = _operands(layout, m, n, k)
    a2, b2 = _operands(layout, m, n, k, seed=5)
    whole = G.mm_x3(a, b, G.Planes()), G.mm_x3(a, b, G.Planes(), a2, b2)
    monkeypatch.setattr(G.Planes, "KEEP_BYTES", 1 << 20)
    monkeypatch.setattr(G.Planes, "bound", lambda self, *_: self.KEEP_BYTES)
    assert G._x3_panels(m, n, k, 1 << 20) != (m, n)
    P = G.Planes()
    assert torch.equal(whole[0], G.mm_x3(a, b, P))
    assert torch.equal(whole[1], G.mm_x3(a, b, P, a2, b2))
    a[m - 1, 3] = float("inf")
    got, ref = G.mm_x3(a, b, G.Planes()), G.mm_any_kernel(a, b)
    assert torch.equal(got[m - 1].view(torch.int32), ref[m - 1].view(torch.int32))
    assert bool(got[:m - 1].isfinite().all())


@pytest.mark.parametrize("train,mode", [("full", "int8"), ("full", "recompute"), ("none", "int8")])
def test_peak_memory_of_a_step(train, mode, monkeypatch):
    """An fp32 step holds at most Planes.KEEP_BYTES of planes and 64 MiB of split
    partials (256 tiles) beside what it holds on the general-layout kernel."""
    from compact_amd import flashffn as F
    from compact_amd import gemm as G
    n, h, d = 8192, 2048, 5632
    x, gy = _rand(n, h, seed=1), _rand(n, h, seed=2)
    ws = [_rand(*s, seed=3) * 0.02 for s in ((d, h), (d, h), (h, d))]
    for t in [x] + ws:
        t.requires_grad_(train == "full")

    def step():
        y = F.FlashFFNv3Function.apply(x, ws[0], None, None, ws[1], None, None, ws[2], None, None,
                                       0.0, 0.0, 0.0, mode, 64)
        return torch.autograd.grad(y, [x] + ws, gy) if train == "full" else y

    def peak():
        step()
        torch.cuda.synchronize()
        base = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        out = step()
        torch.cuda.synchronize()
        del out
        return torch.cuda.max_memory_allocated() - base
    planes = peak()
    monkeypatch.setattr(G, "x3_fits", lambda a, b: False)
    general = peak()
    print(f"{train} {mode}: {general / 2**20:.0f} MiB on the general kernel, {planes / 2**20:.0f}")
    assert planes <= general + G.Planes.KEEP_BYTES + (64 << 20)

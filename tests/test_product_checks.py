"""What the product wrappers refuse and how they repair operands, on the CPU:
tensors are taken for device ones and every library call is recorded and
answered with success, so what runs is the host code in front of the launches."""

import pytest
import torch

from compact_amd import _lib, flashffn as F, gemm as G, kernels as K


class _Library:
    """The entry points by name; calls: (name, arguments)."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return 1024 if name.endswith("_bytes") else 0
        return call


@pytest.fixture
def library(monkeypatch):
    lib = _Library()
    monkeypatch.setattr(_lib, "api", lambda: lib)
    monkeypatch.setattr(_lib, "lib", lambda: lib)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True, raising=False)
    for mod in (G, K):
        monkeypatch.setattr(mod, "_stream", lambda t: 0)
    monkeypatch.setattr(G, "_stream_k", lambda dev: None)
    return lib


# weights (gate, up, down) that do not fit x [64, 512] or each other
MISFITS = {
    "wide_gate_up": ((512, 1024), (512, 1024), (512, 512)),
    "narrow_gate_up": ((512, 448), (512, 448), (512, 512)),
    "wide_up": ((512, 512), (512, 1024), (512, 512)),
    "wide_down": ((512, 512), (512, 512), (512, 576)),
    "narrow_down": ((512, 512), (512, 512), (512, 448)),
}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("misfit", MISFITS)
@pytest.mark.parametrize("function", ["v3", "adapter", "topk"])
def test_functions_refuse_weights_that_do_not_fit(library, function, misfit, dtype):
    """Whatever the type's route, a product whose inner dimensions differ is an
    AssertionError and never a launch over part (or past the end) of an operand."""
    x = torch.zeros(64, 512, dtype=dtype)
    wg, wu, wd = (torch.zeros(s, dtype=dtype, requires_grad=True) for s in MISFITS[misfit])
    with pytest.raises(AssertionError):
        if function == "v3":
            F.FlashFFNv3Function.apply(x, wg, None, None, wu, None, None, wd, None, None)
        elif function == "adapter":
            F.FlashFFNv3AdapterFunction.apply(x, wg, None, None, None, None, wu, None, None, None,
                                              None, wd, None, None, None, None)
        else:
            F.FlashFFNFunction.apply(x, wg, wu, wd)


@pytest.mark.parametrize("shapes", [
    ((64, 128), (192, 64)), ((64, 192), (128, 64)),
    ((64, 128), (128, 64), (64, 128), (64, 64)), ((64, 128), (128, 64), (32, 64), (64, 64)),
    ((64, 128), (128, 64), (64, 64), (64, 128))])
def test_fp32_product_checks_every_extent(library, shapes):
    ts = [torch.zeros(s) for s in shapes]
    with pytest.raises(AssertionError):
        G.mm_x3(ts[0], ts[1], G.Planes(), *ts[2:])
    assert not library.calls


def test_fp32_product_refuses_other_types(library):
    a, b = torch.zeros(64, 128), torch.zeros(128, 64)
    for u, v in ((a.bfloat16(), b), (a, b.bfloat16()), (a.double(), b.double())):
        with pytest.raises(AssertionError):
            G.mm_x3(u, v, G.Planes())
    assert not library.calls


def _terms(n, d, r, dtype, rows=None):
    """(P, B, alpha) of a projection's adapter term."""
    return (torch.zeros(n if rows is None else rows, r, dtype=dtype),
            torch.zeros(d, r, dtype=dtype), 2.0)


@pytest.mark.parametrize("r", [4, 8])
@pytest.mark.parametrize("product,factors", [(torch.bfloat16, torch.float16),
                                             (torch.float16, torch.bfloat16),
                                             (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("call", ["mm2", "gate_up", "gate_up_outlier", "down_dgrad"])
def test_adapter_factors_have_the_products_type(library, call, product, factors, r):
    """A factor of another type would be read with the product's bits."""
    n, h, d = 64, 128, 256
    x, w = torch.zeros(n, h, dtype=product), torch.zeros(d, h, dtype=product)
    p, b, s = _terms(n, d, r, factors)

    def run():
        if call == "mm2":
            G.mm2(x, w.t(), lora=[(p, b.t(), s)])
        elif call == "gate_up":
            G.ffn_gate_up(x, w, w, _lib.CACHE_BF16, 64, lora_gate=(p, b, s))
        elif call == "gate_up_outlier":
            e = torch.empty
            out = (e(n, d), e(n, d), e(n, d // 64), e(n, 8), e(n, d), e(n, d // 64), e(n, 8))
            slot = torch.zeros(d, dtype=torch.int16)
            G.ffn_gate_up_outlier(x, w, w, _lib.CACHE_INT8, 64, slot, slot, 8, out,
                                  lora_gate=(p, b, s))
        else:
            hg = torch.zeros(n, d, dtype=product)
            G.ffn_down_dgrad(x, w.t(), _lib.CACHE_BF16, 64, hg, None, hg, None, False,
                             lora=(p, b.t().contiguous(), s))
    with pytest.raises(AssertionError):
        run()
    assert not library.calls


def test_adapter_rows_cover_the_products_rows(library):
    x, w = torch.zeros(64, 128, dtype=torch.bfloat16), torch.zeros(256, 128, dtype=torch.bfloat16)
    for r in (4, 8):
        p, b, s = _terms(64, 256, r, torch.bfloat16, rows=63)
        with pytest.raises(AssertionError):
            G.mm2(x, w.t(), lora=[(p, b.t(), s)])
    assert not library.calls


@pytest.mark.parametrize("change", ["x1 rows", "x1 columns", "q1 rank", "q1 columns", "p1 rows",
                                    "x1 type", "all of pair 1", "p0 rows", "odd rank"])
def test_dual_pass_of_two_checks_shapes_and_types(library, change):
    """The two tensors' strides may agree where their shapes or types do not."""
    T, N, R, bf = 64, 512, 8, torch.bfloat16
    base = torch.zeros(T, N, dtype=bf), torch.zeros(R, N, dtype=bf), torch.zeros(T, R, dtype=bf)
    x0, q0, p0 = base
    x1, q1, p1 = base
    half = torch.float16
    x1 = {"x1 rows": x0[:32], "x1 columns": x0[:, :256], "x1 type": x0.to(half)}.get(change, x1)
    q1 = {"q1 rank": q0[:4], "q1 columns": q0[:, :256]}.get(change, q1)
    p1 = p0[:32] if change == "p1 rows" else p1
    p0 = p0[:32] if change == "p0 rows" else p0
    if change == "all of pair 1":
        x1, q1, p1 = (t.to(half) for t in base)
    if change == "odd rank":
        q0 = q1 = q0[:4]
        p0 = p1 = torch.zeros(T, 4, dtype=bf)
    with pytest.raises(AssertionError):
        G.skinny_dual_pair(x0, q0, p0, 1.0, x1, q1, p1, 1.0)
    assert not library.calls
    assert G.skinny_dual_pair(*base, 1.0, *base, 1.0) is not None


def _off(t):
    """t's values one element into a buffer of their own: whole rows, a base that
    is not on 16 bytes."""
    flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:]
    return flat.view(t.shape).copy_(t)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_unaligned_factors_are_copied(library, dtype):
    """The kernels read rank factors in 16-byte pieces; a factor viewed out of a
    flat buffer at an odd offset goes in as an aligned copy of itself."""
    x = torch.zeros(64, 512, dtype=dtype)
    wide = torch.zeros(64, 8192, dtype=dtype)
    q, p = torch.zeros(8, 512, dtype=dtype), torch.zeros(64, 8, dtype=dtype)
    qo, po, xo = _off(q), _off(p), _off(x)
    assert all(t.is_contiguous() and t.data_ptr() % 16 for t in (qo, po, xo))
    G.skinny_small(xo, qo, qo)
    G.skinny(_off(wide), _off(torch.zeros(8, 8192, dtype=dtype)))
    G.skinny_t(xo, po)
    G.skinny_dual(xo, qo, po)
    args = {name: a for name, a in library.calls}
    pointers = {"cpt_gemm16_skinny_small": (1, 3, 6), "cpt_gemm16_skinny": (1, 3),
                "cpt_gemm16_skinny_t": (1, 3), "cpt_gemm16_skinny_dual": (1, 3, 6)}
    for name, where in pointers.items():
        assert all(args[name][i] % 16 == 0 for i in where), name
    # an adapter term's P, and its B factor as rows of ranks
    b = _off(torch.zeros(256, 8, dtype=dtype))
    *_, terms, keep = G._lora_args([(po, b.t(), 1.0)], 256, ((512, 256),), x)
    assert terms[0][0] % 16 == 0 and terms[0][1] % 16 == 0 and keep


@pytest.mark.parametrize("r", [1, 2, 8, 24])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("function", ["v3", "adapter"])
def test_b_factors_stored_transposed(library, function, dtype, r):
    """A B factor [d, r] that is the transposed view of [r, d] storage (for rank 1
    a column whose other stride is d) goes into the fused products."""
    n, h, d = 64, 128, 256
    x = torch.zeros(n, h, dtype=dtype)
    wg, wu, wd = (torch.zeros(s, dtype=dtype) for s in ((d, h), (d, h), (h, d)))
    (ag, bg), (au, bu), (ad, bd) = ((torch.zeros(r, i, dtype=dtype, requires_grad=True),
                                     torch.zeros(r, o, dtype=dtype).t().requires_grad_())
                                    for o, i in ((d, h), (d, h), (h, d)))
    assert bg.stride() == (1, d)
    if function == "v3":
        y = F.FlashFFNv3Function.apply(x, wg, ag, bg, wu, au, bu, wd, ad, bd, 2.0, 2.0, 2.0, "bf16")
    else:
        y = F.FlashFFNv3AdapterFunction.apply(x, wg, ag, bg, None, None, wu, au, bu, None, None, wd,
                                              ad, bd, None, None, 2.0, 2.0, 2.0, "bf16")
    y.backward(torch.zeros_like(y))
    assert bg.grad.shape == (d, r)


@pytest.mark.parametrize("ranks", [(8, 17), (16, 12), (24, 4), (8, 24)])
@pytest.mark.parametrize("function", ["v3", "adapter"])
def test_gate_and_up_of_two_ranks(library, function, ranks):
    """Adapters of two ranks of which one is no multiple of 8: the backward's
    dg B_g and du B_u stand side by side only where both halves' rows are aligned."""
    n, h, d, bf = 300, 128, 512, torch.bfloat16
    x = torch.zeros(n, h, dtype=bf, requires_grad=True)
    wg, wu, wd = (torch.zeros(s, dtype=bf) for s in ((d, h), (d, h), (h, d)))
    (ag, bg), (au, bu) = ((torch.zeros(r, h, dtype=bf, requires_grad=True),
                           torch.zeros(r, d, dtype=bf).t().requires_grad_()) for r in ranks)
    if function == "v3":
        y = F.FlashFFNv3Function.apply(x, wg, ag, bg, wu, au, bu, wd, None, None, 2.0, 2.0, 0.0)
    else:
        y = F.FlashFFNv3AdapterFunction.apply(x, wg, ag, bg, None, None, wu, au, bu, None, None, wd,
                                              None, None, None, None, 2.0, 2.0, 0.0)
    y.backward(torch.zeros_like(y))
    assert ag.grad.shape == (ranks[0], h) and bu.grad.shape == (d, ranks[1])


@pytest.mark.parametrize("mode", ["bf16", "recompute"])
@pytest.mark.parametrize("function", ["v3", "adapter"])
@pytest.mark.parametrize("strides", [(1, 1), (256, 1), (7, 1)])
def test_single_rank_down_factor_of_any_strides(library, function, mode, strides):
    """A single-rank A_d [1, d] rides in the down dgrad's epilogue as a row, whatever
    stride its size-1 dimension has (1 where it is a transposed column)."""
    n, h, d, bf = 64, 128, 256, torch.bfloat16
    x = torch.zeros(n, h, dtype=bf, requires_grad=True)
    wg, wu, wd = (torch.zeros(s, dtype=bf) for s in ((d, h), (d, h), (h, d)))
    ad = torch.zeros(d, dtype=bf).as_strided((1, d), strides).requires_grad_()
    bd = torch.zeros(h, 1, dtype=bf, requires_grad=True)
    if function == "v3":
        y = F.FlashFFNv3Function.apply(x, wg, None, None, wu, None, None, wd, ad, bd, 0.0, 0.0, 2.0,
                                       mode)
    else:
        y = F.FlashFFNv3AdapterFunction.apply(x, wg, None, None, None, None, wu, None, None, None,
                                              None, wd, ad, bd, None, None, 0.0, 0.0, 2.0, mode)
    y.backward(torch.zeros_like(y))
    assert ad.grad.shape == (1, d)


def _covered(calls, m, n, base):
    """How often each output of an [m, n] fp32 product at `base` is written."""
    seen = torch.zeros(m, n, dtype=torch.int32)
    for name, a in calls:
        if name == "cpt_gemm_f32x3":
            at, ldc, rows, cols = (a[17] - base) // 4, a[18], a[19], a[20]
            assert ldc == n
            seen[at // n:at // n + rows, at % n:at % n + cols] += 1
    return seen


@pytest.mark.parametrize("left,right", [("nn", "nn"), ("tn", "tt")])
@pytest.mark.parametrize("m,n,k", [(1000, 776, 512), (264, 2048, 320), (2304, 8, 640),
                                   (256, 256, 4096)])
def test_fp32_planes_stay_within_their_bound(library, monkeypatch, m, n, k, left, right):
    """A product whose operands' planes exceed the bound runs in panels that write
    every output once, and holds no more planes at a time than the bound, its larger
    operand's bytes or one 256-wide panel of each operand."""
    limit = 1 << 20
    monkeypatch.setattr(G.Planes, "KEEP_BYTES", limit)
    a = torch.zeros(k, m).t() if left[0] == "t" else torch.zeros(m, k)
    b = torch.zeros(n, k).t() if right[1] == "t" else torch.zeros(k, n)
    P, held = G.Planes(), []
    make = P.of
    P.of = lambda t: (make(t), held.append(P._bytes))[0]
    c = G.mm_x3(a, b, P)
    assert bool((_covered(library.calls, m, n, c.data_ptr()) == 1).all())
    assert max(held) <= max(limit, 4 * max(m, n) * k, 6 * 512 * k)
    assert P._bytes == sum(6 * e[2].numel() for e in P._made.values())
    P.drop(a)
    P.drop(b.t())
    assert not P._made and P._bytes == 0


def test_fp32_planes_of_two_products_are_shared(library):
    """... and made again once others have pushed them out."""
    x, w = torch.zeros(64, 128), torch.zeros(256, 128)
    P = G.Planes()
    G.mm_x3(x, w.t(), P)
    G.mm_x3(x.t(), x, P)
    splits = sum(name == "cpt_split_f32" for name, _ in library.calls)
    assert splits == 2
    P.KEEP_BYTES = 6 * 300 * 128
    G.mm_x3(torch.zeros(128, 128), torch.zeros(128, 128), P)
    assert P._bytes <= P.bound() == P.KEEP_BYTES
    G.mm_x3(x, w.t(), P)
    splits = sum(name == "cpt_split_f32" for name, _ in library.calls)
    assert splits == 6


@pytest.mark.parametrize("m,n,k,planes", [(1, 704, 256, False), (64, 704, 320, False),
                                          (1, 704, 384, True), (2048, 2048, 256, False),
                                          (2048, 5632, 64, False), (2048, 5632, 128, True),
                                          (8, 2048, 64, False), (8, 2048, 2048, True)])
def test_small_fp32_products_keep_the_general_kernel(library, m, n, k, planes):
    """Where its one launch is faster than the splits and what follows them."""
    G.mm_any(torch.zeros(m, k), torch.zeros(n, k).t())
    G.mm_any(torch.zeros(m, k), torch.zeros(n, k).t(), 2.0, G.ANY_SCALE)
    names = {name for name, _ in library.calls}
    assert names == ({"cpt_split_f32", "cpt_gemm_f32x3", "cpt_gemm_any_if"} if planes
                     else {"cpt_gemm_any"})


@pytest.mark.parametrize("n,rows", [(0, 32), (1, 32), (2048, 32), (2049, 33), (8192, 128),
                                    (8193, 128), (100000, 128), (8388480, 128), (8388481, 129)])
def test_column_dot_chunks(library, n, rows):
    """Rows of an fp32 partial: none above 128 while the grid has chunks left."""
    t = torch.zeros(1, 8).expand(n, 8) if n < 1 << 20 else torch.zeros(n, 1, dtype=torch.bfloat16)
    K.col_dot_div(t, t, torch.ones(t.shape[1], dtype=t.dtype))
    (name, args), = library.calls
    assert name == "cpt_col_dot_div_rows" and args[3] == n and args[5] == rows
    assert -(-n // rows) <= 65535

"""Products on 128 x 128 tiles with split k, and fp16 ones (cpt_gemm16,
cpt_ffn_gate_up16), against float64 and against their own unsplit result."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "fp16": torch.float16}
EPS = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11}      # half an ulp, relative


def _rand(*shape, dtype, seed=0, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, device="cuda", generator=g) * scale).to(dtype)


def _gemm16(dt, a, b, a2=None, b2=None, lora=(), splits=1, tiles=128):
    """a [M, K] @ b [K, N] (+ a2 @ b2, + adapter terms) through cpt_gemm16."""
    from compact_amd import _lib
    from compact_amd import gemm as G
    from compact_amd._lib import check
    (M, K), N = a.shape, b.shape[1]
    a, lda, ak = G._layout_a(a)
    b, ldb, bk = G._layout_b(b)
    pair = (None, 0, None, 0, 0)
    if a2 is not None:
        a2, lda2, _ = G._layout_a(a2)
        b2, ldb2, _ = G._layout_b(b2)
        pair = (a2.data_ptr(), lda2, b2.data_ptr(), ldb2, a2.shape[1])
    c = torch.full((M, N), float("nan"), dtype=a.dtype, device=a.device)
    ws = torch.full((max(1, splits) * M * N,), float("nan"), device=a.device)
    r = lora[0][0].shape[1] if lora else 0
    km = 1 if lora and lora[0][1].stride(0) == 1 and r else 0
    t = [(p.data_ptr(), q.data_ptr(), s) for p, q, s in lora] + [(None, None, 0.0)] * 2
    check(_lib.lib().cpt_gemm16(
        _lib.F16 if dt == "fp16" else _lib.BF16, a.data_ptr(), lda, ak, b.data_ptr(), ldb, bk,
        *pair, c.data_ptr(), N, M, N, K, r, r, km, lora[0][1].stride(0) if lora else 0, *t[0],
        *t[1], tiles, splits, ws.data_ptr(), torch.cuda.current_stream().cuda_stream), "gemm16")
    return c


def _close(got, ref, dt, bound):
    """One rounding to the type, plus the fp32 sum's error `bound` = K 2^-24 |A| |B|."""
    err = (got.double() - ref).abs()
    assert bool((err <= 1.01 * EPS[dt] * ref.abs() + bound + 2.0 ** -25).all()), err.max().item()


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("layout", ["nt", "nn", "tn", "tt"])
@pytest.mark.parametrize("m,n,k,splits", [(1, 8, 64, 1), (130, 264, 192, 2), (127, 120, 1024, 5),
                                          (300, 136, 448, 7), (8, 128, 640, 64)])
def test_split_product(dt, layout, m, n, k, splits):
    if layout[0] == "t" and m % 8:
        m = (m + 7) // 8 * 8                        # an MN-major operand's rows are whole vectors
    d = DT[dt]
    a = _rand(m, k, dtype=d, seed=1) if layout[0] == "n" else _rand(k, m, dtype=d, seed=1).t()
    b = _rand(n, k, dtype=d, seed=2).t() if layout[1] == "t" else _rand(k, n, dtype=d, seed=2)
    ref = a.double() @ b.double()
    bound = k * 2.0 ** -24 * (a.double().abs() @ b.double().abs())
    got = _gemm16(dt, a, b, splits=splits)
    _close(got, ref, dt, bound)
    assert torch.equal(got, _gemm16(dt, a, b, splits=splits))


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("k", [1, 63, 65, 1000])
@pytest.mark.parametrize("splits", [1, 3])
def test_partial_last_k_tile(dt, k, splits):
    """Two MN-major operands may end in a partial k-tile: the rows past it, and
    the memory behind them, must not be read into the sum."""
    d = DT[dt]
    abig, bbig = _rand(k + 64, 136, dtype=d, seed=1), _rand(k + 64, 264, dtype=d, seed=2)
    abig[k:] = float("nan")
    bbig[k:] = float("nan")
    a, b = abig[:k].t(), bbig[:k]
    bound = k * 2.0 ** -24 * (a.double().abs() @ b.double().abs())
    _close(_gemm16(dt, a, b, splits=splits), a.double() @ b.double(), dt, bound)


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("splits", [1, 2, 3, 5])
def test_two_pairs_split_across_the_boundary(dt, splits):
    d = DT[dt]
    a, a2 = _rand(77, 320, dtype=d, seed=1), _rand(77, 320, dtype=d, seed=2)
    b, b2 = _rand(320, 264, dtype=d, seed=3), _rand(320, 264, dtype=d, seed=4)
    ref = a.double() @ b.double() + a2.double() @ b2.double()
    bound = 640 * 2.0 ** -24 * (a.double().abs() @ b.double().abs()
                                + a2.double().abs() @ b2.double().abs())
    _close(_gemm16(dt, a, b, a2, b2, splits=splits), ref, dt, bound)


@pytest.mark.parametrize("layout", ["nt", "nn", "tn", "tt"])
@pytest.mark.parametrize("m,n,k,splits", [(1, 8, 128, 2), (260, 264, 448, 3), (520, 136, 1024, 8),
                                          (2048, 4096, 11008, 2)])
def test_split_product_on_large_tiles(layout, m, n, k, splits):
    if layout[0] == "t" and m % 8:
        m = (m + 7) // 8 * 8
    d = DT["bf16"]
    a = _rand(m, k, dtype=d, seed=1) if layout[0] == "n" else _rand(k, m, dtype=d, seed=1).t()
    b = _rand(n, k, dtype=d, seed=2).t() if layout[1] == "t" else _rand(k, n, dtype=d, seed=2)
    ref = a.double() @ b.double()
    bound = k * 2.0 ** -24 * (a.double().abs() @ b.double().abs())
    got = _gemm16("bf16", a, b, splits=splits, tiles=256)
    _close(got, ref, "bf16", bound)
    if layout == "nn":   # two pairs, a range across their boundary, and an adapter term
        p, q = _rand(m, 16, dtype=d, seed=3), _rand(16, n, dtype=d, seed=4)
        got = _gemm16("bf16", a, b, a, b, lora=[(p, q, 0.5)], splits=splits, tiles=256)
        term = 0.5 * (p.double() @ q.double())
        size = 2 * ref.abs() + (2 * ref + term).abs() + 2 * term.abs()
        _close(got, 2 * ref + term, "bf16", 2 * bound + EPS["bf16"] * 1.1 * size)


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("rank", [8, 24, 32])
@pytest.mark.parametrize("q_kmajor", [True, False])
@pytest.mark.parametrize("splits", [1, 4])
def test_adapter_terms(dt, rank, q_kmajor, splits):
    """Each term rounds its product, its scaling and the sum: three roundings
    of the running value and two of the term."""
    d = DT[dt]
    m, n, k = 131, 264, 512
    a, b = _rand(m, k, dtype=d, seed=1), _rand(n, k, dtype=d, seed=2).t()
    lora, ref = [], a.double() @ b.double()
    size = ref.abs()
    for t in range(2):
        p = _rand(m, rank, dtype=d, seed=3 + t)
        q = _rand(n, rank, dtype=d, seed=5 + t).t() if q_kmajor else _rand(rank, n, dtype=d,
                                                                            seed=5 + t)
        term = (0.5 + t) * (p.double() @ q.double())
        lora.append((p, q, 0.5 + t))
        ref, size = ref + term, size + 2 * term.abs() + ref.abs() + term.abs()
    got = _gemm16(dt, a, b, lora=lora, splits=splits)
    bound = EPS[dt] * 1.1 * size + k * 2.0 ** -24 * (a.double().abs() @ b.double().abs())
    _close(got, ref, dt, bound)


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("m,dff", [(1, 8), (129, 136), (300, 520)])
@pytest.mark.parametrize("rank", [0, 8])
@pytest.mark.parametrize("splits", [1, 3])
def test_gate_up(dt, m, dff, rank, splits):
    """h_gate, h_up as the plain product with one term; h_mid the GLU of them."""
    from compact_amd import _lib, kernels
    from compact_amd._lib import check
    d, h = DT[dt], 448
    x = _rand(m, h, dtype=d, seed=1)
    ws = [_rand(dff, h, dtype=d, seed=2 + i, scale=0.1) for i in range(2)]
    xa = _rand(m, 8, dtype=d, seed=4)
    bs = [_rand(dff, 8, dtype=d, seed=5 + i) for i in range(2)]
    out = [torch.full((m, dff), float("nan"), dtype=d, device="cuda") for _ in range(3)]
    work = torch.empty(splits * m * 2 * dff, device="cuda")
    terms = ([xa.data_ptr(), bs[0].data_ptr(), 0.5, xa.data_ptr(), bs[1].data_ptr(), 1.5] if rank
             else [None, None, 0.0] * 2)
    check(_lib.lib().cpt_ffn_gate_up16(
        _lib.F16 if dt == "fp16" else _lib.BF16, x.data_ptr(), ws[0].data_ptr(), ws[1].data_ptr(),
        m, h, dff, *[t.data_ptr() for t in out], rank, rank, *terms, splits, work.data_ptr(),
        torch.cuda.current_stream().cuda_stream), "gate_up16")
    for i in range(2):
        lora = [(xa, bs[i].t(), 0.5 + i)] if rank else []
        ref = _gemm16(dt, x, ws[i].t(), lora=lora, splits=splits)
        assert torch.equal(out[1 + i], ref)
    assert torch.equal(out[0], kernels.silu_mul(out[1], out[2]))


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("m,n,rank", [(2049, 520, 8), (2017, 264, 16), (1340, 264, 24),
                                      (1027, 264, 32)])
@pytest.mark.parametrize("q_kmajor", [True, False])
@pytest.mark.parametrize("splits", [2, 5])
def test_adapter_terms_of_larger_outputs(dt, m, n, rank, q_kmajor, splits):
    """The split sums with the terms on the MFMAs (M N rank above 2^23), ragged in
    rows and columns: test_adapter_terms' bound."""
    d, k = DT[dt], 512
    a, b = _rand(m, k, dtype=d, seed=1), _rand(n, k, dtype=d, seed=2).t()
    lora, ref = [], a.double() @ b.double()
    size = ref.abs()
    for t in range(2):
        p = _rand(m, rank, dtype=d, seed=3 + t)
        q = _rand(n, rank, dtype=d, seed=5 + t).t() if q_kmajor else _rand(rank, n, dtype=d,
                                                                            seed=5 + t)
        term = (0.5 + t) * (p.double() @ q.double())
        lora.append((p, q, 0.5 + t))
        ref, size = ref + term, size + 2 * term.abs() + ref.abs() + term.abs()
    got = _gemm16(dt, a, b, lora=lora, splits=splits)
    bound = EPS[dt] * 1.1 * size + k * 2.0 ** -24 * (a.double().abs() @ b.double().abs())
    _close(got, ref, dt, bound)


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
def test_gate_up_of_larger_outputs(dt):
    test_gate_up(dt, 2049, 520, 8, 3)


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
def test_non_finite_and_subnormal_values(dt):
    """Infinities and NaN travel as in a sum; subnormals of the type count."""
    d = DT[dt]
    a = torch.zeros(64, 128, dtype=d, device="cuda")
    b = torch.eye(128, dtype=d, device="cuda")
    tiny = torch.finfo(d).smallest_normal / 2
    a[0, 3], a[1, 5], a[2, 7], a[3, 9] = float("inf"), float("nan"), tiny, -tiny
    got = _gemm16(dt, a[:, :128], torch.ones(8, 128, dtype=d, device="cuda").t())
    assert bool(torch.isinf(got[0]).all()) and bool(torch.isnan(got[1]).all())
    assert bool((got[2] == tiny).all()) and bool((got[3] == -tiny).all())
    got = _gemm16(dt, b, a.new_full((128, 8), tiny))
    assert bool((got == tiny).all())


def test_split_plan_fills_the_chip_without_empty_ranges():
    from compact_amd import gemm as G
    for m in (1, 4, 64, 200, 512, 1024, 4096):
        for n in (8, 2048, 4096, 11264):
            for nk in (1, 8, 32, 64, 88, 176, 344):
                s = G.split_plan(m, n, nk)
                tiles = -(-m // 128) * -(-n // 128)
                assert 1 <= s <= nk and (s == 1 or (s * tiles <= 256 and nk // s >= 6))
                edge, s = G.tile_plan(m, n, nk)
                tiles = -(-m // edge) * -(-n // edge)
                assert s == 1 or (s * tiles <= 256 and nk // s >= 6)
                assert G.tile_plan(m, n, nk, True)[0] == 128

"""The 128 x 128 tiles of the 16x16x32 loop against its 256 x 256 tiles.

Both sum each output in the same k order, so a product covered by at most 512
small tiles must equal, bit for bit, the same rows of a product large enough
for 256 x 256 tiles (the operands' rows extended by others)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

WIDE = 2048      # 16 small tiles across; TALL rows of them (or of 9) take 256 x 256 tiles
TALL = 60 * 128 + 40


def _rand(*shape, seed=0, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(shape, device="cuda", generator=g) * scale).to(torch.bfloat16)


def _is_small(m, n):
    from compact_amd import gemm as G
    return G.small_tiles(m, n)


@pytest.mark.parametrize("b_kmajor", [True, False])
@pytest.mark.parametrize("m,k,k2", [(1, 64, 0), (127, 128, 0), (128, 192, 0), (129, 1024, 0),
                                    (300, 320, 64), (2048, 256, 512), (2049, 64, 128),
                                    (4096, 320, 0)])
def test_rows_equal_large_tiles(m, k, k2, b_kmajor):
    """A K-major, one and two pairs, 1 to 512 small tiles (both stage counts)."""
    from compact_amd import gemm as G
    a = _rand(TALL, k, seed=1)
    b = _rand(WIDE, k, seed=2) if b_kmajor else _rand(k, WIDE, seed=2).t()
    a2 = _rand(TALL, k, seed=3) if k2 == k else (_rand(TALL, k2, seed=3) if k2 else None)
    b2 = None
    if k2:
        # the pairs share leading dimensions: views of one width
        w = max(k, k2)
        a, a2 = _rand(TALL, w, seed=1)[:, :k], _rand(TALL, w, seed=3)[:, :k2]
        if b_kmajor:
            b, b2 = _rand(WIDE, w, seed=2)[:, :k], _rand(WIDE, w, seed=4)[:, :k2]
        else:
            b2 = _rand(k2, WIDE, seed=4).t()
    assert _is_small(m, WIDE) and not _is_small(TALL, WIDE)
    args = (a, b.t()) if a2 is None else (a, b.t(), a2, b2.t())
    big = G.mm2(*args)
    args = (a[:m], b.t()) if a2 is None else (a[:m], b.t(), a2[:m], b2.t())
    got = G.mm2(*args)
    assert torch.equal(got, big[:m])


@pytest.mark.parametrize("b_kmajor", [True, False])
@pytest.mark.parametrize("m,k", [(8, 64), (136, 128), (2048, 192), (4096, 320)])
def test_mn_major_rows_equal_large_tiles(m, k, b_kmajor):
    """A MN-major (the weight gradients' layout)."""
    from compact_amd import gemm as G
    a = _rand(k, TALL, seed=1)
    b = _rand(WIDE, k, seed=2).t() if b_kmajor else _rand(k, WIDE, seed=2)
    assert torch.equal(G.mm2(a[:, :m].t(), b), G.mm2(a.t(), b)[:m])


@pytest.mark.parametrize("n", [8, 120, 136, 264])
def test_ragged_columns(n):
    """Columns past the last whole tile against a wider product's columns."""
    from compact_amd import gemm as G
    a, b = _rand(TALL, 192, seed=1), _rand(WIDE, 192, seed=2)
    big = G.mm2(a, b.t())
    assert torch.equal(G.mm2(a[:131], b[:n].t()), big[:131, :n])


@pytest.mark.parametrize("rank", [8, 16, 24, 32])
@pytest.mark.parametrize("q_kmajor", [True, False])
def test_adapter_terms_equal_large_tiles(rank, q_kmajor):
    from compact_amd import gemm as G
    m, k = 259, 128
    a, b = _rand(TALL, k, seed=1), _rand(WIDE, k, seed=2)
    terms = []
    for t in range(2):
        q = (_rand(WIDE, rank, seed=5 + t).t() if q_kmajor else _rand(rank, WIDE, seed=5 + t))
        terms.append((_rand(TALL, rank, seed=3 + t), q, 0.5 + t))
    for use in (terms[:1], terms):
        big = G.mm2(a, b.t(), lora=use)
        got = G.mm2(a[:m], b.t(), lora=[(p[:m].contiguous(), q, s) for p, q, s in use])
        assert torch.equal(got, big[:m])


@pytest.mark.parametrize("rank", [0, 8, 32])
@pytest.mark.parametrize("m", [1, 129, 512])
@pytest.mark.parametrize("d", [1032, 2048])
def test_ffn_kernels_equal_large_tiles(m, d, rank):
    """F1 with a bf16 cache or none, B1 on a bf16 cache."""
    from compact_amd import _lib
    from compact_amd import gemm as G
    h = 128
    x, gy = _rand(TALL, h, seed=1), _rand(TALL, h, seed=2)
    wg, wu, wd = (_rand(d, h, seed=3, scale=0.1), _rand(d, h, seed=4, scale=0.1),
                  _rand(h, d, seed=5, scale=0.1))
    kw_big = kw = {}
    dl_big = dl = None
    if rank:
        xa, bg, bu = _rand(TALL, rank, seed=6), _rand(d, rank, seed=7), _rand(d, rank, seed=8)
        kw_big = dict(lora_gate=(xa, bg, 0.5), lora_up=(xa, bu, 1.5))
        kw = dict(lora_gate=(xa[:m], bg, 0.5), lora_up=(xa[:m], bu, 1.5))
        ad = _rand(rank, d, seed=9)
        dl_big, dl = (xa, ad, 0.75), (xa[:m], ad, 0.75)
    assert _is_small(m, 2 * d) and not _is_small(TALL, d)
    big = G.ffn_gate_up(x, wg, wu, _lib.CACHE_BF16, 64, **kw_big)[:3]
    got = G.ffn_gate_up(x[:m], wg, wu, _lib.CACHE_BF16, 64, **kw)[:3]
    assert all(torch.equal(a, b[:m]) for a, b in zip(got, big))
    none = G.ffn_gate_up(x[:m], wg, wu, _lib.CACHE_NONE, 64, **kw)[0]
    assert torch.equal(none, got[0])
    _, hg, hu = big
    big_b = G.ffn_down_dgrad(gy, wd, _lib.CACHE_BF16, 64, hg, None, hu, None, True, lora=dl_big)
    got_b = G.ffn_down_dgrad(gy[:m], wd, _lib.CACHE_BF16, 64, hg[:m], None, hu[:m], None, True,
                             lora=dl)
    assert all(torch.equal(a, b[:m]) for a, b in zip(got_b, big_b))
    # in place over the caller's own cache
    cg, cu = hg[:m].clone(), hu[:m].clone()
    dg, du, _ = G.ffn_down_dgrad(gy[:m], wd, _lib.CACHE_BF16, 64, cg, None, cu, None, False,
                                 lora=dl, inplace=True)
    assert torch.equal(dg, got_b[0]) and torch.equal(du, got_b[1])


@pytest.mark.parametrize("layout", ["nt", "nn", "tn", "tt"])
@pytest.mark.parametrize("m,n", [(5512, 1928), (5128, 2112), (5128, 2104), (1800, 5384),
                                 (11016, 1920)])
@pytest.mark.parametrize("k,k2", [(64, 0), (128, 64), (1088, 128)])
def test_192_column_tiles(layout, m, n, k, k2):
    """Products whose 256 x 256 tiles leave a quarter of a round empty run on 192
    columns: ragged last row and column (8, 184 and 192 columns of the last tile),
    one and two pairs, one round and (11016 rows, MN-major A) two.  The k order is
    that of the 128 x 128 tiles, which take the same columns a part at a time."""
    from compact_amd import gemm as G

    def pair(kk, seed):
        # the pairs share leading dimensions: views of one width
        w = max(k, k2)
        a = (_rand(m, w, seed=seed)[:, :kk] if layout[0] == "n" else _rand(kk, m, seed=seed).t())
        b = (_rand(n, w, seed=seed + 1)[:, :kk].t() if layout[1] == "t"
             else _rand(kk, n, seed=seed + 1))
        return a, b
    args = pair(k, 1) + (pair(k2, 3) if k2 else ())
    wide, narrow = ((m + 255) // 256) * ((n + 255) // 256), ((m + 255) // 256) * ((n + 191) // 192)
    assert not _is_small(m, n) and -(-narrow // 256) <= -(-wide // 256)
    if layout[0] == "n" and wide > 256:
        pytest.skip("K-major A past one round: stream-K shares its tiles (its own k order)")
    got = G.mm2(*args) if k2 else G.mm(*args)
    for r0 in range(0, m, 2048):
        for c0 in range(0, n, 2048):
            part = [t[r0:r0 + 2048] if i % 2 == 0 else t[:, c0:c0 + 2048]
                    for i, t in enumerate(args)]
            assert _is_small(part[0].shape[0], part[1].shape[1])
            ref = G.mm2(*part) if k2 else G.mm2(*part, None, None)
            assert torch.equal(got[r0:r0 + 2048, c0:c0 + 2048], ref)

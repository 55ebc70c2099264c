"""The LoRA backward's two thin products of one tensor in one pass
(cpt_gemm_bf16_skinny_dual): C = x Q^T (the projection) and Z = x^T P (the
token reduction), checked against float32 products of the same bf16
operands (bf16 output rounding: 2^-7 relative plus an fp32 summation
allowance), against the separate skinny kernels within the same bound, for
determinism, and for the Function routed through it against the separate
kernels."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _G():
    from compact_amd import gemm
    return gemm


def rnd(shape, seed, device, scale=1.0):
    g = torch.Generator(device=device).manual_seed(seed)
    return (torch.randn(*shape, device=device, generator=g) * scale).to(torch.bfloat16)


def _close(got, ref, scale):
    got = got.float().cpu()
    tol = 2 ** -7 * ref.abs() + 1e-5 * scale
    return bool(((got - ref).abs() <= tol).all()), float((got - ref).abs().max())


@pytest.mark.parametrize("q_as_b", [False, True])
@pytest.mark.parametrize("T,N,R", [(8192, 11008, 16), (300, 520, 8), (1000, 4096, 32),
                                   (64, 1024, 24), (33, 512, 16)])
def test_skinny_dual_against_fp32(device, T, N, R, q_as_b):
    """q_as_b: Q given as the transposed view of a B factor [N, R] (read in
    place) instead of rank rows [R, N]; same bits either way."""
    G = _G()
    x = rnd((T, N), 1, device)
    q = rnd((R, N), 2, device, 0.05)
    if q_as_b:
        q = q.t().contiguous().t()
    p = rnd((T, R), 3, device, 0.5)
    c, z = G.skinny_dual(x, q, p, 1.0, 2.0)
    c2, z2 = G.skinny_dual(x, q, p, 1.0, 2.0)
    assert torch.equal(c.view(torch.int16), c2.view(torch.int16))
    assert torch.equal(z.view(torch.int16), z2.view(torch.int16))
    xd, qd, pd = x.double().cpu(), q.double().cpu(), p.double().cpu()
    ref_c = xd @ qd.t()
    ref_z = 2.0 * (xd.t() @ pd)
    ok, err = _close(c, ref_c, (xd.abs() @ qd.abs().t()))
    assert ok, err
    ok, err = _close(z, ref_z, 2.0 * (xd.abs().t() @ pd.abs()))
    assert ok, err
    # the separate kernels, within the same bound of each other's reference
    c_sep = G.skinny(x, q, 1.0)
    z_sep = G.skinny_t(x, p, 2.0)
    assert _close(c_sep, ref_c, xd.abs() @ qd.abs().t())[0]
    assert _close(z_sep, ref_z, 2.0 * (xd.abs().t() @ pd.abs()))[0]


def test_skinny_dual_into_a_column_half(device):
    """C written into the column half of a wider buffer (the Function's
    [grad_h_gate B_g | grad_h_up B_u] block); the other half is untouched."""
    G = _G()
    T, N, R = 700, 1536, 16
    x, q, p = rnd((T, N), 4, device), rnd((R, N), 5, device, 0.05), rnd((T, R), 6, device)
    buf = torch.full((T, 2 * R), 7.0, dtype=torch.bfloat16, device=device)
    c, _ = G.skinny_dual(x, q, p, out_c=buf[:, R:])
    alone, _ = G.skinny_dual(x, q, p)
    assert torch.equal(buf[:, R:].view(torch.int16), alone.view(torch.int16))
    assert (buf[:, :R] == 7.0).all()


@pytest.mark.parametrize("mode,group", [("int4", 64), ("int8", 128)])
def test_function_dual_route_matches_separate(device, mode, group):
    """FlashFFNv3Function with LoRA on gate/up/down: the backward through the
    one-pass kernel against the separate projection and reduction kernels:
    y bit-identical (the forward is the same), the B gradients within the
    bf16 rounding of each other, and grad_x and the A gradients (which take
    the projection through further products) within rel 1e-2."""
    import compact_amd
    from compact_amd import flashffn as FF
    from oracle import flashffn_ref as R
    ps = R.synthetic_param_set("all", 1024, 2048, 16, 2.0, seed=7, dtype=torch.bfloat16,
                               device=device, peft_init=True, b_std=0.01)
    gen = torch.Generator(device=device).manual_seed(8)
    x = torch.randn(2, 512, 1024, device=device, generator=gen).to(torch.bfloat16)
    gy = torch.randn(2, 512, 1024, device=device, generator=gen).to(torch.bfloat16)
    res = {}
    for dual in (True, False):
        FF._DUAL_SKINNY = dual
        res[dual] = R.run_function_grads(compact_amd.FlashFFNv3Function.apply, ps, x, gy, mode,
                                         group, True, 0.01)
    FF._DUAL_SKINNY = True
    (g1, y1), (g0, y0) = res[True], res[False]
    assert torch.equal(y1.view(torch.int16), y0.view(torch.int16))
    for k in g1:
        if k.startswith("b_"):
            diff = (g1[k].float() - g0[k].float()).abs()
            assert (diff <= 2 ** -7 * g0[k].float().abs() + 1e-3 * g0[k].float().abs().max()).all(), k
        else:
            rel = ((g1[k].float() - g0[k].float()).norm() / g0[k].float().norm()).item()
            assert rel < 1e-2, (k, rel)


@pytest.mark.parametrize("T,N,r", [(256, 512, 8), (300, 1032, 16), (1024, 2048, 32)])
def test_fp16_adapter_products(T, N, r):
    """fp16 through the projection, the token reduction and the dual pass: one
    fp16 rounding each (alpha * the rounded sum: two) of the fp32 sum."""
    from compact_amd import gemm as G
    g = torch.Generator(device="cuda").manual_seed(0)
    x, q, p = (torch.randn(s, device="cuda", generator=g).half() for s in
               ((T, N), (r, N), (T, r)))
    ref_c, ref_z = x.double() @ q.double().t(), 0.5 * (x.double().t() @ p.double())
    tol_c = N * 2.0 ** -24 * (x.double().abs() @ q.double().abs().t()) + 2.0 ** -25
    tol_z = T * 2.0 ** -24 * (x.double().abs().t() @ p.double().abs()) + 2.0 ** -25
    for c in (G.skinny(x, q), G.skinny_dual(x, q, p, 1.0, 0.5)[0]):
        assert bool(((c.double() - ref_c).abs() <= 2.0 ** -11 * 1.01 * ref_c.abs() + tol_c).all())
    for z in (G.skinny_t(x, p, 0.5), G.skinny_t(x, p, 0.5, trans=True).t(),
              G.skinny_dual(x, q, p, 1.0, 0.5)[1]):
        assert bool(((z.double() - ref_z).abs() <= 2.0 ** -10 * 1.01 * ref_z.abs() + tol_z).all())


@pytest.mark.parametrize("n,h,d", [(1, 64, 128), (65, 192, 320), (259, 256, 512), (300, 200, 336)])
@pytest.mark.parametrize("mode", ["int4", "int8", "bf16", "recompute"])
@pytest.mark.parametrize("rank", [0, 8, 12, 32])
def test_fp16_function_equals_general_layout_kernel(n, h, d, mode, rank, monkeypatch):
    """The fp16 Function on the MFMA tiles against the general-layout kernel:
    the routes differ in the order of fp32 sums only, so in single fp16
    roundings (and codes on a rounding tie)."""
    from compact_amd import flashffn as FF
    from compact_amd import gemm as G
    g = torch.Generator(device="cuda").manual_seed(n + h + rank)

    def rn(*s, std=1.0):
        return (torch.randn(s, device="cuda", generator=g) * std).half().requires_grad_()
    x, gy = rn(n, h), torch.randn(n, h, device="cuda", generator=g).half()
    ws = [rn(d, h, std=0.05), rn(d, h, std=0.05), rn(h, d, std=0.05)]
    ab = [(rn(rank, w.shape[1], std=0.05), rn(w.shape[0], rank, std=0.05)) if rank else (None, None)
          for w in ws]
    leaves = [x] + [t for w, (a, b) in zip(ws, ab) for t in (w, a, b) if t is not None]

    def step():
        args = [t for w, (a, b) in zip(ws, ab) for t in (w, a, b)]
        y = FF.FlashFFNv3Function.apply(x, *args, 0.5, 0.5, 0.5, mode, 64 if d % 64 == 0 else 16)
        return [y] + list(torch.autograd.grad(y, leaves, gy))
    got = step()
    monkeypatch.setattr(G, "f16_fits", lambda a, b: False)
    monkeypatch.setattr(G, "skinny_t_fits", lambda a, b: False)
    monkeypatch.setattr(G, "skinny_dual_ok", lambda *a: False)
    for a, b in zip(got, step()):
        assert a.dtype == torch.float16
        err = (a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-20)
        # a chain of some ten fp16 roundings (2^-11 each); int caches may flip codes on ties
        assert err < (2e-2 if mode == "int4" else 5e-3), err.item()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K", [(1, 8), (15, 264), (17, 512), (300, 1032), (64, 5632)])
@pytest.mark.parametrize("r0,r1", [(8, 0), (1, 0), (8, 8), (16, 16), (24, 3)])
def test_few_token_projection(dt, M, K, r0, r1):
    """The one-launch projection: ragged tokens, K ranges that do not fill the 16
    wavefronts, one and two factors; each factor's columns equal its own call's."""
    from compact_amd import gemm as G
    g = torch.Generator(device="cuda").manual_seed(M + K + r0)
    x, a0, a1 = (torch.randn(s, device="cuda", generator=g).to(dt) for s in
                 ((M, K), (r0, K), (max(r1, 1), K)))
    got = G.skinny_small(x, a0, a1 if r1 else None, 0.5)
    q = torch.cat([a0, a1]) if r1 else a0
    ref = 0.5 * (x.double() @ q.double().t())
    # one rounding (fp16: of the sum and of its half, exact), K 2^-24 |A| |Q|
    half_ulp = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    bound = 0.5 * K * 2.0 ** -24 * (x.double().abs() @ q.double().abs().t()) + 2.0 ** -24
    assert bool(((got.double() - ref).abs() <= 1.01 * half_ulp * ref.abs() + bound).all())
    assert torch.equal(got[:, :r0], G.skinny_small(x, a0, None, 0.5))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b_form", ["rank_rows", "b", "b_ragged"])
@pytest.mark.parametrize("T,N,R", [(1, 512, 8), (65, 520, 16), (300, 1032, 8), (1000, 5632, 16)])
def test_dual_pair_equals_two_calls(device, dt, b_form, T, N, R):
    """Both gradients' dual passes in one launch: the two calls' bits, with Q as
    rank rows and as B with rows that are and are not 16-byte multiples; layouts
    that differ are left to two calls."""
    G = _G()
    xs = [rnd((T, N), s, device).to(dt) for s in (1, 2)]
    qs = [rnd((R, N), s, device, 0.05).to(dt) for s in (3, 4)]
    if b_form == "b":
        qs = [q.t().contiguous().t() for q in qs]
    elif b_form == "b_ragged":
        qs = [torch.empty(N, R + 3, dtype=dt, device=device)[:, :R].copy_(q.t()).t() for q in qs]
    ps = rnd((T, 2 * R), 5, device).to(dt)
    ps = [ps[:, :R], ps[:, R:]]
    c, z0, z1 = G.skinny_dual_pair(xs[0], qs[0], ps[0], 0.5, xs[1], qs[1], ps[1], 2.0)
    for x, q, p, a, half, z in zip(xs, qs, ps, (0.5, 2.0), (c[:, :R], c[:, R:]), (z0, z1)):
        c_alone, z_alone = G.skinny_dual(x, q, p, 1.0, a)
        assert torch.equal(half, c_alone) and torch.equal(z, z_alone)
    wide = torch.zeros(T, N + 8, dtype=dt, device=device)[:, :N].copy_(xs[1])
    if T > 1:
        assert G.skinny_dual_pair(xs[0], qs[0], ps[0], 0.5, wide, qs[1], ps[1], 2.0) is None

"""torch-facing wrappers of the MFMA GEMMs (libcompact_amd.so): the 16x16x32
direct-to-LDS loop for products whose K is a multiple of 64, the 32x32x16
engine otherwise.

mm(a, b)        a @ b for 2-D bf16 tensors; each operand may be row-major or
                a transposed view (K-major / MN-major on the device side).
mm2(a, b, a2, b2)  a @ b + a2 @ b2 in one fp32 accumulation.
mm_engine(a, b) a @ b on the 32x32x16 engine whatever the shape (the fused
                kernels' summation order).
linear(x, w)    x @ w.T (F.linear without bias).
ffn_gate_up     fused dual GEMM + GLU + codec (forward of gate/up + K1).
ffn_down_dgrad  fused grad_y @ w_down + dequantise + SwiGLU backward (+ K2).

LoRA adapter terms (`lora=` / `lora_gate=`, `lora_up=`): PEFT's
`h + s * B(A(x))` applied in the GEMM epilogue, each step rounded to bf16 as
the reference does (src/flashffn.py:1414,1420,1439,1529,1558-1566), for every
rank from 1 to 16, and from 17 to 32 where the product runs on the 16x16x32
loop (`lora_fusable`; a rank that is not a multiple of 8 is zero-padded to the
next multiple of 8).

mm_any          any dtype and any strides (cpt_gemm_any, fp32 MFMA): float32
                (config C1), float16, unaligned bf16 views, rank-1 factors.

These replace the cuBLAS GEMMs the reference issues through F.linear / @
(src/flashffn.py:1410-1439,1503-1587).
"""

from __future__ import annotations

import functools

import torch

from . import _lib
from ._lib import check
from .kernels import _require_device, _stream, _timed


def _layout_a(a: torch.Tensor):
    """(tensor, ld, kmajor) for a logical [M, K] operand: rows 16-byte aligned
    in place, otherwise a contiguous copy."""
    if a.data_ptr() % 16 == 0:
        if a.stride(1) == 1 and a.stride(0) % 8 == 0 and a.stride(0) >= a.shape[1]:
            return a, a.stride(0), 1
        if a.stride(0) == 1 and a.stride(1) % 8 == 0 and a.stride(1) >= a.shape[0]:
            return a, a.stride(1), 0
    a = a.contiguous()
    return a, a.stride(0), 1


def _layout_b(b: torch.Tensor):
    """(tensor, ld, kmajor) for a logical [K, N] operand (kmajor: stored [N][ld]):
    rows 16-byte aligned in place, otherwise a contiguous copy."""
    if b.data_ptr() % 16 == 0:
        if b.stride(0) == 1 and b.stride(1) % 8 == 0 and b.stride(1) >= b.shape[0]:
            return b, b.stride(1), 1
        if b.stride(1) == 1 and b.stride(0) % 8 == 0 and b.stride(0) >= b.shape[1]:
            return b, b.stride(0), 0
    b = b.contiguous()
    return b, b.stride(0), 0


def _with_ld(t: torch.Tensor, ld: int, rows_dim: int) -> torch.Tensor:
    """Copy of 2-D `t` whose storage rows (along `rows_dim`) are `ld` apart."""
    if rows_dim == 0:
        buf = torch.zeros((t.shape[0], ld), dtype=t.dtype, device=t.device)
        buf[:, :t.shape[1]] = t
        return buf[:, :t.shape[1]]
    buf = torch.zeros((t.shape[1], ld), dtype=t.dtype, device=t.device)
    buf[:, :t.shape[0]] = t.t()
    return buf[:, :t.shape[0]].t()


def _common_ld(x, x2, kmajor: int, is_b: bool):
    """The two pairs of mm2 share per-thread offsets, so their operands need
    one leading dimension: re-lay both with the larger one."""
    # storage row axis: A K-major [M][ld] -> dim 0; A MN-major [K][ld] -> dim 1;
    # B K-major [N][ld] -> dim 1; B MN-major [K][ld] -> dim 0
    rows_dim = (0 if kmajor else 1) if not is_b else (1 if kmajor else 0)
    extent = lambda t: t.shape[1 - rows_dim]
    ld = max((extent(x) + 7) // 8 * 8, (extent(x2) + 7) // 8 * 8)
    return _with_ld(x, ld, rows_dim), _with_ld(x2, ld, rows_dim), ld


def _copied(t: torch.Tensor) -> torch.Tensor:
    """t in contiguous rows from a 16-byte aligned base.  (contiguous() copies
    nothing where the rows are whole already, whatever the base: a parameter
    viewed out of a flat buffer.)"""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _check_bf16(*ts):
    for t in ts:
        assert t.dtype == torch.bfloat16, f"MFMA GEMM path is bf16-only, got {t.dtype}"
        assert t.dim() == 2


_DT16 = {torch.bfloat16: _lib.BF16, torch.float16: _lib.F16}


def _check_16(*ts):
    """2-D tensors of one 16-bit type; returns its dtype code."""
    for t in ts:
        assert t.dtype in _DT16 and t.dtype == ts[0].dtype, \
            f"one 16-bit type expected, got {t.dtype} and {ts[0].dtype}"
        assert t.dim() == 2
    return _DT16[ts[0].dtype]


def f16_fits(a: torch.Tensor, b: torch.Tensor) -> bool:
    """a [M, K] @ b [K, N] in fp16 runs on the 128 x 128 tiles (cpt_gemm16):
    16-byte aligned rows, N a multiple of 8, K of 64 unless both operands are
    MN-major, and an MN-major operand within 32-bit offsets."""
    if not (a.dtype == b.dtype == torch.float16 and a.dim() == 2 and b.dim() == 2):
        return False
    (M, K), N = a.shape, b.shape[1]
    if not (M > 0 and K > 0 and N > 0 and N % 8 == 0 and a.data_ptr() % 16 == 0
            and b.data_ptr() % 16 == 0):
        return False
    rows = (K + 256) * 2
    if a.stride(1) == 1 and a.stride(0) % 8 == 0 and a.stride(0) >= K:
        a_mn = False
    elif (a.stride(0) == 1 and M % 8 == 0 and a.stride(1) % 8 == 0 and a.stride(1) >= M
          and rows * a.stride(1) < _SPAN_BYTES):
        a_mn = True
    else:
        return False
    if b.stride(0) == 1 and b.stride(1) % 8 == 0 and b.stride(1) >= K:
        b_mn = False
    elif (b.stride(1) == 1 and b.stride(0) % 8 == 0 and b.stride(0) >= N
          and rows * b.stride(0) < _SPAN_BYTES):
        b_mn = True
    else:
        return False
    return K % 64 == 0 or (a_mn and b_mn)


LORA_MAX_RANK = 32
_NO_TERMS = [(None, None, 0.0)] * 2


def lora_fusable(rank: int, *dims) -> bool:
    """Adapter terms of this rank ride in the epilogue of a GEMM whose summed
    products have the (k, n) `dims` (inner dim, output columns).  One MFMA per
    output block and term over k = 16 (v_mfma_f32_16x16x16_bf16 per 16 x 16
    block on the 16x16x32 loop, v_mfma_f32_32x32x16_bf16 per 32 x 32 block on
    the engine) covers ranks up to 16 on either loop.  Ranks 17 to 32 take a
    second MFMA accumulated onto the first, carried by the 16x16x32 loop's
    kernels only (not the engine's, nor stream-K's): every k a positive
    multiple of 64 and n a multiple of 8."""
    if not 1 <= rank <= LORA_MAX_RANK:
        return False
    return rank <= 16 or (len(dims) > 0 and all(k > 0 and k % 64 == 0 and n % 8 == 0
                                                for k, n in dims))


def _lora_args_whole(terms, n_q, r, x):
    """_lora_args' result where the terms can be used as they are (a rank of
    whole 8-wide chunks, aligned rows, one layout for both), else None."""
    if r % 8:
        return None
    out = []
    dt, m = x.dtype, x.shape[0]
    ldp = ldq = q_km = None
    for pm, q, al in terms:
        sp, sq = pm.stride(), q.stride()
        km = sq[0] == 1 and sq[1] == r
        if ((ldp is not None and (sp[0] != ldp or km != q_km or (not km and sq[0] != ldq)))
                or sp[1] != 1 or sp[0] % 8 or pm.dtype != dt or q.dtype != dt or not pm.is_cuda
                or not q.is_cuda or pm.shape[0] < m or pm.shape[1] != r
                or tuple(q.shape) != (r, n_q)):
            return None
        pp, qp = pm.data_ptr(), q.data_ptr()
        if pp % 16 or (qp % 16 if km else sq[1] != 1):
            return None
        ldp, q_km, ldq = sp[0], km, r if km else sq[0]
        out.append((pp, qp, float(al)))
    if len(out) == 1:
        out.append((None, None, 0.0))
    return r, ldp, int(q_km), ldq, out, terms


def _lora_args(terms, n_q, dims, x, kmajor=None):
    """(rank, ldp, q_kmajor, ldq, [(p, q, alpha) x 2], keep) for up to two
    terms (p [M, r], q the logical [r, N] factor, alpha) of a GEMM with the
    (k, n) `dims` (lora_fusable) and rows and type of its left operand x; `keep`
    holds any re-laid copies alive until the launch.  The kernels fetch P and
    K-major Q in 16-byte chunks of 8 k, so a rank that is not a multiple of 8 is
    zero-padded to the next one (8, 16, 24 or 32): the padded k add exact zeros to
    each fp32 dot product.  kmajor: the layout of Q that the kernel takes, for a
    single rank, whose strides fit both."""
    terms = [t for t in terms if t is not None]
    assert 1 <= len(terms) <= 2
    r = terms[0][0].shape[1]
    fast = _lora_args_whole(terms, n_q, r, x)
    if fast is not None and lora_fusable(r, *dims):
        return fast
    for pm, q, _ in terms:
        _require_device(pm, q)
        assert pm.dtype == q.dtype == x.dtype, \
            f"adapter factors of {pm.dtype} and {q.dtype} in a product of {x.dtype}"
        assert pm.dim() == q.dim() == 2 and pm.shape[0] >= x.shape[0], \
            f"adapter rows {tuple(pm.shape)} for {x.shape[0]} rows"
    assert lora_fusable(r, *dims), \
        f"adapter rank {r} not carried by a GEMM of (k, n) {tuple(dims)} (lora_fusable)"
    if r % 8:
        rp = (r + 7) // 8 * 8
        pad = torch.nn.functional.pad
        padded = []
        for pm, q, al in terms:
            # a factor given as [r, N] rows (an A weight) gains zero rows; one
            # stored [N, r] (a B weight, q its transposed view) zero columns
            rows = q.stride(1) == 1 and q.stride(0) != 1
            if r == 1 and kmajor is not None:
                rows = not kmajor
            if rows:
                q = pad(q, (0, 0, 0, rp - r))
            else:
                q = pad(q.t(), (0, rp - r)).t()
            padded.append((pad(pm, (0, rp - r)), q, al))
        terms, r = padded, rp
    keep, ps, qs = [], [], []
    for pm, q, _ in terms:
        _check_16(pm, q)
        assert pm.shape[1] == r and q.shape[0] == r and q.shape[1] == n_q
        if pm.stride(1) != 1 or pm.stride(0) % 8 or pm.data_ptr() % 16:
            pm = _copied(pm)
        ps.append(pm)
        qs.append(q)
    ldp = ps[0].stride(0)
    if any(x.stride(0) != ldp for x in ps):
        ps = [x.contiguous() for x in ps]
        ldp = r
    # Q: K-major when the [N, r] storage is contiguous, else MN-major rows
    if all(q.stride(0) == 1 and q.stride(1) == r and q.data_ptr() % 16 == 0 for q in qs):
        q_kmajor, ldq = 1, r
    elif all(q.stride(1) == 1 for q in qs) and len({q.stride(0) for q in qs}) == 1:
        q_kmajor, ldq = 0, qs[0].stride(0)
    else:
        qs = [_copied(q.t()).t() for q in qs]
        q_kmajor, ldq = 1, r
    keep += ps + qs
    out = [(ps[i].data_ptr(), qs[i].data_ptr(), float(terms[i][2])) for i in range(len(terms))]
    while len(out) < 2:
        out.append((None, None, 0.0))
    return r, ldp, q_kmajor, ldq, out, keep


SKINNY_MAX_RANK = 32
# blocks of 128 rows x one K range the skinny projection aims for.  In the C3
# step on MI355X (M = 8192: 4 K ranges) h_mid A_d^T took 44.5 us and
# x [A_g; A_u]^T 21.5 us, against 52.0 and 23.6 at 512 blocks (8 ranges) and
# 52.4 / 24.6 at 384, including their reductions.
SKINNY_BLOCKS = 256

# Buffer offsets are 32-bit.  Every kernel's resource starts where a block's
# reads start (a tile's first row, a split's first token or k row), so an
# operand of any size works as long as one block's range spans less than this.
_SPAN_BYTES = 1 << 31


def skinny(a: torch.Tensor, q: torch.Tensor, alpha: float = 1.0,
           name: str = "gemm_skinny", out: torch.Tensor | None = None) -> torch.Tensor:
    """bf16(alpha * a [M, K] @ q[R, K].T) for a rank R <= 32: the tall-skinny
    adapter products (x A^T, grad_y B, ...), streamed once through HBM with K
    split across blocks (fp32 partials summed in a fixed order).  Each output
    column's sum runs in the same order whatever R is, so stacked factors
    give the columns of separate products bit for bit.  out: a bf16 [M, R]
    view with unit column stride and 16-byte aligned rows (e.g. the column
    half of a wider buffer) to write into."""
    _require_device(a, q)
    dt = _check_16(a, q)
    M, K = a.shape
    R = q.shape[0]
    assert q.shape[1] == K and R <= SKINNY_MAX_RANK
    if a.stride(1) != 1 or a.stride(0) % 8 or a.stride(0) < K or a.data_ptr() % 16:
        a = _copied(a)
    if q.stride(1) != 1 or q.stride(0) % 8 or q.stride(0) < K or q.data_ptr() % 16:
        q = _copied(q)
    if out is None and skinny_small_pays(M, K):
        return skinny_small(a, q, None, alpha, name)
    # K ranges for ~SKINNY_BLOCKS blocks of 128 rows (each range >= 256 of
    # K): more ranges cost more partials than they gain in parallelism
    blocks = (M + 127) // 128
    splits = max(1, min(K // 256, (SKINNY_BLOCKS + blocks - 1) // blocks))
    if out is None:
        c = torch.empty((M, R), dtype=a.dtype, device=a.device)
    else:
        c = out
        assert (tuple(c.shape) == (M, R) and c.dtype == a.dtype and c.stride(1) == 1
                and c.stride(0) % 8 == 0 and c.data_ptr() % 16 == 0), "skinny out layout"
    ws = (torch.empty((splits * M * R,), dtype=torch.float32, device=a.device)
          if splits > 1 else None)
    with _timed(name):
        rc = _lib.api().cpt_gemm16_skinny(dt, a.data_ptr(), a.stride(0), q.data_ptr(),
                                          q.stride(0), c.data_ptr(), c.stride(0), M, R, K,
                                          float(alpha), splits,
                                          None if ws is None else ws.data_ptr(), _stream(a))
    check(rc, name)
    return c


# Where the projection is one launch of 16-row blocks whose 16 wavefronts split K
# (skinny_small).  Kernel time on MI355X, us, one factor (two, stacked by a copy
# for the two-launch kernel) against the two-launch kernel's:
#   4 x 2048, rank 8       3.2 (3.9)   /  7.5 (11.1)
#   1808 x 2048, rank 8    4.9 (5.3)   /  7.8 (12.4)
#   4096 x 4096, rank 16   9.3 (13.7)  / 10.4 (17.7)
#   512 x 5632, rank 8     9.7 (11.4)  /  8.1 (13.5)   and a launch fewer
#   512 x 11008, rank 16  20.6 (30.3)  /  8.3 (14.3)
#   8192 x 4096, rank 16  17.1 (26.0)  / 16.0 (23.4)
SKINNY_SMALL_ROWS = 4096
SKINNY_SMALL_K = 6144


def skinny_small_pays(m: int, k: int) -> bool:
    return m <= SKINNY_SMALL_ROWS and k <= SKINNY_SMALL_K


def skinny_small(a: torch.Tensor, q0: torch.Tensor, q1: torch.Tensor | None = None,
                 alpha: float = 1.0, name: str = "gemm_skinny") -> torch.Tensor:
    """a [M, K] @ [q0; q1].T for 16-bit factors of r0 + r1 <= 32 rows, rounded as
    skinny's, one launch; every column's sum runs in the same order whatever
    the ranks are."""
    _require_device(a, q0, q1)
    dt = _check_16(a, q0)
    M, K = a.shape

    def rows(t):
        ok = t.stride(1) == 1 and t.stride(0) % 8 == 0 and t.stride(0) >= K \
            and t.data_ptr() % 16 == 0
        return t if ok else _copied(t)
    a, q0 = rows(a), rows(q0)
    r0, r1 = q0.shape[0], 0
    assert q0.shape[1] == K
    if q1 is not None:
        q1 = rows(q1)
        r1 = q1.shape[0]
        assert q1.dtype == a.dtype and q1.shape[1] == K
    c = torch.empty((M, r0 + r1), dtype=a.dtype, device=a.device)
    with _timed(name):
        rc = _lib.api().cpt_gemm16_skinny_small(
            dt, a.data_ptr(), a.stride(0), q0.data_ptr(), q0.stride(0), r0,
            None if q1 is None else q1.data_ptr(), 0 if q1 is None else q1.stride(0), r1,
            c.data_ptr(), r0 + r1, M, K, alpha, _stream(a))
    check(rc, name)
    return c


def _row_major(t: torch.Tensor) -> bool:
    return t.stride(1) == 1 and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0


def skinny_t(x: torch.Tensor, p: torch.Tensor, alpha: float = 1.0, trans: bool = False,
             name: str = "gemm_skinny_t") -> torch.Tensor:
    """bf16(alpha * x[T, N].T @ p[T, R]) -> [N, R] (or its transpose [R, N]
    with trans) for R <= 32: the adapter-factor gradients that reduce over
    the tokens, x and p token-major."""
    _require_device(x, p)
    dt = _check_16(x, p)
    T, N = x.shape
    R = p.shape[1]
    assert p.shape[0] == T and R <= SKINNY_MAX_RANK
    if not _row_major(x) or x.stride(0) < N:
        x = _copied(x)
    if not _row_major(p) or p.stride(0) < R:
        p = _copied(p)
    splits = skinny_t_splits(T, N)
    # each split reads its tokens (plus 128 of prefetch) within 32-bit offsets
    per = (_SPAN_BYTES // (2 * max(x.stride(0), p.stride(0))) - 129) // 64 * 64
    assert per >= 64, "operand rows too long for 32-bit buffer offsets"
    splits = max(splits, (T + per - 1) // per)
    out = torch.empty((R, N) if trans else (N, R), dtype=x.dtype, device=x.device)
    ws = torch.empty((splits * N * R,), dtype=torch.float32, device=x.device)
    with _timed(name):
        rc = _lib.api().cpt_gemm16_skinny_t(dt, x.data_ptr(), x.stride(0), p.data_ptr(),
                                            p.stride(0), out.data_ptr(), out.stride(0),
                                            1 if trans else 0, T, N, R, float(alpha), splits,
                                            ws.data_ptr(), _stream(x))
    check(rc, name)
    return out


# Blocks of a skinny_dual launch (column blocks x token splits).  In the C3
# step on MI355X, 176 (8 token splits over d_ff 11008, 22 over d_model 4096)
# against 256: 64.6 / 62.7 / 37.1 us against 66.6 / 68.8 / 44.5 us for the
# gate, up and down passes including their reductions (128, 352, 512 and 704
# blocks were no better).  Fewer, longer token splits also cut the Z partials
# by a third.
SKINNY_DUAL_BLOCKS = 176
# tokens per split at least: one piece.  At 1808 tokens 64 against 256: 12.8 /
# 16.9 us over d_ff 5632, 12.1 / 16.2 over d_model 2048 (rank 8); level from 4096
# tokens on, where the blocks bind.
SKINNY_DUAL_TOKENS = 64


def transpose_ok(x: torch.Tensor) -> bool:
    """transpose takes a bf16 row-major [rows, cols] device tensor with rows,
    cols and the row stride multiples of 8 and a 16-byte aligned base."""
    return (x.dtype == torch.bfloat16 and x.is_cuda and x.dim() == 2 and x.stride(1) == 1
            and x.shape[0] % 8 == 0 and x.shape[1] % 8 == 0 and x.stride(0) % 8 == 0
            and x.data_ptr() % 16 == 0)


def transpose(x: torch.Tensor, name: str = "transpose") -> torch.Tensor:
    """x^T as a new row-major [cols, rows] bf16 tensor (cpt_transpose_bf16)."""
    _require_device(x)
    assert transpose_ok(x), "transpose operand"
    rows, cols = x.shape
    out = torch.empty((cols, rows), dtype=x.dtype, device=x.device)
    with _timed(name):
        rc = _lib.api().cpt_transpose_bf16(x.data_ptr(), x.stride(0), rows, cols, out.data_ptr(),
                                           out.stride(0), _stream(x))
    check(rc, name)
    return out


def skinny_dual_ok(x: torch.Tensor, q: torch.Tensor, p: torch.Tensor) -> bool:
    """skinny_dual takes bf16 or fp16 x [T, N] with N a multiple of 8 and a rank
    (q [R, N], p [T, R]) that is a multiple of 8 up to 32."""
    T, N = x.shape
    R = q.shape[0]
    return (x.dtype == q.dtype == p.dtype and x.dtype in _DT16 and x.is_cuda and N % 8 == 0
            and R % 8 == 0 and 0 < R <= SKINNY_MAX_RANK and q.shape[1] == N
            and tuple(p.shape) == (T, R))


def _dual_q(q: torch.Tensor):
    """(q, q_nr, ldq): Q as rank rows [R][ld], or its transpose B [N][ld] as
    stored (no copy)."""
    R, N = q.shape
    if q.stride(1) == 1 and q.stride(0) % 8 == 0 and q.stride(0) >= N and q.data_ptr() % 16 == 0:
        return q, 0, q.stride(0)
    if q.stride(0) == 1 and q.stride(1) >= R and q.data_ptr() % 16 == 0:
        return q, 1, q.stride(1)
    q = _copied(q)
    return q, 0, q.stride(0)


def _dual_splits(T: int, N: int, ld: int) -> int:
    """Token splits: blocks of 512 columns x T / splits tokens, about
    SKINNY_DUAL_BLOCKS of them, each within 32-bit offsets."""
    csplits = (N + 511) // 512
    splits = max(1, min(max(T // SKINNY_DUAL_TOKENS, 1),
                        (SKINNY_DUAL_BLOCKS + csplits - 1) // csplits))
    per = (_SPAN_BYTES // (2 * ld) - 129) // 64 * 64
    assert per >= 64, "operand rows too long for 32-bit buffer offsets"
    return max(splits, (T + per - 1) // per)


def skinny_dual(x: torch.Tensor, q: torch.Tensor, p: torch.Tensor, alpha_c: float = 1.0,
                alpha_z: float = 1.0, out_c: torch.Tensor | None = None,
                name: str = "gemm_skinny_dual"):
    """(bf16(alpha_c * x @ q.T) [T, R], bf16(alpha_z * x.T @ p) [N, R]) in one
    pass over x [T, N] (cpt_gemm_bf16_skinny_dual): the projection and the
    token reduction a LoRA backward takes of one tensor (grad_h B and
    s grad_h^T (x A^T)).  out_c: a bf16 [T, R] view with unit column stride
    and 16-byte aligned rows to write C into."""
    _require_device(x, q, p)
    assert skinny_dual_ok(x, q, p), "skinny_dual operands"
    T, N = x.shape
    R = q.shape[0]
    if not _row_major(x) or x.stride(0) < N:
        x = _copied(x)
    q, q_nr, ldq = _dual_q(q)
    if not _row_major(p) or p.stride(0) < R:
        p = _copied(p)
    splits = _dual_splits(T, N, max(x.stride(0), p.stride(0)))
    if out_c is None:
        c = torch.empty((T, R), dtype=x.dtype, device=x.device)
    else:
        c = out_c
        assert (tuple(c.shape) == (T, R) and c.dtype == x.dtype and c.stride(1) == 1
                and c.stride(0) % 8 == 0 and c.data_ptr() % 16 == 0), "skinny_dual out layout"
    z = torch.empty((N, R), dtype=x.dtype, device=x.device)
    nbytes = _lib.api().cpt_gemm_bf16_skinny_dual_workspace_bytes(T, N, R, splits)
    ws = torch.empty((max(nbytes, 4) // 4,), dtype=torch.float32, device=x.device)
    with _timed(name):
        rc = _lib.api().cpt_gemm16_skinny_dual(
            _DT16[x.dtype], x.data_ptr(), x.stride(0), q.data_ptr(), ldq, q_nr, p.data_ptr(),
            p.stride(0), c.data_ptr(), c.stride(0), float(alpha_c), z.data_ptr(), z.stride(0), 0,
            float(alpha_z), T, N, R, splits, ws.data_ptr(), _stream(x))
    check(rc, name)
    return c, z


def skinny_dual_pair(x0: torch.Tensor, q0: torch.Tensor, p0: torch.Tensor, alpha0: float,
                     x1: torch.Tensor, q1: torch.Tensor, p1: torch.Tensor, alpha1: float,
                     name: str = "gemm_skinny_dual_pair"):
    """skinny_dual of two tensors of one shape, both passes in one launch and
    their split sums in another (bit for bit the two calls' results): returns
    ([x0 q0^T | x1 q1^T] side by side [T, 2 R], alpha0 x0^T p0 [N, R],
    alpha1 x1^T p1 [N, R]), or None where the two do not share a layout."""
    _require_device(x0, q0, p0, x1, q1, p1)
    assert skinny_dual_ok(x0, q0, p0) and skinny_dual_ok(x1, q1, p1), "skinny_dual_pair operands"
    assert x1.shape == x0.shape and q1.shape == q0.shape and x1.dtype == x0.dtype, \
        f"tensors of two shapes or types: {tuple(x0.shape)} {x0.dtype}, {tuple(x1.shape)} {x1.dtype}"
    T, N = x0.shape
    R = q0.shape[0]
    q0, q_nr, ldq = _dual_q(q0)
    q1, *lay1 = _dual_q(q1)
    if (lay1 != [q_nr, ldq] or x0.stride() != x1.stride() or p0.stride() != p1.stride()
            or not _row_major(x0) or not _row_major(x1) or x0.stride(0) < N
            or not _row_major(p0) or not _row_major(p1) or p0.stride(0) < R):
        return None
    splits = _dual_splits(T, N, max(x0.stride(0), p0.stride(0)))
    c = torch.empty((T, 2 * R), dtype=x0.dtype, device=x0.device)
    z0 = torch.empty((N, R), dtype=x0.dtype, device=x0.device)
    z1 = torch.empty((N, R), dtype=x0.dtype, device=x0.device)
    nbytes = _lib.api().cpt_gemm_bf16_skinny_dual_workspace_bytes(T, N, R, splits)
    ws = torch.empty((max(nbytes, 4) // 2,), dtype=torch.float32, device=x0.device)
    with _timed(name):
        rc = _lib.api().cpt_gemm16_skinny_dual2(
            _DT16[x0.dtype], x0.data_ptr(), x1.data_ptr(), x0.stride(0), q0.data_ptr(),
            q1.data_ptr(), ldq, q_nr, p0.data_ptr(), p1.data_ptr(), p0.stride(0), c.data_ptr(),
            c.data_ptr() + 2 * R, 2 * R, 1.0, z0.data_ptr(), z1.data_ptr(), R, 0, float(alpha0),
            float(alpha1), T, N, R, splits, ws.data_ptr(), _stream(x0))
    check(rc, name)
    return c, z0, z1


def skinny_t_splits(T: int, N: int) -> int:
    """Token splits of the token-reduction kernel: ~768 blocks of 64 columns."""
    blocks = (N + 63) // 64
    return max(1, min(max(T // 256, 1), (768 + blocks - 1) // blocks))


def skinny_t_noalloc(x: torch.Tensor, p: torch.Tensor, out: torch.Tensor, alpha: float = 1.0,
                     trans: bool = False, splits: int | None = None,
                     name: str = "gemm_skinny_t_noalloc") -> torch.Tensor:
    """skinny_t into a caller-provided `out` through the allocation-free entry
    point: the split partials use the library's fixed per-GPU scratch, so the
    call allocates nothing (x, p token-major rows 16-byte aligned; out [N, R],
    or [R, N] with trans, rows `out.stride(0)` apart)."""
    _require_device(x, p, out)
    _check_bf16(x, p)
    T, N = x.shape
    R = p.shape[1]
    assert p.shape[0] == T and out.dtype == torch.bfloat16 and out.stride(1) == 1
    assert tuple(out.shape) == ((R, N) if trans else (N, R))
    assert _row_major(x) and _row_major(p), "x and p must have 16-byte aligned rows"
    if splits is None:
        splits = skinny_t_splits(T, N)
    with _timed(name):
        rc = _lib.lib().cpt_gemm_bf16_skinny_t_noalloc(
            x.data_ptr(), x.stride(0), p.data_ptr(), p.stride(0), out.data_ptr(), out.stride(0),
            1 if trans else 0, T, N, R, float(alpha), splits, _stream(x))
    check(rc, f"{name} (split partials beyond the {_lib.NOALLOC_SCRATCH_BYTES >> 20} MiB "
              "scratch?)" if rc == _lib.ERR_TOO_LARGE else name)
    return out


def _max_k_rows(ld: int) -> int:
    """k rows one block may read from an MN-major operand with rows ld apart
    (prefetch overhang of 256 rows included)."""
    return _SPAN_BYTES // (2 * ld) - 257


def _min_splits(K: int, lda: int, ak: int, ldb: int, bk: int) -> int:
    """Fewest k ranges that keep every block of a product within 32-bit
    offsets, given its operand layouts (1 for everything but products over
    very long k, e.g. the weight gradients of ~100k+ tokens whose operands
    exceed 2 GiB)."""
    lim = K
    if not ak:
        lim = min(lim, _max_k_rows(lda))       # A MN-major: [K][lda]
    if not bk:
        lim = min(lim, _max_k_rows(ldb))       # B MN-major: [K][ldb]
    if lim >= K:
        return 1
    assert lim >= 64, "operand rows too long for 32-bit buffer offsets"
    nk, per = (K + 63) // 64, lim // 64
    return (nk + per - 1) // per


def small_tiles(m: int, n: int) -> bool:
    """The 16x16x32 loop covers an [m, n] output with 128 x 128 tiles: at most
    two per CU (launch16 in csrc/gemm.hip; 256 CUs)."""
    return ((m + 127) // 128) * ((n + 127) // 128) <= 512


# Split products (cpt_gemm16): k-tiles per range at least, and k-tiles taken off
# each block at least.  A block alone on its CU takes 0.42 us per k-tile (up to 128
# of them, all that split_plan splits; 0.55 with 256, tile_plan's rate); the first
# tiles' latency is worth about 5, the partials and the second kernel about 20.
# Measured on MI355X, us unsplit / split (both with their launches):
#   512 x 2048, k 5632   (64 tiles, 4 ranges)   39.6 / 24.0
#   512 x 2048, k 11264  (64, 4)                81.3 / 35.8
#   512 x 4096, k 11008  (128, 2)               73.5 / 53.3
#   4 x 2048, k 5632     (16, 14)               40.4 / 18.1
#   1024 x 4096, k 11008 (256, 2 ranges)        83.8 / 100.5   not split
#   4 x 11264, k 2048    (88, 2 ranges)         25.9 / 27.1    not split
SPLIT_MIN_KT = 6
SPLIT_MIN_SAVED = 20


def split_plan(m: int, n: int, nk: int) -> int:
    """k ranges of a product of nk k-tiles on 128 x 128 tiles: where the tiles
    leave half the CUs (of 256) idle, as many as fill them, 1 where the k-tiles
    they take off each block do not pay for the partials."""
    small = ((m + 127) // 128) * ((n + 127) // 128)
    if small == 0 or small > 128:
        return 1
    splits = min(256 // small, nk // SPLIT_MIN_KT)
    return splits if splits > 1 and nk - nk // splits >= SPLIT_MIN_SAVED else 1


@functools.lru_cache(maxsize=4096)
def tile_plan(m: int, n: int, nk: int, half: bool = False) -> tuple[int, int]:
    """(tile edge, k ranges) of a 16-bit product of nk k-tiles: the unsplit
    product (one range: launch16 picks its tiles), 128 x 128 tiles split as
    split_plan has it, or, bf16 only, 256 x 256 tiles with k split to fill the
    CUs, whichever the measured rates make cheapest.

    Rates on MI355X, us per k-tile: 0.55 for 128 x 128 tiles alone on a CU with
    most CUs busy (240 of them, k 11264: 0.50 K-major, 0.52 MN-major B), 1.0 for two
    sharing it, 1.0 to 1.45 for a 256 x 256 tile as the chip fills up;
    8 for a block's ends; a split adds 8 and 1.1 per million partials.  Measured,
    us unsplit (128 x 128 tiles) / split 256 x 256 ones:
      2048 x 4096, k 22016 (128 large tiles, 2 ranges)  382 / 277
      2048 x 4096, k 11008 (128, 2)                     160 / 146
      3000 x 2048, k 11264 (96, 2)                      162 / 127
      1500 x 4096, k 11008 (96, 2)                      161 / 128
      1024 x 4096, k 11008 (64, 4)                       91 / 95     kept unsplit
      4096 x 2048, k 5632  (128, 2)                      87 / 90     kept unsplit
      1808 x 2048, k 11264 (64, 4)                       89 / 89, 92 / 90 kept unsplit"""
    t128 = ((m + 127) // 128) * ((n + 127) // 128)
    t256 = ((m + 255) // 256) * ((n + 255) // 256)
    if t128 == 0:
        return 128, 1
    small = split_plan(m, n, nk)
    if small > 1:
        cost = 0.55 * nk / small + 12 + 1.1e-6 * small * m * n
    elif t128 <= 256:
        cost = 0.55 * nk + 4
    elif t128 <= 512:
        cost = 1.0 * nk + 4
    else:
        return 128, 1
    best = (128, small)
    for s in range(2, min(8, 256 // t256) + 1) if not half else ():
        if nk // s < SPLIT_MIN_KT:
            break
        c = (1.0 + 0.45 * t256 * s / 256) * nk / s + 16 + 1.1e-6 * s * m * n
        if c < 0.95 * cost:
            best, cost = (256, s), c / 0.95
    return best


def mm(a: torch.Tensor, b: torch.Tensor, name: str = "gemm") -> torch.Tensor:
    """a [M, K] @ b [K, N] -> bf16 [M, N] on the MFMA GEMM loops (16x16x32 when
    K is a multiple of 64 and N of 8, else the 32x32x16 engine).  Tall products
    with N <= 32 (the adapter terms' x A^T, grad_y B, ...) go to the skinny
    kernel; products with too few output tiles to fill the chip split K across
    blocks instead (split_plan on the 16x16x32 loop, mm_splitk on the engine),
    as do products whose transposed operands are too long for one block's
    32-bit offsets."""
    M, K = a.shape
    N = b.shape[1]
    if N <= SKINNY_MAX_RANK and K >= 256 and K % 8 == 0 and a.stride(1) == 1:
        return skinny(a, b.t(), 1.0, name)
    if a.dtype == torch.float16:
        return mm2(a, b, None, None, name)
    tiles = ((M + 255) // 256) * ((N + 255) // 256)
    if tiles < 128 and K >= 1024 and (K % 64 or N % 8):
        return mm_splitk(a, b, 1.0, name=name)
    a, lda, ak = _layout_a(a)
    b, ldb, bk = _layout_b(b)
    if _min_splits(K, lda, ak, ldb, bk) > 1:
        return mm_splitk(a, b, 1.0, name=name)
    return mm2(a, b, None, None, name)


# Stream-K workspace per device (cpt_gemm_stream_k_workspace): attached at
# the first product on a device while stream-K is on.
_STREAM_K = {"on": True}
_sk_attached: dict = {}      # device index -> workspace tensor, or None if detached


def set_stream_k(on: bool) -> None:
    """Turn the stream-K schedule of the 16x16x32 loop on or off for later
    products on every device (on by default).  Results are deterministic
    either way; the two summation orders differ in the last bits of the
    tiles the schedule shares."""
    _STREAM_K["on"] = bool(on)
    for idx in list(_sk_attached):
        with torch.cuda.device(idx):
            check(_lib.lib().cpt_gemm_stream_k_workspace(None, 0), "stream_k_workspace")
        del _sk_attached[idx]


def _stream_k(dev: torch.device) -> None:
    """Attach a zero-filled stream-K workspace to `dev` once (the kernels
    leave it zero-filled)."""
    idx = dev.index if dev.index is not None else torch.cuda.current_device()
    if idx in _sk_attached or not _STREAM_K["on"]:
        return
    with torch.cuda.device(idx):
        nbytes = int(_lib.lib().cpt_gemm_stream_k_bytes())
        assert nbytes > 0, "stream-K workspace size"
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
        torch.cuda.synchronize(idx)
        check(_lib.lib().cpt_gemm_stream_k_workspace(ws.data_ptr(), nbytes), "stream_k_workspace")
    _sk_attached[idx] = ws


def stream_k_errors(dev: torch.device) -> int:
    """Waits for a partial that ran out of polls on `dev` since its workspace
    was attached (the word after the flags); 0 unless the schedule broke."""
    ws = _sk_attached.get(dev.index if dev.index is not None else torch.cuda.current_device())
    if ws is None:
        return 0
    return int(ws[-4:].view(torch.int32).item())


def mm2(a, b, a2=None, b2=None, name: str = "gemm", lora=None) -> torch.Tensor:
    """a @ b (+ a2 @ b2) in one fp32 accumulation -> bf16 [M, N], then the
    adapter terms `lora` = [(p [M, r], q [r, N], alpha), ...] (at most two),
    each `out = bf16(out + bf16(alpha * bf16(p @ q)))`.  fp16 likewise, for
    operands that fit the 128 x 128 tiles (f16_fits)."""
    _require_device(a, b)
    dt = _check_16(a, b)
    M, K = a.shape
    K_, N = b.shape
    assert K == K_, f"inner dims differ: {tuple(a.shape)} @ {tuple(b.shape)}"
    a, lda, ak = _layout_a(a)
    b, ldb, bk = _layout_b(b)
    p_a2 = p_b2 = None
    lda2 = ldb2 = K2 = 0
    if a2 is not None:
        _check_16(a, a2, b2)
        assert a2.shape[0] == M and b2.shape[1] == N and a2.shape[1] == b2.shape[0]
        K2 = a2.shape[1]
        a2, lda2, ak2 = _layout_a(a2)
        b2, ldb2, bk2 = _layout_b(b2)
        if ak2 != ak:
            a2 = a2.t().contiguous().t() if ak == 0 else a2.contiguous()
            a2, lda2, ak2 = _layout_a(a2)
        if bk2 != bk:
            b2 = b2.t().contiguous().t() if bk == 1 else b2.contiguous()
            b2, ldb2, bk2 = _layout_b(b2)
        assert ak2 == ak and bk2 == bk
        if lda2 != lda:
            a, a2, lda = _common_ld(a, a2, ak, is_b=False)
            lda2 = lda
        if ldb2 != ldb:
            b, b2, ldb = _common_ld(b, b2, bk, is_b=True)
            ldb2 = ldb
        p_a2, p_b2 = a2.data_ptr(), b2.data_ptr()
    ldc = (N + 7) // 8 * 8
    c = torch.empty((M, ldc), dtype=a.dtype, device=a.device)
    r, ldp, qk, ldq, t = 0, 0, 1, 0, _NO_TERMS
    if lora:
        if ak != 1:
            a = a.contiguous()
            a, lda, ak = _layout_a(a)
            assert a2 is None, "adapter terms with a K-concatenated MN-major A"
        dims = ((K, N),) if a2 is None else ((K, N), (K2, N))
        r, ldp, qk, ldq, t, keep = _lora_args(lora, N, dims, a)
    half = dt == _lib.F16
    tiles, splits = ((128, 1) if (not half and (K % 64 or K2 % 64)) or N % 8 or not K
                     else tile_plan(M, N, (K + 63) // 64 + (K2 + 63) // 64, half))
    if splits > 1 or half:
        ws = (torch.empty((splits * M * N,), dtype=torch.float32, device=a.device)
              if splits > 1 else None)
        with _timed(name):
            rc = _lib.api().cpt_gemm16(
                dt, a.data_ptr(), lda, ak, b.data_ptr(), ldb, bk, p_a2, lda2, p_b2, ldb2,
                K2, c.data_ptr(), ldc, M, N, K, r, ldp, qk, ldq, t[0][0], t[0][1], t[0][2],
                t[1][0], t[1][1], t[1][2], tiles, splits,
                None if ws is None else ws.data_ptr(), _stream(a))
        check(rc, name)
        return c
    _stream_k(a.device)
    with _timed(name):
        if lora:
            rc = _lib.api().cpt_gemm_bf16_lora(
                a.data_ptr(), lda, ak, b.data_ptr(), ldb, bk, p_a2, lda2, p_b2, ldb2, K2,
                c.data_ptr(), ldc, M, N, K, r, ldp, qk, ldq, t[0][0], t[0][1], t[0][2],
                t[1][0], t[1][1], t[1][2], _stream(a))
        else:
            rc = _lib.api().cpt_gemm_bf16(a.data_ptr(), lda, ak, b.data_ptr(), ldb, bk, p_a2,
                                          lda2, p_b2, ldb2, K2, c.data_ptr(), ldc, M, N, K,
                                          _stream(a))
    check(rc, name)
    return c if ldc == N else c[:, :N]


def mm_engine(a: torch.Tensor, b: torch.Tensor, name: str = "gemm_engine") -> torch.Tensor:
    """a [M, K] @ b [K, N] -> bf16 [M, N] on the 32x32x16 engine loop for
    every shape: the fp32 summation order of the fused FFN kernels, so a
    fused kernel equals its unfused composition through this product bit for
    bit.  mm runs every layout on the 16x16x32 loop instead whenever K is a
    multiple of 64 and N of 8 (same bf16 rounding of the fp32 sum, another
    summation order)."""
    _require_device(a, b)
    _check_bf16(a, b)
    M, K = a.shape
    K_, N = b.shape
    assert K == K_, f"inner dims differ: {tuple(a.shape)} @ {tuple(b.shape)}"
    a, lda, ak = _layout_a(a)
    b, ldb, bk = _layout_b(b)
    ldc = (N + 7) // 8 * 8
    c = torch.empty((M, ldc), dtype=torch.bfloat16, device=a.device)
    with _timed(name):
        rc = _lib.api().cpt_gemm_bf16_ex(a.data_ptr(), lda, ak, b.data_ptr(), ldb, bk, c.data_ptr(),
                                         ldc, M, N, K, 1.0, 0, 1, None, _stream(a))
    check(rc, name)
    return c if ldc == N else c[:, :N]


def linear(x: torch.Tensor, w: torch.Tensor, name: str = "gemm") -> torch.Tensor:
    """x [M, K] @ w[N, K].T -> [M, N] (F.linear without bias)."""
    return mm(x, w.t(), name)


def linear_lora(x: torch.Tensor, w: torch.Tensor, xa: torch.Tensor, b: torch.Tensor,
                alpha: float, name: str = "gemm") -> torch.Tensor:
    """PEFT's LoRA Linear without dropout: bf16(bf16(x W^T) + bf16(alpha *
    bf16(xa B^T))) with xa = x A^T [M, r] and B [N, r]."""
    return mm2(x, w.t(), None, None, name, lora=[(xa, b.t(), alpha)])


def ffn_gate_up(x, w_gate, w_up, cache: int, group_size: int, want_h_mid: bool = True,
                lora_gate=None, lora_up=None):
    """Fused dual GEMM + GLU + codec.  Returns (h_mid | None, h_gate | None,
    h_up | None, q_gate | None, s_gate | None, q_up | None, s_up | None).
    CACHE_BF16 keeps h_gate / h_up in x's type (bf16, or fp16 without codec).
    lora_gate / lora_up = (xa [n, r], B [inter, r], s): the projection's LoRA
    term, added to h_gate / h_up before the GLU and the codec."""
    _require_device(x, w_gate, w_up)
    dt = _check_16(x, w_gate, w_up)
    half = dt == _lib.F16
    assert not half or cache in (_lib.CACHE_NONE, _lib.CACHE_BF16), "the codec takes bf16"
    n, hdim = x.shape
    d = w_gate.shape[0]
    assert w_gate.shape == (d, hdim) and w_up.shape == (d, hdim)
    x, w_gate, w_up = x.contiguous(), w_gate.contiguous(), w_up.contiguous()
    dev = x.device
    h_mid = torch.empty((n, d), dtype=x.dtype, device=dev) if want_h_mid else None
    hg = hu = qg = sg = qu = su = None
    if cache == _lib.CACHE_BF16:
        hg = torch.empty((n, d), dtype=x.dtype, device=dev)
        hu = torch.empty((n, d), dtype=x.dtype, device=dev)
    elif cache in (_lib.CACHE_INT4, _lib.CACHE_INT8):
        g = d // group_size
        shape = (n, d // 2) if cache == _lib.CACHE_INT4 else (n, d)
        qdt = torch.uint8 if cache == _lib.CACHE_INT4 else torch.int8
        qg = torch.empty(shape, dtype=qdt, device=dev)
        qu = torch.empty(shape, dtype=qdt, device=dev)
        sg = torch.empty((n, g), dtype=torch.float16, device=dev)
        su = torch.empty((n, g), dtype=torch.float16, device=dev)

    def p(t):
        return None if t is None else t.data_ptr()

    r, ldp, t = 0, 0, _NO_TERMS
    if lora_gate is not None or lora_up is not None:
        # term 0 on the gate columns, term 1 on the up columns (absent: no-op)
        present = [t for t in (lora_gate, lora_up) if t is not None]
        r, ldp, qk, _, t, keep = _lora_args([(xa, bw.t(), s) for xa, bw, s in present], d,
                                            ((hdim, d),), x, kmajor=True)
        assert qk == 1, "the gate/up adapter B factors go K-major"
        if lora_gate is None:
            t = [(None, None, 0.0), t[0]]
    splits = (split_plan(n, 2 * d, hdim // 64)
              if cache in (_lib.CACHE_NONE, _lib.CACHE_BF16) and hdim % 64 == 0 and d % 8 == 0
              else 1)
    with _timed("ffn_gate_up"):
        if splits > 1 or half:
            ws = (torch.empty((splits * n * 2 * d,), dtype=torch.float32, device=dev)
                  if splits > 1 else None)
            rc = _lib.api().cpt_ffn_gate_up16(
                dt, x.data_ptr(), w_gate.data_ptr(), w_up.data_ptr(), n, hdim, d,
                p(h_mid), p(hg), p(hu), r, ldp, t[0][0], t[0][1], t[0][2], t[1][0], t[1][1],
                t[1][2], splits, None if ws is None else ws.data_ptr(), _stream(x))
        elif r:
            rc = _lib.api().cpt_ffn_gate_up_lora(
                x.data_ptr(), w_gate.data_ptr(), w_up.data_ptr(), n, hdim, d, cache, group_size,
                p(h_mid), p(hg), p(hu), p(qg), p(sg), p(qu), p(su), r, ldp, t[0][0], t[0][1],
                t[0][2], t[1][0], t[1][1], t[1][2], _stream(x))
        else:
            rc = _lib.api().cpt_ffn_gate_up(x.data_ptr(), w_gate.data_ptr(), w_up.data_ptr(), n,
                                            hdim, d, cache, group_size, p(h_mid), p(hg), p(hu),
                                            p(qg), p(sg), p(qu), p(su), _stream(x))
    check(rc, "ffn_gate_up")
    return h_mid, hg, hu, qg, sg, qu, su


def ffn_gate_up_outlier_fits(hidden: int) -> bool:
    """The outlier-codec epilogue runs on the 16x16x32 loop: d_model a
    multiple of 64."""
    return hidden > 0 and hidden % 64 == 0


def ffn_gate_up_outlier(x, w_gate, w_up, cache: int, group_size: int, slot_gate, slot_up,
                        k: int, out, lora_gate=None, lora_up=None):
    """Fused dual GEMM + GLU + int codec with config C3's outlier channels
    (cpt_ffn_gate_up_outlier): writes into `out` = (h_mid, q_gate, s_gate,
    o_gate, q_up, s_up, o_up), preallocated (row slices of the Function's
    buffers are fine); the slot maps come from an outlier selection."""
    _require_device(x, w_gate, w_up, slot_gate, slot_up)
    _check_bf16(x, w_gate, w_up)
    n, hdim = x.shape
    d = w_gate.shape[0]
    assert w_gate.shape == (d, hdim) and w_up.shape == (d, hdim)
    assert cache in (_lib.CACHE_INT4, _lib.CACHE_INT8) and k > 0
    x, w_gate, w_up = x.contiguous(), w_gate.contiguous(), w_up.contiguous()
    h_mid, qg, sg, og, qu, su, ou = out
    for t, shape in ((h_mid, (n, d)), (sg, (n, d // group_size)), (su, (n, d // group_size)),
                     (og, (n, k)), (ou, (n, k)),
                     (qg, (n, d // 2) if cache == _lib.CACHE_INT4 else (n, d)),
                     (qu, (n, d // 2) if cache == _lib.CACHE_INT4 else (n, d))):
        assert tuple(t.shape) == shape and t.is_contiguous(), (tuple(t.shape), shape)
    assert slot_gate.dtype == torch.int16 and slot_gate.shape == (d,) and slot_up.shape == (d,)
    rank = ldp = 0
    t = [(None, None, 0.0), (None, None, 0.0)]
    keep = None
    if lora_gate is not None or lora_up is not None:
        present = [tt for tt in (lora_gate, lora_up) if tt is not None]
        rank, ldp, qk, _, t, keep = _lora_args([(xa, bw.t(), sc) for xa, bw, sc in present], d,
                                               ((hdim, d),), x, kmajor=True)
        assert qk == 1, "the gate/up adapter B factors go K-major"
        if lora_gate is None:
            t = [(None, None, 0.0), t[0]]
        elif lora_up is None:
            t = [t[0], (None, None, 0.0)]
    with _timed("ffn_gate_up"):
        rc = _lib.lib().cpt_ffn_gate_up_outlier(
            x.data_ptr(), w_gate.data_ptr(), w_up.data_ptr(), n, hdim, d, cache, group_size,
            h_mid.data_ptr(), qg.data_ptr(), sg.data_ptr(), qu.data_ptr(), su.data_ptr(),
            slot_gate.data_ptr(), og.data_ptr(), slot_up.data_ptr(), ou.data_ptr(), k, rank, ldp,
            t[0][0], t[0][1], t[0][2], t[1][0], t[1][1], t[1][2], _stream(x))
    del keep
    check(rc, "ffn_gate_up_outlier")
    return out


def ffn_down_dgrad(grad_y, w_down, cache: int, group_size: int, c_gate, s_gate, c_up, s_up,
                   want_h_mid: bool, lora=None, outliers=None, inplace: bool = False):
    """Fused grad_y @ w_down + dequantise + SwiGLU backward.
    Returns (grad_h_gate, grad_h_up, h_mid_hat | None).  lora = (gy B_d
    [n, r], A_d [r, inter], s): the down projection's LoRA term of
    grad_h_mid.  outliers = (slot_gate, o_gate, slot_up, o_up): the C3
    outlier channels (int16 slot maps [inter], bf16 blocks [n, k]) that
    replace their dequantised columns.  `inplace=True` (bf16 cache only)
    writes grad_h_gate / grad_h_up over c_gate / c_up, which must be
    contiguous and private to the caller (the in-place GLU backward,
    src/flashffn.py:129-198)."""
    _require_device(grad_y, w_down)
    _check_bf16(grad_y, w_down)
    n, hdim = grad_y.shape
    d = w_down.shape[1]
    assert w_down.shape == (hdim, d)
    grad_y, w_down = grad_y.contiguous(), w_down.contiguous()
    dev = grad_y.device
    if inplace:
        assert cache == _lib.CACHE_BF16 and c_gate.is_contiguous() and c_up.is_contiguous()
        assert tuple(c_gate.shape) == (n, d) and tuple(c_up.shape) == (n, d)
        dg, du = c_gate, c_up
    else:
        dg = torch.empty((n, d), dtype=torch.bfloat16, device=dev)
        du = torch.empty((n, d), dtype=torch.bfloat16, device=dev)
    hm = torch.empty((n, d), dtype=torch.bfloat16, device=dev) if want_h_mid else None

    keep_in = [None if t is None else t.contiguous() for t in (c_gate, s_gate, c_up, s_up)]
    c_gate, s_gate, c_up, s_up = keep_in

    def p(t):
        return None if t is None else t.data_ptr()

    if outliers is not None:
        slot_g, o_g, slot_u, o_u = [t.contiguous() for t in outliers]
        k = o_g.shape[1]
        assert o_u.shape[1] == k and slot_g.numel() == d and slot_u.numel() == d
        rank, ldp, pp, qq, alpha, keep = 0, 0, None, None, 0.0, []
        if lora is not None:
            gyb, a_down, s = lora
            a_down = a_down.contiguous()
            rank, ldp, qk, ldq, t, keep = _lora_args([(gyb, a_down, s)], d, ((hdim, d),),
                                                     grad_y, kmajor=False)
            assert qk == 0 and ldq == d
            pp, qq, alpha = t[0]
        with _timed("ffn_down_dgrad"):
            rc = _lib.lib().cpt_ffn_down_dgrad_outlier(
                grad_y.data_ptr(), w_down.data_ptr(), n, hdim, d, cache, group_size, p(c_gate),
                p(s_gate), slot_g.data_ptr(), o_g.data_ptr(), p(c_up), p(s_up),
                slot_u.data_ptr(), o_u.data_ptr(), k, dg.data_ptr(), du.data_ptr(), p(hm),
                rank, ldp, pp, qq, alpha, _stream(grad_y))
        del keep
    elif lora is not None:
        gyb, a_down, s = lora
        a_down = a_down.contiguous()          # [r, inter] rows: the MN-major factor
        r, ldp, qk, ldq, t, keep = _lora_args([(gyb, a_down, s)], d, ((hdim, d),),
                                              grad_y, kmajor=False)
        assert qk == 0 and ldq == d
        with _timed("ffn_down_dgrad"):
            rc = _lib.api().cpt_ffn_down_dgrad_lora(
                grad_y.data_ptr(), w_down.data_ptr(), n, hdim, d, cache, group_size, p(c_gate),
                p(s_gate), p(c_up), p(s_up), dg.data_ptr(), du.data_ptr(), p(hm), r, ldp,
                t[0][0], t[0][1], t[0][2], _stream(grad_y))
        del keep
    else:
        with _timed("ffn_down_dgrad"):
            rc = _lib.api().cpt_ffn_down_dgrad(grad_y.data_ptr(), w_down.data_ptr(), n, hdim, d,
                                               cache, group_size, p(c_gate), p(s_gate), p(c_up),
                                               p(s_up), dg.data_ptr(), du.data_ptr(), p(hm),
                                               _stream(grad_y))
    check(rc, "ffn_down_dgrad")
    return dg, du, hm


def wgrad_glu(grad_y: torch.Tensor, cache: int, group_size: int, q_gate, s_gate, q_up, s_up,
              name: str = "gemm_wgrad_down_glu") -> torch.Tensor:
    """grad_y^T @ h^ -> bf16 [hidden, inter], h^ = bf16(SiLU(hg^) * hu^) formed
    from the int4/int8 cache inside the GEMM's operand staging: the weight
    gradient of the down projection without K2's h_mid^ (bit-equal to
    mm(grad_y.t(), h_mid_hat), src/flashffn.py:1538-1543)."""
    _require_device(grad_y, q_gate, s_gate, q_up, s_up)
    _check_bf16(grad_y)
    n, hdim = grad_y.shape
    assert cache in (_lib.CACHE_INT4, _lib.CACHE_INT8), f"int4/int8 cache expected, got {cache}"
    d = q_gate.shape[1] * (2 if cache == _lib.CACHE_INT4 else 1)
    assert tuple(q_up.shape) == tuple(q_gate.shape) and q_gate.shape[0] == n
    assert group_size > 0 and d % group_size == 0, \
        f"D={d} not divisible by group_size={group_size}"
    assert tuple(s_gate.shape) == (n, d // group_size) == tuple(s_up.shape), \
        f"scales {tuple(s_gate.shape)} / {tuple(s_up.shape)} != {(n, d // group_size)}"
    q_gate, s_gate, q_up, s_up = (t.contiguous() for t in (q_gate, s_gate, q_up, s_up))
    if grad_y.stride(1) != 1 or grad_y.stride(0) % 8 or grad_y.data_ptr() % 16:
        grad_y = grad_y.contiguous()
    c = torch.empty((hdim, d), dtype=torch.bfloat16, device=grad_y.device)
    with _timed(name):
        rc = _lib.lib().cpt_gemm_wgrad_glu(grad_y.data_ptr(), grad_y.stride(0), cache, group_size,
                                           q_gate.data_ptr(), s_gate.data_ptr(), q_up.data_ptr(),
                                           s_up.data_ptr(), c.data_ptr(), c.stride(0), hdim, d, n,
                                           _stream(grad_y))
    check(rc, name)
    return c


def addmm_(c: torch.Tensor, a: torch.Tensor, b: torch.Tensor, alpha: float,
           name: str = "gemm_lora_add") -> torch.Tensor:
    """In place: c = bf16(c + bf16(alpha * bf16(a @ b))), PEFT's
    `h + s * B(A(x))` in bf16 (src/flashffn.py:1414,1420,1439,1529)."""
    _require_device(c, a, b)
    _check_bf16(c, a, b)
    M, K = a.shape
    K_, N = b.shape
    assert K == K_ and tuple(c.shape) == (M, N) and c.stride(1) == 1
    a, lda, ak = _layout_a(a)
    b, ldb, bk = _layout_b(b)
    with _timed(name):
        rc = _lib.api().cpt_gemm_bf16_ex(a.data_ptr(), lda, ak, b.data_ptr(), ldb, bk, c.data_ptr(),
                                         c.stride(0), M, N, K, float(alpha), 1, 1, None, _stream(a))
    check(rc, name)
    return c


def skinny_t_fits(a: torch.Tensor, b: torch.Tensor) -> bool:
    """a [M, K] @ b [K, N] runs on the token-reduction kernel: both token-major
    (a's transpose and b row-major with 16-byte rows), K >= 256 tokens, M and N
    multiples of 8, one of them a rank up to 32."""
    M, K = a.shape
    N = b.shape[1]
    return (_row_major(a.t()) and _row_major(b) and K >= 256 and M % 8 == 0 and N % 8 == 0
            and (M <= SKINNY_MAX_RANK or N <= SKINNY_MAX_RANK))


def mm_splitk(a: torch.Tensor, b: torch.Tensor, alpha: float = 1.0, splits: int | None = None,
              name: str = "gemm_splitk") -> torch.Tensor:
    """bf16(alpha * (a @ b)) with the K reduction split across blocks (fp32
    partials, fixed-order sum): for the thin adapter gradients that reduce
    over all tokens.  With a token-major operand on each side and M or N <=
    32 (the rank: grad_A = s (grad B)^T x, grad_B = s grad_y^T (x A^T)) the
    token-reduction kernel runs instead of 256 x 256 tiles."""
    _require_device(a, b)
    M, K = a.shape
    K_, N = b.shape
    assert K == K_
    at = a.t()
    if splits is None and skinny_t_fits(a, b):
        if M <= SKINNY_MAX_RANK:
            return skinny_t(b, at, alpha, trans=True, name=name)
        return skinny_t(at, b, alpha, trans=False, name=name)
    _check_bf16(a, b)
    a, lda, ak = _layout_a(a)
    b, ldb, bk = _layout_b(b)
    if splits is None:
        tiles = ((M + 255) // 256) * ((N + 255) // 256)
        splits = max(1, min((K + 63) // 64, (512 + tiles - 1) // tiles))
    splits = max(splits, _min_splits(K, lda, ak, ldb, bk))
    ldc = (N + 7) // 8 * 8
    c = torch.empty((M, ldc), dtype=torch.bfloat16, device=a.device)
    ws = torch.empty((splits * M * N,), dtype=torch.float32, device=a.device)
    with _timed(name):
        rc = _lib.api().cpt_gemm_bf16_ex(a.data_ptr(), lda, ak, b.data_ptr(), ldb, bk, c.data_ptr(),
                                         ldc, M, N, K, float(alpha), 2, splits, ws.data_ptr(),
                                         _stream(a))
    check(rc, name)
    return c if ldc == N else c[:, :N]


# ---------------------------------------------------------------------------
# fp32 products on the bf16 MFMAs (cpt_split_f32, cpt_gemm_f32x3)
# ---------------------------------------------------------------------------

class Planes:
    """The bf16 planes of the fp32 operands of one forward or backward call.

    An operand is split once for the products that follow each other on it,
    whatever view of it they take.  Planes are 1.5 times their operand, so at most
    KEEP_BYTES of them are held, or as many bytes as the call's largest operand:
    the least recently used go first, and are made again if a later product asks.
    320 MiB is what the widest backward of 2048 tokens at 2048 x 5632 shares
    (grad_x's four operands and two before them); held without a bound, a call of
    8192 tokens peaks at 2059 MiB against 727 on the general-layout kernel and 1065
    so, at 8.7 ms against 18.7 and 9.0.  With 320 MiB at 32768 tokens the weight
    gradients' panels are narrow: 45.2 ms against 34.3 without a bound.  An entry
    holds its operand, so no other tensor can take its memory meanwhile; an operand
    must not be written between its products."""

    KEEP_BYTES = 320 << 20
    MAX_FLAGS = 32

    def __init__(self):
        self._made = {}
        self._bytes = 0
        self._largest = 0
        self._flags = None
        self._used = 0

    def bound(self, *operands) -> int:
        """The bytes of planes held at a time, once the call has these operands."""
        for t in operands:
            if t is not None and 4 * t.numel() > self._largest:
                self._largest = 4 * t.numel()
        return max(self.KEEP_BYTES, self._largest)

    def of(self, t: torch.Tensor):
        """(planes bf16 [3, rows, cols], flag int32 [1]) of row-major fp32 t.  The
        caller keeps both until its product is launched."""
        key = (t.data_ptr(), t.shape, t.stride(0))
        hit = self._made.pop(key, None)
        if hit is None:
            nbytes = 6 * t.numel()
            while self._made and self._bytes + nbytes > self.bound():
                self._forget(next(iter(self._made)))
            if self._flags is None or self._used == self.MAX_FLAGS:
                self._flags = torch.zeros((self.MAX_FLAGS,), dtype=torch.int32, device=t.device)
                self._used = 0
            flag = self._flags[self._used:self._used + 1]
            self._used += 1
            planes = torch.empty((3,) + tuple(t.shape), dtype=torch.bfloat16, device=t.device)
            with _timed("split_f32"):
                rc = _lib.api().cpt_split_f32(t.data_ptr(), t.stride(0), t.shape[0], t.shape[1],
                                              planes.data_ptr(), flag.data_ptr(), _stream(t))
            check(rc, "split_f32")
            hit = (planes, flag, t)
            self._bytes += nbytes
        self._made[key] = hit
        return hit[0], hit[1]

    def _forget(self, key):
        self._bytes -= 6 * self._made.pop(key)[2].numel()

    def drop(self, t: torch.Tensor) -> None:
        """Forget t and every view of it: its last product is launched."""
        base = t.untyped_storage().data_ptr()
        for key in [k for k, e in self._made.items()
                    if e[2].untyped_storage().data_ptr() == base]:
            self._forget(key)


def _x3_operand(t: torch.Tensor):
    """(row-major storage of t or of its transpose, whether it is t), or None
    where the split kernel does not take it."""
    if t.stride(1) == 1 and t.stride(0) >= t.shape[1]:
        s, own = t, True
    elif t.stride(0) == 1 and t.stride(1) >= t.shape[0]:
        s, own = t.t(), False
    else:
        return None
    if s.stride(0) % 4 or s.shape[1] % 8 or s.data_ptr() % 16:
        return None
    return s, own


def x3_fits(a: torch.Tensor, b: torch.Tensor) -> bool:
    """a [M, K] @ b [K, N] in fp32 runs on the bf16 MFMAs (mm_x3): row-major or
    transposed operands with 16-byte aligned rows of whole 8-element vectors, N a
    multiple of 8, K of 64 unless both operands are stored k by k."""
    if not (a.dtype == b.dtype == torch.float32 and a.dim() == 2 and b.dim() == 2 and a.is_cuda):
        return False
    (M, K), N = a.shape, b.shape[1]
    if M == 0 or K == 0 or N == 0 or N % 8:
        return False
    oa, ob = _x3_operand(a), _x3_operand(b)
    if oa is None or ob is None:
        return False
    rows = (K + 256) * 2
    if (not oa[1] and rows * M >= _SPAN_BYTES) or (ob[1] and rows * N >= _SPAN_BYTES):
        return False
    return K % 64 == 0 or (not oa[1] and ob[1])


def x3_pays(m: int, n: int, k: int) -> bool:
    """An fp32 product of k (both pairs' together) is faster on the planes than on
    the general-layout kernel, whose time goes with k and its rounds of 128 x 128
    tiles: below this its one launch costs less than two splits, the product and
    the guarded general kernel.  Measured on MI355X, us general / planes with both
    operands to split / with none:
      64 x 704, k 256     32.3 / 42.4 / 22.1    kept general
      64 x 704, k 320     38.9 / 42.6 / 22.7    kept general
      64 x 704, k 448     52.0 / 42.9 / 22.3
      2048 x 2048, k 256  35.0 / 51.9 / 44.5    kept general
      2048 x 5632, k 64   29.5 / 37.7 / 24.0    kept general
      2048 x 5632, k 128  45.6 / 40.8 / 29.9
    and 1 token at 256 x 704, whole steps: forward 147 us general, 165 on the
    planes; full fine-tune 400 and 444."""
    tiles = ((m + 127) // 128) * ((n + 127) // 128)
    return k * max(tiles, 256) >= 352 * 256


def x3_plan(m: int, n: int, nk: int, whole: bool) -> tuple[int, int]:
    """(tile width, k ranges) of an fp32 product of nk k-tiles of plane pairs; 256
    x 256 and 256 x 192 tiles need whole k-tiles.  Times per k-tile with the chip
    full: 1.33 us a 256 x 256 tile, 1.12 a 256 x 192 one, 0.57 a 128 x 128 one, so
    the rounds of blocks decide.  Measured, us on 256 / 192 columns: 2048 x 5632,
    k 2048 (176 / 240 blocks) 269 / 226; 2048 x 2048, k 5632 (4 / 2 ranges) 212 /
    284."""
    small = split_plan(m, n, nk)
    t128 = ((m + 127) // 128) * ((n + 127) // 128) * small
    t256 = ((m + 255) // 256) * ((n + 255) // 256)
    big = max(1, min(256 // t256, nk // SPLIT_MIN_KT))
    cost128 = 0.57 * min(-(-t128 // 256), 1.9 * -(-t128 // 512)) * nk / small
    t192 = ((m + 255) // 256) * ((n + 191) // 192)
    narrow = max(1, min(256 // t192, nk // SPLIT_MIN_KT))
    cost256 = 1.33 * -(-t256 * big // 256) * nk / big
    cost192 = 1.12 * -(-t192 * narrow // 256) * nk / narrow
    if not whole or cost128 <= min(cost256, cost192):
        return 128, small
    return (192, narrow) if cost192 < cost256 else (256, big)


def mm_x3(a, b, planes: Planes, a2=None, b2=None, alpha: float = 1.0,
          name: str = "gemm_f32") -> torch.Tensor:
    """alpha * (a @ b (+ a2 @ b2)) in fp32 from the operands' bf16 planes
    (x3_fits each pair, the pairs in one layout), and, on the device and only if
    a value lies outside the planes' range, again on the general-layout kernel.

    Three times closer to float64 than the general-layout kernel and about
    twice as fast, splitting included (x3_gemm_impl in csrc/gemm.hip)."""
    _require_device(a, b, a2, b2)
    ops = (a, b) if a2 is None else (a, b, a2, b2)
    assert all(t.dtype == torch.float32 and t.dim() == 2 for t in ops), \
        f"2-D float32 operands expected, got {[t.dtype for t in ops]}"
    (M, K), N = a.shape, b.shape[1]
    assert b.shape[0] == K, f"inner dims differ: {tuple(a.shape)} @ {tuple(b.shape)}"
    assert a2 is None or (a2.shape[0] == M and tuple(b2.shape) == (a2.shape[1], N)), \
        f"second pair {tuple(a2.shape)} @ {tuple(b2.shape)} of an [{M}, {N}] product"

    c = torch.empty((M, N), dtype=torch.float32, device=a.device)
    pm, pn = _x3_panels(M, N, K if a2 is None else K + a2.shape[1], planes.bound(a, b, a2, b2))
    for m in range(0, M, pm):
        for n in range(0, N, pn):
            if pm >= M and pn >= N:
                _x3_launch(c, a, b, a2, b2, planes, alpha, name)
                break
            row, col = slice(m, m + pm), slice(n, n + pn)
            _x3_launch(c[row, col], a[row], b[:, col], None if a2 is None else a2[row],
                       None if a2 is None else b2[:, col], planes, alpha, name)
    return c


def _x3_panels(m: int, n: int, k: int, limit: int) -> tuple[int, int]:
    """(rows, columns) of the panels that an [m, n] product of k runs in, so that
    the planes of one panel's operands stay within `limit` bytes (or are 256
    wide): the wider side is halved first."""
    pm, pn = m, n
    while 6 * (pm + pn) * k > limit and max(pm, pn) > 256:
        if pm >= pn:
            pm = (pm // 2 + 255) // 256 * 256
        else:
            pn = (pn // 2 + 255) // 256 * 256
    return pm, pn


def _x3_launch(c, a, b, a2, b2, planes: Planes, alpha: float, name: str) -> None:
    """One panel of mm_x3 into the view c."""
    (M, K), N = a.shape, b.shape[1]
    held = []

    def operand(t, left):
        s, own = _x3_operand(t)
        p, flag = planes.of(s)
        held.append((p, flag))
        # [M][K] or [N][K] storage is K-major
        return p.data_ptr(), s.shape[0] * s.shape[1], s.shape[1], int(own == left), flag.data_ptr()
    pa, sa, lda, ak, fa = operand(a, True)
    pb, sb, ldb, bk, fb = operand(b, False)
    pa2 = pb2 = fa2 = fb2 = None
    sa2 = sb2 = K2 = 0
    if a2 is not None:
        K2 = a2.shape[1]
        pa2, sa2, lda2, ak2, fa2 = operand(a2, True)
        pb2, sb2, ldb2, bk2, fb2 = operand(b2, False)
        assert (lda2, ldb2, ak2, bk2) == (lda, ldb, ak, bk), "the pairs share one layout"
    tiles, splits = x3_plan(M, N, 6 * ((K + 63) // 64 + (K2 + 63) // 64),
                            K % 64 == 0 and K2 % 64 == 0)
    ws = (torch.empty((splits * M * N,), dtype=torch.float32, device=a.device)
          if splits > 1 else None)
    st = _stream(a)
    L = _lib.api()
    ldc = c.stride(0)
    with _timed(name):
        rc = L.cpt_gemm_f32x3(pa, sa, lda, ak, pb, sb, ldb, bk, pa2, sa2, pb2, sb2, K2, fa, fb,
                              fa2, fb2, c.data_ptr(), ldc, M, N, K, float(alpha), tiles, splits,
                              None if ws is None else ws.data_ptr(), st)
        check(rc, name)
        for i, (u, v) in enumerate(((a, b), (a2, b2))[:1 if a2 is None else 2]):
            rc = L.cpt_gemm_any_if(fa, fb, fa2, fb2, _lib.F32, u.data_ptr(), u.stride(0),
                                   u.stride(1), v.data_ptr(), v.stride(0), v.stride(1),
                                   c.data_ptr(), ldc, 1, M, N, u.shape[1], float(alpha),
                                   ANY_ADD if i else ANY_SCALE, st)
            check(rc, name)


# epilogues of the general-layout GEMM (cpt_gemm_any)
ANY_STORE, ANY_ADD, ANY_SCALE = 0, 1, 2
_ANY_DT = {torch.float32: _lib.F32, torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}


def mm_any(a: torch.Tensor, b: torch.Tensor, alpha: float = 1.0, mode: int = ANY_STORE,
           out: torch.Tensor | None = None, name: str = "gemm_any",
           planes: Planes | None = None) -> torch.Tensor:
    """a [M, K] @ b [K, N] for float32 / float16 / bfloat16 operands of any
    strides, in the modes of mm_any_kernel: the products the bf16 engine does
    not take (config C1's float32, unaligned views, rank-1 factors).  fp32
    operands that fit (x3_fits) go to the bf16 MFMAs where that pays (x3_pays),
    sharing the planes that the caller's other products made."""
    if (mode != ANY_ADD and a.dtype == torch.float32 and x3_fits(a, b)
            and x3_pays(a.shape[0], b.shape[1], a.shape[1])):
        return mm_x3(a, b, planes or Planes(), alpha=alpha if mode == ANY_SCALE else 1.0,
                     name=name)
    return mm_any_kernel(a, b, alpha, mode, out, name)


def mm_any_kernel(a: torch.Tensor, b: torch.Tensor, alpha: float = 1.0, mode: int = ANY_STORE,
                  out: torch.Tensor | None = None, name: str = "gemm_any") -> torch.Tensor:
    """a [M, K] @ b [K, N] on the general-layout kernel, the fp32 MFMA
    (cpt_gemm_any).
    mode ANY_STORE: rd(a @ b); ANY_SCALE: rd(alpha * rd(a @ b)); ANY_ADD: in
    place, out = rd(out + rd(alpha * rd(a @ b))), with rd the rounding to the
    operands' dtype (the reference's eager op order)."""
    _require_device(a, b)
    assert a.dim() == 2 and b.dim() == 2, "2-D operands expected"
    assert a.dtype == b.dtype and a.dtype in _ANY_DT, f"unsupported dtypes {a.dtype}, {b.dtype}"
    M, K = a.shape
    K_, N = b.shape
    assert K == K_, f"inner dims differ: {tuple(a.shape)} @ {tuple(b.shape)}"
    if mode == ANY_ADD:
        assert out is not None and tuple(out.shape) == (M, N) and out.dtype == a.dtype
    else:
        out = torch.empty((M, N), dtype=a.dtype, device=a.device)
    with _timed(name):
        rc = _lib.api().cpt_gemm_any(_ANY_DT[a.dtype], a.data_ptr(), a.stride(0), a.stride(1),
                                     b.data_ptr(), b.stride(0), b.stride(1), out.data_ptr(),
                                     out.stride(0), out.stride(1), M, N, K, float(alpha), mode,
                                     _stream(a))
    check(rc, name)
    return out

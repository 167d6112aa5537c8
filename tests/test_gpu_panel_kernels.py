"""Panel and small-node kernels at the edges of their ranges (GPU)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _dev(later, A, pad=0):
    X = later.colmajor(A.shape[0], A.shape[1], ld=A.shape[0] + pad)
    X.copy_(torch.from_numpy(np.ascontiguousarray(A)))
    return X


def _np(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


# Block MGS: full blocks, a merged tail (five rows per lane), a lone short
# block, a partly filled last wave.  Scaling the panel by a power of two
# scales every intermediate exactly (no overflow, no underflow that reaches a
# sum), so Q must keep its bits and R must scale exactly, although +-2^52
# takes the column norms out of the range of the fast square root.
@pytest.mark.parametrize("m,w", [(256, 32), (287, 32), (1000, 29), (40, 1), (33, 32), (600, 6)])
@pytest.mark.parametrize("p", [-52, 52])
def test_mgs_panel_scales_exactly(later, oracle, m, w, p):
    A = oracle.gen_uniform(m, w, 3, 1)
    a, b = _dev(later, A), _dev(later, np.ldexp(A, p).astype(np.float32))
    ra, rb = later.caqr_panel(a), later.caqr_panel(b)
    assert np.array_equal(_np(a), _np(b))
    assert np.array_equal(np.ldexp(_np(ra), p), _np(rb))
    Qo, Ro = oracle.caqr32(A)
    assert oracle.rel_err(_np(ra), Ro) < 2e-6 and oracle.rel_err(_np(a), Qo) < 4e-6


# Tree apply: the next level's product folded in (two levels), a level left to
# its own launch (three), w that does not divide 256 (rows of one stack block
# in two blocks of the next level), a workgroup per block (256 blocks and
# more) with a merged tail.
@pytest.mark.parametrize("m,w", [(520, 20), (5000, 20), (9000, 31), (65536 + 9, 20), (70003, 29), (132000, 32)])
@pytest.mark.parametrize("fp64", [0, 1])
def test_tsqr_apply_levels(later, oracle, m, w, fp64):
    A = oracle.gen_uniform(m, w, 5, 2)
    X = _dev(later, A, pad=1)
    R = later.caqr_panel(X, fp64=fp64)
    Q, R = _np(X), _np(R)
    Qo, Ro = oracle.caqr32(A)
    assert oracle.rel_err(R, Ro) < 2e-6 and oracle.rel_err(Q, Qo) < 4e-6
    assert oracle.orth(Q) < (2e-6 if fp64 else 4e-6) * np.sqrt(w)


# The 16-blocked Cholesky factor: dependent columns (a zero column, a repeated
# one) at the edges of its blocks, widths that end inside each block, on the
# fused launch and (200000 rows) the separate factor launch.  The dependent
# column of Q is zero, the rest orthonormal, A = QR still holds: the bounds of
# the other wide-leaf tests.
@pytest.mark.parametrize("m", [1500, 200000])
@pytest.mark.parametrize("w,dup", [(17, (None, 16)), (16, (0, 15)), (48, (31, 32)), (64, (None, 0)), (64, (15, 16)),
                                   (64, (5, 63)), (33, (None, 32)), (49, (47, 48)), (32, (2, 17))])
def test_cholesky_leaf_blocks_breakdown(later, oracle, m, w, dup):
    A = oracle.gen_uniform(m, w, 7, 3)
    A[:, dup[1]] = 0.0 if dup[0] is None else A[:, dup[0]]
    X = _dev(later, A)
    o = later.opts("mixed")
    work = later.workspace(m, w, o)
    R = later.rgsqrf(X, o=o, work=work)
    torch.cuda.synchronize()
    assert later.read_status(work) & 1
    Q, R = _np(X), _np(R)
    keep = [j for j in range(w) if j != dup[1]]
    assert np.all(Q[:, dup[1]] == 0) and np.isfinite(Q).all() and np.isfinite(R).all()
    assert oracle.orth(Q[:, keep]) < 2e-6 * np.sqrt(w) and oracle.backward(A, Q, R) < 1e-6


# FP32 products of narrow nodes: tile edges, K blocks of 128 and splits, any
# leading dimension (dword-aligned vector loads).  Each product is a chain of K
# fused multiply-adds (and a sum of split partials in FP64), so an element is
# within (K + 2) 2^-24 of its terms' magnitudes.
@pytest.mark.parametrize("m", [1, 15, 17, 128, 129, 257, 4099])
@pytest.mark.parametrize("n1,n2,pad", [(1, 1, 0), (31, 33, 1), (32, 32, 2), (64, 96, 3), (128, 127, 0), (65, 128, 1)])
def test_narrow_products(later, oracle, m, n1, n2, pad):
    u = 2.0 ** -24
    Q, B, C = oracle.gen_uniform(m, n1, 1, 1), oracle.gen_uniform(m, n2, 2, 2), oracle.gen_uniform(n1, n2, 3, 3)
    q, b, c = _dev(later, Q, pad), _dev(later, B, pad), _dev(later, C, pad)
    P = _np(later.gemm_proj(q, b, later.colmajor(n1, n2, ld=n1 + pad), later.GEMM_F32))
    Q, B, C = Q.astype(np.float64), B.astype(np.float64), C.astype(np.float64)
    assert np.all(np.abs(P - Q.T @ B) <= (m + 2) * u * (np.abs(Q).T @ np.abs(B)) + 1e-45)
    U = _np(later.gemm_update(q, c, b, later.GEMM_F32))
    assert np.all(np.abs(U - (B - Q @ C)) <= (n1 + 2) * u * (np.abs(Q) @ np.abs(C) + np.abs(B)) + 1e-45)


# Triangular solve at the edges of its 64-row blocks and of its two column
# arrays, and with a zero on the diagonal (its unknown is 0).  The sums are FP64
# and x is rounded to FP32 once, so the residual is within 2^-24 (plus n FP64
# roundings) of |R| |x| in every component.
@pytest.mark.parametrize("n,k", [(1, 1), (63, 2), (65, 1), (129, 3), (1024, 3), (1025, 1)])
@pytest.mark.parametrize("zero", [False, True])
def test_trsm_upper_blocks(later, oracle, n, k, zero):
    R = np.triu(oracle.gen_uniform(n, n, 4, 4)) + 4.0 * np.sqrt(n) * np.eye(n, dtype=np.float32)
    R = R.astype(np.float32)
    B = oracle.gen_uniform(n, k, 5, 5)
    j = n // 2
    if zero:
        R[j, j] = 0.0
    X = _dev(later, B, 1)
    later.trsm_upper(_dev(later, R, 1), X)
    X = _np(X).astype(np.float64)
    rows = [i for i in range(n) if not (zero and i == j)]
    if zero:
        assert np.all(X[j] == 0.0)
    R = R.astype(np.float64)
    res = np.abs(R @ X - B)[rows]
    assert np.all(res <= (2.0 ** -24 + n * 2.0 ** -50) * (np.abs(R) @ np.abs(X))[rows] + 1e-30)


# Products whose operands are converted on the way to LDS: slab counts around
# the untested loop's start, ragged K, tile rows and columns, leading dimension
# and address at any dword (K-major both, then rows of A along M).  An element
# is a chain of K fused products (and a few FP64 sums) of operands kept to 24
# (F32, F16X6), 22 (F16X3) or 11 bits (F16): K + 2 units of 2^-24 of its terms'
# magnitudes, 16 more for the dropped low pieces, 2^-10 for one piece.
@pytest.mark.parametrize("k", [128, 129, 160, 161, 321, 575, 640, 1089])
@pytest.mark.parametrize("n1,n2,pad", [(64, 192, 0), (131, 129, 1), (300, 257, 3)])
@pytest.mark.parametrize("prec,extra", [("GEMM_F32", 0.0), ("GEMM_F16X6", 16.0), ("GEMM_F16X3", 16.0),
                                        ("GEMM_F16", 2.0 ** 14)])
def test_staged_products(later, oracle, k, n1, n2, pad, prec, extra):
    u, p = 2.0 ** -24, getattr(later, prec)
    A, B = oracle.gen_uniform(k, n1, 1, 1), oracle.gen_uniform(k, n2, 2, 2)
    a, b = _dev(later, A, pad), _dev(later, B, pad)
    P = _np(later.gemm_proj(a, b, later.colmajor(n1, n2, ld=n1 + pad), p))
    A, B = A.astype(np.float64), B.astype(np.float64)
    assert np.all(np.abs(P - A.T @ B) <= (k + 2 + extra) * u * (np.abs(A).T @ np.abs(B)) + k * 2.0 ** -22 * (extra > 16))
    Q, C, D = oracle.gen_uniform(n1, k, 3, 3), oracle.gen_uniform(k, n2, 4, 4), oracle.gen_uniform(n1, n2, 5, 5)
    q, c, d = _dev(later, Q, pad), _dev(later, C, pad), _dev(later, D, pad)
    U = _np(later.gemm_update(q, c, d, p))
    Q, C, D = (x.astype(np.float64) for x in (Q, C, D))
    assert np.all(np.abs(U - (D - Q @ C)) <= (k + 2 + extra) * u * (np.abs(Q) @ np.abs(C)) + 2 * u * np.abs(D)
                  + k * 2.0 ** -22 * (extra > 16))


# Tall Cholesky leaves: four blocks and more for some workgroups of the grid
# (512 blocks of 64 rows are one each), a ragged last block, widths short of
# the kernel's, odd leading dimensions.  FP64 Grams and two passes: Q within
# the FP32 rounding of its entries.
@pytest.mark.parametrize("m", [98304, 131072 + 64 * 5 + 17, 262144 + 3])
@pytest.mark.parametrize("w,pad", [(64, 0), (64, 1), (63, 3), (32, 1), (20, 0)])
def test_tall_cholesky_leaf(later, oracle, m, w, pad):
    A = oracle.gen_uniform(m, w, 9, 4)
    X = _dev(later, A, pad)
    o = later.opts("mixed")
    work = later.workspace(m, w, o)
    R = later.rgsqrf(X, o=o, work=work)
    torch.cuda.synchronize()
    Q, R = _np(X), _np(R)
    assert later.read_status(work) == 0
    assert oracle.orth(Q) < 2e-6 * np.sqrt(w) and oracle.backward(A, Q, R) < 1e-6


# Streamed products of pre-split operands: wave tiles inside C and at its edges
# (64 and 32 rows of a wave), exponents of B at any dword address, an update and
# a projection with and without splits.  Bounds as above.
@pytest.mark.parametrize("m,n1,n2", [(512, 192, 160), (3000, 257, 130), (1100, 320, 97)])
@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("prec,extra", [("GEMM_F16X6", 16.0), ("GEMM_F16X3", 16.0), ("GEMM_F16", 2.0 ** 14)])
def test_streamed_products(later, oracle, m, n1, n2, pad, prec, extra):
    u, p = 2.0 ** -24, getattr(later, prec)
    Q, B, C = oracle.gen_uniform(m, n1, 1, 1), oracle.gen_uniform(m, n2, 2, 2), oracle.gen_uniform(n1, n2, 3, 3)
    q, b, c = _dev(later, Q, pad), _dev(later, B, pad), _dev(later, C, pad)
    P = _np(later.gemm_proj(q, b, later.colmajor(n1, n2, ld=n1 + pad), p, pieces=True))
    U = _np(later.gemm_update(q, c, b, p, pieces=True))
    Q, B, C = (x.astype(np.float64) for x in (Q, B, C))
    assert np.all(np.abs(P - Q.T @ B) <= (m + 2 + extra) * u * (np.abs(Q).T @ np.abs(B)) + m * 2.0 ** -22 * (extra > 16))
    assert np.all(np.abs(U - (B - Q @ C)) <= (n1 + 2 + extra) * u * (np.abs(Q) @ np.abs(C)) + 2 * u * np.abs(B)
                  + n1 * 2.0 ** -22 * (extra > 16))


# A node whose second half is a Cholesky leaf: update and first Gram in one
# pass.  Against the same steps one by one (leaf, projection, update, leaf), for
# both kernel widths, fewer and more blocks than workgroups, ragged rows and any
# leading dimension: the same bits.
@pytest.mark.parametrize("m", [128, 161, 4099, 33000, 131072 + 70, 300003])
@pytest.mark.parametrize("n,pad", [(65, 1), (96, 0), (97, 3), (127, 2), (128, 0), (128, 1)])
@pytest.mark.parametrize("panel", ["PANEL_CHOLQR1", "PANEL_CHOLQR2"])
def test_update_with_leaf_gram(later, oracle, m, n, pad, panel):
    o = later.opts("mixed", reorth=0, panel=getattr(later, panel))
    A = _dev(later, oracle.gen_uniform(m, n, 11, 6), pad)
    X, R = _dev(later, _np(A), pad), later.colmajor(n, n, ld=n + pad)
    later.rgsqrf(A, o=o, R=R)
    S = later.colmajor(n, n, ld=n + pad)
    X1, X2 = X[:, :64], X[:, 64:]
    later.rgsqrf(X1, R=S[:64, :64], o=o)
    later.gemm_proj(X1, X2, S[:64, 64:], later.GEMM_F32)
    later.gemm_update(X1, S[:64, 64:], X2, later.GEMM_F32)
    later.rgsqrf(X2, R=S[64:, 64:], o=o)
    assert np.array_equal(_np(A), _np(X))
    assert np.array_equal(np.triu(_np(R)), np.triu(_np(S)))


# Projections of many splits (97 and more): their reduction's rounds, ragged
# elements of its last workgroup, FP32 and FP64 partials.  Bounds as above (a
# split's FP32 chain is shorter than m; FP64 folds keep chains to 256).
@pytest.mark.parametrize("m", [24900, 40001, 131072 + 5])
@pytest.mark.parametrize("n1,n2", [(64, 64), (33, 17), (1, 3), (128, 100)])
@pytest.mark.parametrize("prec,chunk", [("GEMM_F32", 0), ("GEMM_F16X6", 256)])
def test_many_splits(later, oracle, m, n1, n2, prec, chunk):
    A, B = oracle.gen_uniform(m, n1, 1, 1), oracle.gen_uniform(m, n2, 2, 2)
    C = _np(later.gemm_proj(_dev(later, A, 1), _dev(later, B), later.colmajor(n1, n2, ld=n1 + 1),
                            getattr(later, prec), chunk))
    A, B = A.astype(np.float64), B.astype(np.float64)
    k = chunk + 16 if chunk else 2048
    assert np.all(np.abs(C - A.T @ B) <= (k + 2) * 2.0 ** -24 * (np.abs(A).T @ np.abs(B)))


# Column exponents on both sides of the tall kernel's line, with the largest
# entry in the first row, the last row or the last whole vector, columns far from
# 1 and any address: a wrong exponent overflows FP16 or loses the column.  Bound
# as above (FP64 folds every 256 rows).
@pytest.mark.parametrize("m", [16384, 16385, 32768 + 5, 70001])
@pytest.mark.parametrize("pad", [0, 1, 2])
def test_tall_column_exponents(later, oracle, m, pad):
    A, B = oracle.gen_uniform(m, 40, 1, 1), oracle.gen_uniform(m, 6, 2, 2)
    for j, (i, p) in enumerate([(0, 40), (m - 1, -40), (m - 6, 20), (m // 2, -20), (1, 0), (m - 2, 3)]):
        B[i, j] = 1000.0
        B[:, j] = np.ldexp(B[:, j], p)
    C = _np(later.gemm_proj(_dev(later, A, pad), _dev(later, B, pad), later.colmajor(40, 6), later.GEMM_F16X6, 256))
    A, B = A.astype(np.float64), B.astype(np.float64)
    assert np.all(np.abs(C - A.T @ B) <= (256 + 18) * 2.0 ** -24 * (np.abs(A).T @ np.abs(B)))

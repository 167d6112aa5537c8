"""The triangular solve: zero diagonals, many right-hand sides (GPU)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _dev(later, A, pad=0):
    X = later.colmajor(A.shape[0], A.shape[1], ld=A.shape[0] + pad)
    X.copy_(torch.from_numpy(np.ascontiguousarray(A)))
    return X


def _system(oracle, n, k, seed=31):
    R = (np.triu(oracle.gen_uniform(n, n, seed, 1)) + 4.0 * np.sqrt(n) * np.eye(n)).astype(np.float32)
    return R, oracle.gen_uniform(n, k, seed, 2)


# The unknown of a zero on the diagonal is +0 whatever its right-hand side holds
# (negative, infinite, NaN), and the rows above are solved with that 0: their
# residual is within 2^-24 (plus n FP64 roundings) of |R| |x|.
@pytest.mark.parametrize("n", [1, 16, 17, 40, 64, 65, 200])
@pytest.mark.parametrize("value", [-1.0, np.inf, -np.inf, np.nan])
def test_zero_diagonal_unknown_is_zero(later, oracle, n, value):
    R, B = _system(oracle, n, 3)
    zeros = sorted({n // 2, n - 1, 0})
    for j in zeros:
        R[j, j] = 0.0
        B[j] = value
    X = _dev(later, B, 1)
    later.trsm_upper(_dev(later, R), X)
    torch.cuda.synchronize()
    X = X.cpu().numpy()
    assert np.array_equal(X[zeros], np.zeros((len(zeros), 3))) and not np.signbit(X[zeros]).any()
    rows = [i for i in range(n) if i not in zeros]
    R, X = R.astype(np.float64), X.astype(np.float64)
    res = np.abs(R @ X - np.where(np.isfinite(B), B, 0.0))[rows]
    assert np.all(res <= (2.0 ** -24 + n * 2.0 ** -50) * (np.abs(R) @ np.abs(X))[rows] + 1e-30)


# Every right-hand side gets the same bits however many there are: a workgroup
# each, a wave for two and a wave for four, at the edges of their ranges, with
# zeros on the diagonal and a partly filled last wave.
@pytest.mark.parametrize("n", [1, 8, 16, 17, 63, 64, 65, 130, 256, 512, 513, 600])
@pytest.mark.parametrize("k", [513, 1537, 4097])
@pytest.mark.parametrize("zero", [False, True])
def test_same_bits_for_many_right_hand_sides(later, oracle, n, k, zero):
    R, B = _system(oracle, n, k)
    if zero:
        R[n // 2, n // 2] = 0.0
    R, X = _dev(later, R, 3), _dev(later, B, 1)
    later.trsm_upper(R, X)
    for a in sorted({0, 254, 255, 511, k - 5, k - 1}):
        b = min(a + 2, k)
        Y = _dev(later, B[:, a:b])
        later.trsm_upper(R, Y)
        torch.cuda.synchronize()
        assert np.array_equal(X.cpu().numpy()[:, a:b], Y.cpu().numpy()), (a, b)


# Residuals as above, with one right-hand side and with many.
@pytest.mark.parametrize("k", [1, 2000])
def test_many_right_hand_sides_residual(later, oracle, k):
    n = 100
    R, B = _system(oracle, n, k)
    X = _dev(later, B)
    later.trsm_upper(_dev(later, R), X)
    torch.cuda.synchronize()
    X, R = X.cpu().numpy().astype(np.float64), R.astype(np.float64)
    assert np.all(np.abs(R @ X - B) <= (2.0 ** -24 + n * 2.0 ** -50) * (np.abs(R) @ np.abs(X)) + 1e-30)

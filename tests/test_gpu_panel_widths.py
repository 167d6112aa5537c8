"""Tall panels at the widths where the block and tree kernels change over (GPU)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

WIDTHS = [1, 3, 4, 5, 7, 8, 9, 12, 15, 16, 17, 31]


def _panel(later, A, fp64, pad=0):
    X = later.colmajor(A.shape[0], A.shape[1], ld=A.shape[0] + pad)
    X.copy_(torch.from_numpy(np.ascontiguousarray(A)))
    R = later.caqr_panel(X, fp64=fp64)
    torch.cuda.synchronize()
    return X.cpu().numpy(), R.cpu().numpy()


# One block: a column of MGS does not depend on those behind it, so a narrow
# panel has the bits of the first columns of a 32-column one.
@pytest.mark.parametrize("m", [32, 200, 256])
@pytest.mark.parametrize("fp64", [0, 1])
def test_block_widths_keep_bits(later, oracle, m, fp64):
    A = oracle.gen_uniform(m, 32, 41, 1)
    Q, R = _panel(later, A, fp64)
    for w in WIDTHS:
        q, r = _panel(later, A[:, :w], fp64, 1)
        assert np.array_equal(q, Q[:, :w]) and np.array_equal(r, R[:w, :w]), w


# A merged tail (five rows per lane), two and three levels, a 64-row tile and a
# whole block per workgroup: the bounds of the other panel tests.
@pytest.mark.parametrize("m", [257, 520, 5000, 70003])
@pytest.mark.parametrize("fp64", [0, 1])
def test_tree_widths(later, oracle, m, fp64):
    for w in WIDTHS:
        A = oracle.gen_uniform(m, w, 42, w)
        Q, R = _panel(later, A, fp64, 1)
        Qo, Ro = oracle.caqr32(A)
        assert oracle.rel_err(R, Ro) < 2e-6 and oracle.rel_err(Q, Qo) < 4e-6, w
        assert oracle.orth(Q) < (2e-6 if fp64 else 4e-6) * np.sqrt(w), w

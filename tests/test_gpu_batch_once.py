"""The batched QR's FP32 kernels with one projection (reorth = 0), where a panel
behind the first may have to be factored a second time (GPU)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

NARROW, WIDE = 1, 4


def _run(later, mats, variant, form="fp32", reorth=0, pad=0):
    As, Rs = [], []
    for A in mats:
        X = later.colmajor(A.shape[0], A.shape[1], ld=A.shape[0] + pad)
        X.copy_(torch.from_numpy(np.ascontiguousarray(A)))
        As.append(X)
        Rs.append(later.colmajor(A.shape[1], A.shape[1], ld=A.shape[1] + pad))
    tuning = None if variant is None else [variant] * later.BATCH_BUCKETS
    plan = later.BatchWg(As, Rs, later.opts(form, reorth=reorth), tuning=tuning)
    plan.execute()
    torch.cuda.synchronize()
    status = plan.status.cpu().numpy().copy()
    plan.close()
    return [(q.cpu().numpy().copy(order="F"), r.cpu().numpy().copy(order="F")) for q, r in zip(As, Rs)], status


def _kappa(m, n, decades, seed):
    """Singular values over `decades` powers of ten."""
    rng = np.random.default_rng(seed)
    U, _ = np.linalg.qr(rng.standard_normal((m, n)))
    V, _ = np.linalg.qr(rng.standard_normal((n, n)))
    return (U * np.logspace(0, -decades, n) @ V.T).astype(np.float32)


# Panels that are factored twice: near-square matrices, columns of magnitude 1
# and 1000 in turn, singular values over six decades, a zero column behind the
# first panel.  A = QR to the rounding of the batch's other tests (1e-6), R
# within kappa 1e-6 of FP64 LAPACK's, everything finite, the status bit for the
# zero column only; on the kernel that the built-in table takes and on the wide
# one.
@pytest.mark.parametrize("form", ["fp32", "mixed"])
@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("variant", [None, WIDE])
def test_one_projection_second_factor(later, oracle, form, pad, variant):
    mats = [oracle.gen_uniform(m, n, 17, i) for i, (m, n) in
            enumerate([(65, 65), (96, 96), (128, 128), (130, 129), (200, 200), (256, 256), (257, 193)])]
    for m, n in [(1000, 128), (515, 256)]:
        mats.append((oracle.gen_uniform(m, n, 18, n) * np.where(np.arange(n) % 2, 1000.0, 1.0)).astype(np.float32))
    mats.append(_kappa(400, 150, 6, 6))
    dep = oracle.gen_uniform(600, 150, 19, 3)
    dep[:, 90] = 0.0
    mats.append(dep)
    outs, status = _run(later, mats, variant, form, 0, pad)
    assert list(status) == [0] * (len(mats) - 1) + [1]
    for i, (A, (Q, R)) in enumerate(zip(mats, outs)):
        assert np.isfinite(Q).all() and np.isfinite(R).all() and np.array_equal(R, np.triu(R)), (i, A.shape)
        assert oracle.backward(A, Q, R) < 1e-6, (i, A.shape, oracle.backward(A, Q, R))
        if i < len(mats) - 1:
            _, R64 = oracle.lapack_qr64(A)
            assert oracle.rel_err(R, R64) < 1e-6 * np.linalg.cond(R64) + 1e-6, (i, A.shape)
    assert np.all(outs[-1][0][:, 90] == 0)


# One projection out of 64-column blocks one after another, as on the narrow
# kernel: the loss of orthogonality grows with kappa, not its square, so it is
# no worse than twice the narrow kernel's on the same input (other roundings),
# with the 3e-5 of two projections as the floor.
@pytest.mark.parametrize("pad", [0, 1])
def test_one_projection_orthogonality(later, oracle, pad):
    mats = [oracle.gen_uniform(m, n, 21, i) for i, (m, n) in enumerate([(130, 129), (200, 200), (256, 256), (700, 193)])]
    mats += [oracle.gen_uniform(m, n, 22, n) + np.float32(3) for m, n in [(300, 256), (400, 200), (1000, 129)]]
    mats += [_kappa(m, n, d, n + int(d)) for m, n in [(200, 200), (515, 256), (400, 150)] for d in (2, 4, 6)]
    outs, status = _run(later, mats, WIDE, pad=pad)
    ref, _ = _run(later, mats, NARROW, pad=pad)
    assert not status.any()
    for i, (A, (Q, _), (Qn, _)) in enumerate(zip(mats, outs, ref)):
        assert oracle.orth(Q) < 2.0 * oracle.orth(Qn) + 3e-5, (i, A.shape, oracle.orth(Q), oracle.orth(Qn))


# Columns that share a direction (a common mean): the first columns of Q carry
# the large terms of an update, and the others' are added before them, so their
# roundings stay at their own magnitude.  The backward error is within twice the
# narrow kernel's, which starts each sum from the panel's own entry.
@pytest.mark.parametrize("reorth", [0, 2])
def test_correlated_columns_backward(later, oracle, reorth):
    mats = [oracle.gen_uniform(m, n, 23, n) + np.float32(3) for m, n in [(96, 96), (300, 256), (400, 200), (1000, 129)]]
    mats += [_kappa(m, n, 6, n) for m, n in [(200, 200), (515, 256)]]
    outs, status = _run(later, mats, WIDE, reorth=reorth)
    ref, _ = _run(later, mats, NARROW, reorth=reorth)
    assert not status.any()
    for i, (A, (Q, R), (Qn, Rn)) in enumerate(zip(mats, outs, ref)):
        assert oracle.backward(A, Q, R) < 2.0 * oracle.backward(A, Qn, Rn), (i, A.shape, oracle.backward(A, Q, R))


# Columns scaled by powers of two scale every sum and product exactly, so Q keeps
# its bits and R's columns scale exactly, as long as no decision depends on the
# columns' norms.
@pytest.mark.parametrize("reorth", [0, 2])
def test_column_scaling_is_exact(later, oracle, reorth):
    mats = [oracle.gen_uniform(m, n, 24, i) for i, (m, n) in enumerate([(500, 96), (64, 64), (130, 129), (1000, 256)])]
    by = [np.where(np.arange(A.shape[1]) % 2, 1024.0, 0.125).astype(np.float32) for A in mats]
    outs, _ = _run(later, mats, WIDE, reorth=reorth)
    scaled, status = _run(later, [A * d for A, d in zip(mats, by)], WIDE, reorth=reorth)
    assert not status.any()
    for (Q, R), (Qs, Rs), d in zip(outs, scaled, by):
        assert np.array_equal(Q, Qs) and np.array_equal(R * d, Rs)
        assert oracle.orth(Qs) < 1e-3


# With two projections what is left of Q in a panel may grow by the panel's
# condition: panels just under the limit of a second factorisation (singular
# values of the whole matrix over two and three decades).  Orthogonality within
# 1.3 times the narrow kernel's, whose panels are half as wide.
@pytest.mark.parametrize("m,n,decades", [(1000, 128, 2), (515, 256, 3), (4000, 256, 3)])
def test_two_projections_orthogonality(later, oracle, m, n, decades):
    mats = [_kappa(m, n, decades, s) for s in (1, 2)]
    outs, status = _run(later, mats, WIDE, reorth=2)
    ref, _ = _run(later, mats, NARROW, reorth=2)
    assert not status.any()
    for (Q, _), (Qn, _) in zip(outs, ref):
        assert oracle.orth(Q) < 1.3 * oracle.orth(Qn), (oracle.orth(Q), oracle.orth(Qn))

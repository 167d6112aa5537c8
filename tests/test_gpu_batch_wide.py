"""The batched QR's wide kernel (variant 4: 64-column panels against all
earlier columns) at the edges of its chunks, panels and column slots (GPU)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

WIDE = 4


def _run(later, mats, form="mixed", pad=0, variant=WIDE):
    As, Rs = [], []
    for A in mats:
        X = later.colmajor(A.shape[0], A.shape[1], ld=A.shape[0] + pad)
        X.copy_(torch.from_numpy(np.ascontiguousarray(A)))
        As.append(X)
        Rs.append(later.colmajor(A.shape[1], A.shape[1], ld=A.shape[1] + pad))
    plan = later.BatchWg(As, Rs, later.opts(form, reorth=later.REORTH_PASS), tuning=[variant] * later.BATCH_BUCKETS)
    outs = []
    for _ in range(2):
        for X, A in zip(As, mats):
            X.copy_(torch.from_numpy(np.ascontiguousarray(A)))
        plan.execute()
        torch.cuda.synchronize()
        outs.append([(q.cpu().numpy().copy(order="F"), r.cpu().numpy().copy(order="F")) for q, r in zip(As, Rs)])
    status = plan.status.cpu().numpy()
    plan.close()
    for (q0, r0), (q1, r1) in zip(*outs):
        assert np.array_equal(q0, q1) and np.array_equal(r0, r1)
    return outs[0], status


# The gates of the narrow kernel's test: orthogonality 3e-5, backward error
# 1e-6, R within kappa 1e-6 of FP64 LAPACK.
@pytest.mark.parametrize("pad", [0, 1, 4])
def test_wide_edges(later, oracle, pad):
    shapes = [(4, 1), (5, 4), (31, 16), (32, 32), (33, 20), (63, 63), (64, 64), (65, 64), (65, 65), (127, 100),
              (128, 128), (130, 129), (160, 127), (200, 192), (257, 193), (300, 255), (256, 256), (515, 256), (3, 2),
              (1, 1), (700, 300)]
    mats = [oracle.gen_uniform(m, n, 11, i) for i, (m, n) in enumerate(shapes)]
    outs, status = _run(later, mats, pad=pad)
    assert not status.any()
    for A, (Q, R), s in zip(mats, outs, shapes):
        Q64, R64 = oracle.lapack_qr64(A)
        assert np.array_equal(R, np.triu(R)), s
        assert oracle.orth(Q) < 3e-5 and oracle.backward(A, Q, R) < 1e-6, (s, oracle.orth(Q), oracle.backward(A, Q, R))
        assert oracle.rel_err(R, R64) < 1e-6 * np.linalg.cond(R64) + 1e-6, s


# Graded columns (kappa 1e6, in the panels and across them): the normalised
# panel is projected and factored again, so orthogonality does not follow
# kappa.  A dependent column gives a zero column and the status bit.
def test_wide_ill_conditioned_and_dependent(later, oracle):
    rng = np.random.default_rng(5)
    mats = []
    for m, n in [(500, 100), (1000, 200), (300, 64), (400, 256)]:
        U, _ = np.linalg.qr(rng.standard_normal((m, n)))
        V, _ = np.linalg.qr(rng.standard_normal((n, n)))
        mats.append((U * np.logspace(0, -6, n) @ V.T).astype(np.float32))
    dep = oracle.gen_uniform(600, 150, 3, 3)
    dep[:, 90] = 0.0
    mats.append(dep)
    outs, status = _run(later, mats)
    assert list(status) == [0, 0, 0, 0, 1]
    for A, (Q, R) in zip(mats[:4], outs):
        assert oracle.orth(Q) < 3e-5 and oracle.backward(A, Q, R) < 1e-6, (A.shape, oracle.orth(Q))
    Q, R = outs[4]
    keep = [j for j in range(150) if j != 90]
    assert np.all(Q[:, 90] == 0) and np.isfinite(Q).all() and np.isfinite(R).all()
    assert oracle.orth(Q[:, keep]) < 3e-5 and oracle.backward(dep, Q, R) < 1e-6


# Tasks of both kernels in one plan (two launches, a queue each).
def test_wide_and_narrow_in_one_plan(later, oracle):
    shapes = [(600, 20)] * 40 + [(300, 100)] * 3 + [(500, 300)] * 2
    mats = [oracle.gen_uniform(m, n, 2, i) for i, (m, n) in enumerate(shapes)]
    outs, status = _run(later, mats, form="fp32", variant=-1)
    assert not status.any()
    for A, (Q, R) in zip(mats, outs):
        assert oracle.orth(Q) < 3e-5 and oracle.backward(A, Q, R) < 1e-6

"""A batch whose tasks take both kernels of the one-launch batched QR (GPU)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# (m, n): up to 32 columns, 33 to 256, more; a small share of narrow ones.
SHAPES = [(600, 20), (64, 16), (1000, 32), (90, 5), (3, 2)] + [(700 + 9 * i, 100 + 7 * i) for i in range(20)] + [(500, 300)]


def _inputs(later, shapes=SHAPES):
    src = [later.generate_uniform(m, n, seed=5, mat=i) for i, (m, n) in enumerate(shapes)]
    return src, [later.colmajor(m, n) for m, n in shapes], [later.colmajor(n, n) for _, n in shapes]


def _run(plan, src, As, Rs):
    for a, s in zip(As, src):
        a.copy_(s)
    plan.execute()
    torch.cuda.synchronize()
    return [(a.cpu().numpy().copy(), r.cpu().numpy().copy()) for a, r in zip(As, Rs)]


def _equal(x, y):
    return all(np.array_equal(a, c) and np.array_equal(b, d) for (a, b), (c, d) in zip(x, y))


# A matrix gets the same bits alone, in a batch and in another order, and the
# same with no table as with one of -1.
@pytest.mark.parametrize("form", ["mixed", "fp32"])
def test_same_bits_alone_and_in_a_batch(later, form):
    o = later.opts(form)
    src, As, Rs = _inputs(later)
    plan = later.BatchWg(As, Rs, o)
    mix = _run(plan, src, As, Rs)
    assert not plan.status.any()
    plan.close()
    plan = later.BatchWg(As, Rs, o, tuning=[-1] * later.BATCH_BUCKETS)
    assert _equal(mix, _run(plan, src, As, Rs))
    plan.close()
    plan = later.BatchWg(As[::-1], Rs[::-1], o)
    assert _equal(mix[::-1], _run(plan, src[::-1], As[::-1], Rs[::-1]))
    plan.close()
    for i in range(len(SHAPES)):
        plan = later.BatchWg(As[i:i + 1], Rs[i:i + 1], o)
        assert _equal(mix[i:i + 1], _run(plan, src[i:i + 1], As[i:i + 1], Rs[i:i + 1])), SHAPES[i]
        plan.close()


# Both kernels follow what was enqueued before on the caller's stream and come
# before what is enqueued after, eagerly and in a captured graph, replayed with
# other work between the replays.
def test_stream_order_and_capture(later):
    src, As, Rs = _inputs(later)
    plan = later.BatchWg(As, Rs, later.opts("mixed"))
    want = _run(plan, src, As, Rs)
    got = [(torch.empty_like(a), torch.empty_like(r)) for a, r in zip(As, Rs)]

    def step():
        torch._foreach_copy_(As, src)
        plan.execute()
        torch._foreach_copy_([x for g in got for x in g], [x for p in zip(As, Rs) for x in p])

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        step()
    s.synchronize()
    assert _equal(want, [(a.cpu().numpy(), r.cpu().numpy()) for a, r in got])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    for rep in range(4):
        for a, r in got:
            a.zero_(), r.zero_()
        if rep % 2:
            _run(plan, src, As, Rs)
        graph.replay()
        torch.cuda.synchronize()
        assert _equal(want, [(a.cpu().numpy(), r.cpu().numpy()) for a, r in got]), rep
    plan.close()


# A plan may be closed behind its last launch: what was enqueued still runs, and
# later work on the stream follows it.
def test_close_behind_a_launch(later):
    src, As, Rs = _inputs(later)
    plan = later.BatchWg(As, Rs, later.opts("mixed"))
    want = _run(plan, src, As, Rs)
    for a, s in zip(As, src):
        a.copy_(s)
    plan.execute()
    plan.close()
    got = [(a.clone(), r.clone()) for a, r in zip(As, Rs)]
    torch.cuda.synchronize()
    assert _equal(want, [(a.cpu().numpy(), r.cpu().numpy()) for a, r in got])

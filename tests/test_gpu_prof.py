"""Kernel-class timing: every product of the recursion is in its class (GPU)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _nodes(n, leaf):
    """(n1, n2) of every node above the leaves, split at 32 ceil(n / 64)."""
    if n <= leaf:
        return []
    n1 = 32 * -(-n // 64)
    return [(n1, n - n1)] + _nodes(n1, leaf) + _nodes(n - n1, leaf)


# One update and one projection a node, 2 m n1 n2 operations each, whether the
# update is a launch of its own or also forms the next leaf's Gram.
@pytest.mark.parametrize("form,leaf", [("mixed", 64), ("fp32", 32), ("reference", 32)])
@pytest.mark.parametrize("m,n", [(2000, 65), (2000, 96), (2000, 128), (1500, 333), (20000, 128)])
def test_products_are_all_in_their_class(later, form, leaf, m, n):
    A = later.generate_uniform(m, n, seed=1, mat=0)
    o = later.opts(form, reorth=0)
    work = later.workspace(m, n, o)
    torch.cuda.synchronize()
    later.prof_begin()
    later.rgsqrf(A, o=o, work=work, hwork=None)
    prof = later.prof_end()
    nodes = _nodes(n, leaf)
    want = sum(2.0 * m * n1 * n2 for n1, n2 in nodes)
    update = [prof["gemm_update"], prof["gemm_update_x3"]]
    assert prof["gemm_proj"]["launches"] == len(nodes) and prof["gemm_proj"]["flops"] == want
    assert sum(u["launches"] for u in update) == len(nodes) and sum(u["flops"] for u in update) == want
    assert all(p["ms"] > 0.0 for p in prof.values() if p["launches"])

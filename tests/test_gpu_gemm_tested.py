"""Projections of operands several times the cache, on tested loads (GPU)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# Aligned operands past the size rule take the tested loads, the same values at an
# odd leading dimension the ring; the split plan and the order of the products are
# the same, so are the bits.
@pytest.mark.parametrize("prec,m,n1,n2", [("GEMM_F16", 300003, 512, 400), ("GEMM_BF16", 131072, 1024, 1000),
                                          ("GEMM_F16X3", 262143, 1024, 900)])
def test_tested_loads_keep_bits(later, prec, m, n1, n2):
    out = []
    for ld in ((m + 3) // 4 * 4, (m + 3) // 4 * 4 + 1):
        Q = later.generate_uniform(m, n1, seed=1, mat=1, out=later.colmajor(m, n1, ld=ld))
        B = later.generate_uniform(m, n2, seed=1, mat=2, out=later.colmajor(m, n2, ld=ld))
        out.append(later.gemm_proj(Q, B, later.colmajor(n1, n2), getattr(later, prec)))
    assert torch.equal(out[0], out[1])
    want = Q[:, :8].double().t().contiguous() @ B[:, :8].double().contiguous()
    scale = Q[:, :8].abs().double().t().contiguous() @ B[:, :8].abs().double().contiguous()
    bits = 2.0 ** -10 if prec == "GEMM_F16" else 2.0 ** -7 if prec == "GEMM_BF16" else 2.0 ** -18
    assert bool(((out[0][:8, :8].double() - want).abs() <= bits * scale).all())

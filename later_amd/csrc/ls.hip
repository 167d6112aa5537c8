// Least-squares solve on top of the QR: X = R^{-1} Q^T B.
//
// Q^T B is the node projection GEMM (gemm.hip).  The triangular solve is a
// blocked back substitution standing in for the reference's recursive TRSM
// (BLAS/later_rtrsm.cu:75-187): one workgroup per right-hand side keeps the
// column in LDS in FP64 and works up R in 64-row blocks.
#include <type_traits>

#include "common.h"
#include "gemm.h"

namespace {

constexpr int TB = 64;          // diagonal block
constexpr int kWaves = 8;
constexpr int NT = 64 * kWaves;
constexpr int kMaxN = 8192;     // FP64 column in LDS: 64 KiB

// Block b's rows need the products with every later block's x.  While wave 0
// solves block b (lane i owns row i of the diagonal block in registers, x_r is
// read from lane r after one multiplication by the reciprocal of its
// diagonal), the other waves sum block b - 1's products with the blocks after
// b, and every wave's share of block b's own columns is already in flight; one
// barrier after x_b is known those are added, and wave 0 goes on.
// Bound: wave 0's chain, 64 x (multiply, broadcast, multiply-add) a block: 512
// unknowns 49 us, where loads and a division on the chain took 398.
template <int NMAX>
__global__ __launch_bounds__(NT) void trsm_upper_kernel(int n, const float *R, int64_t ldr, float *B, int64_t ldb,
                                                        int *status)
{
    __shared__ double x[NMAX], part[kWaves][TB];
    float *b = B + (int64_t)blockIdx.x * ldb;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int nblk = (n + TB - 1) / TB;
    // Wave 0: row `lane` of the diagonal block (its part right of the
    // diagonal) and the diagonal entry.
    float dn[TB], diag_n = 1.0f;
    auto load_diag = [&](int j0) {
        const int row = min(j0 + lane, n - 1);
#pragma unroll
        for (int r = 0; r < TB; ++r) dn[r] = R[row + (int64_t)min(j0 + r, n - 1) * ldr];
        diag_n = R[row + (int64_t)row * ldr];
    };
    if (wave == 0) load_diag((nblk - 1) * TB);
    for (int i = threadIdx.x; i < n; i += NT) x[i] = (double)b[i];
    part[wave][lane] = 0.0;
    __syncthreads();
    constexpr int kShare = TB / kWaves;
    for (int blk = nblk - 1; blk >= 0; --blk) {
        const int j0 = blk * TB, jn = min(TB, n - j0);
        const int up = j0 - TB + lane;  // this lane's row of the block above
        float f[kShare];
        double acc = 0.0;
        if (blk > 0) {
#pragma unroll
            for (int q = 0; q < kShare; ++q) {
                const int c = kShare * wave + q;
                const float v = R[up + (int64_t)(j0 + min(c, jn - 1)) * ldr];
                f[q] = c < jn ? v : 0.0f;
            }
        }
        if (wave == 0) {
            float d[TB];
#pragma unroll
            for (int r = 0; r < TB; ++r) d[r] = lane < r ? dn[r] : 0.0f;
            const float diag = diag_n;
            if (blk > 0) load_diag(j0 - TB);
            double xi = lane < jn ? x[j0 + lane] : 0.0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) xi -= part[w][lane];
            // A zero on the diagonal: its unknown is 0, whatever the right-hand
            // side holds (a product with 0 would keep its sign, or be NaN).
            const bool zero = !(diag != 0.0f) && lane < jn;
            if (zero && status) atomicOr(status, 2);
            const double inv = zero ? 0.0 : 1.0 / (double)diag;
            double res = 0.0;
            auto solve = [&](auto zeros) {
#pragma unroll
                for (int r = TB - 1; r >= 0; --r) {
                    if (r < jn) {
                        double t = xi * inv;
                        if constexpr (decltype(zeros)::value) t = zero ? 0.0 : t;
                        const double xr = readlane_d(t, r);
                        res = lane == r ? xr : res;
                        xi = fma(-(double)d[r], xr, xi);
                    }
                }
            };
            if (__builtin_amdgcn_ballot_w64(zero) == 0) solve(std::false_type());
            else solve(std::true_type());
            if (lane < jn) x[j0 + lane] = res;
        } else if (blk > 0) {
            constexpr int kU = 8;
            for (int c0 = j0 + jn + wave - 1; c0 < n; c0 += kU * (kWaves - 1)) {
                float v[kU];
#pragma unroll
                for (int u = 0; u < kU; ++u) v[u] = R[up + (int64_t)min(c0 + u * (kWaves - 1), n - 1) * ldr];
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    const int c = c0 + u * (kWaves - 1);
                    if (c < n) acc = fma((double)v[u], x[c], acc);
                }
            }
        }
        __syncthreads();
        if (blk > 0) {
#pragma unroll
            for (int q = 0; q < kShare; ++q)
                if (kShare * wave + q < jn) acc = fma((double)f[q], x[j0 + kShare * wave + q], acc);
            part[wave][lane] = acc;
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < n; i += NT) b[i] = (float)x[i];
}

} // namespace

int trsm_upper(hipStream_t s, int n, int k, const float *R, int64_t ldr, float *B, int64_t ldb, int *status)
{
    if (n < 1 || k < 1 || n > kMaxN) return LATER_ERR_SHAPE;
    // The smaller column array leaves room for several workgroups a CU (servers
    // solve on several streams at once).
    if (n <= 1024)
        hipLaunchKernelGGL(trsm_upper_kernel<1024>, dim3(k), dim3(NT), 0, s, n, R, ldr, B, ldb, status);
    else
        hipLaunchKernelGGL(trsm_upper_kernel<kMaxN>, dim3(k), dim3(NT), 0, s, n, R, ldr, B, ldb, status);
    HIP_OK(hipGetLastError());
    return LATER_OK;
}

LATER_API int later_trsm_upper(laterCtxt ctxt, int n, int k, const float *R, int ldr, float *B, int ldb)
{
    if (n < 1 || k < 1 || ldr < n || ldb < n || !R || !B) return LATER_ERR_SHAPE;
    if (n > kMaxN) return LATER_ERR_SHAPE;
    return trsm_upper(ctx_stream(ctxt), n, k, R, ldr, B, ldb, nullptr);
}

LATER_API int later_ls_workspace(int m, int n, int k, const later_opts *opts, int64_t *lwork)
{
    int64_t lw = 0, lh = 0;
    int rc = later_rgsqrf_workspace(m, n, opts, &lw, &lh);
    if (rc) return rc;
    // later_gels reuses `work` after the QR: the status header (64 floats),
    // the exponents of B's columns, then the split-K partials of Q^T B.
    const int64_t proj = 64 + ((int64_t)k + 63) / 64 * 64 + gemm_proj_work_floats(m, n, k, 256);
    if (lwork) *lwork = (lw > proj ? lw : proj);
    return LATER_OK;
}

// Solves min ||A X - B||: A (m x n) <- Q, R (n x n) <- R, X (n x k) <- solution.
// B is read only.  Q^T B uses FP16 hi/lo products with FP64-folded chunks.
LATER_API int later_gels(laterCtxt ctxt, int m, int n, int k, float *A, int lda, float *R, int ldr, const float *B,
                         int ldb, float *X, int ldx, float *work, int64_t lwork, const later_opts *opts,
                         later_info *info)
{
    if (m < 1 || n < 1 || k < 1 || m < n || lda < m || ldr < n || ldb < m || ldx < n || !A || !R || !B || !X)
        return LATER_ERR_SHAPE;
    if (n > kMaxN) return LATER_ERR_SHAPE;
    int64_t need = 0;
    int rc = later_ls_workspace(m, n, k, opts, &need);
    if (rc) return rc;
    if (!work || lwork < need) return LATER_ERR_WORKSPACE;
    rc = later_rgsqrf_ex(ctxt, m, n, A, lda, R, ldr, work, lwork, nullptr, 0, opts, info);
    if (rc) return rc;
    hipStream_t s = ctx_stream(ctxt);
    // X = Q^T B (FP16 hi/lo split products, column scaling of B, FP64 chunks).
    int *bexp = (int *)work + 64;
    rc = gemm_colexp(s, m, k, B, ldb, bexp, nullptr);
    if (rc) return rc;
    const int64_t off = 64 + ((int64_t)k + 63) / 64 * 64;
    rc = gemm_proj(s, GEMM_F16X3, m, n, k, A, lda, B, ldb, X, ldx, 256, bexp, 14, work + off, lwork - off, nullptr);
    if (rc) return rc;
    return trsm_upper(s, n, k, R, ldr, X, ldx, (int *)work);
}

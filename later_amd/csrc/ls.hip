// Least-squares solve on top of the QR: X = R^{-1} Q^T B.
//
// Q^T B is the node projection GEMM (gemm.hip).  The triangular solve is a
// blocked back substitution standing in for the reference's recursive TRSM
// (BLAS/later_rtrsm.cu:75-187): one workgroup per right-hand side, or one wave
// for several, keeps the columns in LDS in FP64 and works up R in 64-row blocks.
#include <type_traits>

#include "common.h"
#include "gemm.h"

namespace {

constexpr int TB = 64;          // diagonal block
constexpr int kWaves = 8;
constexpr int NT = 64 * kWaves;
constexpr int kMaxN = 8192;     // FP64 column in LDS: 64 KiB

// One wave's solve of N right-hand sides with a diagonal block: lane i holds row
// i (d: its entries right of the diagonal, zeros elsewhere), inv its diagonal's
// reciprocal and xi its right-hand sides; x_r is read from lane r.
template <int N, int T>
__device__ __forceinline__ void solve_block(int jn, const float (&d)[T], double inv, bool zero, double (&xi)[N],
                                            double (&res)[N])
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int c = 0; c < N; ++c) res[c] = 0.0;
    auto solve = [&](auto zeros) {
#pragma unroll
        for (int r = T - 1; r >= 0; --r) {
            if (r < jn) {
#pragma unroll
                for (int c = 0; c < N; ++c) {
                    double t = xi[c] * inv;
                    if constexpr (decltype(zeros)::value) t = zero ? 0.0 : t;
                    const double xr = readlane_d(t, r);
                    res[c] = lane == r ? xr : res[c];
                    xi[c] = fma(-(double)d[r], xr, xi[c]);
                }
            }
        }
    };
    if (__builtin_amdgcn_ballot_w64(zero) == 0) solve(std::false_type());
    else solve(std::true_type());
}

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
            double xs[1] = {xi}, res[1];
            solve_block(jn, d, inv, zero, xs, res);
            if (lane < jn) x[j0 + lane] = res[0];
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

// The same for many right-hand sides: one wave takes N of them and does what
// the workgroup above does, its waves' sums each in the same order, so that x
// has the same bits.  Where the CUs are full of right-hand sides the waves that
// follow a solver only take registers from other solvers (n = 64, 8192 of them:
// 187 us on the kernel above, 17.5 here).  T: rows of a diagonal block, 16 for
// systems that one such block holds.
template <int N, int T>
__global__ __launch_bounds__(64) void trsm_upper_many_kernel(int n, int k, const float *R, int64_t ldr, float *B,
                                                             int64_t ldb, int *status)
{
    extern __shared__ __attribute__((aligned(16))) double xs[];  // x of column c at N c .. N c + N - 1
    constexpr int kStep = kWaves - 1, kShare = T / kWaves, kU = 4;
    const int lane = threadIdx.x, k0 = N * blockIdx.x;
    const int nblk = (n + T - 1) / T;
    for (int i = lane; i < n; i += 64)
#pragma unroll
        for (int c = 0; c < N; ++c) xs[N * i + c] = (double)B[(int64_t)min(k0 + c, k - 1) * ldb + i];
    __syncthreads();
    double acc[kWaves][N];
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
#pragma unroll
        for (int c = 0; c < N; ++c) acc[w][c] = 0.0;
    for (int blk = nblk - 1; blk >= 0; --blk) {
        const int j0 = blk * T, jn = min(T, n - j0);
        const int row = min(j0 + lane, n - 1), up = j0 - T + lane;
        float d[T];
#pragma unroll
        for (int r = 0; r < T; ++r) d[r] = R[row + (int64_t)min(j0 + r, n - 1) * ldr];
        const float diag = R[row + (int64_t)row * ldr];
        double xi[N], res[N];
#pragma unroll
        for (int c = 0; c < N; ++c) {
            xi[c] = lane < jn ? xs[N * row + c] : 0.0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) xi[c] -= acc[w][c];
        }
#pragma unroll
        for (int r = 0; r < T; ++r) d[r] = lane < r ? d[r] : 0.0f;
        const bool zero = !(diag != 0.0f) && lane < jn;
        if (zero && status) atomicOr(status, 2);
        solve_block(jn, d, zero ? 0.0 : 1.0 / (double)diag, zero, xi, res);
        if (lane < jn)
#pragma unroll
            for (int c = 0; c < N; ++c) xs[N * row + c] = res[c];
        __syncthreads();
        if (blk == 0) break;
        float f[T];
#pragma unroll
        for (int r = 0; r < T; ++r) f[r] = R[up + (int64_t)(j0 + min(r, jn - 1)) * ldr];
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
#pragma unroll
            for (int c = 0; c < N; ++c) acc[w][c] = 0.0;
        for (int c0 = j0 + jn; c0 < n; c0 += kU * kStep) {
            float v[kU * kStep];
#pragma unroll
            for (int u = 0; u < kU * kStep; ++u) v[u] = R[up + (int64_t)min(c0 + u, n - 1) * ldr];
#pragma unroll
            for (int u = 0; u < kU * kStep; ++u)
                if (c0 + u < n)
#pragma unroll
                    for (int c = 0; c < N; ++c)
                        acc[1 + u % kStep][c] = fma((double)v[u], xs[N * (c0 + u) + c], acc[1 + u % kStep][c]);
        }
#pragma unroll
        for (int r = 0; r < T; ++r)
            if (r < jn)
#pragma unroll
                for (int c = 0; c < N; ++c)
                    acc[r / kShare][c] = fma((double)f[r], xs[N * (j0 + r) + c], acc[r / kShare][c]);
    }
    for (int i = lane; i < n; i += 64)
#pragma unroll
        for (int c = 0; c < N; ++c)
            if (k0 + c < k) B[(int64_t)(k0 + c) * ldb + i] = (float)xs[N * i + c];
}

} // namespace

int trsm_upper(hipStream_t s, int n, int k, const float *R, int64_t ldr, float *B, int64_t ldb, int *status)
{
    if (n < 1 || k < 1 || n > kMaxN) return LATER_ERR_SHAPE;
    // Up to 16 unknowns a block of 16 rows holds them all: a fixed cost of 2.6 us
    // where blocks of 64 rows have 5.7 (8 unknowns, 1 right-hand side; 1000 of them
    // 3.6 and 6.6, 20000 7.7 and 19).
    //
    // A workgroup a right-hand side while the CUs hold them in a few rounds (one
    // workgroup a CU: its registers), then one wave for two of them, which takes
    // 1 to 5 times as long and goes round after 4096 (us, 256 / 512 / 1024 / 2048 right-hand
    // sides: n = 64 8.8 / 13.9 / 25 / 48 and 9.2 / 9.3 / 9.5 / 9.1; n = 256 22 / 42 / 80 /
    // 157 and 48 / 50 / 50 / 52; n = 1024 120 / 229 / 457 / 909 and 557 / 559 / 555 / 561), or for
    // four (16384: n = 64 34 and 30, n = 512 596 and 459, n = 1024 2691 and 2919).  Above
    // 3072 unknowns the columns' LDS leaves too few waves (n = 4096, 1280: 10.6
    // and 17.2 ms).
    const int rounds = (k + 255) / 256;
    const bool many = n <= 3072 && rounds > (n < 576 ? 1 + n / 192 : 4);
    if (n <= 16 && k <= 4096)
        hipLaunchKernelGGL((trsm_upper_many_kernel<1, 16>), dim3(k), dim3(64), n * sizeof(double), s, n, k, R, ldr, B, ldb,
                           status);
    else if (n <= 16)
        hipLaunchKernelGGL((trsm_upper_many_kernel<4, 16>), dim3((k + 3) / 4), dim3(64), 4 * n * sizeof(double), s, n, k, R,
                           ldr, B, ldb, status);
    else if (many && k > 4096 && n <= 512)
        hipLaunchKernelGGL((trsm_upper_many_kernel<4, TB>), dim3((k + 3) / 4), dim3(64), 4 * n * sizeof(double), s, n, k, R, ldr,
                           B, ldb, status);
    else if (many)
        hipLaunchKernelGGL((trsm_upper_many_kernel<2, TB>), dim3((k + 1) / 2), dim3(64), 2 * n * sizeof(double), s, n, k, R, ldr,
                           B, ldb, status);
    // The smaller column array leaves LDS to other streams' kernels (servers
    // solve on several at once).
    else if (n <= 1024)
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

// FP32 products of the narrow nodes: projections C = Q^T B and updates
// B -= Q C whose result or depth is at most 128 columns wide.
//
// At these widths a node is a chain of short launches, so what counts is the
// time from launch to last store, not the rate: every operand of a tile is
// requested before the first wait, the tiles are small enough that a node of
// a few thousand rows covers the chip, and each wave runs one or two 16 x 16
// tiles (v_mfma_f32_16x16x4f32, 32 cycles a step against 64 of the 32 x 32
// form) from LDS without a barrier per slab.  Both MFMA shapes add their
// products to the accumulator one k after another with one rounding each, so
// an element's value does not depend on the tile shape: the results are the
// bits of the general kernel (gemm.hip), with its split plan and partials.
#include "common.h"
#include "gemm.h"

namespace {

constexpr int kThreads = 256;
constexpr int kKB = 128;         // rows of K per LDS block of the projection
constexpr int kLdP = kKB + 4;    // its column stride (floats)

// 16-byte vector of floats with only the alignment of a float (the target
// allows dword-aligned multi-dword global accesses), for any lda.
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

// A column-major operand block in LDS, column c at c * ld: its k values in
// chunks of four, chunk 4 t + g holding k = 16 t + g, + 4, + 8, + 12 (the four
// values lane group g of a 16x16x4 MFMA takes in steps 4 t .. 4 t + 3, so one
// 16-byte read serves four steps), stored at chunk 4 t + (g ^ (t / 4 % 4)): both
// the writes (16 lanes: 16 consecutive t of one column) and the reads (16
// lanes: 16 columns) then cover all banks once.
__device__ __forceinline__ int chunk_of(int t, int g) { return 4 * (4 * t + (g ^ ((t >> 2) & 3))); }

// k = k0 + 16 t .. + 15 of column `col` (rows kmax and beyond: zeros).
struct Run16 {
    floatx4u v[4];
    __device__ __forceinline__ void load(const float *P, int64_t ld, int col, int k0, int kmax)
    {
        const float *p = P + (int64_t)col * ld + k0;
        if (k0 + 16 <= kmax) {
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = *(const floatx4u *)(p + 4 * u);
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[u][e] = k0 + 4 * u + e < kmax ? p[4 * u + e] : 0.0f;
        }
    }
    __device__ __forceinline__ void store(float *column, int t) const
    {
#pragma unroll
        for (int g = 0; g < 4; ++g) *(floatx4 *)(column + chunk_of(t, g)) = floatx4{v[0][g], v[1][g], v[2][g], v[3][g]};
    }
};

// Split-K projection, one 32 x 32 tile of C and one split per workgroup: each
// wave one 16 x 16 tile over the split's whole depth.  256 rows of both
// operands are requested at once and pass through LDS in two halves (34 KB:
// four workgroups a CU).  blockIdx.x is the split, so that the tiles of one
// split (which read the same rows) land on one XCD when the number of splits
// is a multiple of 8.
__global__ __launch_bounds__(kThreads, 4) void proj_narrow_kernel(int M, int N, int K, int kper, const float *Q,
                                                                  int64_t ldq, const float *B, int64_t ldb, float *C,
                                                                  int64_t ldc, float *partial)
{
    __shared__ __attribute__((aligned(16))) float lds[64 * kLdP];  // 32 columns of Q, 32 of B
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int ti = (M + 31) / 32, i0 = 32 * ((int)blockIdx.y % ti), j0 = 32 * ((int)blockIdx.y / ti);
    const int kbeg = blockIdx.x * kper, kend = min(K, kbeg + kper);
    Run16 r[4];
    auto load = [&](int k0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = (t >> 4) + 16 * u, k = k0 + 16 * (t & 15);
            if (u < 2) r[u].load(Q, ldq, min(i0 + c, M - 1), min(k, kend), kend);
            else r[u].load(B, ldb, min(j0 + c - 32, N - 1), min(k, kend), kend);
        }
    };
    load(kbeg);
    floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    const int li = lane & 15, g = lane >> 4, wi = 16 * (wv >> 1), wj = 16 * (wv & 1);
    const float *qc = lds + (wi + li) * kLdP, *bc = lds + (32 + wj + li) * kLdP;
    for (int k0 = kbeg; k0 < kend; k0 += 2 * kKB) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const int kh = k0 + half * kKB;
            if (kh >= kend) break;
            if (kh > kbeg) __syncthreads();  // the previous rows have been read
            if (((t & 15) >> 3) == half) {
#pragma unroll
                for (int u = 0; u < 4; ++u) r[u].store(lds + ((t >> 4) + 16 * u) * kLdP, t & 7);
            }
            __syncthreads();
            if (half == 1 && k0 + 2 * kKB < kend) load(k0 + 2 * kKB);
            const int nt = min(kKB, kend - kh + 15) / 16;
            floatx4 a = *(const floatx4 *)(bc + chunk_of(0, g)), b = *(const floatx4 *)(qc + chunk_of(0, g));
            for (int s = 0; s < nt; ++s) {
                const int sn = min(s + 1, kKB / 16 - 1);
                const floatx4 an = *(const floatx4 *)(bc + chunk_of(sn, g)),
                              bn = *(const floatx4 *)(qc + chunk_of(sn, g));
#pragma unroll
                for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b[u], acc, 0, 0, 0);
                a = an;
                b = bn;
            }
        }
    }
    // Lane l, entry r: row l % 16, column 4 (l / 16) + r of the wave's tile.
    const int row = i0 + wi + li;
    if (row < M) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int col = j0 + wj + 4 * g + e;
            if (col < N) {
                if (partial) partial[((int64_t)blockIdx.x * N + col) * M + row] = acc[e];
                else C[(int64_t)col * ldc + row] = acc[e];
            }
        }
    }
}

// B (M x N) += alpha Q C for a depth K of at most KM (a multiple of 16): a
// workgroup takes 32 rows x 64 columns at a time (each wave 16 x 32), with C
// staged in LDS once and Q's rows read straight into the MFMA operand (lane l
// of step s: row l % 16, k = 4 s + l / 16).  The next rows' Q and B are
// requested before the current product.
template <int KM>
__global__ __launch_bounds__(kThreads, 2) void update_narrow_kernel(int M, int N, int K, const float *Q, int64_t ldq,
                                                                 const float *C, int64_t ldc, float *B, int64_t ldb,
                                                                 float alpha, int f64)
{
    constexpr int LD = KM + 4, S = KM / 4;
    __shared__ __attribute__((aligned(16))) float lds[64 * LD];
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int li = lane & 15, g = lane >> 4, wi = 16 * (wv >> 1), wj = 32 * (wv & 1);
    const int j0 = 64 * blockIdx.y;
    const int nblk = (M + 31) / 32;
    float q[S], c[2][4];
    auto load = [&](int blk) {
        const int row = min(32 * blk + wi + li, M - 1);
#pragma unroll
        for (int s = 0; s < S; ++s) q[s] = Q[row + (int64_t)min(4 * s + g, K - 1) * ldq];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e) c[x][e] = B[row + (int64_t)min(j0 + wj + 16 * x + 4 * g + e, N - 1) * ldb];
    };
    load(blockIdx.x);
    constexpr int RPC = KM / 16;                                     // runs of 16 k per column
    constexpr int NR = (64 * RPC + kThreads - 1) / kThreads;         // runs per thread
    Run16 r[NR];
#pragma unroll
    for (int u = 0; u < NR; ++u) {
        const int id = min(t + kThreads * u, 64 * RPC - 1);
        r[u].load(C, ldc, min(j0 + id / RPC, N - 1), min(16 * (id % RPC), K), K);
    }
#pragma unroll
    for (int u = 0; u < NR; ++u) {
        const int id = min(t + kThreads * u, 64 * RPC - 1);
        r[u].store(lds + (id / RPC) * LD, id % RPC);
    }
    __syncthreads();
    const float *w0 = lds + (wj + li) * LD, *w1 = w0 + 16 * LD;
    for (int blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
        float qv[S], cv[2][4];
#pragma unroll
        for (int s = 0; s < S; ++s) qv[s] = 4 * s + g < K ? q[s] : 0.0f;
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int e = 0; e < 4; ++e) cv[x][e] = c[x][e];
        if (blk + (int)gridDim.x < nblk) load(blk + gridDim.x);
        floatx4 acc[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
        for (int s = 0; s < KM / 16; ++s) {
            const floatx4 a0 = *(const floatx4 *)(w0 + chunk_of(s, g)), a1 = *(const floatx4 *)(w1 + chunk_of(s, g));
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[u], qv[4 * s + u], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[u], qv[4 * s + u], acc[1], 0, 0, 0);
            }
        }
        const int row = 32 * blk + wi + li;
        if (row < M) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int col = j0 + wj + 16 * x + 4 * g + e;
                    if (col >= N) continue;
                    B[row + (int64_t)col * ldb] = f64 ? (float)((double)cv[x][e] + (double)alpha * (double)acc[x][e])
                                                      : fmaf(alpha, acc[x][e], cv[x][e]);
                }
        }
    }
}

} // namespace

// Measured against the general kernel's 64 x 64 tiles (us, 16384 rows unless
// said): 32 x 32 8.9 against 13.5, 64 x 64 9.5 / 13.6, 32 x 128 9.3 / 13.8, with
// the reduction of the partials.  Where both sides are wide, a 32 x 32 tile
// reads its rows more often than a 64 x 64 one; that is paid back while the
// launch is latency-bound: 64 x 64 at 32768 rows 13.9 / 16.2, at 65536 22.6 /
// 21.4; 128 x 128 at 8192 10.6 / 12.9, at 16384 15.9 / 15.3; 96 x 64 at 16384
// 14.0 / 15.5, at 32768 21.4 / 18.2.  At equal traffic it is ahead at every
// height (32 x 128 at 524288: 91 / 103, 64 x 32 at 1048576 114 / 119).
bool gemm_proj_narrow(hipStream_t s, int m, int n1, int n2, const float *Q, int64_t ldq, const float *B, int64_t ldb,
                      float *C, int64_t ldc, int nsplit, int kper, float *partial)
{
    if (n1 > 128 || n2 > 128) return false;
    const int64_t tiles = ceil_div64(n1, 32) * ceil_div64(n2, 32);
    const int64_t reads = 64 * tiles, reads64 = 128 * ceil_div64(n1, 64) * ceil_div64(n2, 64);  // columns read per row
    if (reads > reads64 && tiles * m > (1 << 17)) return false;
    hipLaunchKernelGGL(proj_narrow_kernel, dim3((unsigned)nsplit, (unsigned)tiles), dim3(kThreads), 0, s, n1, n2, m, kper,
                       Q, ldq, B, ldb, C, ldc, partial);
    return true;
}

// Against the general kernel (us): depth 32 ahead or level while the operands
// fit the 256 MB cache (32 columns: 16384 rows 4.2 / 4.8, 262144 23.6 / 26.3; 128
// columns: 262144 rows 54 / 57, 524288 202 / 149: past it, its 64-byte row
// segments lose to whole 256-byte tiles); depth 64 up to two workgroups a CU (64
// columns: 8192 rows 4.4 / 5.4, 16384 5.7 / 5.9, 32768 8.8 / 8.2); deeper, up to
// one (128 columns: 4096 rows 6.0 / 7.2, 8192 7.9 / 7.6, 16384 13.1 / 11.1).
bool gemm_update_narrow(hipStream_t s, int M, int N, int K, float alpha, const float *Q, int64_t ldq, const float *C,
                        int64_t ldc, float *B, int64_t ldb, bool f64)
{
    const int64_t cols = ceil_div64(N, 64), blocks = ceil_div64(M, 32);
    if (K > 128 || cols > 65535) return false;
    if (K <= 32 ? (int64_t)M * N > (1 << 25) : blocks * cols > (K <= 64 ? 512 : 256)) return false;
    const dim3 grid((unsigned)(blocks < 2048 ? blocks : 2048), (unsigned)cols);
    const int d = f64 ? 1 : 0;
    if (K <= 32)
        hipLaunchKernelGGL(update_narrow_kernel<32>, grid, dim3(kThreads), 0, s, M, N, K, Q, ldq, C, ldc, B, ldb, alpha, d);
    else if (K <= 64)
        hipLaunchKernelGGL(update_narrow_kernel<64>, grid, dim3(kThreads), 0, s, M, N, K, Q, ldq, C, ldc, B, ldb, alpha, d);
    else
        hipLaunchKernelGGL(update_narrow_kernel<128>, grid, dim3(kThreads), 0, s, M, N, K, Q, ldq, C, ldc, B, ldb, alpha, d);
    return true;
}

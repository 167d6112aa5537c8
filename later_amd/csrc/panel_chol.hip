// Tall-skinny panel by Cholesky QR, twice (CholQR2), with FP64 Gram factors.
//
// An alternative to the block-MGS TSQR tree for the leaves of the accurate
// forms, with no sequential loop over columns across the grid.  For an m x w
// panel (w <= 64; kernels for widths 32 and 64), per pass (the partition of
// the rows depends on m only, so every result is bit-reproducible):
//   gram    G workgroups each form the Gram matrix of their 64-row blocks
//           with FP64 MFMA (products of FP32 values are exact in FP64) from
//           coalesced loads staged in LDS, and store the packed upper
//           triangle as a partial (a fixed-tree reduction kernel adds them
//           when there are more than 32);
//   factor  one workgroup adds the partials in a fixed order, factors
//           G = R^T R and inverts R (FP64, in 16-column blocks), and stores
//           R^{-1} (and R);
//   apply   the same grid forms q = a R^{-1} for its rows on FP64
//           MFMA and store Q in FP32; in the first of two passes they also
//           form the partial Grams of the stored Q1 for the second, which
//           repeats the factor and apply on Q1 and sets R = R2 R1.
// All of the small-matrix arithmetic is FP64, so multiplying by the explicit
// inverse adds errors of order u_64 kappa, far below the FP32 rounding of Q.
// Workgroups never wait for each other: the kernel boundaries order the
// partials and the factor, so there are no atomics and no device-scope
// fences (which would write back and invalidate the L2 of every XCD).  The
// factor runs once per pass instead of in every apply workgroup, so the
// apply kernels hold little LDS and several of them share a CU.
//
// One pass of Cholesky QR loses orthogonality like kappa^2 u_64 (the Gram and
// its factor are FP64) plus the FP32 rounding of Q; the second pass starts
// from kappa(Q1) ~ 1 and restores O(u) for kappa(panel) up to ~1e7.  Panels
// known to be near-orthonormal (a repeated factorisation of a Q) take one
// pass (`once`).
// A pivot that is not positive and finite, or that cancels to below
// 64 u_64 of the column's squared norm (numerical rank deficiency in the FP64
// Gram), sets status bit 0 and yields a zero column, like the MGS panel.
#include <type_traits>

#include "chol_dev.h"
#include "common.h"
#include "panel.h"
#include "prof.h"

namespace {

typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));  // one dwordx4 load at any dword address

// Sum of more than kDirect partial Grams, in a fixed tree: workgroup b owns
// entries 32b .. 32b+31; thread (q, e) adds groups q*G/8 .. (q+1)*G/8 - 1 in
// order, then the eight part sums are added in order of q.  The result is
// stored as the full matrix, so that no reader has to unpack it.
template <int W>
__global__ __launch_bounds__(256) void chol_reduce_kernel(const double *part, int ngroups, int w, double *out)
{
    __shared__ double ps[8][32];
    const int e = blockIdx.x * 32 + (threadIdx.x & 31), q = threadIdx.x >> 5;
    const int per = (ngroups + 7) / 8, g0 = q * per, g1 = min(ngroups, g0 + per);
    double s = 0.0;
    if (e < Shape<W>::P) {
        constexpr int kB = 32;  // one round of loads for up to 256 partials
        for (int g = g0; g < g1; g += kB) {
            double v[kB];
#pragma unroll
            for (int u = 0; u < kB; ++u) v[u] = part[(int64_t)min(g + u, g1 - 1) * Shape<W>::P + e];
#pragma unroll
            for (int u = 0; u < kB; ++u)
                if (g + u < g1) s += v[u];
        }
    }
    ps[q][threadIdx.x & 31] = s;
    __syncthreads();
    if (threadIdx.x < 32 && e < Shape<W>::P) {
        double t = ps[0][threadIdx.x];
#pragma unroll
        for (int k = 1; k < 8; ++k) t += ps[k][threadIdx.x];
        int i, j;
        unpack(e, i, j);
        if (i >= w || j >= w) t = (i == j) ? 1.0 : 0.0;
        out[i * W + j] = t;
        out[j * W + i] = t;
    }
}

// Rows r0 .. r0 + 63 of the panel's (up to W) columns, loaded with 16-byte
// loads (16 lanes cover the 64 rows of one column) into registers, then
// stored column-major into LDS (stride kRows + 4) for the Gram MFMA
// operands; zeros past m and past w.
template <int W> struct BlockRegs {
    static constexpr int NV = W / 16;  // float4 per thread
    floatx4 v[NV];
    __device__ __forceinline__ void load(const float *A, int64_t lda, int m, int w, int r0)
    {
        const int t = threadIdx.x, row = r0 + 4 * (t & 15);
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = (t >> 4) + 16 * j;
            const float *src = A + (int64_t)min(c, w - 1) * lda + min(row, m - 1);
            if (c < w && row + 4 <= m && ((((uintptr_t)src) & 15) == 0)) {
                v[j] = *(const floatx4 *)src;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[j][e] = (c < w && row + e < m) ? A[(int64_t)min(c, w - 1) * lda + min(row + e, m - 1)] : 0.0f;
            }
        }
    }
    // Either form; last: the last block inside (inside_last).
    __device__ __forceinline__ void load_block(const float *A, int64_t lda, int m, int w, int b, int last)
    {
        if (b <= last) load_inside(A, lda, b * kRows);
        else load(A, lda, m, w, b * kRows);
    }
    // All W columns of 64 rows that all lie inside the panel, at any dword
    // alignment and without a branch (a branch around a load makes the
    // compiler wait at the join for every load in flight).
    __device__ __forceinline__ void load_inside(const float *A, int64_t lda, int r0)
    {
        const int t = threadIdx.x;
        const float *src = A + (int64_t)(t >> 4) * lda + r0 + 4 * (t & 15);
#pragma unroll
        for (int j = 0; j < NV; ++j) v[j] = *(const floatx4u *)(src + 16 * j * lda);  // (the same step for all lanes)
    }
    __device__ __forceinline__ void store_ld(float *Qs, int ld) const
    {
        const int t = threadIdx.x;
#pragma unroll
        for (int j = 0; j < NV; ++j)
            *(floatx4 *)&Qs[((t >> 4) + 16 * j) * ld + 4 * (t & 15)] = v[j];
    }
    __device__ __forceinline__ void store(float *Qs) const { store_ld(Qs, kRows + 4); }
};

// The last of the 64-row blocks 0, 1, .. that lie inside a panel of full
// width (-1: none).
__device__ __forceinline__ int inside_last(int m, int w, int W) { return w == W ? m / kRows - 1 : -1; }

// Partial Gram of the rows of this workgroup (64-row blocks b, b + G, ...)
// into p1[blockIdx.x]: coalesced loads two blocks ahead, the block staged in
// LDS, FP64 MFMA per 16-row group of each wave.  Bound by FP64 MFMA (68 us for
// 1048576 x 64); with the loads of blocks inside the panel free of branches
// they are two blocks ahead in fact: 136 -> 105 us.
template <int W>
__global__ __launch_bounds__(kThreads) void chol_gram_kernel(int m, int w, const float *A, int64_t lda, float *ws)
{
    constexpr int kQs = W * (kRows + 4) * 4, kCb = kGramLds<W>;
    __shared__ __attribute__((aligned(16))) char smem[kQs > kCb ? kQs : kCb];
    float *Qs = (float *)smem;
    const CholWork cw = carve<W>(ws);
    const int nblk = (m + kRows - 1) / kRows;
    const int G = gridDim.x;
    const int wv = threadIdx.x >> 6;
    Gram<W> g;
    gram_zero<W>(g);
    BlockRegs<W> r0, r1;
    auto block = [&](const BlockRegs<W> &r) {
        __syncthreads();  // the previous block has been read
        r.store(Qs);
        __syncthreads();
    };
    auto product = [&]() {
#pragma unroll
        for (int sg = 0; sg < kTT; ++sg) gram_lds<W>(g, Qs, (wv * kTT + sg) * 16);
    };
    int b = blockIdx.x;
    const int last = inside_last(m, w, W);  // blocks up to here need no test
    if (b + 3 * G <= last) {
        r0.load_inside(A, lda, b * kRows);
        __builtin_amdgcn_sched_barrier(0);  // r0 first: the loop's waits count on the order
        r1.load_inside(A, lda, (b + G) * kRows);
#pragma unroll 1
        for (; b + 3 * G <= last; b += 2 * G) {
            block(r0);
            r0.load_inside(A, lda, (b + 2 * G) * kRows);
            product();
            block(r1);
            r1.load_inside(A, lda, (b + 3 * G) * kRows);
            product();
        }
    } else {
        if (b < nblk) r0.load_block(A, lda, m, w, b, last);
        if (b + G < nblk) r1.load_block(A, lda, m, w, b + G, last);
    }
    for (int it = 0; b < nblk; b += G, ++it) {
        if (it & 1) block(r1); else block(r0);
        if (b + 2 * G < nblk) {
            if (it & 1) r1.load_block(A, lda, m, w, b + 2 * G, last);
            else r0.load_block(A, lda, m, w, b + 2 * G, last);
        }
        product();
    }
    __syncthreads();
    gram_finish_shared<W>(g, (double *)smem, cw.p1 + (int64_t)blockIdx.x * Shape<W>::P);
}

// A -= Q C (Q: m x k, k <= 64; C: k x w) and the partial Gram of the result,
// in one pass over both: the update of a node whose second half is a leaf, and
// that leaf's first launch.  The Gram kernel's blocks and grid, so the partials
// are the same; the product is a chain of FP32 MFMA steps over k and one fused
// multiply-add with A, as in the separate update, so A keeps its bits too.
// Each wave forms the 16 rows whose Gram it takes, so between the two products
// the rows go through LDS without a barrier.  Q's and A's rows come in 256-byte
// runs a block ahead (4600 cycles of MFMA a block and wave, two waves a SIMD); C stays in LDS in operand order (lane l of step
// 4 s + u: column l % 16, k = 16 s + 4 u + l / 16).
// Bound by memory when tall.  1048576 x 64 with k = 64: 233 us, against 188 for
// the update and 104 for the Gram; 262144 rows 59 against 45 and 29; 8192 rows
// 9.7 against 5.1 and 5.8, with a launch less.
template <int W>
__global__ __launch_bounds__(kThreads, 2) void chol_update_gram_kernel(int m, int w, float *A, int64_t lda, float *ws, int k,
                                                                    const float *Q, int64_t ldq, const float *C,
                                                                    int64_t ldc)
{
    constexpr int KM = 64, LDC = KM + 4, CT = Shape<W>::CT;
    constexpr int kAs = KM * (kRows + 16) * 4, kQs = W * (kRows + 4) * 4, kCs = W * LDC * 4, kCb = kGramLds<W>;
    constexpr int kBytes = (kAs + kQs + kCs) > kCb ? (kAs + kQs + kCs) : kCb;
    __shared__ __attribute__((aligned(16))) char smem[kBytes];
    float *As = (float *)smem, *Qs = (float *)(smem + kAs), *Cs = (float *)(smem + kAs + kQs);
    const CholWork cw = carve<W>(ws);
    const int nblk = (m + kRows - 1) / kRows;
    const int G = gridDim.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
    const int lrow = wv * 16 + li;  // row within the block
    Gram<W> g;
    gram_zero<W>(g);
    struct Rows {
        BlockRegs<KM> q;
        BlockRegs<W> a;
    } r;
    int b = blockIdx.x;
    const int last = k == KM ? inside_last(m, w, W) : -1;
    auto load = [&](Rows &r, int b) {
        r.q.load_block(Q, ldq, m, k, b, last);
        r.a.load_block(A, lda, m, w, b, last);
    };
    auto block = [&]() {
        __syncthreads();  // the previous block has been read
        r.q.store_ld(As, kRows + 16);
        r.a.store(Qs);
        __syncthreads();
    };
    auto product = [&](auto inside) {
        const int row = b * kRows + lrow;
        floatx4 acc[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[c] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < KM / 16; ++s) {
            float q[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) q[u] = As[(16 * s + 4 * u + lk) * (kRows + 16) + lrow];
            floatx4 a[CT];
#pragma unroll
            for (int c = 0; c < CT; ++c) a[c] = *(const floatx4 *)&Cs[(16 * c + li) * LDC + 16 * s + 4 * lk];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int c = 0; c < CT; ++c) acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[c][u], q[u], acc[c], 0, 0, 0);
        }
        // acc[c][e]: row l % 16 of the wave's, column 16 c + 4 (l / 16) + e
        float *out = A + row + 4 * lk * lda;
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int col = 16 * c + 4 * lk + e;
                const bool ok = decltype(inside)::value || (row < m && col < w);
                float *x = &Qs[col * (kRows + 4) + lrow];
                const float v = ok ? fmaf(-1.0f, acc[c][e], *x) : 0.0f;
                if (ok) out[(16 * c + e) * lda] = v;
                *x = v;
            }
        __builtin_amdgcn_wave_barrier();  // the wave's own rows: its LDS accesses stay in order
        gram_lds<W>(g, Qs, wv * 16);
    };
    static_assert(kTT == 1, "a wave updates the 16 rows whose Gram it forms");
    load(r, b);
    {
        constexpr int N = W * KM / kThreads, S = kThreads / KM;
        const int kk = threadIdx.x % KM, c0 = threadIdx.x / KM;
        float x[N];
#pragma unroll
        for (int n = 0; n < N; ++n) x[n] = C[min(kk, k - 1) + (int64_t)min(c0 + S * n, w - 1) * ldc];
#pragma unroll
        for (int n = 0; n < N; ++n)
            Cs[(c0 + S * n) * LDC + (kk & ~15) + 4 * (kk & 3) + ((kk >> 2) & 3)] =
                (kk < k && c0 + S * n < w) ? x[n] : 0.0f;
    }
    auto step = [&]() {
        block();
        r.q.load_inside(Q, ldq, (b + G) * kRows);
        r.a.load_inside(A, lda, (b + G) * kRows);
        product(std::true_type());
        b += G;
    };
    if (b <= last) {  // apart, as in the apply kernel; all there is below 512 blocks
        block();
        if (b + G < nblk) load(r, b + G);
        product(std::true_type());
        b += G;
    }
#pragma unroll 1
    while (b + G <= last) step();
#pragma unroll 1
    for (; b < nblk; b += G) {
        block();
        if (b + G < nblk) load(r, b + G);
        product(std::false_type());
    }
    __syncthreads();
    gram_finish_shared<W>(g, (double *)smem, cw.p1 + (int64_t)blockIdx.x * Shape<W>::P);
}

// The factor of one Cholesky QR pass, by one workgroup, from the G partial
// Grams (or their reduced sum when G > kDirect):
//   PASS 1: R1 -> r1; PASS 0: R = R1 (ldr, FP32); PASS 2: R = R2 R1.
// R^{-1} goes to ri for the apply kernel.  A panel known to be
// near-orthonormal (PASS 0 or 2) whose Gram deviation E = G - I has
// max |E| <= 1e-5 uses R = I + U, R^{-1} = I - U with U = triu(E, 1) +
// diag(E) / 2, which agree with the Cholesky factor and its inverse to
// O(w |E|^2) <= 6.4e-9, far below the FP32 rounding of Q.
template <int PASS, int W>
__global__ __launch_bounds__(kThreads) void chol_factor_kernel(int w, float *ws, int G, float *R, int64_t ldr,
                                                            int *status)
{
    constexpr int LDG = Shape<W>::LDG;
    __shared__ double Gs[W * LDG], Rs[W * W], Ris[W * W], d0[W];
    __shared__ float emax_w[4];
    const CholWork cw = carve<W>(ws);
    const int t = threadIdx.x;
    const float e = G > kDirect ? load_gram<W>(cw.g, Gs) : sum_partials<W>(PASS == 2 ? cw.p2 : cw.p1, G, w, Gs);
    const float emax = gram_dev_max(e, emax_w);
    bool first_order = false;
    if constexpr (PASS != 1) {
        first_order = emax <= 1e-5f;  // NaN compares false: Cholesky path
        if (first_order) {
            for (int q = t; q < W * W; q += kThreads) {
                const int i = q / W, j = q % W;
                const double u = (i < j) ? Gs[i * LDG + j] : (i == j ? 0.5 * (Gs[i * LDG + i] - 1.0) : 0.0);
                Rs[i * W + j] = (i == j ? 1.0 : 0.0) + u;
                Ris[i * W + j] = (i == j ? 1.0 : 0.0) - u;
            }
        }
    }
    if (!first_order) {
        const bool bad = factor<W>(Gs, Rs, Ris, d0);
        if (bad && t == 0 && status) atomicOr(status, 1);
    }
    __syncthreads();
    for (int e = t; e < W * W; e += kThreads) cw.ri[e] = Ris[e];
    if constexpr (PASS == 1) {
        for (int e = t; e < W * W; e += kThreads) cw.r1[e] = Rs[e];
    } else {
        // R (FP32, ldr): R1 itself (PASS 0) or R2 R1 (PASS 2, both upper, FP64
        // then rounded once).
        for (int e = t; e < w * w; e += kThreads) {
            const int i = e % w, j = e / w;
            double s = 0.0;
            if constexpr (PASS == 2) {
                for (int k = i; k <= j; ++k) s = fma(Rs[i * W + k], cw.r1[k * W + j], s);
            } else {
                s = Rs[i * W + j];
            }
            R[i + (int64_t)j * ldr] = (i <= j) ? (float)s : 0.0f;
        }
    }
}

// Q = A R^{-1} over the rows of this workgroup (64-row blocks b, b + G, ...),
// with R^{-1} from ri.  Each block is loaded with coalesced 16-byte row
// loads two blocks ahead (as in the Gram kernel) and staged column-major in
// LDS with a row stride of kRows + 16 floats, so that a wave's MFMA operand
// reads (16 rows x 4 columns) cover 64 distinct banks.  The product runs on
// FP64 MFMA as D = R^{-T} A^T per 16 x 16 tile: the A operand (slices of
// R^{-1}) stays in registers, the B operand is the block's rows, and the
// four column tiles' accumulation chains are interleaved k-step by k-step
// (up to four independent MFMAs in flight); D's lanes walk 16 consecutive
// rows of one column (64-byte stores).  PASS 1 also forms the partial Gram
// of the stored Q1 rows into p2[blockIdx.x].  The grid is the Gram kernel's, two
// workgroups a CU, which is what the registers hold: 1048576 x 64 takes 120 us,
// 127 in two rounds on 1024 workgroups (262144 rows 35 and 39).  Bound by memory
// (110 us at a copy's rate); 152 us with branches around the loads and stores.
constexpr int kApplyLd = kRows + 16;

template <int PASS, int W>
__global__ __launch_bounds__(kThreads) void chol_apply_kernel(int m, int w, float *A, int64_t lda, float *ws)
{
    constexpr int CT = Shape<W>::CT, KS = Shape<W>::KS;
    constexpr int kAs = W * kApplyLd * 4;                       // the block, for the product
    constexpr int kQs = (PASS == 1) ? W * (kRows + 4) * 4 : 0;  // the stored Q1 rows, for their Gram
    constexpr int kCb = (PASS == 1) ? kGramLds<W> : 0;
    constexpr int kBytes = (kAs + kQs) > kCb ? (kAs + kQs) : kCb;
    __shared__ __attribute__((aligned(16))) char smem[kBytes];
    float *As = (float *)smem;
    float *Qs = (float *)(smem + kAs);
    const CholWork cw = carve<W>(ws);
    const int nblk = (m + kRows - 1) / kRows;
    const int G = gridDim.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;

    BlockRegs<W> r0, r1;
    int b = blockIdx.x;
    // A-operand slices of R^{-1}: rv[ct][s] = R^{-1}[4 s + l/16][16 ct + l%16]
    // (zero for k > column, so column tile ct needs k-steps 0 .. 4 ct + 3).
    double rv[CT][KS];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int s2 = 0; s2 < 4 * (ct + 1); ++s2)
            rv[ct][s2] = cw.ri[(4 * s2 + (lane >> 4)) * W + 16 * ct + (lane & 15)];

    Gram<W> g;
    if constexpr (PASS == 1) gram_zero<W>(g);
    auto block = [&](const BlockRegs<W> &r) {
        __syncthreads();  // the previous block's operands have been read
        r.store_ld(As, kApplyLd);
        __syncthreads();
    };
    // Q of the staged block b (inside: its rows and columns all exist).
    auto product = [&](int b, auto inside) {
        const int lrow = wv * 16 + (lane & 15);  // row within the block
        const int row = b * kRows + lrow;
        float av[KS];
#pragma unroll
        for (int s2 = 0; s2 < KS; ++s2) av[s2] = As[(4 * s2 + (lane >> 4)) * kApplyLd + lrow];
        doublex4 d[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) d[ct] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s2 = 0; s2 < KS; ++s2)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
                if (s2 < 4 * (ct + 1)) d[ct] = __builtin_amdgcn_mfma_f64_16x16x4f64(rv[ct][s2], (double)av[s2], d[ct], 0, 0, 0);
        // d[ct][r] = Q[row][16 ct + l/16 + 4 r]
        float *out = A + row + (lane >> 4) * lda;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int col = 16 * ct + (lane >> 4) + 4 * q;
                const bool ok = decltype(inside)::value || (row < m && col < w);
                const float v = ok ? (float)d[ct][q] : 0.0f;
                if (ok) out[(16 * ct + 4 * q) * lda] = v;
                if constexpr (PASS == 1) Qs[col * (kRows + 4) + lrow] = v;
            }
        if constexpr (PASS == 1) {
            // Gram of the stored (FP32) Q1 rows of this block.
            __syncthreads();
#pragma unroll
            for (int sg = 0; sg < kTT; ++sg) gram_lds<W>(g, Qs, (wv * kTT + sg) * 16);
        }
    };
    const int last = inside_last(m, w, W);
    if (b + 3 * G <= last) {
        r0.load_inside(A, lda, b * kRows);
        __builtin_amdgcn_sched_barrier(0);  // r0 first: the loop's waits count on the order
        r1.load_inside(A, lda, (b + G) * kRows);
        auto pair = [&]() {
            block(r0);
            r0.load_inside(A, lda, (b + 2 * G) * kRows);
            product(b, std::true_type());
            block(r1);
            r1.load_inside(A, lda, (b + 3 * G) * kRows);
            product(b + G, std::true_type());
            b += 2 * G;
        };
        // The first pair stands apart: the loop's waits are set by the path
        // with the fewest requests behind a block's loads, and before the
        // first pair no stores are.
        pair();
#pragma unroll 1
        while (b + 3 * G <= last) pair();
    } else {
        if (b < nblk) r0.load_block(A, lda, m, w, b, last);
        if (b + G < nblk) r1.load_block(A, lda, m, w, b + G, last);
    }
#pragma unroll 1
    for (int it = 0; b < nblk; b += G, ++it) {
        if (it & 1) block(r1); else block(r0);
        if (b + 2 * G < nblk) {
            if (it & 1) r1.load_block(A, lda, m, w, b + 2 * G, last);
            else r0.load_block(A, lda, m, w, b + 2 * G, last);
        }
        product(b, std::false_type());
    }
    if constexpr (PASS == 1) {
        __syncthreads();
        gram_finish_shared<W>(g, (double *)smem, cw.p2 + (int64_t)blockIdx.x * Shape<W>::P);
    }
}

// One Cholesky QR pass over the rows of this workgroup, the factor formed
// by every workgroup (panels of at most kFusedBlocks 64-row blocks: one
// launch less than the separate factor kernel).
//   PASS 1: Gram of A -> R1 (stored to r1 by workgroup 0); Q1 = A R1^{-1}
//           stored; partials p2 of the stored Q1.
//   PASS 2: Gram of Q1 -> R2; Q = Q1 R2^{-1} stored; R = R2 R1 (ldr, FP32).
//   PASS 0: the only pass (panels with condition number near 1): Gram of A
//           -> R1; Q = A R1^{-1} stored; R = R1.
// The product with R^{-1} runs on FP64 MFMA as D = R^{-T} A^T per 16 x 16
// tile: the A operand (slices of R^{-1}) stays in registers for the whole
// block, the B operand is the block's rows, and D's lanes walk 16
// consecutive rows of one column (64-byte stores).
template <int PASS, int W>
__global__ __launch_bounds__(kThreads) void chol_apply_fused_kernel(int m, int w, float *A, int64_t lda, float *ws, float *R,
                                                          int64_t ldr, int *status)
{
    constexpr int CT = Shape<W>::CT, KS = Shape<W>::KS, LDG = Shape<W>::LDG;
    __shared__ __attribute__((aligned(16))) char smem[ApplyLds<W>::kBytes];
    double *Gs = (double *)smem;      // W x (W + 1)
    double *Rs = Gs + W * LDG;        // W x W
    double *Ris = Rs + W * W;         // W x W
    double *d0 = Ris + W * W;         // W
    float *Qs = (float *)smem;        // W x (kRows + 4), after the factor
    double *Cb = (double *)smem;      // after the last block
    const CholWork cw = carve<W>(ws);
    const int nblk = (m + kRows - 1) / kRows;
    const int G = gridDim.x;
    const int t = threadIdx.x;
    const int lane = t & 63, wv = t >> 6;

    // The first block's rows are in flight while the factor is formed.
    float av[kTT][KS];
    load_block_mfma<W>(A, lda, m, w, blockIdx.x * kRows, av);

    __shared__ float emax_w[4];
    const float e = G > kDirect ? load_gram<W>(cw.g, Gs) : sum_partials<W>(PASS == 2 ? cw.p2 : cw.p1, G, w, Gs);
    const float emax = gram_dev_max(e, emax_w);
    // A-operand slices of R^{-1}: rv[ct][s] = R^{-1}[4 s + l/16][16 ct + l%16]
    // (zero for k > column, so column tile ct needs k-steps 0 .. 4 ct + 3).
    double rv[CT][KS];
    auto slices = [&](auto at) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int s2 = 0; s2 < 4 * (ct + 1); ++s2) rv[ct][s2] = at(4 * s2 + (lane >> 4), 16 * ct + (lane & 15));
    };
    // The panel (Q1, or a near-orthonormal input) has Gram I + E.  When
    // max |E| <= 1e-5, R2 = I + U and R2^{-1} = I - U with
    // U = triu(E, 1) + diag(E) / 2 agree with the Cholesky factor and its
    // inverse to O(w |E|^2) <= 6.4e-9, far below the FP32 rounding of Q;
    // otherwise (and for a zero column of Q1) the Cholesky runs.  Every
    // workgroup sees the same E, so all take the same branch (NaN compares
    // false).  The inverse's slices then come straight from the Gram: the
    // launch is a chain of latencies, and without R and R^{-1} passed through
    // LDS, a second sweep for E and the unpacking of the reduced Gram it takes
    // 13.3 us on average over a first and a second pass where it took 16.0
    // (8192 x 64).
    const bool first_order = PASS != 1 && emax <= 1e-5f;
    auto upper = [&](int i, int j) { return i < j ? Gs[i * LDG + j] : (i == j ? 0.5 * (Gs[i * LDG + i] - 1.0) : 0.0); };
    if (first_order) {
        slices([&](int i, int j) { return (i == j ? 1.0 : 0.0) - upper(i, j); });
        if constexpr (PASS == 2) {
            for (int q = t; q < W * W; q += kThreads) Rs[q] = (q / W == q % W ? 1.0 : 0.0) + upper(q / W, q % W);
            __syncthreads();
        }
    } else {
        const bool bad = factor<W>(Gs, Rs, Ris, d0);
        if (bad && t == 0 && blockIdx.x == 0 && status) atomicOr(status, 1);
        __syncthreads();
        slices([&](int i, int j) { return Ris[i * W + j]; });
    }
    if constexpr (PASS == 1) {
        if (blockIdx.x == 0)
            for (int q = t; q < W * W; q += kThreads) cw.r1[q] = Rs[q];
    } else {
        // R (FP32, ldr): R1 itself (PASS 0) or R2 R1 (PASS 2, both upper,
        // FP64 then rounded once), four columns per round, column j by
        // workgroup (j / 4) mod G, with column j of R1 staged in LDS (over
        // the Gram, no longer needed).
        for (int j0 = blockIdx.x * 4; j0 < w; j0 += G * 4) {
            const int c = t >> 6, j = j0 + c, i = t & 63;
            if constexpr (PASS == 2) {
                __syncthreads();  // every wave has its slices; the round before has been read
                if (j < w && i < W) Gs[c * LDG + i] = (i <= j) ? cw.r1[i * W + j] : 0.0;
                __syncthreads();
            }
            if (j < w && i < w) {
                double s = 0.0;
                if constexpr (PASS == 2) {
                    // Full k range: R2's lower and the staged column's
                    // below-j entries are zeros, so the sum is the same.
#pragma unroll
                    for (int k = 0; k < W; ++k) s = fma(Rs[i * W + k], Gs[c * LDG + k], s);
                } else if (first_order) {
                    s = (i == j ? 1.0 : 0.0) + upper(i, j);
                } else {
                    s = Rs[i * W + j];
                }
                R[i + (int64_t)j * ldr] = (i <= j) ? (float)s : 0.0f;
            }
        }
    }

    Gram<W> g;
    gram_zero<W>(g);
#pragma unroll 1
    for (int b = blockIdx.x; b < nblk; b += G) {
        __syncthreads();  // the factor, or Qs of the previous block, has been read
        const int r0 = b * kRows;
#pragma unroll
        for (int tt = 0; tt < kTT; ++tt) {
            const int lrow = (wv * kTT + tt) * 16 + (lane & 15);  // row within the block
            const int row = r0 + lrow;
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                doublex4 d = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int s2 = 0; s2 < 4 * (ct + 1); ++s2)
                    d = __builtin_amdgcn_mfma_f64_16x16x4f64(rv[ct][s2], (double)av[tt][s2], d, 0, 0, 0);
                // d[r] = Q[row][16 ct + l/16 + 4 r]
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int col = 16 * ct + (lane >> 4) + 4 * r;
                    const bool ok = row < m && col < w;
                    const float q = ok ? (float)d[r] : 0.0f;
                    if (ok) A[row + (int64_t)col * lda] = q;
                    if constexpr (PASS == 1) Qs[col * (kRows + 4) + lrow] = q;
                }
            }
        }
        if (b + G < nblk) load_block_mfma<W>(A, lda, m, w, (b + G) * kRows, av);
        if constexpr (PASS == 1) {
            // Gram of the stored (FP32) Q1 rows of this block.
            __syncthreads();
#pragma unroll
            for (int sg = 0; sg < kTT; ++sg) gram_lds<W>(g, Qs, (wv * kTT + sg) * 16);
        }
    }
    if constexpr (PASS == 1) {
        __syncthreads();
        gram_finish_shared<W>(g, Cb, cw.p2 + (int64_t)blockIdx.x * Shape<W>::P);
    }
}

constexpr int kFusedBlocks = 256;

template <int W>
int launch_cholqr(hipStream_t s, int m, int w, float *A, int lda, float *R, int ldr, float *work, int *status,
                  int G, bool once, const PanelUpdate *up)
{
    const CholWork cw = carve<W>(work);
    const int nblk = (m + kRows - 1) / kRows;
    // Up to kFusedBlocks blocks every apply workgroup forms the factor itself
    // (the latency of a separate factor launch outweighs the redundancy);
    // taller panels factor once and apply on the Gram's grid.
    const bool fused = nblk <= kFusedBlocks;
    const dim3 rgrid((Shape<W>::P + 31) / 32);
    int n = 0;
    if (up) {
        // Timed with the other updates, by the update's own work (its time
        // holds the Gram's).
        const int tok = prof_start(s);
        hipLaunchKernelGGL(chol_update_gram_kernel<W>, dim3(G), dim3(kThreads), 0, s, m, w, A, (int64_t)lda, work, up->k,
                           up->Q, up->ldq, up->C, up->ldc);
        prof_stop(tok, s, PROF_GEMM_UPDATE, 2.0 * m * w * up->k,
                  4.0 * ((double)m * up->k + 2.0 * m * w + (double)up->k * w));
    } else {
        hipLaunchKernelGGL(chol_gram_kernel<W>, dim3(G), dim3(kThreads), 0, s, m, w, (const float *)A, (int64_t)lda, work);
    }
    ++n;
    if (G > kDirect) {
        hipLaunchKernelGGL(chol_reduce_kernel<W>, rgrid, dim3(256), 0, s, cw.p1, G, w, cw.g);
        ++n;
    }
    auto pass = [&](auto P) {
        constexpr int PASS = decltype(P)::value;
        if (fused) {
            hipLaunchKernelGGL((chol_apply_fused_kernel<PASS, W>), dim3(G), dim3(kThreads), 0, s, m, w, A,
                               (int64_t)lda, work, R, (int64_t)ldr, status);
            ++n;
        } else {
            hipLaunchKernelGGL((chol_factor_kernel<PASS, W>), dim3(1), dim3(kThreads), 0, s, w, work, G, R,
                               (int64_t)ldr, status);
            hipLaunchKernelGGL((chol_apply_kernel<PASS, W>), dim3(G), dim3(kThreads), 0, s, m, w, A,
                               (int64_t)lda, work);
            n += 2;
        }
    };
    if (once) {
        pass(std::integral_constant<int, 0>());
        return n;
    }
    pass(std::integral_constant<int, 1>());
    if (G > kDirect) {
        hipLaunchKernelGGL(chol_reduce_kernel<W>, rgrid, dim3(256), 0, s, cw.p2, G, w, cw.g);
        ++n;
    }
    pass(std::integral_constant<int, 2>());
    return n;
}

} // namespace

int64_t panel_chol_work_floats(int w) { return w <= 32 ? work_floats<32>() : work_floats<64>(); }

int panel_cholqr2(hipStream_t s, int m, int w, float *A, int lda, float *R, int ldr, float *work, int64_t lwork,
                  int *status, int *launches, bool once, const PanelUpdate *up)
{
    if (up && (up->k < 1 || up->k > kWMax)) return LATER_ERR_SHAPE;
    if (w < 1 || w > kWMax || m < w) return LATER_ERR_SHAPE;
    if (lwork < panel_chol_work_floats(w)) return LATER_ERR_WORKSPACE;
    const int nblk = (m + kRows - 1) / kRows;
    const int G = nblk < kMaxGroups ? nblk : kMaxGroups;
    const int n = (w <= 32) ? launch_cholqr<32>(s, m, w, A, lda, R, ldr, work, status, G, once, up)
                            : launch_cholqr<64>(s, m, w, A, lda, R, ldr, work, status, G, once, up);
    HIP_OK(hipGetLastError());
    if (launches) *launches += n;
    return LATER_OK;
}

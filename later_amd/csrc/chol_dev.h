// Device helpers of the Cholesky QR panels (FP64 MFMA Gram, FP64
// Cholesky with its inverse), shared by the grid-wide panel kernels
// (panel_chol.hip) and the one-workgroup-per-matrix batched kernel
// (batch_wg.hip).
#pragma once
#include <type_traits>

#include "common.h"

namespace {

typedef double doublex4 __attribute__((ext_vector_type(4)));

constexpr int kWMax = 64;                 // max panel width
constexpr int kThreads = 256;             // threads per workgroup (four waves)
constexpr int kTT = 1;                    // 16-row tiles per wave in a block
constexpr int kRows = 64 * kTT;           // rows per block (workgroup b takes blocks b, b + G, ...)
constexpr int kMaxGroups = 512;           // Gram workgroups (and partials) per launch: two per CU
constexpr int kDirect = 32;               // up to this many partials, every workgroup adds them itself
constexpr double kPivotRel = 64.0 * 2.220446049250313e-16;

// Sizes of the width-W kernels (W = 32 or 64).
template <int W> struct Shape {
    static constexpr int CT = W / 16;             // 16-column tiles
    static constexpr int NT = CT * (CT + 1) / 2;  // distinct 16 x 16 tiles of the symmetric Gram
    static constexpr int P = W * (W + 1) / 2;     // packed upper triangle
    static constexpr int LDG = W + 1;             // row stride of the Gram in LDS
    static constexpr int KS = W / 4;              // MFMA k-steps over the columns
};

// Index of Gram tile (a, b), a <= b < CT, in row-major upper-triangular order.
template <int CT> __host__ __device__ constexpr int tile_index(int a, int b)
{
    return a * CT - a * (a - 1) / 2 + (b - a);
}

// Workspace of the width-W kernels (doubles; the partials have stride P).
struct CholWork {
    double *p1;  // kMaxGroups x P: partial Grams of A
    double *p2;  // kMaxGroups x P: partial Grams of Q1
    double *r1;  // W x W, row-major: R1 (upper)
    double *g;   // W x W: a reduced Gram (more than kDirect partials), both triangles, the identity's outside w x w
    double *ri;  // the same place: the inverse factor the apply kernel multiplies by (one workgroup reads g, then
                 // writes ri)
};

template <int W> __host__ __device__ inline CholWork carve(float *ws)
{
    constexpr int P = Shape<W>::P;
    CholWork c;
    c.p1 = (double *)ws;
    c.p2 = c.p1 + (int64_t)kMaxGroups * P;
    c.r1 = c.p2 + (int64_t)kMaxGroups * P;
    c.g = c.ri = c.r1 + W * W;
    return c;
}

template <int W> constexpr int64_t work_floats()
{
    return ((int64_t)2 * kMaxGroups * Shape<W>::P + 2 * W * W) * 2 + 64;
}

// Packed index e of the upper triangle (column-major, i <= j) -> (i, j).
__device__ __forceinline__ void unpack(int e, int &i, int &j)
{
    int c = (int)((sqrtf(8.0f * (float)e + 1.0f) - 1.0f) * 0.5f);
    while (c * (c + 1) / 2 > e) --c;
    while ((c + 1) * (c + 2) / 2 <= e) ++c;
    j = c;
    i = e - c * (c + 1) / 2;
}

// The distinct 16 x 16 tiles (a, b), a <= b, of a W x W Gram.
template <int W> struct Gram {
    doublex4 t[Shape<W>::NT];
};

template <int W> __device__ __forceinline__ void gram_zero(Gram<W> &g)
{
#pragma unroll
    for (int q = 0; q < Shape<W>::NT; ++q) g.t[q] = doublex4{0.0, 0.0, 0.0, 0.0};
}

// v_mfma_f64_16x16x4f64: A (16 x 4) lane l holds A[l%16][l/16], B (4 x 16)
// lane l holds B[l/16][l%16], D (16 x 16) lane l item r holds
// D[l/16 + 4r][l%16] (rows interleaved, unlike the FP32 16 x 16 forms).  For
// the Gram, the k index is a row of the panel: the lane's value of column
// c = 16 t + l%16 at row k serves as both A[c][k] and B[k][c].  a[t][p] holds
// column tile t at four rows (one per MFMA).
template <int W> __device__ __forceinline__ void gram_step(Gram<W> &g, const double (*a)[4])
{
    constexpr int CT = Shape<W>::CT;
#pragma unroll
    for (int p = 0; p < 4; ++p)
#pragma unroll
        for (int x = 0; x < CT; ++x)
#pragma unroll
            for (int y = x; y < CT; ++y)
                g.t[tile_index<CT>(x, y)] =
                    __builtin_amdgcn_mfma_f64_16x16x4f64(a[x][p], a[y][p], g.t[tile_index<CT>(x, y)], 0, 0, 0);
}

// Adds the four waves' Grams, (w0 + w2) + (w1 + w3), in two lane-aligned
// LDS rounds (every wave reads back exactly the slots it wrote: no bank
// conflicts), and wave 0 stores this workgroup's packed partial from its
// registers.  Cb: 2 x NT x 4 x 64 doubles of LDS.
template <int W> __device__ __forceinline__ void gram_finish(const Gram<W> &g, double *Cb, double *part)
{
    constexpr int NT = Shape<W>::NT, CT = Shape<W>::CT;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    Gram<W> s = g;
    if (wv >= 2) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) Cb[(((wv - 2) * NT + t) * 4 + r) * 64 + lane] = g.t[t][r];
    }
    __syncthreads();
    if (wv < 2) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) s.t[t][r] += Cb[((wv * NT + t) * 4 + r) * 64 + lane];
    }
    __syncthreads();
    if (wv == 1) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) Cb[(t * 4 + r) * 64 + lane] = s.t[t][r];
    }
    __syncthreads();
    if (wv == 0) {
        // Lane l, item r of tile (a, b) holds entry (16 a + l/16 + 4 r, 16 b + l%16).
#pragma unroll
        for (int a = 0; a < CT; ++a)
#pragma unroll
            for (int b = a; b < CT; ++b) {
                const int t = tile_index<CT>(a, b);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = 16 * a + (lane >> 4) + 4 * r, j = 16 * b + (lane & 15);
                    if (i <= j) part[j * (j + 1) / 2 + i] = s.t[t][r] + Cb[(t * 4 + r) * 64 + lane];
                }
            }
    }
}

// The four waves' Grams added as above, in one round for the grid-wide
// kernels: every wave writes the tiles it does not own (tile t belongs to wave
// t % 4), and the owners add them up and store their part of the partial.  One
// barrier instead of three and the stores on four waves (Gram of 8192 x 64:
// 6.7 -> 6.1 us).  Cb: 3 x NT x 4 x 64 doubles of LDS.
template <int W> __device__ __forceinline__ void gram_finish_shared(const Gram<W> &g, double *Cb, double *part)
{
    constexpr int NT = Shape<W>::NT, CT = Shape<W>::CT;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    auto slot = [&](int t, int from) { return Cb + (((from - (from > t % 4)) * NT + t) * 4) * 64 + lane; };
#pragma unroll
    for (int t = 0; t < NT; ++t)
        if (t % 4 != wv) {
            double *c = slot(t, wv);
#pragma unroll
            for (int r = 0; r < 4; ++r) c[r * 64] = g.t[t][r];
        }
    __syncthreads();
    // Lane l, item r of tile (a, b) holds entry (16 a + l/16 + 4 r, 16 b + l%16).
#pragma unroll
    for (int a = 0; a < CT; ++a)
#pragma unroll
        for (int b = a; b < CT; ++b) {
            const int t = tile_index<CT>(a, b);
            if (t % 4 != wv) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                auto of = [&](int w) { return w == t % 4 ? g.t[t][r] : slot(t, w)[r * 64]; };
                const double v = (of(0) + of(2)) + (of(1) + of(3));
                const int i = 16 * a + (lane >> 4) + 4 * r, j = 16 * b + (lane & 15);
                if (i <= j) part[j * (j + 1) / 2 + i] = v;
            }
        }
}

// Largest |G - I| entry that a thread has seen, over the workgroup's four
// waves (e4: 4 floats of LDS; a barrier inside).
__device__ __forceinline__ float gram_dev_max(float e, float *e4)
{
#pragma unroll
    for (int mask = 32; mask > 0; mask >>= 1) e = fmaxf(e, __shfl_xor(e, mask, 64));
    if ((threadIdx.x & 63) == 0) e4[threadIdx.x >> 6] = e;
    __syncthreads();
    return fmaxf(fmaxf(e4[0], e4[1]), fmaxf(e4[2], e4[3]));
}

// G (LDS, W x (W + 1)) = a reduced Gram (CholWork.g).  Returns the largest
// |G - I| entry among the thread's own.
template <int W> __device__ __forceinline__ float load_gram(const double *g, double *Gs)
{
    constexpr int N = W * W / 2 / kThreads, LDG = Shape<W>::LDG;
    double2 v[N];
#pragma unroll
    for (int x = 0; x < N; ++x) v[x] = ((const double2 *)g)[threadIdx.x + x * kThreads];
    float e = 0.0f;
#pragma unroll
    for (int x = 0; x < N; ++x) {
        const int q = threadIdx.x + x * kThreads, i = q / (W / 2), j = 2 * (q % (W / 2));
        Gs[i * LDG + j] = v[x].x;
        Gs[i * LDG + j + 1] = v[x].y;
        e = fmaxf(e, (float)fabs(v[x].x - (i == j ? 1.0 : 0.0)));
        e = fmaxf(e, (float)fabs(v[x].y - (i == j + 1 ? 1.0 : 0.0)));
    }
    return e;
}

// G (LDS, W x (W + 1)) = sum over g < ngroups of the packed partials, in order
// g = 0, 1, ...; entries outside the w x w block are the identity's.  Returns
// the largest |G - I| entry among the thread's own.
template <int W>
__device__ __forceinline__ float sum_partials(const double *part, int ngroups, int w, double *Gs)
{
    constexpr int P = Shape<W>::P, LDG = Shape<W>::LDG;
    constexpr int kPer = (P + kThreads - 1) / kThreads;  // 3 or 9
    int ei[kPer];
    double s[kPer];
    float dev = 0.0f;
#pragma unroll
    for (int x = 0; x < kPer; ++x) {
        ei[x] = min((int)threadIdx.x + x * kThreads, P - 1);
        s[x] = 0.0;
    }
    // Many loads in flight per thread: the partials were written by other
    // XCDs and come from memory, so each round costs a full memory latency.
    constexpr int kBatch = W == 32 ? 16 : 4;
    for (int g0 = 0; g0 < ngroups; g0 += kBatch) {
        double v[kPer][kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const int g = min(g0 + u, ngroups - 1);
#pragma unroll
            for (int x = 0; x < kPer; ++x) v[x][u] = part[(int64_t)g * P + ei[x]];
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
#pragma unroll
            for (int x = 0; x < kPer; ++x)
                if (g0 + u < ngroups) s[x] += v[x][u];
    }
#pragma unroll
    for (int x = 0; x < kPer; ++x) {
        const int e = threadIdx.x + x * kThreads;
        if (e < P) {
            int i, j;
            unpack(e, i, j);
            double val = s[x];
            if (i >= w || j >= w) val = (i == j) ? 1.0 : 0.0;
            Gs[i * LDG + j] = val;
            Gs[j * LDG + i] = val;
            dev = fmaxf(dev, (float)fabs(val - (i == j ? 1.0 : 0.0)));
        }
    }
    return dev;
}

__device__ __forceinline__ double readlane_f64(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// v += (lane K of each 16-lane row of l) b, for N values each of s and m
// against the same l = s: one v_fmac_f64 with a DPP row broadcast per value.
// (A DPP read needs two instructions after the write of its register: the
// callers' order gives that inside a pivot, the trailing s_nop across pivots.)
template <int K, int N>
__device__ __forceinline__ void rank1_rows(double *s, double *m, double a, double b)
{
#define LATER_ROW(S, M)                                                                    \
    "v_fmac_f64_dpp %" #M ", %" #S ", %[b] row_newbcast:%c[k] row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f64_dpp %" #S ", %" #S ", %[a] row_newbcast:%c[k] row_mask:0xf bank_mask:0xf\n\t"
    if constexpr (N == 1)
        asm(LATER_ROW(0, 1) "s_nop 1" : "+v"(s[0]), "+v"(m[0]) : [a] "v"(a), [b] "v"(b), [k] "n"(K));
    else if constexpr (N == 2)
        asm(LATER_ROW(0, 2) LATER_ROW(1, 3) "s_nop 1"
            : "+v"(s[0]), "+v"(s[1]), "+v"(m[0]), "+v"(m[1]) : [a] "v"(a), [b] "v"(b), [k] "n"(K));
    else if constexpr (N == 3)
        asm(LATER_ROW(0, 3) LATER_ROW(1, 4) LATER_ROW(2, 5) "s_nop 1"
            : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(m[0]), "+v"(m[1]), "+v"(m[2])
            : [a] "v"(a), [b] "v"(b), [k] "n"(K));
    else if constexpr (N == 4)
        asm(LATER_ROW(0, 4) LATER_ROW(1, 5) LATER_ROW(2, 6) LATER_ROW(3, 7) "s_nop 1"
            : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]), "+v"(m[0]), "+v"(m[1]), "+v"(m[2]), "+v"(m[3])
            : [a] "v"(a), [b] "v"(b), [k] "n"(K));
    else if constexpr (N > 4) {
        rank1_rows<K, 4>(s, m, a, b);
        rank1_rows<K, N - 4>(s + 4, m + 4, a, b);
    }
#undef LATER_ROW
}

// Elimination of a 16 x 16 block S = L D L^T in LDS by one wave: U = D L^T,
// M = L^{-1} and 1/sqrt(d_k), so that R = D^{-1/2} U and R^{-T} = D^{-1/2} M
// (Gauss-Jordan on [S | I]).  Each 16-lane row of the wave holds all of it
// (lane j: column j of the trailing matrix and of the identity's rows), so a
// pivot's row is already in every lane and its multipliers are a DPP row
// broadcast inside the multiply-add: no value crosses through scalar
// registers.  Only 1/d_k is on the serial chain; the square roots are taken at
// once afterwards, one per lane.
// S: row stride LDS_; least[k]: what pivot k has to exceed.  U (row stride 16), M (row stride kLdM) get rows k, isq[k]
// the scale; a bad pivot k gets scale 0 (which zeroes row k of R and column k
// of R^{-1}, so column k of Q) and drops row k from the later columns'
// elimination.  Returns true if a pivot was bad.
constexpr int kLdM = 17;

template <int K>
__device__ __forceinline__ void eliminate16_from(double *s, double *m, const double *least)
{
    const double p = dpp_d<0x150 + K>(s[K]);  // row_newbcast:K
    // 1/p: hardware estimate and two Newton steps.
    double y = __builtin_amdgcn_rcp(p);
    y = fma(fma(-p, y, 1.0), y, y);
    y = fma(fma(-p, y, 1.0), y, y);
    y = p > least[K] ? y : 0.0;
    rank1_rows<K, 15 - K>(s + K + 1, m + K + 1, -(s[K] * y), -(m[K] * y));
    if constexpr (K + 1 < 16) eliminate16_from<K + 1>(s, m, least);
}

template <int LDS_>
__device__ __forceinline__ bool eliminate16_wave(const double *S, const double *least, double *U, double *M,
                                                 double *isq)
{
    constexpr int kW = 16;
    const int lane = threadIdx.x & 63, j = lane & (kW - 1);
    double s[kW], m[kW], lk[kW];
#pragma unroll
    for (int i = 0; i < kW; ++i) {
        s[i] = S[i * LDS_ + j];
        m[i] = i == j ? 1.0 : 0.0;
        lk[i] = least[i];
    }
    eliminate16_from<0>(s, m, lk);
    if (lane < kW) {
#pragma unroll
        for (int i = 0; i < kW; ++i) {
            U[i * kW + j] = s[i];
            M[i * kLdM + j] = m[i];
        }
    }
    // Lane j's own pivot; estimate of 1/sqrt and two Newton steps.
    const double d = U[j * kW + j];
    const bool ok = d > least[j] && d <= 1.7976931348623157e308;
    const double p = ok ? d : 1.0;
    double y = __builtin_amdgcn_rsq(p);
    y = y * fma(-0.5 * p * y, y, 1.5);
    y = y * fma(-0.5 * p * y, y, 1.5);
    if (lane < kW) isq[j] = ok ? y : 0.0;
    return __builtin_amdgcn_ballot_w64(!ok) != 0;
}

// G = R^T R and R^{-1} for the W x W Gram in LDS (Gs, row stride W + 1; R and
// Ri row stride W), blocked by 16: the elimination of [G | I] with the
// diagonal blocks on wave 0 (eliminate16_wave) and every other product on FP64
// MFMA.  Step b: X_bb = R_bb^{-T}; R_bj = X_bb G_bj (j > b) and
// X_bj = X_bb Y_bj (j < b); then G_ij -= R_bi^T R_bj (b < i <= j) and
// Y_ij -= R_bi^T X_bj (i > b >= j).  X (= R^{-T}) and Y share the lower
// blocks of Gs; Ris holds U, M and the scales of the current step until the
// end.  Wave 0 updates the next diagonal block and goes on to its
// elimination while the other waves update the rest, so the serial path is
// the W / 16 eliminations and one product before and after each.  A pivot is
// compared with the diagonal of G.  Destroys Gs.  nb: the blocks to factor
// (the columns behind them are left undefined).  Called by every thread of the
// workgroup (four waves or more); returns (on wave 0) whether a pivot was bad.
// Bound: the dependent FP64 chain of the pivots (about 100 cycles each) and
// the issue of the rank-1 rows beside it.  W = 64: 10 us, where two 32 x 32
// one-wave eliminations, fully unrolled with scalar broadcasts and each
// pivot's square root on the chain, took 19 us (a first-pass leaf of 8192 x 64:
// factor and apply 30 -> 21 us).
template <int W>
__device__ __forceinline__ bool factor(double *Gs, double *Rs, double *Ris, double *d0, int nb = W / 16)
{
    constexpr int LDG = Shape<W>::LDG;
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int li = lane & 15, lk = lane >> 4;
    double *U = Ris, *M = Ris + 256, *isq = Ris + 256 + 16 * kLdM;
    static_assert(256 + 16 * kLdM + 16 <= W * W, "scratch in Ris");
    if (t < W) {
        const double g = Gs[t * LDG + t];
        d0[t] = g > 0.0 ? kPivotRel * g : __longlong_as_double(0x7ff0000000000000ll);
    }
    // Zero blocks of R below the diagonal ones.
    for (int e = t; e < W * W; e += kThreads)
        if (e / W / 16 > e % W / 16) Rs[e] = 0.0;
    __syncthreads();
    // One 16 x 16 tile: T = c + a b over k = 0 .. 15 (v_mfma_f64_16x16x4f64: lane
    // l, entry r of the result is tile element (l / 16 + 4 r, l % 16)).
    // a(x, k) by the caller; b[k][y] at B + k ldb + y.
    auto product = [&](const double (&av)[4], const double *B, int ldb, doublex4 c) {
        double bv[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) bv[s] = B[(4 * s + lk) * ldb + li];
#pragma unroll
        for (int s = 0; s < 4; ++s) c = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s], bv[s], c, 0, 0, 0);
        return c;
    };
    // Tile (i, j) of the trailing update of step b: both halves read row b of
    // R (R_bj) or of X (X_bj, whose blocks lie in Gs).
    auto trailing = [&](int b, int i, int j) {
        double *T = Gs + 16 * i * LDG + 16 * j;
        doublex4 c = doublex4{0.0, 0.0, 0.0, 0.0};
        if (!(i > j && j == b)) {  // Y_ib starts here
#pragma unroll
            for (int r = 0; r < 4; ++r) c[r] = T[(lk + 4 * r) * LDG + li];
        }
        double av[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) av[s] = -Rs[(16 * b + 4 * s + lk) * W + 16 * i + li];
        c = i <= j ? product(av, Rs + 16 * b * W + 16 * j, W, c) : product(av, Gs + 16 * b * LDG + 16 * j, LDG, c);
#pragma unroll
        for (int r = 0; r < 4; ++r) T[(lk + 4 * r) * LDG + li] = c[r];
    };
    bool bad = false;
#pragma unroll 1
    for (int b = 0; b < nb; ++b) {
        if (wv == 0) {
            if (b > 0) trailing(b - 1, b, b);
            bad |= eliminate16_wave<LDG>(Gs + 16 * b * LDG + 16 * b, d0 + 16 * b, U, M, isq);
        } else if (b > 0) {
            int n = 0;
#pragma unroll 1
            for (int i = b; i < nb; ++i)
#pragma unroll 1
                for (int j = 0; j < nb; ++j)
                    if ((i <= j || j < b) && !(i == b && j == b)) {
                        if (n == wv - 1) trailing(b - 1, i, j);
                        n = n == 2 ? 0 : n + 1;
                    }
        }
        __syncthreads();
        if (wv == 3) {
            // R_bb and X_bb (over G_bb).
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = lk + 4 * u;
                const double s = isq[k];
                Rs[(16 * b + k) * W + 16 * b + li] = li < k ? 0.0 : U[k * 16 + li] * s;
                Gs[(16 * b + k) * LDG + 16 * b + li] = M[k * kLdM + li] * s;
            }
        } else if (wv < nb - 1) {
            // Row b of R and of X: block j on wave (j - b - 1) mod nb, so that
            // the next diagonal block's factor R_b,b+1 is wave 0's.
            const int j = (b + 1 + wv) % nb;
            double av[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) av[s] = M[li * kLdM + 4 * s + lk] * isq[li];
            const doublex4 c = product(av, Gs + 16 * b * LDG + 16 * j, LDG, doublex4{0.0, 0.0, 0.0, 0.0});
            double *T = j > b ? Rs + 16 * b * W + 16 * j : Gs + 16 * b * LDG + 16 * j;
            const int ld = j > b ? W : LDG;
#pragma unroll
            for (int r = 0; r < 4; ++r) T[(lk + 4 * r) * ld + li] = c[r];
        }
        __syncthreads();
    }
    // R^{-1} = X^T, zeros below the diagonal.
    for (int e = t; e < W * W; e += kThreads) {
        const int i = e / W, j = e % W;
        Ris[e] = i <= j ? Gs[j * LDG + i] : 0.0;
    }
    return bad;
}

// Gram MFMA operands of one 16-row group at local row r0 + 4 (l/16) of a
// column-major LDS block Qs[col][kRows + 4].
template <int W> __device__ __forceinline__ void gram_lds(Gram<W> &g, const float *Qs, int r0)
{
    constexpr int CT = Shape<W>::CT;
    const int lane = threadIdx.x & 63;
    const int c = lane & 15, r = r0 + 4 * (lane >> 4);
    double a[CT][4];
#pragma unroll
    for (int x = 0; x < CT; ++x) {
        const floatx4 v = *(const floatx4 *)&Qs[(16 * x + c) * (kRows + 4) + r];
#pragma unroll
        for (int p = 0; p < 4; ++p) a[x][p] = (double)v[p];
    }
    gram_step<W>(g, a);
}

// Rows of one block in the operand layout of the apply MFMA: wave wv owns
// kTT 16-row tiles; lane l holds, for tile t and k-step s,
// A[r0 + 16 (kTT wv + t) + l%16][4 s + l/16] (zero past m or w).
template <int W>
__device__ __forceinline__ void load_block_mfma(const float *A, int64_t lda, int m, int w, int r0, float (*av)[W / 4])
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int kk = lane >> 4;
#pragma unroll
    for (int t = 0; t < kTT; ++t) {
        const int row = r0 + (wv * kTT + t) * 16 + (lane & 15);
        const int rc = min(row, m - 1);
#pragma unroll
        for (int s2 = 0; s2 < W / 4; ++s2) {
            const int col = 4 * s2 + kk;
            const float x = A[rc + (int64_t)min(col, w - 1) * lda];
            av[t][s2] = (row < m && col < w) ? x : 0.0f;
        }
    }
}

// LDS of gram_finish_shared.
template <int W> constexpr int kGramLds = 3 * Shape<W>::NT * 4 * 64 * 8;

// LDS of the apply kernel: the factor's matrices while it is formed, then
// (PASS 1) the block of stored Q1 rows, then the Gram reduction buffer.
template <int W> struct ApplyLds {
    static constexpr int kFactor = (W * Shape<W>::LDG + 2 * W * W + W) * 8;
    static constexpr int kQs = W * (kRows + 4) * 4;
    static constexpr int kCb = kGramLds<W>;
    static constexpr int kBytes = kFactor > kQs ? (kFactor > kCb ? kFactor : kCb) : (kQs > kCb ? kQs : kCb);
};

} // namespace

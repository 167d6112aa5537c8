// Tall-skinny panel: TSQR tree of block modified Gram-Schmidt factorisations.
//
// Follows the structure of mgs_caqr_panel_256x32 (QR/panel.cu:65-134): every
// 256-row block is factored by MGS, the blocks' R factors are stacked and the
// stack is factored recursively, then each block's Q is multiplied by its
// rows of the stack's Q.  The block kernel is laid out for 64-lane
// wavefronts instead of the reference's 32x32 thread block of 32-lane warps
// (QR/panel.cu:246-325): wave v owns columns 4v .. 4v + 3 and lane l holds rows
// l, l+64, ... of them in registers, so the column norm and the projections are
// single-wave reductions, and a finished column passes to the waves behind
// through LDS with a count, without a barrier.
//
// The kernels come for panels of up to 8, 16 and 32 columns (KC): a narrow
// panel on the widest one keeps waves and registers for columns it does not
// have (FP64 sums, 1000000 rows: 1 column 59 us, 9 columns 151; 22 and 86 here).
#include <type_traits>

#include "common.h"
#include "panel.h"
#include "prof.h"

namespace {

constexpr int kCols = 32;                 // max panel width
constexpr int kCPW = 4;                   // columns per wave: wave v owns kCPW v .. kCPW v + kCPW - 1
constexpr int kMaxRows = 320;             // rows of a block: 256, or up to 256 + 31 with a merged tail

// sqrt(s) and its reciprocal, both correctly rounded (0 for the reciprocal
// and ok = false unless the root is positive and finite).  For s well inside
// the normal range the root is the hardware estimate (within 1 ulp) moved by
// one ulp where the sign of the exact residual of its neighbour says so, and
// the reciprocal is refined from the estimate of 1/sqrt(s), which is ready
// at the same time, by three exact-residual steps: about half the dependent
// operations of a square root followed by a division.
__device__ __forceinline__ bool norm_of(float s, float &nrm, float &inv)
{
    const unsigned u = __builtin_amdgcn_readfirstlane(__float_as_uint(s));
    const float y = __builtin_amdgcn_sqrtf(s);
    float r = __builtin_amdgcn_rsqf(s);
    const float yd = __uint_as_float(__float_as_uint(y) - 1u), yu = __uint_as_float(__float_as_uint(y) + 1u);
    const float ed = fmaf(-yd, y, s), eu = fmaf(-yu, y, s);
    nrm = ed <= 0.0f ? yd : y;
    nrm = eu > 0.0f ? yu : nrm;
#pragma unroll
    for (int i = 0; i < 3; ++i) r = fmaf(fmaf(-nrm, r, 1.0f), r, r);
    inv = r;
    if (__builtin_expect(u - 0x10000000u < 0x6E000000u - 0x10000000u, 1)) return true;  // 2^-95 <= s < 2^93
    nrm = sqrtf(s);
    const bool ok = (nrm > 0.0f) && (nrm < INFINITY);
    inv = ok ? 1.0f / nrm : 0.0f;
    return ok;
}
// FP64: the reciprocal root by two Newton steps from the estimate and the root
// from it with one correction, each within an ulp or two of FP64 (Q and R are
// rounded to FP32 once afterwards).
__device__ __forceinline__ bool norm_of(double s, double &nrm, double &inv)
{
    const unsigned e = (unsigned)__builtin_amdgcn_readfirstlane(__double2hiint(s)) >> 20;
    double y = __builtin_amdgcn_rsq(s);
    const double h = 0.5 * s;
    y = y * fma(-h * y, y, 1.5);
    y = y * fma(-h * y, y, 1.5);
    const double g = s * y;
    nrm = fma(fma(-g, g, s), 0.5 * y, g);
    inv = y;
    if (__builtin_expect(e - 23u < 2000u, 1)) return true;  // positive, 2^-1000 <= s < 2^1000
    nrm = sqrt(s);
    const bool ok = (nrm > 0.0) && (nrm < INFINITY);
    inv = ok ? 1.0 / nrm : 0.0;
    return ok;
}

// Block MGS as a pipeline of waves.  Wave v holds its kCPW consecutive columns
// in registers (lane l: rows l, l + 64, ...), applies q_0, q_1, ... to them as
// the earlier waves publish them in LDS, then normalises its own columns one
// after another (three of four hand-overs stay inside the wave) and publishes
// each as soon as it is final.  A wave waits only for waves with smaller
// numbers, by polling the count of published columns, so no wave is held at a
// barrier by one that is not on the chain.  The operations on every column and
// their order are those of plain MGS: for k = 0, 1, ...: d = q_k . a,
// a -= q_k d.
// Bound: the serial chain of w norms (dot, wave sum, square root, reciprocal):
// 12 us for 256 x 32, where one barrier per column and a column dealt to
// every eighth wave took 24 us (same bits; FP64 sums 21 and 30 us).
// RPL: rows per lane, 4 for blocks of up to 256 rows, 5 with a merged tail.
template <int KC> constexpr int kThreads = 64 * KC / kCPW;
template <typename Acc, int RPL, int KC>
__device__ __forceinline__ void mgs_block_body(int m, int w, float *A, int64_t lda, float *Rout, int64_t ldr,
                                               int bh, int nblk, int *status, const int b)
{
    __shared__ float qs[KC][64 * RPL];
    __shared__ float Rs[KC][KC + 1];
    __shared__ int published;

    const int r0 = b * bh;
    // The last block takes every remaining row (a tail shorter than w is merged).
    const int mm = (b == nblk - 1) ? (m - r0) : bh;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int c0 = kCPW * wave;
    auto *Ab = gmem(A) + r0;  // global view (the grouped kernel reads A from a table)

    // Loads from clamped in-bounds addresses, selected afterwards, so that all
    // of them issue before the first wait.
    float a[kCPW][RPL];
#pragma unroll
    for (int c = 0; c < kCPW; ++c) {
        const int jc = min(c0 + c, w - 1);
#pragma unroll
        for (int t = 0; t < RPL; ++t) a[c][t] = Ab[min(lane + 64 * t, mm - 1) + (int64_t)jc * lda];
    }
    if (threadIdx.x == 0) published = 0;
#pragma unroll
    for (int c = 0; c < kCPW; ++c)
#pragma unroll
        for (int t = 0; t < RPL; ++t)
            if (!(c0 + c < w && lane + 64 * t < mm)) a[c][t] = 0.0f;
    __syncthreads();

    // Columns C0 .. of this wave: d = q . a, a -= q d.
    auto dot = [&](const float (&q)[RPL], int c) -> Acc {
        Acc d = (Acc)q[0] * (Acc)a[c][0];
#pragma unroll
        for (int t = 1; t < RPL; ++t) d = fma((Acc)q[t], (Acc)a[c][t], d);
        return d;
    };
    auto subtract = [&](const float (&q)[RPL], int c, Acc d) {
#pragma unroll
        for (int t = 0; t < RPL; ++t) {
            a[c][t] = (float)fma(-(Acc)q[t], d, (Acc)a[c][t]);
            asm volatile("" : "+v"(a[c][t]));  // here, not sunk below the stores that follow
        }
    };
    auto norm_terms = [&](int c) -> Acc {
        Acc s = (Acc)a[c][1] * (Acc)a[c][1];
        s = fma((Acc)a[c][0], (Acc)a[c][0], s);
#pragma unroll
        for (int t = 2; t < RPL; ++t) s = fma((Acc)a[c][t], (Acc)a[c][t], s);
        return s;
    };
    // All of them by q.
    auto project = [&](const float (&q)[RPL], Acc *d) {
        Acc v[kCPW];
#pragma unroll
        for (int c = 0; c < kCPW; ++c) v[c] = dot(q, c);
        wave_sums(v);
#pragma unroll
        for (int c = 0; c < kCPW; ++c) {
            subtract(q, c, v[c]);
            d[c] = v[c];
        }
    };
    // Columns C0 .. by q, the next pivot's column C0 first: its squared norm is
    // summed together with the other columns' products.  Returns that norm.
    auto project_next = [&](const float (&q)[RPL], auto first, Acc *d) -> Acc {
        constexpr int C0 = decltype(first)::value, N = kCPW - C0;
        Acc h[1] = {dot(q, C0)};
        wave_sums(h);
        subtract(q, C0, h[0]);
        d[C0] = h[0];
        Acc v[N];
        v[0] = norm_terms(C0);
#pragma unroll
        for (int c = 1; c < N; ++c) v[c] = dot(q, C0 + c);
        wave_sums(v);
#pragma unroll
        for (int c = 1; c < N; ++c) {
            subtract(q, C0 + c, v[c]);
            d[C0 + c] = v[c];
        }
        return v[0];
    };
    auto load_q = [&](float (&q)[RPL], int k) {
#pragma unroll
        for (int t = 0; t < RPL; ++t) q[t] = qs[k][lane + 64 * t];
    };
    auto count = [&]() { return __hip_atomic_load(&published, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
    // The count and, behind it in the same LDS queue, q_k: valid when the count
    // says so.
    auto peek = [&](float (&q)[RPL], int k) -> int {
        const int n = count();
        asm volatile("" ::: "memory");
        load_q(q, k);
        asm volatile("" ::: "memory");
        return n;
    };
    // q_k, waiting for it: the wave whose turn is next reads it with every
    // look at the count, the ones behind it only look.
    auto take = [&](float (&q)[RPL], int k) {
        if (c0 - k > kCPW)
            while (__builtin_amdgcn_readfirstlane(count()) <= k) {}
        asm volatile("" ::: "memory");
        while (__builtin_amdgcn_readfirstlane(peek(q, k)) <= k) {}
    };

    Acc s0 = 0;
    if (c0 < w && c0 > 0) {
        float q[RPL], qn[RPL];
        take(q, 0);
        for (int k = 0; k + 1 < c0; ++k) {
            const int n = peek(qn, k + 1);
            Acc d[kCPW];
            project(q, d);
            if (lane == 0) {
#pragma unroll
                for (int c = 0; c < kCPW; ++c) Rs[k][c0 + c] = (float)d[c];
            }
            if (__builtin_amdgcn_readfirstlane(n) <= k + 1) take(qn, k + 1);
#pragma unroll
            for (int t = 0; t < RPL; ++t) q[t] = qn[t];
        }
        __builtin_amdgcn_s_setprio(3);
        Acc d[kCPW];
        s0 = project_next(q, std::integral_constant<int, 0>(), d);
        if (lane == 0) {
#pragma unroll
            for (int c = 0; c < kCPW; ++c) Rs[c0 - 1][c0 + c] = (float)d[c];
        }
    } else if (c0 == 0) {
        Acc v[1] = {norm_terms(0)};
        wave_sums(v);
        s0 = v[0];
    }
    // This wave's own columns, ahead of the waves that only follow; R's
    // entries and Q are stored when the chain has left this wave.
    __builtin_amdgcn_s_setprio(3);
    Acc r[kCPW][kCPW];
    bool bad = false;
    auto own = [&](auto col, Acc s) -> Acc {
        constexpr int I = decltype(col)::value;
        const int k = c0 + I;
        if (k >= w) return s;
        Acc nrm, inv;
        const bool ok = norm_of(s, nrm, inv);
        bad |= !ok;
        r[I][I] = ok ? nrm : (Acc)0;
#pragma unroll
        for (int t = 0; t < RPL; ++t) {
            a[I][t] = (float)((Acc)a[I][t] * inv);
            qs[k][lane + 64 * t] = a[I][t];
        }
        // A wave's LDS operations are carried out in order: whoever sees the
        // count sees q_k.
        asm volatile("" ::: "memory");
        if (lane == 0) __hip_atomic_store(&published, k + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if constexpr (I + 1 < kCPW) return project_next(a[I], std::integral_constant<int, I + 1>(), r[I]);
        else return s;
    };
    static_assert(kCPW == 4, "four columns per wave");
    const Acc s1 = own(std::integral_constant<int, 0>(), s0);
    const Acc s2 = own(std::integral_constant<int, 1>(), s1);
    const Acc s3 = own(std::integral_constant<int, 2>(), s2);
    own(std::integral_constant<int, 3>(), s3);
    __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int i = 0; i < kCPW; ++i) {
        if (c0 + i >= w) break;
        if (lane == 0) {
#pragma unroll
            for (int c = i; c < kCPW; ++c) Rs[c0 + i][c0 + c] = (float)r[i][c];
        }
#pragma unroll
        for (int t = 0; t < RPL; ++t)
            if (lane + 64 * t < mm) Ab[lane + 64 * t + (int64_t)(c0 + i) * lda] = a[i][t];
    }
    if (bad && lane == 0 && status) atomicOr(status, 1);
    __syncthreads();
    // R block (w x w, zeros below the diagonal) at rows b*w of Rout.
    auto *Rb = gmem(Rout) + (int64_t)b * w;
    for (int i = threadIdx.x; i < w * w; i += kThreads<KC>) {
        const int x = i % w, y = i / w;
        Rb[x + (int64_t)y * ldr] = (x <= y) ? Rs[x][y] : 0.0f;
    }
}

template <typename Acc, int RPL, int KC>
__global__ __launch_bounds__(kThreads<KC>) void mgs_block_kernel(int m, int w, float *A, int lda, float *Rout,
                                                                 int ldr, int bh, int nblk, int *status)
{
    mgs_block_body<Acc, RPL, KC>(m, w, A, lda, Rout, ldr, bh, nblk, status, blockIdx.x);
}

template <typename Acc>
__global__ __launch_bounds__(kThreads<kCols>) void mgs_block_grouped_kernel(const PanelArgs *args, const int2 *tasks)
{
    const int2 t = tasks[blockIdx.x];
    const PanelArgs a = args[t.x];
    mgs_block_body<Acc, 5, kCols>(a.m, a.w, a.A, a.lda, a.W, a.ldw, kPanelBlockRows, a.nblk, a.status, t.y);
}

// f(columns) with the narrowest of the widths that the kernels come in.
template <typename F> void by_width(int w, F f)
{
    if (w <= 8) f(std::integral_constant<int, 8>());
    else if (w <= 16) f(std::integral_constant<int, 16>());
    else f(std::integral_constant<int, kCols>());
}

// Rows per lane of the largest block: 4 unless a short tail is merged.
template <typename Acc>
void launch_mgs(hipStream_t s, int m, int w, float *A, int lda, float *Rout, int ldr, int bh, int nblk, int *status)
{
    by_width(w, [&](auto cols) {
        constexpr int KC = decltype(cols)::value;
        if (m - (nblk - 1) * bh <= 256)
            hipLaunchKernelGGL((mgs_block_kernel<Acc, 4, KC>), dim3(nblk), dim3(kThreads<KC>), 0, s, m, w, A, lda, Rout,
                               ldr, bh, nblk, status);
        else
            hipLaunchKernelGGL((mgs_block_kernel<Acc, 5, KC>), dim3(nblk), dim3(kThreads<KC>), 0, s, m, w, A, lda, Rout,
                               ldr, bh, nblk, status);
    });
}

// A_b <- A_b * W_b for every row block b, W_b = rows b*w .. b*w+w-1 of the
// stacked factor (ld ldw).  Each thread owns whole rows, so the in-place
// update never reads a value another thread writes (the reference relies on
// an aliased batched Sgemm here, QR/panel.cu:97-102).
template <typename Acc>
__device__ __forceinline__ void tsqr_apply_body(int m, int w, float *A, int64_t lda, const float *W, int64_t ldw,
                                                int bh, int nblk, const int b)
{
    __shared__ float Ws[kCols][kCols];
    const int r0 = b * bh;
    const int mm = (b == nblk - 1) ? (m - r0) : bh;
    const auto *Wb = gmem(W) + (int64_t)b * w;
    for (int i = threadIdx.x; i < w * w; i += 256) {
        const int x = i % w, y = i / w;
        Ws[x][y] = Wb[x + (int64_t)y * ldw];
    }
    __syncthreads();
    auto *Ab = gmem(A) + r0;
    for (int row = threadIdx.x; row < mm; row += 256) {
        // Unconditional loads (clamped column) so all of them are in flight at once.
        float v[kCols];
#pragma unroll
        for (int k = 0; k < kCols; ++k) v[k] = Ab[row + (int64_t)min(k, w - 1) * lda];
#pragma unroll
        for (int k = 0; k < kCols; ++k)
            if (k >= w) v[k] = 0.0f;
#pragma unroll 4
        for (int j = 0; j < w; ++j) {
            Acc s = 0;
#pragma unroll
            for (int k = 0; k < kCols; ++k)
                if (k < w) s += (Acc)v[k] * (Acc)Ws[k][j];
            Ab[row + (int64_t)j * lda] = (float)s;
        }
    }
}

template <typename Acc>
__global__ __launch_bounds__(256) void tsqr_apply_grouped_kernel(const PanelArgs *args, const int2 *tasks)
{
    const int2 t = tasks[blockIdx.x];
    const PanelArgs a = args[t.x];
    tsqr_apply_body<Acc>(a.m, a.w, a.A, a.lda, a.W, a.ldw, kPanelBlockRows, a.nblk, t.y);
}

// The same product for a panel of its own launch, in the same order of
// summation over k (the same bits).  Two layouts: CG = 4 gives a workgroup 64
// rows, each wave a quarter of the output columns (a 16384-row panel then
// covers the chip); CG = 1 gives it a whole 256-row block, each wave 64 rows
// and every column (an eighth of the W traffic per row, no barrier between
// reading and writing A: for panels with a block for every CU).
// FUSED: W is itself still to be multiplied by its rows of the next level's
// Q, W2 (blocks of 256 rows of W, W2's rows b2 w ..); the workgroup forms its
// w x w product W_b W2_b2 first, rounded to FP32 as the separate launch would
// store it, which saves that launch and a round trip of the stack.
// W is kept k-contiguous in LDS and read as broadcast 16-byte vectors, all of
// A's loads are in flight before the first wait: 16384 x 32 takes 7.1 us with
// the next level's product in it and 4.9 us without, where two launches took
// 14.5 us each with runtime-strided staging and scalar LDS reads.
template <typename Acc, int CG, bool FUSED, int KC>
__global__ __launch_bounds__(256) void tsqr_apply_kernel(int m, int w, float *A, int lda, const float *W, int ldw,
                                                         int nblk, const float *W2, int ldw2, int nblk2)
{
    constexpr int bh = kPanelBlockRows;
    __shared__ __attribute__((aligned(16))) Acc Ws[KC][KC];  // [j][k]
    __shared__ float S1[FUSED ? KC : 1][KC + 1], S2[FUSED ? 2 : 1][FUSED ? KC : 1][KC + 1];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = (CG == 4) ? min((int)blockIdx.x * 64 / bh, nblk - 1) : (int)blockIdx.x;
    const int rend = (b == nblk - 1) ? m : (b + 1) * bh;  // rows of the block end here
    const int row0 = (CG == 4) ? (int)blockIdx.x * 64 : b * bh + 64 * wv;

    float v[KC];
    auto load_rows = [&](int r0) {
        const float *src = A + min(r0 + lane, rend - 1);
#pragma unroll
        for (int k = 0; k < KC; ++k) v[k] = src[(int64_t)min(k, w - 1) * lda];
    };
    if (CG == 4 || row0 < rend) load_rows(row0);

    // Thread (x, y0) holds entries (x, y0 + YS u) of the w x w factors (KC = 8:
    // some hold none).
    constexpr int YS = 256 / KC, NU = (KC + YS - 1) / YS;
    const int x = tid & (KC - 1), y0 = tid >> (KC == 8 ? 3 : KC == 16 ? 4 : 5);
    if constexpr (!FUSED) {
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int y = y0 + YS * u;
            const float t = W[(int64_t)b * w + min(x, w - 1) + (int64_t)min(y, w - 1) * ldw];
            if (KC >= YS || y < KC) Ws[y][x] = (x < w && y < w) ? (Acc)t : (Acc)0;
        }
    } else {
        // Rows g = b w + i of W lie in block min(g / 256, nblk2 - 1) of the
        // next level: one block, or two where w does not divide 256.
        const int b0 = min(b * w / bh, nblk2 - 1), b1 = min((b * w + w - 1) / bh, nblk2 - 1);
        float t1[NU], t2[NU], t3[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int xc = min(x, w - 1), yc = min(y0 + YS * u, w - 1);
            t1[u] = W[(int64_t)b * w + xc + (int64_t)yc * ldw];
            t2[u] = W2[(int64_t)b0 * w + xc + (int64_t)yc * ldw2];
            t3[u] = W2[(int64_t)b1 * w + xc + (int64_t)yc * ldw2];
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int y = y0 + YS * u;
            if (KC >= YS || y < KC) {
                S1[x][y] = t1[u];
                S2[0][x][y] = t2[u];
                S2[1][x][y] = t3[u];
            }
        }
        __syncthreads();
        const int sel = (b * w + x) / bh > b0 && b1 > b0 ? 1 : 0;
        Acc s[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) s[u] = (Acc)0;
        const int yc = KC < YS ? min(y0, KC - 1) : y0;
#pragma unroll 8
        for (int k = 0; k < w; ++k) {
            const Acc l = (Acc)S1[x][k];
#pragma unroll
            for (int u = 0; u < NU; ++u) s[u] = fma(l, (Acc)S2[sel][k][yc + YS * u], s[u]);
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int y = y0 + YS * u;
            if (KC >= YS || y < KC) Ws[y][x] = (x < w && y < w) ? (Acc)(float)s[u] : (Acc)0;
        }
    }
#pragma unroll
    for (int k = 0; k < KC; ++k)
        if (k >= w) v[k] = 0.0f;
    // With CG = 4 this also orders every wave's reads of the tile before any
    // wave's writes to it.
    __syncthreads();

    constexpr int PW = KC / CG;  // columns of a wave
    constexpr int NJ = PW < 4 ? PW : 4, VW = 16 / sizeof(Acc);  // columns in flight, values of W per LDS read
    typedef Acc vec_t __attribute__((ext_vector_type(VW)));
    auto product = [&](int r0) {
        const int row = r0 + lane;
        const int jbeg = (CG == 4) ? PW * wv : 0, jend = min(w, jbeg + PW);
        for (int j = jbeg; j < jend; j += NJ) {
            Acc s[NJ];
#pragma unroll
            for (int c = 0; c < NJ; ++c) s[c] = (Acc)0;
#pragma unroll
            for (int k = 0; k < KC; k += VW) {
                vec_t wk[NJ];
#pragma unroll
                for (int c = 0; c < NJ; ++c) wk[c] = *(const vec_t *)&Ws[j + c][k];
#pragma unroll
                for (int e = 0; e < VW; ++e)
#pragma unroll
                    for (int c = 0; c < NJ; ++c) s[c] = fma((Acc)v[k + e], wk[c][e], s[c]);
            }
            if (row < rend) {
#pragma unroll
                for (int c = 0; c < NJ; ++c)
                    if (j + c < w) A[row + (int64_t)(j + c) * lda] = (float)s[c];
            }
        }
    };
    if constexpr (CG == 4) {
        product(row0);
    } else {
        for (int r0 = row0; r0 < rend; r0 += 256) {  // a second round only for a merged tail
            if (r0 != row0) {
                load_rows(r0);
#pragma unroll
                for (int k = 0; k < KC; ++k)
                    if (k >= w) v[k] = 0.0f;
            }
            product(r0);
        }
    }
}

// A_b <- A_b W_b (W2 given: W_b W2_b2 in place of W_b) over the m x w panel.
template <typename Acc>
void launch_apply(hipStream_t s, int m, int w, float *A, int lda, const float *W, int ldw, int nblk, const float *W2,
                  int ldw2, int nblk2)
{
    // A workgroup per block once that gives every CU one: below, the four
    // times finer grid hides the latency of the loads (16384 rows: 7.1 us).
    const bool whole = nblk >= 256;
    const dim3 grid(whole ? nblk : (m + 63) / 64);
    by_width(w, [&](auto cols) {
#define LATER_APPLY(CG, F)                                                                                         \
    hipLaunchKernelGGL((tsqr_apply_kernel<Acc, CG, F, decltype(cols)::value>), grid, dim3(256), 0, s, m, w, A, lda, W, \
                       ldw, nblk, W2, ldw2, nblk2)
        if (whole && W2) LATER_APPLY(1, true);
        else if (whole) LATER_APPLY(1, false);
        else if (W2) LATER_APPLY(4, true);
        else LATER_APPLY(4, false);
#undef LATER_APPLY
    });
}

struct Blocks {
    int nblk;
};

Blocks plan_blocks(int m, int w)
{
    const int bh = kPanelBlockRows;
    int nb = m / bh, r = m % bh;
    if (nb == 0) return {1};
    return {nb + ((r >= w) ? 1 : 0)};
}

} // namespace

int panel_blocks(int m, int w) { return plan_blocks(m, w).nblk; }

int mgs_grouped(hipStream_t s, bool fp64, const PanelArgs *args, const int2 *tasks, int ntasks)
{
    if (ntasks <= 0) return LATER_OK;
    if (fp64) hipLaunchKernelGGL(mgs_block_grouped_kernel<double>, dim3(ntasks), dim3(kThreads<kCols>), 0, s, args, tasks);
    else hipLaunchKernelGGL(mgs_block_grouped_kernel<float>, dim3(ntasks), dim3(kThreads<kCols>), 0, s, args, tasks);
    HIP_OK(hipGetLastError());
    return LATER_OK;
}

int apply_grouped(hipStream_t s, bool fp64, const PanelArgs *args, const int2 *tasks, int ntasks)
{
    if (ntasks <= 0) return LATER_OK;
    if (fp64) hipLaunchKernelGGL(tsqr_apply_grouped_kernel<double>, dim3(ntasks), dim3(256), 0, s, args, tasks);
    else hipLaunchKernelGGL(tsqr_apply_grouped_kernel<float>, dim3(ntasks), dim3(256), 0, s, args, tasks);
    HIP_OK(hipGetLastError());
    return LATER_OK;
}

int64_t panel_work_floats_any(int m)
{
    // A ragged leaf can be narrower than 32 columns; its tree can need a
    // stack where the 32-wide tree has none (a short tail is merged only when
    // it has fewer rows than the panel has columns).
    int64_t mx = 0;
    for (int w = 1; w <= kCols; ++w) {
        const int64_t f = panel_work_floats(m, w);
        if (f > mx) mx = f;
    }
    return mx;
}

int64_t panel_work_floats(int m, int w)
{
    if (w < 1) w = 1;
    int64_t tot = 0;
    int64_t mm = m;
    for (;;) {
        Blocks p = plan_blocks((int)mm, w);
        if (p.nblk <= 1) break;
        tot += (int64_t)p.nblk * w * w;
        mm = (int64_t)p.nblk * w;
    }
    return tot;
}

namespace {

// The MGS launches of the tree below an m x w panel; *stack, *ldst: its
// level's stacked factors, whose Q rows the panel's blocks are multiplied by
// (none when the panel is a single block).  apply_here: multiply the panel
// too; otherwise the caller folds that product into its own.
int tsqr_level(hipStream_t s, int m, int w, float *A, int lda, float *R, int ldr, float *work, int64_t lwork,
               bool fp64, int *status, int *launches, bool apply_here, const float **stack_out, int *ldst_out)
{
    *stack_out = nullptr;
    *ldst_out = 0;
    const Blocks p = plan_blocks(m, w);
    const int bh = kPanelBlockRows;
    if (p.nblk <= 1) {
        if (m > kMaxRows) return LATER_ERR_SHAPE;
        if (fp64) launch_mgs<double>(s, m, w, A, lda, R, ldr, bh, 1, status);
        else launch_mgs<float>(s, m, w, A, lda, R, ldr, bh, 1, status);
        if (launches) ++*launches;
        HIP_OK(hipGetLastError());
        return LATER_OK;
    }
    const int ldst = p.nblk * w;
    const int64_t need = (int64_t)ldst * w;
    if (lwork < need) return LATER_ERR_WORKSPACE;
    float *stack = work;
    const int tok = prof_start(s);
    if (fp64) launch_mgs<double>(s, m, w, A, lda, stack, ldst, bh, p.nblk, status);
    else launch_mgs<float>(s, m, w, A, lda, stack, ldst, bh, p.nblk, status);
    prof_stop(tok, s, PROF_PANEL, 4.0 * m * w * w, 8.0 * m * w + 4.0 * ldst * w);
    if (launches) ++*launches;
    HIP_OK(hipGetLastError());
    // Levels are applied in pairs: this one's product takes the next one's in.
    const float *stack2 = nullptr;
    int ldst2 = 0;
    const int rc = tsqr_level(s, ldst, w, stack, ldst, R, ldr, work + need, lwork - need, fp64, status, launches,
                              !apply_here, &stack2, &ldst2);
    if (rc) return rc;
    *stack_out = stack;
    *ldst_out = ldst;
    if (!apply_here) return LATER_OK;
    const int nblk2 = plan_blocks(ldst, w).nblk;
    if (fp64) launch_apply<double>(s, m, w, A, lda, stack, ldst, p.nblk, stack2, ldst2, nblk2);
    else launch_apply<float>(s, m, w, A, lda, stack, ldst, p.nblk, stack2, ldst2, nblk2);
    if (launches) ++*launches;
    HIP_OK(hipGetLastError());
    return LATER_OK;
}

} // namespace

int panel_tsqr(hipStream_t s, int m, int w, float *A, int lda, float *R, int ldr, float *work,
               int64_t lwork, bool fp64, int *status, int *launches)
{
    if (w < 1 || w > kCols || m < w) return LATER_ERR_SHAPE;
    const float *stack;
    int ldst;
    return tsqr_level(s, m, w, A, lda, R, ldr, work, lwork, fp64, status, launches, true, &stack, &ldst);
}

// The batched QR's kernel for FP32 products and matrices of up to 256 columns:
// a persistent 512-thread workgroup per CU, each taking whole matrices from
// the queue.
//
// Per matrix (m x n, column-major, in place: A <- Q, R n x n), left-looking
// block Gram-Schmidt with reorthogonalisation (BCGS2) over panels P of 64
// columns, with all earlier columns Q (a multiple of 64) at once.  A panel is
// three sweeps over the rows, 32 at a time, instead of the four that a
// projection and an update per pass would take:
//   S1 = Q^T P;    P -= Q S1, S2 = Q^T P;    P -= Q S2, G = P^T P
// then P = Q_P R_PP by Cholesky QR on G (FP64, chol_dev.h) and one more sweep
// P <- P R^{-1}.  Without reorthogonalisation P is projected out of Q's
// 64-column blocks one after another, a block's update and the next one's
// projection in a sweep:
//   S1 = Q1^T P;    P -= Q1 S1, S2 = Q2^T P;    ...;    P -= Qb Sb, G = P^T P
// (block by block the loss of orthogonality grows with kappa 2^-24, all at once
// with kappa^2 2^-24: 515 x 256 of kappa 1e4 2.2e-3 and 0.32; 1024 matrices of up
// to 4096 x 256 take 2.57 and 2.51 ms).
// That is all for a panel whose factor is well conditioned: with an FP64 Gram
// of FP32 data one Cholesky QR leaves kappa^2 2^-53, far below the rounding of
// Q's entries to FP32, and what is left of Q in P grows by kappa at most (kappa
// of the panel with its columns scaled to norm 1: neither the factor nor a
// projection depends on their norms).  A panel with a bad pivot or kappa (its
// Frobenius bound, condition2) above a limit is factored again: 2 w where
// reorthogonalisation has left Q's rounding in P to grow, and then the
// normalised panel is projected out of Q once more; 2^12 where there is no Q or
// one projection only, and kappa^2 2^-53 alone counts.  (At 4 w a 4000 x 256
// matrix of kappa 1e3 is left 6.8e-6 from orthogonal, 4.4e-6 on the narrow kernel
// and 2.3e-6 here; at 1.5 w near-square batches pay, 160 x 160 11% over the narrow
// kernel.  Unscaled and at 4 w throughout, 512 matrices of 500 x 96 with columns
// of magnitude 1 and 1000 took 755 us, 420 now; 2048 of 64 x 64 722, 425 now.)
//
// A chunk of 32 rows of [Q P] is staged in LDS column by column (stride 36:
// 16-byte reads of 16 columns and 4-byte reads of 16 rows of every fourth
// column both cover the banks once), two buffers, the loads of the two chunks
// behind in registers.  All products run on v_mfma_f32_16x16x4f32: its k index is
// permuted within each 16 (lane group g takes k = 16 t + 4 g + u in step u)
// so that the operand that lies along k is one 16-byte read for four steps.
// Bound: the matrix cores of one CU (FP32 4 m n^2 at 614 GFLOP/s, FP64 Gram and
// apply at 258; 57% busy on a 4096 x 256 matrix, the rest the barriers between
// the phases of a chunk), and the largest matrix of a batch on its workgroup:
// 4096 x 256 takes 3.45 ms, 9.3 on the narrow kernel; 1024 matrices of up to
// that size 3.7 ms, 9.9 there.
#include <type_traits>

#include "batch_wg.h"
#include "chol_dev.h"
#include "common.h"

namespace {

constexpr int kT = 512;                      // threads: eight waves, two per SIMD
constexpr int kB = 64;                       // panel columns
constexpr int kR = 32;                       // rows per chunk
constexpr int kLdC = kR + 4;                 // column stride of a chunk (floats)
constexpr int kMaxQ = kWideCols - kB;        // earlier columns of the last panel
constexpr int kLdS = kMaxQ + 4;              // column stride of S (floats)
constexpr int kTiles = kMaxQ / 64;           // 16-column tiles of Q per wave
constexpr int kLoads = kWideCols * kR / 4 / kT;  // 16-byte loads per thread and chunk

// LDS (bytes): S (column n at n kLdS floats), then two chunks; over them, while
// a factor is formed, Gs, Rs and Ris; while it is applied, R^{-1} at the start
// and the chunks behind it; the saved R1 and the pivot bounds apart.
constexpr int kSBytes = kB * kLdS * 4;
constexpr int kChunkBytes = kWideCols * kLdC * 4;
constexpr int kGs = kB * (kB + 1) * 8, kMat = kB * kB * 8;
constexpr int kOffR1 = kSBytes + 2 * kChunkBytes;
constexpr int kLds = kOffR1 + kMat + kB * 8;
static_assert(kGs + 2 * kMat <= kOffR1 && kMat + 2 * kChunkBytes <= kOffR1, "regions before R1");
static_assert(kMaxQ * kB * 4 <= 2 * kChunkBytes, "the waves' half sums of S fit the chunk buffers");
static_assert(4 * 3 * 4 * 64 * 8 <= 2 * kChunkBytes && kGs <= kSBytes, "and those of the Gram; Gs over S");
static_assert(kLds + 1024 <= 163840, "LDS");

typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

// What a sweep reads: K earlier columns Q, the first ku of which it updates with
// and those from kp on it projects on, and the panel P.
struct Panel {
    int m, w;             // rows, columns of P
    int K, ku, kp;        // multiples of 64
    const float *Q, *P;
    int64_t lda;
};

// Columns c0 .. c0 + 64 sets - 1 of [Q P], `subs` groups of 32 rows at a time: a
// chunk fills its four 64-column slots of the buffer whatever the window's
// width, so the bytes in flight do not shrink with it.

struct Window {
    int c0, sets, subs;
    __device__ __forceinline__ Window(const Panel &p, bool with_q)
    {
        c0 = with_q ? 0 : p.K;
        sets = with_q ? p.K / 64 + 1 : 1;
        subs = sets == 1 ? 4 : sets == 2 ? 2 : 1;
    }
    // LDS offset (floats) of 32-row group `sub`, column c.
    __device__ __forceinline__ int at(int sub, int c) const { return (64 * sets * sub + c) * kLdC; }
};

// This thread's part of a chunk: slot i holds rows 4 (t % 8) .. + 3 of the
// column t / 8 of its set and row group.
struct Part {
    floatx4u v[kLoads];
};

// The window's chunks through the two LDS buffers, two more in registers;
// f(chunk, r0, full) runs between the barriers that make a chunk visible and
// free its buffer (full: all of its rows are inside the matrix).  Every slot is
// one 16-byte load at dword alignment, without a branch: a branch with loads of
// its own in this loop makes the compiler wait for every load in flight where
// the paths join, which costs a memory latency per chunk.  So columns past the
// panel are clamped, and rows past the end too: the last rows' vector starts at
// row m - 4 and is shifted when it is stored (m >= 4).
template <typename F> __device__ __forceinline__ void for_chunks(const Panel &p, const Window &x, float *buf, F f)
{
    typedef const __attribute__((address_space(1))) float *gptr;
    const int t = threadIdx.x, nc = p.K + p.w;
    const int rows = kR * x.subs, n = (p.m + rows - 1) / rows, nfull = p.m / rows;
    gptr src[kLoads];
    int rg[kLoads];
    bool in[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int sub = i / x.sets, c = x.c0 + (t >> 3) + 64 * (i - sub * x.sets);
        rg[i] = kR * min(sub, x.subs - 1) + 4 * (t & 7);
        in[i] = c < nc && sub < x.subs;
        src[i] = c < p.K ? gmem(p.Q) + (int64_t)c * p.lda : gmem(p.P) + (int64_t)(min(c, nc - 1) - p.K) * p.lda;
    }
    const bool ragged = p.w < kB;
    auto load = [&](Part &part, int i) {
#pragma unroll
        for (int q = 0; q < kLoads; ++q)
            part.v[q] = *(const __attribute__((address_space(1))) floatx4u *)(src[q] + min(i * rows + rg[q], p.m - 4));
    };
    auto store = [&](const Part &part, float *C, int i) {
#pragma unroll
        for (int q = 0; q < kLoads; ++q) {
            floatx4 y = floatx4(part.v[q]);
            if (i >= nfull) {
                const int s = i * rows + rg[q] - (p.m - 4);  // > 0: rows s .. 3 of the vector, then zeros
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float z = s <= 0 ? y[e] : 0.0f;
#pragma unroll
                    for (int d = 1; d < 4 - e; ++d) z = s == d ? y[e + d] : z;
                    y[e] = z;
                }
            }
            if (ragged && !in[q]) y = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            *(floatx4 *)(C + ((t >> 3) + 64 * q) * kLdC + 4 * (t & 7)) = y;
        }
    };
    Part a, b;
    load(a, 0);
    load(b, 1);
    auto step = [&](Part &part, int i) {
        float *C = buf + (i & 1) * (kWideCols * kLdC);
        store(part, C, i);
        __syncthreads();  // chunk i is there, and chunk i - 1 has been read
        load(part, i + 2);
        f(C, i * rows, i < nfull);
    };
    for (int i = 0; i < n; i += 2) {
        step(a, i);
        if (i + 1 < n) step(b, i + 1);
    }
    __syncthreads();
}

// Sixteen k, the last of each lane group first.
__device__ __forceinline__ floatx4 mfma4_down(floatx4 a, floatx4 b, floatx4 c)
{
#pragma unroll
    for (int u = 3; u >= 0; --u) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b[u], c, 0, 0, 0);
    return c;
}

// Gram tile q of wave position v4 (0 .. 3): the ten 16 x 16 tiles (x <= y) of a
// 64 x 64 Gram in row order, three, three, two and two.
__device__ __forceinline__ bool gram_tile(int v4, int q, int &x, int &y)
{
    const int first = v4 < 2 ? 3 * v4 : 2 * v4 + 2, count = v4 < 2 ? 3 : 2;
    const int e = min(first + q, 9);
    x = e < 4 ? 0 : e < 7 ? 1 : e < 9 ? 2 : 3;
    y = x + e - (x == 0 ? 0 : x == 1 ? 4 : x == 2 ? 7 : 9);
    return q < count;
}

// One sweep over the rows of [Q P].  update: P -= Q S over Q's first ku columns
// (S in LDS; P written back); then of the updated rows, project: S' = Q^T P over
// S, for Q's columns from kp on, or otherwise G = P^T P to Gs (row stride 65,
// identity outside w x w).  Wave v: row half v / 4 of a chunk; of the products,
// Q tiles v % 4 + 4 i against the four tiles
// of P, tile v % 4 of P in the update, the Gram tiles of gram_tile.  (One
// instance per kind of sweep: with both results' accumulators live, registers
// spill into the loop, and a reload waits for the loads in flight.)
template <bool update, bool project>
__device__ __forceinline__ void sweep(const Panel &p, float *P, char *lds)
{
    constexpr bool gram = !project;
    float *S = (float *)lds, *buf = (float *)(lds + kSBytes);
    const int lane = threadIdx.x & 63, v = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, g = lane >> 4, v4 = v & 3, h = 16 * (v >> 2);
    const int ku = p.ku, kp = p.kp, qt = (p.K - kp) / 64;
    floatx4 acc[kTiles][4];
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    doublex4 gt[3];
    int gx[3], gy[3];
    bool gok[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        gt[q] = doublex4{0.0, 0.0, 0.0, 0.0};
        gok[q] = gram_tile(v4, q, gx[q], gy[q]);
    }
    const Window x(p, update || project);
    const int pc = update || project ? p.K : 0;  // P's first column in the window
    for_chunks(p, x, buf, [&](float *C, int r0, bool full) {
        if (update) {
#pragma unroll 1
            for (int sub = 0; sub < x.subs; ++sub) {
                // D[n][row] += S[k][n] Q[row][k]: lane n = l % 16 of S, row l % 16
                // of Q; the operands of the next 32 k are read ahead.  The sum
                // runs from the last column of Q to the first: where columns
                // share a direction the first carry the large terms, and the
                // rest are then added before them, at their own magnitude
                // (columns with a common mean, 515 x 256: backward error 2.2e-7
                // in ascending order, 5.8e-8 so; uniform ones the same).
                const float *sn = S + (16 * v4 + li) * kLdS + 4 * g, *qr = C + x.at(sub, 4 * g) + h + li;
                float *pr = C + x.at(sub, pc + 16 * v4 + 4 * g) + h + li;
                floatx4 d = floatx4{0.0f, 0.0f, 0.0f, 0.0f}, sv[2], qv[2], sw[2], qw[2], old;
#pragma unroll
                for (int e = 0; e < 4; ++e) old[e] = pr[e * kLdC];
                auto fetch = [&](floatx4 (&sx)[2], floatx4 (&qx)[2], int k) {
#pragma unroll
                    for (int y = 0; y < 2; ++y) {
                        sx[y] = *(const floatx4 *)(sn + k + 16 * y);
#pragma unroll
                        for (int u = 0; u < 4; ++u) qx[y][u] = qr[(k + 16 * y + u) * kLdC];
                    }
                };
                fetch(sv, qv, ku - 32);
#pragma unroll 1
                for (int k = ku - 64; k >= 0; k -= 64) {
                    fetch(sw, qw, k);
                    d = mfma4_down(sv[1], qv[1], d);
                    d = mfma4_down(sv[0], qv[0], d);
                    fetch(sv, qv, max(k - 32, 0));
                    d = mfma4_down(sw[1], qw[1], d);
                    d = mfma4_down(sw[0], qw[0], d);
                }
                const int row = r0 + kR * sub + h + li, col = 16 * v4 + 4 * g;
                auto *dst = gmem(P) + row + (int64_t)col * p.lda;
                const bool all = full && p.w == kB;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    old[e] -= d[e];
                    pr[e * kLdC] = old[e];
                }
                if (all) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) dst[e * p.lda] = old[e];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (row < p.m && col + e < p.w) dst[e * p.lda] = old[e];
                }
            }
            __syncthreads();
        }
        if (project) {
#pragma unroll 1
            for (int sub = 0; sub < x.subs; ++sub) {
                floatx4 b[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) b[j] = *(const floatx4 *)(C + x.at(sub, pc + 16 * j + li) + h + 4 * g);
#pragma unroll
                for (int i = 0; i < kTiles; ++i)
                    if (i < qt) {
                        const floatx4 a = *(const floatx4 *)(C + x.at(sub, kp + 16 * (v4 + 4 * i) + li) + h + 4 * g);
#pragma unroll
                        for (int u = 0; u < 4; ++u)
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b[j][u], acc[i][j], 0, 0, 0);
                    }
            }
        }
        if (gram) {
#pragma unroll 1
            for (int sub = 0; sub < x.subs; ++sub) {
                floatx4 a[3], b[3];
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    a[q] = *(const floatx4 *)(C + x.at(sub, pc + 16 * gx[q] + li) + h + 4 * g);
                    b[q] = *(const floatx4 *)(C + x.at(sub, pc + 16 * gy[q] + li) + h + 4 * g);
                }
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    if (gok[q]) {
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            gt[q] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[q][u], (double)b[q][u], gt[q], 0, 0, 0);
                    }
            }
        }
    });
    // The two row halves are added through the (now free) chunk buffers.
    if (project) {
#pragma unroll
        for (int i = 0; i < kTiles; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (i < qt && h) *(floatx4 *)(buf + (((v4 + 4 * i) * 4 + j) * 64 + lane) * 4) = acc[i][j];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kTiles; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (i < qt && !h) {
                    // Lane l, entry e: row 16 tile + 4 (l / 16) + e of S', column 16 j + l % 16.
                    const floatx4 s = acc[i][j] + *(const floatx4 *)(buf + (((v4 + 4 * i) * 4 + j) * 64 + lane) * 4);
                    *(floatx4 *)(S + (16 * j + li) * kLdS + 16 * (v4 + 4 * i) + 4 * g) = s;
                }
        __syncthreads();
    }
    if (gram) {
        double *part = (double *)buf, *Gs = (double *)lds;
        // part: 40 KB at the chunk buffers; Gs: 33 KB from the start, over S.
        if (h) {
#pragma unroll
            for (int q = 0; q < 3; ++q)
                if (gok[q])
#pragma unroll
                    for (int e = 0; e < 4; ++e) part[((v4 * 3 + q) * 4 + e) * 64 + lane] = gt[q][e];
        }
        __syncthreads();
        if (!h) {
#pragma unroll
            for (int q = 0; q < 3; ++q)
                if (gok[q])
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int i = 16 * gx[q] + g + 4 * e, j = 16 * gy[q] + li;
                        double s = gt[q][e] + part[((v4 * 3 + q) * 4 + e) * 64 + lane];
                        if (i >= p.w || j >= p.w) s = i == j ? 1.0 : 0.0;
                        Gs[i * (kB + 1) + j] = s;
                        if (gx[q] != gy[q]) Gs[j * (kB + 1) + i] = s;
                    }
        }
        __syncthreads();
    }
}

// P <- P R^{-1} (R^{-1} row-major kB x kB in LDS at Ris, upper) on FP64 MFMA: wave
// v the row half v / 4 and column tile v % 4, or 3 - v % 4 for the second half
// (tile j costs j + 1: the SIMDs' shares are then equal).
__device__ __forceinline__ void apply_inverse(const Panel &p, float *P, const double *Ris, float *buf)
{
    const int lane = threadIdx.x & 63, v = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, g = lane >> 4, h = 16 * (v >> 2), ct = h ? 3 - (v & 3) : (v & 3);
    double rv[4][4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) rv[t][u] = t <= ct ? Ris[(16 * t + 4 * g + u) * kB + 16 * ct + li] : 0.0;
    const Window x(p, false);
    for_chunks(p, x, buf, [&](float *C, int r0, bool full) {
#pragma unroll 1
        for (int sub = 0; sub < x.subs; ++sub) {
            doublex4 d = doublex4{0.0, 0.0, 0.0, 0.0};
            float y[4][4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int u = 0; u < 4; ++u) y[t][u] = t <= ct ? C[x.at(sub, 16 * t + 4 * g + u) + h + li] : 0.0f;
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (t <= ct) {
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        d = __builtin_amdgcn_mfma_f64_16x16x4f64(rv[t][u], (double)y[t][u], d, 0, 0, 0);
                }
            const int row = r0 + kR * sub + h + li, col = 16 * ct + g;
            auto *dst = gmem(P) + row + (int64_t)col * p.lda;
            if (full && p.w == kB) {
#pragma unroll
                for (int e = 0; e < 4; ++e) dst[4 * e * p.lda] = (float)d[e];
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (row < p.m && col + 4 * e < p.w) dst[4 * e * p.lda] = (float)d[e];
            }
        }
    });
}

// ||R D^{-1}||_F^2 ||D R^{-1}||_F^2 of the w x w factor, D the norms of the
// panel's columns (d0: their squares times kPivotRel), by every thread.  The
// first factor's columns have norm 1.
__device__ __forceinline__ double condition2(const double *Ris, const double *d0, int w)
{
    __shared__ double red[kT / 64];
    double v[1] = {0.0};
    for (int e = threadIdx.x; e < kB * kB; e += kT) {
        const int i = e / kB, j = e % kB;
        if (i <= j && j < w) v[0] = fma(Ris[e] * d0[i], Ris[e], v[0]);
    }
    wave_sums(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v[0];
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < kT / 64; ++q) s += red[q];
    __syncthreads();
    return s * w / kPivotRel;
}

// (An instance with reorthogonalisation and one without: one for both spills
// more, 1024 matrices 3.70 ms for 3.65, and 2.80 for 2.57 without.)
template <bool reorth> __device__ __forceinline__ void wide_factor(const WgTask &tk, char *lds)
{
    const int m = tk.m, n = tk.n;
    const int64_t ldr = tk.ldr;
    auto *R = gmem(tk.R);
    for (int64_t e = threadIdx.x; e < (int64_t)n * n; e += kT) {
        const int i = (int)(e % n), j = (int)(e / n);
        if (i > j) R[i + (int64_t)j * ldr] = 0.0f;
    }
    float *S = (float *)lds;
    double *Gs = (double *)lds, *Rs = Gs + kB * (kB + 1), *Ris = Rs + kB * kB;
    double *R1 = (double *)(lds + kOffR1), *d0 = R1 + kB * kB;
    __shared__ int bad_s;
    bool any_bad = false;
    for (int c0 = 0; c0 < n; c0 += kB) {
        float *P = tk.A + (int64_t)c0 * tk.lda;
        Panel p;
        p.m = m;
        p.w = min(kB, n - c0);
        p.P = P;
        p.lda = tk.lda;
        const int gw = reorth ? c0 : kB;  // columns of Q in a projection
        for (int pass = 0;; ++pass) {
            // Projections of P: twice on all of Q, or once on each block; those
            // of the normalised panel (pass 1): once on all of Q, or none.
            const int ng = c0 == 0 ? 0 : reorth ? 2 - pass : pass ? 0 : c0 / kB;
            for (int g = 0; g < ng; ++g) {
                const int q0 = reorth ? 0 : kB * g;  // its first column
                p.kp = reorth || g == 0 ? 0 : kB;
                p.K = gw + p.kp;
                p.ku = gw;
                p.Q = tk.A + (int64_t)(q0 - p.kp) * tk.lda;
                if (g == 0) sweep<false, true>(p, P, lds);
                else sweep<true, true>(p, P, lds);
                // R's rows above the panel: S, + S, + S R1.
                for (int e = threadIdx.x; e < gw * p.w; e += kT) {
                    const int k = e % gw, j = e / gw;
                    auto *d = R + q0 + k + (int64_t)(c0 + j) * ldr;
                    if (pass == 0) {
                        const float s = S[j * kLdS + k];
                        *d = reorth && g ? *d + s : s;
                    } else {
                        double s = 0.0;
                        for (int i = 0; i <= j; ++i) s = fma((double)S[i * kLdS + k], R1[i * kB + j], s);
                        *d = (float)((double)*d + s);
                    }
                }
            }
            // The last projection's update (S is still in LDS) and G, or G alone.
            p.kp = 0;
            p.K = p.ku = ng ? gw : 0;
            p.Q = tk.A + (int64_t)(reorth || ng == 0 ? 0 : kB * (ng - 1)) * tk.lda;
            if (ng) sweep<true, false>(p, P, lds);
            else sweep<false, false>(p, P, lds);
            const bool bad = factor<kB>(Gs, Rs, Ris, d0, (p.w + 15) / 16);
            if (threadIdx.x == 0) bad_s = bad ? 1 : 0;
            __syncthreads();
            any_bad |= bad_s != 0;
            const double limit = reorth && c0 > 0 ? 4.0 * p.w * p.w : 0x1p24;
            const bool again = pass == 0 && (bad_s != 0 || !(condition2(Ris, d0, p.w) <= limit));
            if (again) {
                for (int e = threadIdx.x; e < kB * kB; e += kT) R1[e] = Rs[e];
            } else {
                for (int e = threadIdx.x; e < p.w * p.w; e += kT) {
                    const int i = e % p.w, j = e / p.w;
                    double s = 0.0;
                    if (pass == 0) s = Rs[i * kB + j];
                    else
                        for (int k = i; k <= j; ++k) s = fma(Rs[i * kB + k], R1[k * kB + j], s);
                    R[c0 + i + (int64_t)(c0 + j) * ldr] = (i <= j) ? (float)s : 0.0f;
                }
            }
            // R^{-1} to the start of the LDS, the chunks behind it.
            double keep[kB * kB / kT];
#pragma unroll
            for (int q = 0; q < kB * kB / kT; ++q) keep[q] = Ris[threadIdx.x + q * kT];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < kB * kB / kT; ++q) Gs[threadIdx.x + q * kT] = keep[q];
            __syncthreads();
            apply_inverse(p, P, Gs, (float *)(lds + kMat));
            if (!again) break;
        }
    }
    if (any_bad && threadIdx.x == 0 && tk.status) atomicOr(tk.status, 1);
}

template <bool reorth> __global__ __launch_bounds__(kT) void batch_wide_kernel(const WgTask *tasks, int ntasks, WgQueue *q)
{
    __shared__ __attribute__((aligned(16))) char lds[kLds];
    for (;;) {
        const unsigned int t = wg_next_task(q);
        if (t >= (unsigned int)ntasks) break;
        const WgTask tk = tasks[t];
        if (threadIdx.x == 0 && tk.status) *tk.status = 0;
        __syncthreads();
        wide_factor<reorth>(tk, lds);
        __syncthreads();
    }
    wg_leave(q);
}

} // namespace

int batch_wide_launch(hipStream_t s, const WgTask *tasks, int ntasks, WgQueue *q, int grid, bool reorth)
{
    if (reorth) hipLaunchKernelGGL(batch_wide_kernel<true>, dim3(grid), dim3(kT), 0, s, tasks, ntasks, q);
    else hipLaunchKernelGGL(batch_wide_kernel<false>, dim3(grid), dim3(kT), 0, s, tasks, ntasks, q);
    HIP_OK(hipGetLastError());
    return LATER_OK;
}

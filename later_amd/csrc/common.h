// Shared definitions for the MI355X (gfx950) HIP sources of the QR library.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/later.h"

#define LATER_API extern "C" __attribute__((visibility("default")))

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef int intx4 __attribute__((ext_vector_type(4)));
typedef int intx16 __attribute__((ext_vector_type(16)));

#define HIP_OK(expr)                                     \
    do {                                                 \
        hipError_t e_ = (expr);                          \
        if (e_ != hipSuccess) return LATER_ERR_DEVICE;   \
    } while (0)

static inline hipStream_t ctx_stream(const laterCtxt &c) { return (hipStream_t)c.stream; }

// Sum over the 64 lanes of a wavefront with DPP operations: quad_perm
// [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror and row_mirror leave every
// lane of a 16-lane row holding that row's sum (the pairings are symmetric,
// so all lanes hold the same bits); row_bcast15 adds row 0 to row 1 and row 2
// to row 3, row_bcast31 adds those two, and lane 63 is read into scalars: the
// sum is (row 0 + row 1) + (row 2 + row 3), uniform and bit-reproducible.
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ int dpp_i(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xF, false);
}

template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ double dpp_d(double v)
{
    const int lo = dpp_i<CTRL, ROWS>(__double2loint(v));
    const int hi = dpp_i<CTRL, ROWS>(__double2hiint(v));
    return __hiloint2double(hi, lo);
}

__device__ __forceinline__ float readlane_f(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

__device__ __forceinline__ double readlane_d(double v, int l)
{
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}

// N wave sums at once.  FP32: one v_add_f32_dpp per step and value (rows
// outside a row mask keep their value), the N values interleaved: a DPP read
// needs two instructions between it and the write of its register, which the
// other values supply when N >= 3.
template <int N> __device__ __forceinline__ void wave_sums(float (&v)[N])
{
    static_assert(N >= 1 && N <= 4, "one to four sums");
#define LATER_DPP_SUM(STEP)                                                        \
    STEP("quad_perm:[1,0,3,2] row_mask:0xf") STEP("quad_perm:[2,3,0,1] row_mask:0xf") \
    STEP("row_half_mirror row_mask:0xf") STEP("row_mirror row_mask:0xf")              \
    STEP("row_bcast:15 row_mask:0xa") STEP("row_bcast:31 row_mask:0xc")
#define LATER_DPP_ADD(i, CTRL) "v_add_f32_dpp %" #i ", %" #i ", %" #i " " CTRL " bank_mask:0xf\n\t"
#define LATER_DPP_1(CTRL) "s_nop 1\n\t" LATER_DPP_ADD(0, CTRL)
#define LATER_DPP_2(CTRL) "s_nop 0\n\t" LATER_DPP_ADD(0, CTRL) LATER_DPP_ADD(1, CTRL)
#define LATER_DPP_3(CTRL) LATER_DPP_ADD(0, CTRL) LATER_DPP_ADD(1, CTRL) LATER_DPP_ADD(2, CTRL)
#define LATER_DPP_4(CTRL) LATER_DPP_3(CTRL) LATER_DPP_ADD(3, CTRL)
    if constexpr (N == 1) asm(LATER_DPP_SUM(LATER_DPP_1) : "+v"(v[0]));
    else if constexpr (N == 2) asm("s_nop 0\n\t" LATER_DPP_SUM(LATER_DPP_2) : "+v"(v[0]), "+v"(v[1]));
    else if constexpr (N == 3) asm("s_nop 1\n\t" LATER_DPP_SUM(LATER_DPP_3) : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]));
    else asm("s_nop 1\n\t" LATER_DPP_SUM(LATER_DPP_4) : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
#undef LATER_DPP_SUM
#undef LATER_DPP_ADD
#undef LATER_DPP_1
#undef LATER_DPP_2
#undef LATER_DPP_3
#undef LATER_DPP_4
#pragma unroll
    for (int c = 0; c < N; ++c) v[c] = readlane_f(v[c], 63);
}

template <int N> __device__ __forceinline__ void wave_sums(double (&v)[N])
{
#pragma unroll
    for (int c = 0; c < N; ++c) v[c] += dpp_d<0xB1>(v[c]);   // quad_perm [1,0,3,2]
#pragma unroll
    for (int c = 0; c < N; ++c) v[c] += dpp_d<0x4E>(v[c]);   // quad_perm [2,3,0,1]
#pragma unroll
    for (int c = 0; c < N; ++c) v[c] += dpp_d<0x141>(v[c]);  // row_half_mirror
#pragma unroll
    for (int c = 0; c < N; ++c) v[c] += dpp_d<0x140>(v[c]);  // row_mirror
#pragma unroll
    for (int c = 0; c < N; ++c) v[c] += dpp_d<0x142, 0xA>(v[c]);  // row_bcast15
#pragma unroll
    for (int c = 0; c < N; ++c) v[c] += dpp_d<0x143, 0xC>(v[c]);  // row_bcast31
#pragma unroll
    for (int c = 0; c < N; ++c) v[c] = readlane_d(v[c], 63);
}

// Global-address-space view of a device pointer.  A pointer the compiler
// cannot trace to a kernel argument (one read from a task table, or a
// parameter of a function that is not inlined) is generic, and its loads and
// stores become flat instructions; those count in lgkmcnt as well as vmcnt,
// so every wait for an LDS access also waits for them, and loads issued
// ahead of their use stop overlapping anything.  Accesses through this view
// are global loads and stores.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T *gmem(T *p)
{
    return (__attribute__((address_space(1))) T *)p;
}

__host__ __device__ static inline int64_t ceil_div64(int64_t a, int64_t b) { return (a + b - 1) / b; }

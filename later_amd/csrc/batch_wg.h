// Task table and queue of the one-launch batched QR, shared by its two
// kernels (batch_wg.hip, batch_wide.hip).
#pragma once
#include "common.h"

struct WgTask {
    int m, n, variant, pad;
    float *A;
    int64_t lda;
    float *R;
    int64_t ldr;
    int *status;
};

struct WgQueue {
    unsigned int head, done;
};

// Next task of the queue for this workgroup (ntasks or more: none left), and
// the count-out at its end: the last workgroup to leave resets the queue for
// the next launch.  Both by every thread.
__device__ __forceinline__ unsigned int wg_next_task(WgQueue *q)
{
    __shared__ unsigned int cur;
    if (threadIdx.x == 0) cur = atomicAdd(&q->head, 1u);
    __syncthreads();
    const unsigned int t = cur;
    __syncthreads();
    return t;
}

__device__ __forceinline__ void wg_leave(WgQueue *q)
{
    if (threadIdx.x == 0) {
        const unsigned int d = atomicAdd(&q->done, 1u);
        if (d == gridDim.x - 1) {
            atomicExch(&q->head, 0u);
            atomicExch(&q->done, 0u);
        }
    }
}

// FP32-product tasks of up to kWideCols columns on 512-thread workgroups, one
// per CU (batch_wide.hip).
constexpr int kWideCols = 256;
int batch_wide_launch(hipStream_t s, const WgTask *tasks, int ntasks, WgQueue *q, int grid, bool reorth);

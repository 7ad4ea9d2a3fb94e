#pragma once
// The two small jobs beside the BCE forward (ffi_forward.hip): marking the
// positives' bits before it, summing its loss partials and clearing the bits
// after it.  haste_ffi_forward_bce runs them as kernels of their own; a training
// step runs them as extra workgroups of the feature transpose and of the
// weight update, whose launches it makes anyway.
#include "common.hpp"

namespace haste {

struct BceJob {
    const int32_t* labels;  // [nnz, 2] (row, label)
    int64_t nnz;
    uint32_t* ybits;        // [B, ldyw] label bits
    int64_t ldyw;
    int B;
    int64_t O;
    const float* part;      // n loss partials
    int64_t n;
    float* loss;
    int nblk;               // workgroups of 256 threads
};

// Workgroup blk: the bits of 256 of the positives, ored into the (all zero)
// bitmap.  Pairs outside [0, B) x [0, O) are ignored.
__device__ __forceinline__ void mark_labels(const BceJob& j, int64_t blk) {
    const int64_t i = blk * 256 + threadIdx.x;
    if (i >= j.nnz) return;
    const int r = j.labels[2 * i], c = j.labels[2 * i + 1];
    if (r < 0 || r >= j.B || c < 0 || c >= j.O) return;
    atomicOr(j.ybits + (int64_t)r * j.ldyw + c / 32, 1u << (c % 32));
}

// Workgroup blk clears the label words of 256 of the pairs; workgroup 0 also sums
// the partials into *loss: each thread a strided subset in order, then a fixed
// tree over the threads.  s: 256 floats of LDS.
__device__ __forceinline__ void sum_loss(const BceJob& j, int64_t blk, float* s) {
    const int64_t li = blk * 256 + threadIdx.x;
    if (li < j.nnz) {
        const int r = j.labels[2 * li], c = j.labels[2 * li + 1];
        if (r >= 0 && r < j.B && c >= 0 && c < j.O) j.ybits[(int64_t)r * j.ldyw + c / 32] = 0u;
    }
    if (blk != 0) return;
    // the partials in batches of 8 loads in flight, summed in index order
    float v = 0.0f;
    for (int64_t i0 = threadIdx.x; i0 < j.n; i0 += 8 * 256) {
        float pv[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) pv[k] = i0 + k * 256 < j.n ? j.part[i0 + k * 256] : 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) v += pv[k];
    }
    s[threadIdx.x] = v;
    __syncthreads();
    for (int m = 128; m >= 1; m >>= 1) {
        if ((int)threadIdx.x < m) s[threadIdx.x] += s[threadIdx.x + m];
        __syncthreads();
    }
    if (threadIdx.x == 0) *j.loss = s[0];
}

// The job of a call on a haste_ffi_forward_bce workspace (ffi_forward.hip).
BceJob bce_job(const int32_t* labels, int64_t nnz, void* workspace, float* loss, int64_t B,
               int64_t O, int64_t G);
int check_bce_job(const char* fn, const int32_t* labels, int64_t nnz, const void* workspace,
                  int64_t ws_bytes, int64_t B, int64_t O, int64_t G);

}  // namespace haste

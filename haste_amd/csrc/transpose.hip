// Feature transpose X [B, D] -> X^T [D, ldt] (2-byte elements), the layout the
// FFI kernels gather from (a feature index selects one contiguous row of B
// values).  64 x 64 tiles staged through LDS; 16-byte loads and stores where a
// row chunk of 8 elements is in bounds and aligned, element accesses otherwise.
// Columns B..ldt-1 of X^T are written as zero, so kernels that read whole
// 8-column chunks never see uninitialised padding.
#include "bce_job.hpp"

namespace haste {
namespace {

constexpr int kT = 64;

__global__ __launch_bounds__(256) void transpose_kernel(const uint16_t* __restrict__ x,
                                                        int64_t ldx, uint16_t* __restrict__ xT,
                                                        int64_t ldt, int64_t B, int64_t D,
                                                        int32_t vec, int gy, BceJob job) {
    if ((int)blockIdx.y >= gy) {  // the label job's workgroups
        mark_labels(job, ((int64_t)blockIdx.y - gy) * gridDim.x + blockIdx.x);
        return;
    }
    __shared__ uint16_t tile[kT][kT + 2];
    const int64_t b0 = (int64_t)blockIdx.x * kT;  // output columns (batch)
    const int64_t d0 = (int64_t)blockIdx.y * kT;  // output rows (features)
    const int tid = threadIdx.x;
    // load x[b0 + r][d0 + c .. c+7] -> tile[r][c..c+7]
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int r = tid / 8 + 32 * h, c = (tid % 8) * 8;
        const int64_t b = b0 + r, d = d0 + c;
        uint16_t v[8];
        if (vec && b < B && d + 8 <= D) {
            u32x4 q = *reinterpret_cast<const u32x4*>(x + b * ldx + d);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[2 * e] = (uint16_t)(q[e] & 0xFFFFu);
                v[2 * e + 1] = (uint16_t)(q[e] >> 16);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (b < B && d + e < D) ? x[b * ldx + d + e] : 0;
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) tile[r][c + e] = v[e];
    }
    __syncthreads();
    // store xT[d0 + r][b0 + c .. c+7] = tile[c..c+7][r]; columns >= B are zero
    const int64_t ncol = ldt;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int r = tid / 8 + 32 * h, c = (tid % 8) * 8;
        const int64_t d = d0 + r, b = b0 + c;
        if (d >= D || b >= ncol) continue;
        uint16_t v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = (b + e < B) ? tile[c + e][r] : 0;
        if (vec && b + 8 <= ncol) {
            u32x4 q;
#pragma unroll
            for (int e = 0; e < 4; ++e) q[e] = (uint32_t)v[2 * e] | ((uint32_t)v[2 * e + 1] << 16);
            *reinterpret_cast<u32x4*>(xT + d * ldt + b) = q;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (b + e < ncol) xT[d * ldt + b + e] = v[e];
        }
    }
}

}  // namespace
}  // namespace haste

namespace haste {
namespace {

// job.nblk > 0: its workgroups follow the transpose's, in further rows of the grid.
int transpose(const char* fn, const uint16_t* x, int64_t ldx, uint16_t* xT, int64_t ldt, int64_t B,
              int64_t D, const BceJob& job, void* stream) {
    HASTE_CHECK_ARG(B >= 0 && D >= 0, "%s: negative size", fn);
    HASTE_CHECK_ARG(ldx >= D && ldt >= B, "%s: need ldx >= D and ldt >= B (ldx=%lld ldt=%lld)", fn,
                    (long long)ldx, (long long)ldt);
    if (D == 0 || ldt == 0) return HASTE_OK;
    HASTE_CHECK_ARG(xT != nullptr && (B == 0 || x != nullptr), "%s: null pointer", fn);
    const int64_t gx = ceil_div(ldt, (int64_t)kT);
    const int64_t gy = ceil_div(D, (int64_t)kT);
    const int64_t gl = ceil_div((int64_t)job.nblk, gx);
    HASTE_CHECK_ARG(gx < 65536 * 32 && gy + gl < 65536, "%s: matrix too large", fn);
    const int vec = aligned16(x) && aligned16(xT) && ldx % 8 == 0 && ldt % 8 == 0;
    transpose_kernel<<<dim3((unsigned)gx, (unsigned)(gy + gl)), dim3(256), 0,
                       static_cast<hipStream_t>(stream)>>>(x, ldx, xT, ldt, B, D, vec, (int)gy, job);
    HASTE_CHECK_LAUNCH(fn);
    return HASTE_OK;
}

}  // namespace
}  // namespace haste

extern "C" int haste_transpose_features(const uint16_t* x, int64_t ldx, uint16_t* xT, int64_t ldt,
                                        int64_t B, int64_t D, void* stream) {
    return haste::transpose("haste_transpose_features", x, ldx, xT, ldt, B, D, haste::BceJob{},
                            stream);
}

extern "C" int haste_transpose_features_labels(const uint16_t* x, int64_t ldx, uint16_t* xT,
                                               int64_t ldt, int64_t B, int64_t D,
                                               const int32_t* labels, int64_t nnz,
                                               void* bce_workspace, int64_t bce_ws_bytes,
                                               int64_t O, int64_t G, void* stream) {
    const char* fn = "haste_transpose_features_labels";
    HASTE_CHECK_ARG(B > 0 && B <= 0x7FFFFFFF && D > 0, "%s: invalid sizes", fn);
    const int rc = haste::check_bce_job(fn, labels, nnz, bce_workspace, bce_ws_bytes, B, O, G);
    if (rc != HASTE_OK) return rc;
    return haste::transpose(fn, x, ldx, xT, ldt, B, D,
                            haste::bce_job(labels, nnz, bce_workspace, nullptr, B, O, G), stream);
}

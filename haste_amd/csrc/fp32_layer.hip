// Passes of an fp32 layer that torch would make in several kernels (gfx950): the
// fp16 copy of grad_output in rows the backward kernels read in place, and the
// SGD step on fp32 tensors.  Both are bound by HBM.
#include <algorithm>

#include "common.hpp"

namespace haste {
namespace {

constexpr int kThreads = 256;

// out[r, 8p .. 8p+7] = RNE(in[r, ...]) (0 past the row): a thread one 8-element
// piece, 2^tx threads to a row, so that short rows share a workgroup (60,000 rows
// of 100: 28 us with a workgroup to a row, below the launch's 9 here).  in's rows start on
// 4-byte boundaries only (its loads are unaligned 16-byte ones), out's on
// 128-byte lines, so that the backward kernels take their aligned builds: torch's
// cast left rows at in's stride, where the weight gradient took 36.5 us, here 29.8
// (B = 256, O = 131,073, G = 32, F = 64), at the cost of torch's cast (28 us, 7.2 TB/s).
__global__ __launch_bounds__(kThreads) void cast_rows_f16_kernel(const float* __restrict__ in,
                                                                 int64_t ldi,
                                                                 uint16_t* __restrict__ out,
                                                                 int64_t ldo, int64_t rows,
                                                                 int64_t cols, int tx) {
    typedef f32x4 __attribute__((aligned(4))) f32x4_u;
    const int x = threadIdx.x & ((1 << tx) - 1), y = threadIdx.x >> tx;
    const int64_t r = (int64_t)blockIdx.y * (kThreads >> tx) + y;
    const int64_t c = (((int64_t)blockIdx.x << tx) + x) * 8;
    if (r >= rows || c >= cols) return;
    const float* p = in + r * ldi + c;
    f32x4 a = {0.f, 0.f, 0.f, 0.f}, b = {0.f, 0.f, 0.f, 0.f};
    if (c + 8 <= cols) {
        a = *reinterpret_cast<const f32x4_u*>(p);
        b = *reinterpret_cast<const f32x4_u*>(p + 4);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            a[e] = c + e < cols ? p[e] : 0.f;
            b[e] = c + 4 + e < cols ? p[4 + e] : 0.f;
        }
    }
    *reinterpret_cast<u32x4*>(out + r * ldo + c) =
        u32x4{pack2_rne<F16>(a[0], a[1]), pack2_rne<F16>(a[2], a[3]), pack2_rne<F16>(b[0], b[1]),
              pack2_rne<F16>(b[2], b[3])};
}

// The SGD step on fp32 tensors, in one pass over p, g (and m) where the torch
// ops of optim_sr.py:73-84 take one pass per op.  The roundings are those of the
// ops: g' = fma(wd, p, g) if wd != 0; m' = round(mu * m) + g'; p' = fma(-lr, m' or
// g', p).  W and bias of that layer: four launches and 36 us -> one, 17 us.
constexpr int kMaxSegs = 8;
constexpr int kVec = 4;
struct F32Seg {
    float* w;
    const float* g;
    float* m;
    int64_t n, blk0;
    int vec;
};
struct F32Batch {
    F32Seg s[kMaxSegs];
    int count;
};

template <bool MOM, bool WD>
__device__ __forceinline__ float sgd_f32_one(float w, float g, float* m, float lr, float wd,
                                             float mu) {
    if constexpr (WD) g = __builtin_fmaf(wd, w, g);
    if constexpr (MOM) {
        float t = mu * *m;
        asm volatile("" : "+v"(t));  // a rounded product: not contracted into the sum
        g = t + g;
        *m = g;
    }
    return __builtin_fmaf(-lr, g, w);
}

template <bool MOM, bool WD>
__global__ __launch_bounds__(kThreads) void sgd_f32_kernel(const F32Batch b, float lr, float wd,
                                                           float mu) {
    int t = 0;
#pragma unroll
    for (int k = 1; k < kMaxSegs; ++k)
        if (k < b.count && (int64_t)blockIdx.x >= b.s[k].blk0) t = k;
    const F32Seg s = b.s[t];
    const int64_t i = (((int64_t)blockIdx.x - s.blk0) * kThreads + threadIdx.x) * kVec;
    if (s.vec && i + kVec <= s.n) {
        f32x4 w = *reinterpret_cast<const f32x4*>(s.w + i);
        const f32x4 g = *reinterpret_cast<const f32x4*>(s.g + i);
        f32x4 m = {0.f, 0.f, 0.f, 0.f};
        if constexpr (MOM) m = *reinterpret_cast<const f32x4*>(s.m + i);
#pragma unroll
        for (int e = 0; e < kVec; ++e) {
            float mv = m[e];
            w[e] = sgd_f32_one<MOM, WD>(w[e], g[e], &mv, lr, wd, mu);
            m[e] = mv;
        }
        *reinterpret_cast<f32x4*>(s.w + i) = w;
        if constexpr (MOM) *reinterpret_cast<f32x4*>(s.m + i) = m;
        return;
    }
    for (int64_t k = i; k < std::min<int64_t>(s.n, i + kVec); ++k) {
        float mv = MOM ? s.m[k] : 0.f;
        s.w[k] = sgd_f32_one<MOM, WD>(s.w[k], s.g[k], &mv, lr, wd, mu);
        if constexpr (MOM) s.m[k] = mv;
    }
}

}  // namespace
}  // namespace haste

extern "C" int haste_cast_rows_f16(const float* in, int64_t ldi, uint16_t* out, int64_t ldo,
                                   int64_t rows, int64_t cols, void* stream) {
    const char* fn = "haste_cast_rows_f16";
    HASTE_CHECK_ARG(rows >= 0 && cols >= 0, "%s: negative size", fn);
    if (rows == 0 || cols == 0) return HASTE_OK;
    HASTE_CHECK_ARG(in && out && ldi >= cols && ldo >= (cols + 7) / 8 * 8 && ldo % 8 == 0 &&
                        haste::aligned16(out) && reinterpret_cast<uintptr_t>(in) % 4 == 0,
                    "%s: null pointer, short stride or misaligned rows (ldi=%lld ldo=%lld "
                    "cols=%lld)", fn, (long long)ldi, (long long)ldo, (long long)cols);
    int tx = 0;
    while (tx < 8 && (int64_t)8 << tx < cols) ++tx;
    const int64_t bx = haste::ceil_div(cols, (int64_t)8 << tx);
    const int64_t by = haste::ceil_div(rows, (int64_t)haste::kThreads >> tx);
    HASTE_CHECK_ARG(rows < 65536 && bx < 0x7FFFFFFF, "%s: matrix too large", fn);
    haste::cast_rows_f16_kernel<<<dim3((unsigned)bx, (unsigned)by), dim3(haste::kThreads), 0,
                                  static_cast<hipStream_t>(stream)>>>(in, ldi, out, ldo, rows, cols,
                                                                      tx);
    HASTE_CHECK_LAUNCH(fn);
    return HASTE_OK;
}

extern "C" int haste_sgd_step_f32_multi(const haste_sgd_tensor* tensors, int32_t count, float lr,
                                        float wd, float mu, int32_t use_mom, void* stream) {
    const char* fn = "haste_sgd_step_f32_multi";
    HASTE_CHECK_ARG(count >= 0 && (count == 0 || tensors != nullptr), "%s: bad tensor list", fn);
    hipStream_t st = static_cast<hipStream_t>(stream);
    for (int base = 0; base < count; base += haste::kMaxSegs) {
        haste::F32Batch b{};
        int64_t blocks = 0;
        for (int k = base; k < std::min<int>(count, base + haste::kMaxSegs); ++k) {
            const haste_sgd_tensor& t = tensors[k];
            HASTE_CHECK_ARG(t.n >= 0 && (t.n == 0 || (t.w && t.g && (!use_mom || t.m))),
                            "%s: tensor %d: null pointer or negative size", fn, k);
            if (t.n == 0) continue;
            haste::F32Seg& s = b.s[b.count++];
            s = haste::F32Seg{reinterpret_cast<float*>(t.w), static_cast<const float*>(t.g), t.m,
                              t.n, blocks, 0};
            s.vec = haste::aligned16(s.w) && haste::aligned16(s.g) &&
                    (!use_mom || haste::aligned16(s.m));
            blocks += haste::ceil_div(t.n, (int64_t)haste::kThreads * haste::kVec);
        }
        if (b.count == 0) continue;
        HASTE_CHECK_ARG(blocks < 0x7FFFFFFF, "%s: tensors too large", fn);
        const dim3 grid((unsigned)blocks), th(haste::kThreads);
        if (use_mom && wd != 0.0f)
            haste::sgd_f32_kernel<true, true><<<grid, th, 0, st>>>(b, lr, wd, mu);
        else if (use_mom)
            haste::sgd_f32_kernel<true, false><<<grid, th, 0, st>>>(b, lr, wd, mu);
        else if (wd != 0.0f)
            haste::sgd_f32_kernel<false, true><<<grid, th, 0, st>>>(b, lr, wd, mu);
        else
            haste::sgd_f32_kernel<false, false><<<grid, th, 0, st>>>(b, lr, wd, mu);
        HASTE_CHECK_LAUNCH(fn);
    }
    return HASTE_OK;
}

// The fused weight update that also computes the logits (ffi_bwd_w_kernel with
// FWD): its instantiations and dispatch.
#include "bwdw_kernel.hpp"

namespace haste {
namespace {

template <int G, int FP>
int launch_fwd_sgd(const int32_t* idx, const uint16_t* xT, int64_t ldx, const uint16_t* dY,
                   int64_t lddy, int64_t B, int64_t D, int64_t F, int64_t O, const SgdArgs& sg,
                   hipStream_t st) {
    if (B * lddy * 2 > kMallBytes)
        return launch<BF16, G, FP, true, true, false, true>(
            idx, xT, ldx, dY, lddy, nullptr, HASTE_DTYPE_F32, nullptr, HASTE_DTYPE_F32, B, D, F, O,
            sg, st);
    return launch<BF16, G, FP, true, false, false, true>(
        idx, xT, ldx, dY, lddy, nullptr, HASTE_DTYPE_F32, nullptr, HASTE_DTYPE_F32, B, D, F, O, sg,
        st);
}

template <int G>
int dispatch_fp(const int32_t* idx, const uint16_t* xT, int64_t ldx, const uint16_t* dY,
                int64_t lddy, int64_t B, int64_t D, int64_t F, int64_t O, const SgdArgs& sg,
                hipStream_t st) {
    if (F <= 32) return launch_fwd_sgd<G, 32>(idx, xT, ldx, dY, lddy, B, D, F, O, sg, st);
    if (F <= 64) return launch_fwd_sgd<G, 64>(idx, xT, ldx, dY, lddy, B, D, F, O, sg, st);
    if (F <= 128) return launch_fwd_sgd<G, 128>(idx, xT, ldx, dY, lddy, B, D, F, O, sg, st);
    if constexpr (G <= 64)
        return launch_fwd_sgd<G, 256>(idx, xT, ldx, dY, lddy, B, D, F, O, sg, st);
    set_error("haste_ffi_forward_bwd_weights_sgd_dx: no build for G = %d, F = %lld", G, (long long)F);
    return HASTE_ERR_UNSUPPORTED;
}

}  // namespace

bool fwd_sgd_fits(const void* dY, int64_t lddy, int64_t ldl, int64_t F, int64_t G) {
    return lddy % 8 == 0 && aligned16(dY) && (G < 128 || F <= 128) &&
           64 * ldl * 2 <= kMaxRsrcBytes;
}

// Where the joined launch is faster than forward, backward to features and update
// in turn.  Measured over some 2,500 shapes, B = 1 .. 1024 and O = 500 .. 1,600,000 (time of
// the step, joined / in turn: mean, extremes; 1,450 of them also with other data
// through the caches before each step, "cold"): 0.93 (0.72 - 1.07) where true, and
// where not
//  - under 100 groups with large batches and fan-ins, 1.02 (0.91 - 1.19): a group's
//    chunks are one serial chain, longer in the joined kernel, on a chip that idles;
//  - little work per group beside the joined kernel's fewer waves, with dY within the
//    last-level cache: G = 128 with short rows from O = 300,000, 1.03 (0.97 - 1.08, cold
//    1.02), and batches of one chunk at G = 64 with F half filling its tiles, 1.03 (0.99
//    - 1.05, cold 1.05), or from 48M weights, 1.03 (0.97 - 1.07, cold 1.02).
// A dY over that cache draws even (1.00, 0.86 - 1.09) where the same dY was read a step
// ago, as its tail is then found there, and gains cold (0.95; 690 us in turn, 643 joined
// at O = 670,091, G = F = 64, B = 512).
bool fwd_sgd_pays(int64_t lddy, int64_t B, int64_t F, int64_t O, int64_t G) {
    if (O < 100 * G) return B * F < 48 * 1024;
    if (B * lddy * 2 > kMallBytes) return true;
    if (G == 128) return F >= 64 || O < 300000;
    const bool one_chunk = B <= 64 && F > 64 && F <= 128 && G > 16;
    return !one_chunk || (O * F < 48000000 && (G == 32 || F > 112 || O < 50000));
}

int fwd_sgd_dispatch(const int32_t* idx, const uint16_t* xT, int64_t ldx, const uint16_t* dY,
                     int64_t lddy, int64_t B, int64_t D, int64_t F, int64_t O, int64_t G,
                     const SgdArgs& sg, hipStream_t st) {
    switch (G) {
    case 16: return dispatch_fp<16>(idx, xT, ldx, dY, lddy, B, D, F, O, sg, st);
    case 32: return dispatch_fp<32>(idx, xT, ldx, dY, lddy, B, D, F, O, sg, st);
    case 64: return dispatch_fp<64>(idx, xT, ldx, dY, lddy, B, D, F, O, sg, st);
    default: return dispatch_fp<128>(idx, xT, ldx, dY, lddy, B, D, F, O, sg, st);
    }
}

}  // namespace haste

extern "C" int haste_ffi_forward_bwd_weights_joined(const void* dY, int64_t lddy, int64_t ldl,
                                                    int64_t B, int64_t F, int64_t O, int64_t G) {
    return haste::fwd_sgd_fits(dY, lddy, ldl, F, G) && haste::fwd_sgd_pays(lddy, B, F, O, G);
}

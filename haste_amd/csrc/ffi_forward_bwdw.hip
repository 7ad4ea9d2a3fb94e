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

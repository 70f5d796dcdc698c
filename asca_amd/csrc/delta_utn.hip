// Gated delta rule in the blocked form at dh = 16, 32, 96 and 128.
#include "ut64_kernels.h"

namespace asca {

int launch_ut_fwd_n(const void* q, const void* k, const void* v, bool bf, bool al, const float* alpha,
                    const float* beta, float* o, const DeltaWs& ws, int B, int T, int H, int dh, hipStream_t st) {
    switch (dh) {
        case 16: return ut_fwd_variant<1>(q, k, v, bf, al, alpha, beta, o, ws, B, T, H, st);
        case 32: return ut_fwd_variant<2>(q, k, v, bf, al, alpha, beta, o, ws, B, T, H, st);
        case 96: return ut_fwd_variant<6>(q, k, v, bf, al, alpha, beta, o, ws, B, T, H, st);
        case 128: return ut_fwd_variant<8>(q, k, v, bf, al, alpha, beta, o, ws, B, T, H, st);
        default: return fail(ASCA_ERR_UNSUPPORTED, "ut_fwd: dh=%d", dh);
    }
}

int launch_ut_bwd_n(const ut64::BArgs& a, int dh, bool bf, bool fused, bool al, hipStream_t st) {
    switch (dh) {
        case 16: return ut_bwd_variant<1>(a, bf, fused, al, st);
        case 32: return ut_bwd_variant<2>(a, bf, fused, al, st);
        case 96: return ut_bwd_variant<6>(a, bf, fused, al, st);
        case 128: return ut_bwd_variant<8>(a, bf, fused, al, st);
        default: return fail(ASCA_ERR_UNSUPPORTED, "ut_bwd: dh=%d", dh);
    }
}

}  // namespace asca

// Gated delta rule in the blocked form: dh = 64 and 48 off the hot path (bf16
// rows, raw gradients, rows not aligned to 16 bytes), and the choice of the
// head width, in a translation unit of their own so that they keep the default
// instruction scheduler (the hot path's setting does not compile them).
#include "ut64_kernels.h"

namespace asca {

int launch_ut_fwd_other(const void* q, const void* k, const void* v, bool bf, bool al, const float* alpha,
                        const float* beta, float* o, const DeltaWs& ws, int B, int T, int H, int dh, hipStream_t st) {
    switch (dh) {
        case 48: return ut_fwd_variant<3>(q, k, v, bf, al, alpha, beta, o, ws, B, T, H, st);
        case 64:
            return al ? launch_ut_fwd_t<UtDims<4>::F, true, true>(q, k, v, alpha, beta, o, ws, B, T, H, st)
                      : launch_ut_fwd_t<UtDims<4>::F, true, false>(q, k, v, alpha, beta, o, ws, B, T, H, st);
        default: return launch_ut_fwd_n(q, k, v, bf, al, alpha, beta, o, ws, B, T, H, dh, st);
    }
}

int launch_ut_bwd_other(const ut64::BArgs& a, int dh, bool bf, bool fused, bool al, hipStream_t st) {
    switch (dh) {
        case 48: return ut_bwd_variant<3>(a, bf, fused, al, st);
        case 64: return ut_bwd_variant<4>(a, bf, fused, al, st);
        default: return launch_ut_bwd_n(a, dh, bf, fused, al, st);
    }
}

}  // namespace asca

// Gated delta rule in the blocked (UT) form: the launchers, and the f32 dh = 64
// forward and fused backward on 16-byte-aligned rows (the training hot
// path).  The kernels are in ut64_kernels.h; the other head widths and
// variants are launched from delta_ut64_b.hip and delta_utn.hip.
#include "ut64_kernels.h"

namespace asca {

static bool aligned(const void* p, unsigned a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

bool ut_fits(int T, int H, int dh, long ld) {
    // the buffer resources over a unit's rows, gates, u tiles, checkpoints and
    // records take 32-bit byte sizes and offsets
    const long NC = (T + ut64::C - 1) / ut64::C;
    return (long)T * max((long)H * dh, ld) < (1L << 30) && (long)T * 2 * H < (1L << 30) &&
           (NC + 1) * dh * dh < (1L << 30) && NC * ut64::R_SZ < (1L << 30);
}

int launch_ut_fwd(const void* q, const void* k, const void* v, bool bf, const float* alpha, const float* beta,
                  float* o, const DeltaWs& ws, int B, int T, int H, int dh, hipStream_t st) {
    if (ws.ck != D64_CK || !ws.rec) return fail(ASCA_ERR_INVALID, "ut_fwd: workspace layout mismatch");
    if (!ut_fits(T, H, dh, 0)) return fail(ASCA_ERR_UNSUPPORTED, "ut_fwd: one sequence's rows exceed 32-bit byte offsets");
    const unsigned ia = bf ? 8 : 16;
    const bool al = aligned(q, ia) && aligned(k, ia) && aligned(v, ia) && aligned(o, 16);
    if (dh == 64 && !bf)
        return al ? launch_ut_fwd_t<UtDims<4>::F, false, true>(q, k, v, alpha, beta, o, ws, B, T, H, st)
                  : launch_ut_fwd_t<UtDims<4>::F, false, false>(q, k, v, alpha, beta, o, ws, B, T, H, st);
    return launch_ut_fwd_other(q, k, v, bf, al, alpha, beta, o, ws, B, T, H, dh, st);
}

// The gate sums of every block and, for column splits, their partial dq, dk, dalpha, dbeta.
static size_t gate_sums(int B, int T, int H, int dh) {
    return ut_bwd_scratch_floats((long)B * H * ut_col_splits(dh), (T + ut64::C - 1) / ut64::C);
}
size_t ut_bwd_scratch(int B, int T, int H, int dh) {
    const size_t vs = ut_col_splits(dh), rows = (size_t)B * T;
    return gate_sums(B, T, H, dh) + (vs > 1 ? vs * 2 * rows * ((size_t)H * dh + H) : 0);
}

int launch_ut_bwd(bool fused, const void* q, const void* k, const void* v, bool bf, const float* alpha,
                  const float* beta, const void* d_o, const DeltaWs& ws, float* scratch, const float* qn,
                  const float* kn, float* gq, float* gk, float* gv, long ldx, float* ga, float* gb, long ldg, int B,
                  int T, int H, int dh, hipStream_t st) {
    if (!ws.rec) return fail(ASCA_ERR_INVALID, "ut_bwd: workspace layout mismatch");
    if (!ut_fits(T, H, dh, max(ldx, ldg)))
        return fail(ASCA_ERR_UNSUPPORTED, "ut_bwd: one sequence's rows exceed 32-bit byte offsets");
    ut64::BArgs a;
    a.q = q; a.k = k; a.v = v; a.alpha = alpha; a.beta = beta; a.d_o = d_o; a.u = ws.sk; a.ckpt = ws.ckpt;
    a.rec = ws.rec; a.qn = qn; a.kn = kn; a.gq = gq; a.gk = gk; a.gv = gv; a.ga = ga; a.gb = gb;
    a.ldx = ldx; a.ldv = ldx; a.ldg = ldg; a.d = (long)H * dh; a.B = B; a.T = T; a.H = H; a.nslots = ws.nslots;
    a.NC = (T + ut64::C - 1) / ut64::C;
    a.x_vs = a.g_vs = 0;
    a.vs = 0;
    // a caller that lends the forward's workspace only for reading gives no scratch
    const int vs = ut_col_splits(dh);
    const size_t rows = (size_t)B * T, n = rows * a.d, gs = gate_sums(B, T, H, dh);
    StreamScratch sc;
    int rc = ASCA_OK;
    if (!scratch) {
        if ((rc = sc.get(ut_bwd_scratch(B, T, H, dh), st))) return rc;
        scratch = sc.ws.p;
    }
    a.gsc = scratch;
    float *px = nullptr, *pg = nullptr;
    if (vs > 1) {
        px = scratch + gs;
        pg = px + 2 * vs * n;
        a.gq = px;
        a.gk = px + vs * n;
        a.ldx = a.d;
        a.x_vs = (long)n;
        a.ga = pg;
        a.gb = pg + H;
        a.ldg = 2L * H;
        a.g_vs = (long)rows * 2 * H;
    }
    a.di = (int)a.d; a.ldxi = (int)a.ldx; a.ldvi = (int)a.ldv; a.ldgi = (int)a.ldg;
    const unsigned ia = bf ? 8 : 16;
    const bool al = aligned(q, ia) && aligned(k, ia) && aligned(v, ia) && aligned(d_o, ia) && aligned(a.gq, 16) &&
                    aligned(a.gk, 16) && aligned(gv, 16) && ldx % 4 == 0;
    if (dh == 64 && !bf && fused && al)
        rc = launch_ut_bwd_t<UtDims<4>::B, false, true, true>(a, st);
    else
        rc = launch_ut_bwd_other(a, dh, bf, fused && vs == 1, al, st);
    if (!rc && vs > 1)
        rc = launch_delta_combine(fused, vs, px, pg, static_cast<const float*>(q), static_cast<const float*>(k), alpha,
                                  beta, qn, kn, gq, gk, ldx, ga, gb, ldg, (long)rows, H, dh, st);
    const int rr = sc.release(st);
    return rc ? rc : rr;
}

}  // namespace asca

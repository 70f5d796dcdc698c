// Kernels of the gated delta rule at dh = 16, 32, 48, 64, 96 and 128, f32 (rows f32 or
// bf16): the recurrence advanced 16 steps at a time on the matrix cores, with the
// state resident in registers.
//
// Same math, outputs and tolerances as DeltaBlock::scan_cpu / bptt_cpu
// (rust/src/delta.rs:244-334, :421-613).  Over a block of C = 16 steps the
// recurrence S_t = alpha_t S_{t-1} + k_t u_t^T, u_t = beta_t (v_t - alpha_t
// S_{t-1}^T k_t) unrolls into the UT (WY) form of docs/SPEC_V2.md:50-69: with
// gamma_t = prod_{s<=t} alpha_s and Gamma[t][m] = prod_{m<s<=t} alpha_s (running
// products inside the block, never a division, so alpha = 0 is exact),
//
//     L  = strict_tril(diag(beta) (Gamma o K K^T)),   T = (I + L)^-1
//     U  = T diag(beta) (V - diag(gamma) K S)           (the 16 u_t rows)
//     O  = diag(gamma) Q S + tril(Gamma o Q K^T) U       (the 16 o_t rows)
//     S' = gamma_15 S + K^T diag(Gamma[15][:]) U.
//
// One block per (sequence, head) unit (dh / 32 blocks of 32 value columns above
// dh = 64), in the reference's h*B + b order; chain waves, at dh = 64 four, one per
// SIMD, each owning value columns 16w .. 16w + 15 of S.  Column i
// of S meets only k, q, the gates and its own v_i, so a wave advances its dh x 16
// slab of S alone: dh / 16 16x16 accumulator tiles of the 16x16x4 f32 MFMA (lane l
// holds S[16r + 4(l/16) + j][16w + l%16] in register j of tile r).  Because the
// accumulator's row index is the MFMA's contraction index (with the k order
// permuted inside each 4-row group), the state feeds the products K S and
// Q S directly and the block update lands in the same registers: the state
// never leaves them.  Per block and wave that is 16 + 16 + 4 + 4 + 16 = 56 MFMAs at
// dh = 64 (K S, Q S, T R, M U, the update).
//
// The state-independent per-block matrices (T, M, gamma, beta, Gamma[15][:])
// are formed one group of blocks ahead (four at dh = 64), one block per helper wave (the Gram
// products K K^T and Q K^T on the MFMA, T by back substitution one row per lane),
// and handed over in LDS with one barrier per group.
//
// The kernel templates and their launch templates live in this header, included
// by delta_ut64.hip (the f32 dh = 64 forward and its fused, 16-byte-aligned
// backward: the hot path, compiled with its own scheduler setting) and by
// delta_ut64_b.hip and delta_utn.hip (the other variants and head widths,
// compiled with the default one).
#pragma once
#include <type_traits>

#include "common.h"
#include "delta.h"
#include "runtime.h"

namespace asca {
namespace ut64 {

constexpr int C = 16;          // steps per block; a checkpoint every 2 C steps

// A head width: dh = 16 NR, whose value columns run on VS = NR / NV blocks of
// NV chain waves (16 columns each), beside NH helper waves of NR / NH key tiles
// each.  dh <= 64 takes one block per unit with a chain and a helper wave per
// 16 columns.  Above, one block's LDS does not hold the backward, and a unit's
// block would leave most CUs idle: NV = 2, the forward with two helper waves (a
// wave per SIMD), the backward's partial dq, dk, dalpha, dbeta of the splits
// added by delta_combine_k.  Bound: the chain of blocks (forward 1.4-1.9 us, backward
// 2-6 us per 16 steps from dh = 16 to 128); the per-step kernels of these widths
// (delta.hip: they keep sequences of a few steps) walk the steps one by one: forward and fused backward of B8 T1000 H8 dh128
// 2627 -> 534 us, B4 T128 H4 dh32 76 -> 33, B32 T512 H8 dh48 667 -> 171, B32 T512
// H8 dh96 7424 -> 700.  Each width is ten kernels with a register allocation of its
// own to look after; 80 and 112 and the widths between have not been made.
template <int NR_, int NV_, int NH_>
struct Dim {
    static constexpr int NR = NR_, NV = NV_, NH = NH_;
    static constexpr int KS = NR / NH, VS = NR / NV;
    static_assert(NR % NV == 0, "tile split");
    // whether a non-finite value is kept to the steps that the recurrence takes it
    // to (any_bad below); the dh = 64 kernels spread it over its block of 16 steps
    static constexpr bool CAUSAL = NR != 4;
    // whether sums of a few terms are added up apart from the large value that they
    // join, in short chains (mfma_sum; T held without its unit diagonal)
    static constexpr bool FINE = NR != 4;
    static constexpr int DH = 16 * NR, DH2 = DH * DH;
    static constexpr int NWT = NV + NH, NT = 64 * NWT;   // waves, threads of a block
    // row pitches in LDS (4 mod 32 at 64 columns: the 16-byte reads of 16 rows
    // at one offset spread over the banks) of the key-wide and value-wide rows
    static constexpr int RK = 16 * NR + 4, RV = 16 * NV + 4;
    static constexpr int U_BLK = NR * 256;               // a block's u rows (U_TILE)
    // forward LDS (floats)
    static constexpr int NSLOT = 2 * NH;                 // prepared matrices: two groups of NH blocks
    static constexpr int P_SZ = 576;
    static constexpr int F_SCR = NSLOT * P_SZ;           // per helper: L^T scratch [16][16]
    static constexpr int F_STG = F_SCR + NH * 256;       // [2][S_BUF]
    static constexpr int G_ROWS = NH * C;                // rows of one group
    static constexpr int S_Q = G_ROWS * RK, S_V = 2 * G_ROWS * RK;
    static constexpr int S_BUF = G_ROWS * (2 * RK + RV);
    static constexpr int OTP = 20;
    static constexpr int F_OT = F_STG + 2 * S_BUF;       // per chain wave: o, u and state tiles [3][16][20]
    static constexpr int F_ALL = F_OT + NV * 3 * C * OTP;
    static constexpr size_t F_LDS = (size_t)F_ALL * 4;
};

// D += A B on a 16x16x4 f32 MFMA: lane l gives A[l % 16][l / 16] and
// B[l / 16][l % 16] and holds D[4 (l / 16) + r][l % 16] in register r.
ASCA_DEV f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// element i of the sum of N accumulators, pairwise
template <int N>
ASCA_DEV float acc_sum(const f32x4 (&a)[N], int i) {
    if constexpr (N == 1) return a[0][i];
    else if constexpr (N == 2) return a[0][i] + a[1][i];
    else if constexpr (N == 3) return (a[0][i] + a[1][i]) + a[2][i];
    else return (a[0][i] + a[1][i]) + (a[2][i] + a[3][i]);
}
// Non-finite values.  The triangular products of a block (T R, M U, M^T dO, T^T dU,
// (Gamma o dM) K, ...) multiply masked zeros with every row of the block, and zero
// times an infinity or NaN is NaN: one at step t would reach outputs and gradients
// of the block's other steps that do not depend on it.  So where such a product's
// sum is not finite (rare: one check per block), it is formed again with only the
// terms that belong to it, at the end of the step (a branch inside one holds up what
// the scheduler would move past it).  The checks cost B4 T128 H4 dh32 31.6 -> 32.5
// us, B8 T1000 H8 dh128 528 -> 531 us.
ASCA_DEV bool any_bad(float x) { return __builtin_expect(__any(!__builtin_isfinite(x)), 0); }
// FINE sums.  A product over 16 k (a[i], b[i]: its four MFMAs) from zero in NC chains,
// so that its terms are rounded against their own sum: where it joins a larger value,
// once against that instead of sixteen times.  Sums of 16 terms that join one (T R,
// M^T dO, T^T dU, the Gamma o dM and dA parts of dq and dk), the Gram products and
// dO U^T, Y U^T are formed so.  Error against float64 (forward and fused backward,
// 2-norm over all outputs, 1e-7) of the per-step kernels, of one chain for every sum,
// of these: dh16 1.19 1.43 1.18, dh32 1.22 1.44 1.20, dh48 1.24 1.46 1.23, dh96 1.21
// 1.49 1.21, dh128 1.23 1.53 1.23 (o alone at dh128: 1.11 1.44 1.17).  Time against
// one chain, forward + backward: B8 T512 H8 dh16 42.5 + 59.8 -> 41.6 + 61.9 us, B4 T128
// H4 dh32 11.2 + 21.4 -> 11.4 + 21.9, B16 T512 H8 dh48 44.1 + 98.5 -> 43.6 + 99.5, B8
// T512 H8 dh96 65.4 + 144 -> 66.9 + 150, B8 T1000 H8 dh128 152 + 370 -> 157 + 374.
template <int NC = 2>
ASCA_DEV f32x4 mfma_sum(const float (&a)[4], const float (&b)[4]) {
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    if constexpr (NC == 4)
        return (mfma4(a[0], b[0], z) + mfma4(a[1], b[1], z)) + (mfma4(a[2], b[2], z) + mfma4(a[3], b[3], z));
    else
        return mfma4(a[1], b[1], mfma4(a[0], b[0], z)) + mfma4(a[3], b[3], mfma4(a[2], b[2], z));
}
ASCA_DEV f32x4 mfma_sum(const float4& a, const float (&b)[4]) {
    const float x[4] = {a.x, a.y, a.z, a.w};
    return mfma_sum(x, b);
}
template <int NC = 2>
ASCA_DEV f32x4 mfma_sum(const float4& a, const float4& b) {
    const float x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
    return mfma_sum<NC>(x, y);
}
// A product and (E) its rounding error: h + e.
template <bool E>
struct Prod {
    float h, e;
    ASCA_DEV float value() const { return E ? h + e : h; }
};
template <bool E>
ASCA_DEV Prod<E> operator*(Prod<E> a, Prod<E> b) {
    const float p = a.h * b.h;
    if constexpr (!E) return {p, 0.0f};
    return {p, fmaf(a.h, b.h, -p) + fmaf(a.h, b.e, a.e * b.h)};
}
// even (or low) and odd (high) 16-lane rows' (32-lane halves') values, in both
ASCA_DEV void row_pair16(float x, float& lo, float& hi) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    lo = __uint_as_float(r[0]);
    hi = __uint_as_float(r[1]);
}
ASCA_DEV void row_pair32(float x, float& lo, float& hi) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    lo = __uint_as_float(r[0]);
    hi = __uint_as_float(r[1]);
}
ASCA_DEV float readlane_f(float x, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l)); }
ASCA_DEV float el(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// Orders the wave's own LDS writes before its reads of other lanes' values.  The
// LDS executes one wave's instructions in issue order, so only the compiler has
// to keep them in program order: a compiler barrier, no wait.
ASCA_DEV void wave_sync() { asm volatile("" ::: "memory"); }

// Rows of q, k, v, dO are f32 or (BF) bf16, widened exactly.  Four consecutive
// elements as loaded, and widened:
template <bool BF>
struct RawRow {
    float4 x;
};
template <>
struct RawRow<true> {
    uint2 x;
};
ASCA_DEV float4 widen(const RawRow<false>& r) { return r.x; }
ASCA_DEV float4 widen(const RawRow<true>& r) {
    return make_float4(__uint_as_float(r.x.x << 16), __uint_as_float(r.x.x & 0xffff0000u),
                       __uint_as_float(r.x.y << 16), __uint_as_float(r.x.y & 0xffff0000u));
}
// ... from element offset vo + so (so uniform) of a resource
template <bool BF>
ASCA_DEV RawRow<BF> row_ld(Rsrc r, unsigned vo, unsigned so) {
    RawRow<BF> w;
    if constexpr (BF) {
        typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
        const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(r, (int)(2u * vo), (int)(2u * so), 0);
        w.x = make_uint2(x[0], x[1]);
    } else {
        w.x = buf_load4(r, 4u * vo, 4u * so);
    }
    return w;
}
// ... from element `off` of an array of any alignment
template <bool BF>
ASCA_DEV RawRow<BF> row_ld_any(const void* p, long off) {
    RawRow<BF> w;
    if constexpr (BF) {
        const uint16_t* e = reinterpret_cast<const uint16_t*>(p) + off;
        w.x = make_uint2(e[0] | (unsigned)e[1] << 16, e[2] | (unsigned)e[3] << 16);
    } else {
        const float* e = reinterpret_cast<const float*>(p) + off;
        w.x = make_float4(e[0], e[1], e[2], e[3]);
    }
    return w;
}
template <bool BF>
ASCA_DEV const void* at_el(const void* p, long off) {
    return reinterpret_cast<const char*>(p) + off * (BF ? 2 : 4);
}

// One block's state-independent matrices in LDS (floats).
constexpr int P_T = 0;      // T = (I + L)^-1 (FINE: T - I), row-major [16][16]
constexpr int P_M = 256;    // M = tril(Gamma o Q K^T), row-major [16][16]
constexpr int P_GAM = 512;  // gamma_t
constexpr int P_BET = 528;  // beta_t (0 past the sequence end)
constexpr int P_GC = 544;   // Gamma[15][m] = prod_{m<s<=15} alpha_s
constexpr int P_AL = 560;   // alpha_t (1 past the sequence end)
constexpr int P_SZ = 576;

// Buffer resources over the unit's part of every array the forward reads or
// writes, made once per kernel: a load's or store's lane offset is then
// loop-invariant and the block's offset a uniform register.  Rows past the
// sequence end lie outside the row resources: they load as 0 (their gates make
// such steps inert) and their stores are dropped.
struct FRes {
    Rsrc q, k, v, o, al, be, u, ck, rec;
};

template <class D>
struct PrepIn {
    float4 kr[D::NR], qr[D::NR];  // K, Q rows n = lane % 16: columns 16r + 4(lane/16) .. +3
    float a, b;           // alpha, beta of step n (as loaded)
};

// Forms block p's matrices from its loads into the slot `ps`.  Steps past the
// sequence end get alpha = 1, beta = 0: they leave the state, T and the
// products of the live steps unchanged.  `scr` is the wave's own scratch.
// Record of a block for the backward (1344 floats): K K^T, Q K^T, T, M and
// Gamma (zero above the diagonal) in the accumulator layout, 16 bytes per lane (float4 index 64 m + lane holds
// matrix m's elements [4 (lane/16) + j][lane % 16], j = 0..3), then the per-step gate
// vectors gamma_t, beta_t gamma_t, Gamma[15][t], beta_t (16 floats each; steps past the
// sequence end as alpha = 1, beta = 0), so that no wave of the backward forms them again.
constexpr int R_A = 0, R_BQ = 256, R_T = 512, R_M = 768, R_G = 1024, R_V = 1280, R_SZ = 1344;
// U_TILE: the u rows for the backward, per unit and block (U_BLK floats): the
// 16 x 16 tiles of value columns 16w .. one after another, each row-major, so a
// chain wave writes its block's u as one contiguous 1 KB.
constexpr int RV_GAM = R_V, RV_BG = R_V + 16, RV_GC = R_V + 32, RV_BET = R_V + 48;
static_assert(R_SZ == D64_REC, "record size");
static_assert(C == D64_BLK && D64_CK == 2 * C, "a checkpoint before every other block");

template <class D>
ASCA_DEV void prep_compute(const PrepIn<D>& pi, int p, int T, float* __restrict__ ps, float* __restrict__ scr,
                           Rsrc rrec, int lane) {
    const unsigned srec = 4u * (unsigned)(p * R_SZ);   // the block's record
    const int n = lane & 15, g = lane >> 4;
    const bool live = p * C + n < T;
    const float a = live ? pi.a : 1.0f;
    const float b = live ? pi.b : 0.0f;
    // Gram products: A[t][m] = k_t . k_m, Bq[t][m] = q_t . k_m (lane: t = 4g + i, m = n)
    f32x4 A = {0.f, 0.f, 0.f, 0.f}, Bq = A;
#pragma unroll
    for (int r = 0; r < D::NR; ++r) {
        if constexpr (D::FINE) {
            constexpr int NC = D::NR < 4 ? 4 : 2;  // (four chains spill at dh = 128)
            A += mfma_sum<NC>(pi.kr[r], pi.kr[r]);
            Bq += mfma_sum<NC>(pi.qr[r], pi.kr[r]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                A = mfma4(el(pi.kr[r], i), el(pi.kr[r], i), A);
                Bq = mfma4(el(pi.qr[r], i), el(pi.kr[r], i), Bq);
            }
        }
    }
    // gam: lane n's gamma_n; G[i] = Gamma[4g + i][n] for 4g + i >= n; pr = Gamma[15][n]
    float gam, G[4] = {1.f, 1.f, 1.f, 1.f}, pr = 1.0f;
    if constexpr (D::FINE) {
        // with their rounding errors at the column splits, where a helper has the time
        // (dh128 forward 155 -> 157 us; at dh16 it is what the chain waits for, 42 -> 47)
        using P = Prod<(D::VS > 1)>;
        P x = {a, 0.0f};
        x = P{dpp_or<0x111>(1.0f, x.h), dpp_or<0x111>(0.0f, x.e)} * x;
        x = P{dpp_or<0x112>(1.0f, x.h), dpp_or<0x112>(0.0f, x.e)} * x;
        x = P{dpp_or<0x114>(1.0f, x.h), dpp_or<0x114>(0.0f, x.e)} * x;
        x = P{dpp_or<0x118>(1.0f, x.h), dpp_or<0x118>(0.0f, x.e)} * x;
        gam = x.value();
        // products over the lane group's own steps 4g .. 4g + i past n, then those of
        // the groups before it and of all four
        P l[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float as = __shfl(a, 4 * g + i);
            const P y = {4 * g + i > n ? as : 1.0f, 0.0f};
            l[i] = i ? l[i - 1] * y : y;
        }
        P even, odd, low, high;
        row_pair16(l[3].h, even.h, odd.h);
        row_pair16(l[3].e, even.e, odd.e);
        const P two = even * odd;
        row_pair32(two.h, low.h, high.h);
        row_pair32(two.e, low.e, high.e);
        pr = (low * high).value();
        const P one = {1.0f, 0.0f}, three = low * even, pre = g == 0 ? one : g == 1 ? even : g == 2 ? low : three;
#pragma unroll
        for (int i = 0; i < 4; ++i) G[i] = (pre * l[i]).value();
    } else {
        gam = prefix_prod<16>(a);
#pragma unroll
        for (int s = 0; s < C; ++s) {
            const float as = readlane_f(a, s);
            pr = s > n ? pr * as : pr;
            if ((s >> 2) == g) G[s & 3] = pr;
        }
    }
    if (g == 0) {
        ps[P_GAM + n] = gam;
        ps[P_BET + n] = b;
        ps[P_GC + n] = pr;
        if constexpr (D::CAUSAL) ps[P_AL + n] = a;
    }
    buf_store1(rrec, 4u * (R_V + lane), g == 0 ? gam : g == 1 ? b * gam : g == 2 ? pr : b, srec);
    const float4 bt = *reinterpret_cast<const float4*>(ps + P_BET + 4 * g);
    float Lv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int t = 4 * g + i;
        Lv[i] = n < t ? el(bt, i) * G[i] * A[i] : 0.f;
        ps[P_M + t * 16 + n] = n <= t ? G[i] * Bq[i] : 0.f;
    }
    // scr holds L row-major: scr[m*16 + j] = L[m][j]
#pragma unroll
    for (int i = 0; i < 4; ++i) scr[(4 * g + i) * 16 + n] = Lv[i];
    // row n of T = (I + L)^-1 from x^T (I + L) = e_n^T, columns from the last:
    // x_j = [j == n] - sum_{m > j} x_m L[m][j]
    // Right-looking: once x_m is final it is taken out of every x_j, j < m (the
    // terms of each x_j in descending m), so x_j is one FMA behind x_{j+1}
    // instead of at the end of a chain of 15 - j, with 16 live partial sums.
    float x[C];
#pragma unroll
    for (int j = 0; j < C; ++j) x[j] = n == j ? 1.f : 0.f;
    float4 rw[2][4];
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) rw[C & 1][q4] = *reinterpret_cast<const float4*>(scr + (C - 1) * 16 + 4 * q4);
#pragma unroll
    for (int m = C - 1; m >= 1; --m) {
        // row m - 1 read one step ahead (broadcast: every lane the same address)
        if (m > 1) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
                if (4 * q4 < m - 1) rw[m & 1][q4] = *reinterpret_cast<const float4*>(scr + (m - 1) * 16 + 4 * q4);
        }
#pragma unroll
        for (int j = 0; j < m; ++j) x[j] -= x[m] * el(rw[(m + 1) & 1][j >> 2], j & 3);
        __builtin_amdgcn_sched_barrier(0);   // keep the solve's steps in order (bounds the live registers)
    }
    // T row-major for the forward, then in the accumulator layout for the record
    auto put_t = [&] {
        if (g == 0) {
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4)
                *reinterpret_cast<float4*>(ps + P_T + n * 16 + 4 * q4) =
                    make_float4(x[4 * q4], x[4 * q4 + 1], x[4 * q4 + 2], x[4 * q4 + 3]);
        }
        if constexpr (D::FINE) {
            wave_sync();
            ps[P_T + 17 * n] = 0.0f;
            wave_sync();
        }
    };
    auto record_t = [&] {
        const float* tp = ps + P_T + 64 * g + n;
        buf_store4(rrec, 16u * ((R_T >> 2) + lane), make_float4(tp[0], tp[16], tp[32], tp[48]), srec);
    };
    put_t();
    buf_store4(rrec, 16u * ((R_A >> 2) + lane), make_float4(A[0], A[1], A[2], A[3]), srec);
    buf_store4(rrec, 16u * ((R_BQ >> 2) + lane), make_float4(Bq[0], Bq[1], Bq[2], Bq[3]), srec);
    record_t();
    const float* mp = ps + P_M + 64 * g + n;
    buf_store4(rrec, 16u * ((R_M >> 2) + lane), make_float4(mp[0], mp[16], mp[32], mp[48]), srec);
    buf_store4(rrec, 16u * ((R_G >> 2) + lane),
               make_float4(n <= 4 * g ? G[0] : 0.f, n <= 4 * g + 1 ? G[1] : 0.f, n <= 4 * g + 2 ? G[2] : 0.f,
                           n <= 4 * g + 3 ? G[3] : 0.f),
               srec);
    if constexpr (D::CAUSAL) {
        if (any_bad((Lv[0] + Lv[1]) + (Lv[2] + Lv[3]))) {  // row n of T from the rows of L up to n
#pragma unroll
            for (int j = 0; j < C; ++j) x[j] = n == j ? 1.f : 0.f;
#pragma unroll
            for (int m = C - 1; m >= 1; --m) {
#pragma unroll
                for (int j = 0; j < m; ++j) {
                    const float y = x[j] - x[m] * scr[m * 16 + j];
                    x[j] = m <= n ? y : x[j];
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            put_t();
            wave_sync();
            record_t();
        }
    }
}

// Staging of a group's k, q, v rows in LDS: NH blocks x 16 rows, two buffers
// alternating by group.
constexpr int OTP = 20;

// Helper hw stages block c0 + hw of the group: its 16 rows of k, q and (this
// block's value columns, from column v0) v.  Rows past the sequence end load as
// 0 or repeat the last row (their gates make them inert).
template <class D, bool BF>
struct Stage {
    RawRow<BF> k[D::NR], q[D::NR], v[D::NV];
};

template <class D, bool BF, bool AL>
ASCA_DEV void stage_load(Stage<D, BF>& st, int c, const void* q, const void* k, const void* v, const FRes& R,
                         long ubase, long d, int T, int v0, int lane) {
    const unsigned so = (unsigned)(c * C * d);
#pragma unroll
    for (int s = 0; s < D::NR; ++s) {
        const int e = lane + 64 * s, row = e / (4 * D::NR), col = 4 * (e % (4 * D::NR));
        if constexpr (AL) {
            const unsigned vo = (unsigned)(row * d + col);
            st.k[s] = row_ld<BF>(R.k, vo, so);
            st.q[s] = row_ld<BF>(R.q, vo, so);
        } else {
            const long off = ubase + min(c * C + row, T - 1) * d + col;
            st.k[s] = row_ld_any<BF>(k, off);
            st.q[s] = row_ld_any<BF>(q, off);
        }
        if (s < D::NV) {
            const int vrow = e / (4 * D::NV), vcol = v0 + 4 * (e % (4 * D::NV));
            if constexpr (AL)
                st.v[s] = row_ld<BF>(R.v, (unsigned)(vrow * d + vcol), so);
            else
                st.v[s] = row_ld_any<BF>(v, ubase + min(c * C + vrow, T - 1) * d + vcol);
        }
    }
}

template <class D, bool BF>
ASCA_DEV void stage_store(const Stage<D, BF>& st, float* __restrict__ buf, int w, int lane) {
#pragma unroll
    for (int s = 0; s < D::NR; ++s) {
        const int e = lane + 64 * s, row = 16 * w + e / (4 * D::NR), col = 4 * (e % (4 * D::NR));
        *reinterpret_cast<float4*>(buf + row * D::RK + col) = widen(st.k[s]);
        *reinterpret_cast<float4*>(buf + D::S_Q + row * D::RK + col) = widen(st.q[s]);
        if (s < D::NV) {
            const int vrow = 16 * w + e / (4 * D::NV), vcol = 4 * (e % (4 * D::NV));
            *reinterpret_cast<float4*>(buf + D::S_V + vrow * D::RV + vcol) = widen(st.v[s]);
        }
    }
}

// Checkpoint slot layout (dh^2 floats), the state before a block as the
// backward's key-slab waves read it, 16 bytes per lane: float4 index
// (r*NR + c)*64 + lane holds S[16r + lane%16][16c + 4(lane/16) + j], j = 0..3
// (key tile r, value tile c).  The forward's chain wave of value tile c holds it with
// keys and values swapped within each 16 x 16 tile, so every tile is transposed
// through the wave's LDS scratch `st` on its way out.
template <class D>
ASCA_DEV void ck_store(const FRes& R, int slot, const f32x4 (&S)[D::NR], float* __restrict__ st, int vt, int lane) {
    const int n = lane & 15, g = lane >> 4;
#pragma unroll
    for (int r = 0; r < D::NR; ++r) {
#pragma unroll
        for (int i = 0; i < 4; ++i) st[(4 * g + i) * OTP + n] = S[r][i];
        const float4 t4 = *reinterpret_cast<const float4*>(st + n * OTP + 4 * g);
        buf_store4(R.ck, 16u * ((r * D::NR + vt) * 64 + lane), t4, 4u * (unsigned)(slot * D::DH2));
    }
}

// A block's o and u rows leave as 16-byte stores: the 16 x 16 tiles go through the
// wave's LDS scratch `ot` (lane: row lane / 4, columns 4 (lane % 4) .. +3).
template <class D, bool FULL, bool AL>
ASCA_DEV void store_ou(const f32x4& O, const f32x4& U, float* __restrict__ ot, int c, float* __restrict__ o,
                       const FRes& res, long ubase, long d, int T, int vt, int lane) {
    const int n = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ot[(4 * g + i) * OTP + n] = O[i];
        ot[C * OTP + (4 * g + i) * OTP + n] = U[i];
    }
    const int rr = lane >> 2, cc = 4 * (lane & 3);
    const float4 o4 = *reinterpret_cast<const float4*>(ot + rr * OTP + cc);
    const float4 u4 = *reinterpret_cast<const float4*>(ot + C * OTP + rr * OTP + cc);
    if constexpr (AL) {
        // rows past the sequence end fall outside the resource: dropped
        buf_store4(res.o, 4u * (unsigned)(rr * d + 16 * vt + cc), o4, 4u * (unsigned)(c * C * d));
    } else {
        const long t = (long)c * C + rr;
        if (FULL || t < T) {
            float* po = o + ubase + t * d + 16 * vt + cc;
            po[0] = o4.x; po[1] = o4.y; po[2] = o4.z; po[3] = o4.w;
        }
    }
    // u tile: 1 KB contiguous per wave and block (layout at U_TILE)
    buf_store4(res.u, 4u * (unsigned)(vt * 256 + rr * 16 + cc), u4, 4u * (unsigned)(c * D::U_BLK));
}

// The `nt` steps of a block one after another (see any_bad): S advanced in place,
// the o and u rows in the accumulator layout.  Per step the lane's keys of S^T k and
// S^T q, added over the four lanes of column n.
template <class D>
ASCA_DEV void chain_by_steps(f32x4 (&S)[D::NR], f32x4& O, f32x4& U, const float* __restrict__ kb,
                             const float* __restrict__ qb, const float* __restrict__ vb,
                             const float* __restrict__ ps, int nt, int w, int lane) {
    const int n = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) O[i] = U[i] = 0.0f;
#pragma unroll 1
    for (int t = 0; t < nt; ++t) {
        const float a = ps[P_AL + t], b = ps[P_BET + t];
        float4 kr[D::NR];
        float sk = 0.0f, o = 0.0f;
#pragma unroll
        for (int r = 0; r < D::NR; ++r) {
            kr[r] = *reinterpret_cast<const float4*>(kb + t * D::RK + 16 * r + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) sk = fmaf(el(kr[r], i), S[r][i], sk);
        }
        sk = add_xor32(add_xor16(sk));
        const float u = b * (vb[t * D::RV + 16 * w + n] - a * sk);
#pragma unroll
        for (int r = 0; r < D::NR; ++r) {
            const float4 qr = *reinterpret_cast<const float4*>(qb + t * D::RK + 16 * r + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                S[r][i] = fmaf(el(kr[r], i), u, a * S[r][i]);
                o = fmaf(el(qr, i), S[r][i], o);
            }
        }
        o = add_xor32(add_xor16(o));
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (t == 4 * g + i) {
                O[i] = o;
                U[i] = u;
            }
    }
}

// One block of 16 steps for the wave's dh x 16 slab of S (value tile vt, the
// block's w-th): outputs o, the u rows
// (for the backward), the checkpoint (state before the block, even blocks) and the block
// update.  `kb` points at the block's first staged k row
// (q and v rows follow at qb, vb).
template <class D, bool FULL, bool AL>
ASCA_DEV float chain_step(f32x4 (&S)[D::NR], const float* __restrict__ kb, const float* __restrict__ qb,
                         const float* __restrict__ vb, const float* __restrict__ ps,
                         float* __restrict__ ot, int c, float* __restrict__ o, const FRes& res, bool ckw, long ubase,
                         long d, int T, int w, int vt, int lane) {
    constexpr int NR = D::NR, RK = D::RK;
    const int n = lane & 15, g = lane >> 4;
    float4 kc[NR], qc[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        kc[r] = *reinterpret_cast<const float4*>(kb + n * RK + 16 * r + 4 * g);
        qc[r] = *reinterpret_cast<const float4*>(qb + n * RK + 16 * r + 4 * g);
    }
    const float4 gm = *reinterpret_cast<const float4*>(ps + P_GAM + 4 * g);
    const float4 bt = *reinterpret_cast<const float4*>(ps + P_BET + 4 * g);
    const float4 gc = *reinterpret_cast<const float4*>(ps + P_GC + 4 * g);
    const float4 tr = *reinterpret_cast<const float4*>(ps + P_T + n * 16 + 4 * g);
    const float4 mr = *reinterpret_cast<const float4*>(ps + P_M + n * 16 + 4 * g);
    const float g15 = ps[P_GAM + 15];
    float vv[4], kt[NR][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        vv[i] = vb[(4 * g + i) * D::RV + 16 * w + n];
#pragma unroll
        for (int r = 0; r < NR; ++r) kt[r][i] = kb[(4 * g + i) * RK + 16 * r + n];
    }
    // K S and Q S, the key tiles dealt to NA accumulators: shorter chains of
    // rounded sums (at dh = 128, with the Gram products' likewise, o is 1.4e-7 off
    // float64 instead of 2.2e-7, as the per-step kernels' sums over eight lanes)
    constexpr int NA = NR == 4 ? 2 : NR < 4 ? NR : 4;
    f32x4 ka[NA], qa[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) ka[a] = qa[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r0 = 0; r0 < NR; r0 += NA)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int a = 0; a < NA; ++a) {
                const int r = r0 + a;
                if (r < NR) {
                    ka[a] = mfma4(el(kc[r], i), S[r][i], ka[a]);
                    qa[a] = mfma4(el(qc[r], i), S[r][i], qa[a]);
                }
            }
    float R[4], qs[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        R[i] = el(bt, i) * (vv[i] - el(gm, i) * acc_sum(ka, i));
        qs[i] = acc_sum(qa, i);
    }
    f32x4 U = {0.f, 0.f, 0.f, 0.f};
    if constexpr (D::FINE) {
        U = mfma_sum(tr, R);
#pragma unroll
        for (int i = 0; i < 4; ++i) U[i] += R[i];
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) U = mfma4(el(tr, i), R[i], U);
    }
    f32x4 O;
#pragma unroll
    for (int i = 0; i < 4; ++i) O[i] = el(gm, i) * qs[i];
#pragma unroll
    for (int i = 0; i < 4; ++i) O = mfma4(el(mr, i), U[i], O);
    if (ckw) ck_store<D>(res, c >> 1, S, ot + 2 * C * OTP, vt, lane);
    store_ou<D, FULL, AL>(O, U, ot, c, o, res, ubase, d, T, vt, lane);
    float Ut[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) Ut[i] = el(gc, i) * U[i];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        S[r] *= g15;
#pragma unroll
        for (int i = 0; i < 4; ++i) S[r] = mfma4(kt[r][i], Ut[i], S[r]);
    }
    return O[0];  // (a U that is not finite is in every row of M U)
}

// A helper wave's gate loads: lane l holds alpha, beta of step 16 c + (l % 16).
// Steps past the sequence end load 0 (prep_compute makes them alpha = 1, beta = 0).
ASCA_DEV void gate_load(float& a, float& b, int c, const FRes& R, int H, int lane) {
    const unsigned vo = 4u * (unsigned)((lane & 15) * H), so = 4u * (unsigned)(c * C * H);
    a = buf_load1(R.al, vo, so);
    b = buf_load1(R.be, vo, so);
}

// The helper wave's prep of block p from its staged rows (rows 16 hw .. of `buf`).
template <class D>
ASCA_DEV void helper_prep(int p, const float* __restrict__ buf, float a, float b, float* __restrict__ ps,
                          float* __restrict__ scr, Rsrc rrec, int T, int hw, int lane) {
    const int n = lane & 15, g = lane >> 4;
    PrepIn<D> pi;
#pragma unroll
    for (int r = 0; r < D::NR; ++r) {
        pi.kr[r] = *reinterpret_cast<const float4*>(buf + (C * hw + n) * D::RK + 16 * r + 4 * g);
        pi.qr[r] = *reinterpret_cast<const float4*>(buf + D::S_Q + (C * hw + n) * D::RK + 16 * r + 4 * g);
    }
    pi.a = a;
    pi.b = b;
    prep_compute<D>(pi, p, T, ps, scr, rrec, lane);
}

// Block of NV + NH waves.  Waves 0 .. NV-1 run the chain: wave w owns value
// columns 16vt .. 16vt + 15 and advances the state block by block from the
// staged rows and the prepared matrices.  The helpers behind them: during group g
// helper hw stages block NH(g+1) + hw's k, q, v rows into the other buffer and
// forms that block's matrices, so the chain waves' matrix cores share their SIMD
// with the helpers' products and the helpers' VALU and LDS work fills the chain's
// dependency stalls.  One barrier per group of NH blocks.
template <class D, bool BF, bool AL>
__global__ __launch_bounds__(D::NT) void ut_fwd_k(const void* __restrict__ q, const void* __restrict__ k,
                                                  const void* __restrict__ v, const float* __restrict__ alpha,
                                                  const float* __restrict__ beta, float* __restrict__ o,
                                                  float* __restrict__ ws_u, float* __restrict__ ckpt,
                                                  float* __restrict__ rec, int B, int T, int H, int nslots) {
    constexpr int NH = D::NH, NV = D::NV;
    static_assert(D::F_LDS <= 160 * 1024, "forward LDS");
    extern __shared__ float lds[];
    // h*B + b, and the column split: a unit's blocks lie B*H apart (on one XCD
    // where that is a multiple of 8)
    const int vs = D::VS > 1 ? blockIdx.x / (B * H) : 0;
    const int unit = blockIdx.x - vs * (B * H);
    const int h = unit / B, b = unit - h * B;
    // the wave index, uniform in a scalar register (so are the block indices and
    // buffer offsets derived from it)
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const long d = (long)H * D::DH;
    const long ubase = (long)b * T * d + (long)h * D::DH;
    const int NC = (T + C - 1) / C;
    const int v0 = vs * NV * 16;
    FRes R;
    {
        const unsigned els = (unsigned)((T - 1) * d + D::DH);   // the unit's columns of rows t < T
        const unsigned rows = (BF ? 2u : 4u) * els;
        R.q = make_rsrc(at_el<BF>(q, ubase), rows);
        R.k = make_rsrc(at_el<BF>(k, ubase), rows);
        R.v = make_rsrc(at_el<BF>(v, ubase), rows);
        R.o = make_rsrc(o + ubase, 4u * els);
        const long gbase = (long)b * T * H + h;
        const unsigned grow = 4u * (unsigned)((T - 1) * H + 1);
        R.al = make_rsrc(alpha + gbase, grow);
        R.be = make_rsrc(beta + gbase, grow);
        R.u = make_rsrc(ws_u + (long)unit * NC * D::U_BLK, 4u * (unsigned)(NC * D::U_BLK));
        R.ck = make_rsrc(ckpt + (long)unit * nslots * D::DH2, 4u * (unsigned)(nslots * D::DH2));
        // the records are the same in every split: the first writes them
        R.rec = make_rsrc(rec + (long)unit * NC * R_SZ, vs == 0 ? 4u * (unsigned)(NC * R_SZ) : 0u);
    }

    if (w >= NV) {
        const int hw = w - NV;
        float* scr = lds + D::F_SCR + hw * 256;
        Stage<D, BF> stg;
        float ga, gb;
        stage_load<D, BF, AL>(stg, min(hw, NC - 1), q, k, v, R, ubase, d, T, v0, lane);
        gate_load(ga, gb, min(hw, NC - 1), R, H, lane);
        stage_store(stg, lds + D::F_STG, hw, lane);
        if (hw < NC) helper_prep<D>(hw, lds + D::F_STG, ga, gb, lds + hw * P_SZ, scr, R.rec, T, hw, lane);
        stage_load<D, BF, AL>(stg, min(NH + hw, NC - 1), q, k, v, R, ubase, d, T, v0, lane);
        gate_load(ga, gb, min(NH + hw, NC - 1), R, H, lane);
        lds_barrier();
        for (int c0 = 0; c0 < NC; c0 += NH) {
            const int pn = c0 + NH + hw;
            float* nbuf = lds + D::F_STG + (((c0 / NH) + 1) & 1) * D::S_BUF;
            stage_store(stg, nbuf, hw, lane);
            const float a = ga, bb = gb;
            stage_load<D, BF, AL>(stg, min(pn + NH, NC - 1), q, k, v, R, ubase, d, T, v0, lane);
            gate_load(ga, gb, min(pn + NH, NC - 1), R, H, lane);
            if (pn < NC) helper_prep<D>(pn, nbuf, a, bb, lds + (pn % D::NSLOT) * P_SZ, scr, R.rec, T, hw, lane);
            lds_barrier();
        }
        return;
    }

    const int vt = vs * NV + w;
    float* ot = lds + D::F_OT + w * 3 * C * OTP;
    f32x4 S[D::NR];
#pragma unroll
    for (int r = 0; r < D::NR; ++r) S[r] = f32x4{0.f, 0.f, 0.f, 0.f};
    lds_barrier();
    const int NCF = T / C;
    for (int c0 = 0; c0 < NC; c0 += NH) {
        const float* buf = lds + D::F_STG + ((c0 / NH) & 1) * D::S_BUF;
        f32x4 S0[D::CAUSAL ? D::NR : 1];  // the state before the group
        if constexpr (D::CAUSAL)
#pragma unroll
            for (int r = 0; r < D::NR; ++r) S0[r] = S[r];
        float bad = 0.0f;  // NaN once a block of the group has sums that are not finite
        if (c0 + NH <= NCF) {
#pragma unroll
            for (int j = 0; j < NH; ++j) {
                const float o0 = chain_step<D, true, AL>(
                    S, buf + j * C * D::RK, buf + D::S_Q + j * C * D::RK, buf + D::S_V + j * C * D::RV,
                    lds + ((c0 + j) % D::NSLOT) * P_SZ, ot, c0 + j, o, R, ((NH % 2 ? c0 + j : j) & 1) == 0, ubase, d,
                    T, w, vt, lane);
                if constexpr (D::CAUSAL) bad = fmaf(o0, 0.0f, bad);
            }
        } else {
            for (int j = 0; j < NH && c0 + j < NC; ++j) {
                const float o0 = chain_step<D, false, AL>(
                    S, buf + j * C * D::RK, buf + D::S_Q + j * C * D::RK, buf + D::S_V + j * C * D::RV,
                    lds + ((c0 + j) % D::NSLOT) * P_SZ, ot, c0 + j, o, R, ((c0 + j) & 1) == 0, ubase, d, T, w, vt, lane);
                if constexpr (D::CAUSAL) bad = fmaf(o0, 0.0f, bad);
            }
        }
        if constexpr (D::CAUSAL) {
            if (any_bad(bad)) {
#pragma unroll
                for (int r = 0; r < D::NR; ++r) S[r] = S0[r];
#pragma unroll 1
                for (int j = 0; j < NH && c0 + j < NC; ++j) {
                    const int c = c0 + j;
                    if ((c & 1) == 0) ck_store<D>(R, c >> 1, S, ot + 2 * C * OTP, vt, lane);
                    f32x4 O, U;
                    chain_by_steps<D>(S, O, U, buf + j * C * D::RK, buf + D::S_Q + j * C * D::RK,
                                      buf + D::S_V + j * C * D::RV, lds + (c % D::NSLOT) * P_SZ, min(C, T - c * C), w,
                                      lane);
                    store_ou<D, false, AL>(O, U, ot, c, o, R, ubase, d, T, vt, lane);
                }
            }
        }
        lds_barrier();
    }
    ck_store<D>(R, (NC + 1) >> 1, S, ot + 2 * C * OTP, vt, lane);
}

// ================================================================= backward
//
// Reverse over the blocks, with X = dL/dS' the gradient of the state after the
// block (zero after the last step, as bptt_cpu starts, delta.rs:475-587), the
// block's gradients follow from the UT form (the oracle's chunked restatement):
//
//     dU = M^T dO + diag(Gamma[15][:]) K X,      Y = T^T dU,     dv = diag(beta) Y
//     X_prev = gamma_15 X + (diag(gamma) Q)^T dO - K^T diag(beta gamma) Y
//     dM = tril(dO U^T),   dL = -strict_tril(Y U^T),   dA = dL o beta_row o Gamma
//     dq = diag(gamma) dO S^T + (Gamma o dM) K
//     dk = -diag(beta gamma) Y S^T + diag(Gamma[15][:]) U X^T + (Gamma o dM)^T Q + (dA + dA^T) K
//     dbeta, dgamma, dGamma from row sums, dalpha from running products (no division).
//
// Eight waves per unit.  The four chain waves own value columns 16w .. 16w + 15
// of X (accumulator tiles, like the forward's state) and run only the X
// recurrence (K X, M^T dO, T^T dU, the update: 56 MFMAs per block) plus dv and
// their share of dO U^T and Y U^T.  They hand X (before its update) and Y over
// in LDS, and stage the k, q, dO, u rows of the block after theirs.  The four
// helper waves own key columns 16hw .. 16hw + 15 of dq and dk:
// one block behind the chain they form dO S^T, Y S^T, U X^T over all value
// columns (S from the forward's checkpoint, advanced by one block for odd
// blocks), dq and dk and their row
// sums; one more block behind, the L2-norm backward of dq, dk (from the row dots
// of all four helpers) and the stores.  One barrier per block.  The gate gradients
// need sums over all four helpers and all value columns: the helpers leave
// theirs in the workspace's backward scratch, and after the block loop all
// eight waves form dalpha, dbeta of every block from them.
// a helper's five row sums over its keys: q.dq, k.dk (to the epilogue, in LDS
// [hw][2][16]) and q.F, k.Zt, k.D (to the gate gradients, in the backward scratch)
constexpr int EP_RQ = 0, EP_RK = 1, EP_QF = 2, EP_ZK = 3, EP_KD = 4;
// per unit and block in the backward's scratch (GS_SZ floats): what the gate
// gradients need, written by the helpers with the block's products, read after
// the block loop
constexpr int GS_ROW = 0;                    // [hw][3][16]: q.F, k.Zt, k.D row sums per helper (at most 4)
constexpr int GS_DSS = 192;                  // [hw]: <X, S> per helper
constexpr int GS_YV = 196;                   // [16]: row sums of Y o V
constexpr int GS_DM = 256;                   // dM, accumulator layout [lane][4]
constexpr int GS_DL = 512;                   // dL
constexpr int GS_SZ = 768;
constexpr int NSB = 3;                       // stage buffers: block c in buffer c % 3
constexpr int WSCR = 2 * C * OTP + 128;      // per wave: two transpose tiles and a vector area
constexpr int SVO = 2 * C * OTP;             // the vector area's offset
// Backward LDS (floats).
template <class D>
struct BL {
    static constexpr int NR = D::NR, NV = D::NV, NH = D::NH;
    // a block's staged rows: k, q (key-wide), dO, u (this block's value columns)
    static constexpr int SB_K = 0, SB_Q = C * D::RK, SB_DO = 2 * C * D::RK, SB_U = SB_DO + C * D::RV;
    static constexpr int SB_BUF = SB_U + C * D::RV;
    // handed over by the chain: X tiles [r][w][lane][4] (checkpoint order); Y tiles
    // [w][lane] float4 = Y[n][16w + 4g ..]; per chain wave dO_w U_w^T and Y_w U_w^T
    // (accumulator layout) and the row sums of Y_w o V_w [w][16]
    static constexpr int HO_DS = 0, HO_Y = NR * NV * 256, HO_DM = HO_Y + NV * 256, HO_DL = HO_DM + NV * 256;
    static constexpr int HO_YV = HO_DL + NV * 256, HO_SZ = HO_YV + NV * 16;
    static constexpr int EP_SZ = NH * 2 * 16;
    static constexpr int B_STG = 0;
    static constexpr int B_HO = B_STG + NSB * SB_BUF;
    static constexpr int B_EP = B_HO + 2 * HO_SZ;
    static constexpr int B_SCR = B_EP + 2 * EP_SZ;
    static constexpr int B_LOOP = B_SCR + D::NWT * WSCR;
    static constexpr int B_TAIL = D::NWT * 4 * WSCR;     // the gate tail's scratch, over the loop's
    static constexpr int B_END = B_LOOP > B_TAIL ? B_LOOP : B_TAIL;
    static constexpr size_t B_LDS = (size_t)B_END * 4;
    static_assert(B_LDS <= 160 * 1024 && B_HO % 4 == 0 && B_EP % 4 == 0 && B_SCR % 4 == 0, "backward LDS");
};

// 16x16 tile in the accumulator layout (lane (g, n) holds X[4g + j][n]) ->
// lane (g, n) receives X[n][4g .. 4g + 3].
ASCA_DEV float4 tile_t(const f32x4& x, float* __restrict__ st, int lane) {
    const int n = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) st[(4 * g + j) * OTP + n] = x[j];
    wave_sync();
    const float4 r = *reinterpret_cast<const float4*>(st + n * OTP + 4 * g);
    wave_sync();
    return r;
}

// Values held by lane t of each 16-lane row (the same in every row) -> lane
// (g, n) receives those of lanes 4g .. 4g + 3.
ASCA_DEV float4 rows4(float x, float* __restrict__ sv, int lane) {
    if (lane < 16) sv[lane] = x;
    wave_sync();
    const float4 r = *reinterpret_cast<const float4*>(sv + 4 * (lane >> 4));
    wave_sync();
    return r;
}

// rows4 for several values at once (one LDS round trip).
template <int NQ>
ASCA_DEV void rows4x(const float (&x)[NQ], float4 (&out)[NQ], float* __restrict__ sv, int lane) {
    if (lane < 16) {
#pragma unroll
        for (int e = 0; e < NQ; ++e) sv[16 * e + lane] = x[e];
    }
    wave_sync();
#pragma unroll
    for (int e = 0; e < NQ; ++e) out[e] = *reinterpret_cast<const float4*>(sv + 16 * e + 4 * (lane >> 4));
    wave_sync();
}

// Two 16x16 accumulator tiles transposed at once (see tile_t).
ASCA_DEV void tile_t2(const f32x4& x, const f32x4& y, float4& xt, float4& yt, float* __restrict__ st, int lane) {
    const int n = lane & 15, g = lane >> 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        st[(4 * g + j) * OTP + n] = x[j];
        st[C * OTP + (4 * g + j) * OTP + n] = y[j];
    }
    wave_sync();
    xt = *reinterpret_cast<const float4*>(st + n * OTP + 4 * g);
    yt = *reinterpret_cast<const float4*>(st + C * OTP + n * OTP + 4 * g);
    wave_sync();
}

// Exclusive suffix product over each 16-lane row: lane m gets prod_{m<s<16} x_s.
ASCA_DEV float suffix_excl_prod(float x) {
    x *= dpp_or<0x101>(1.0f, x);
    x *= dpp_or<0x102>(1.0f, x);
    x *= dpp_or<0x104>(1.0f, x);
    x *= dpp_or<0x108>(1.0f, x);
    return dpp_or<0x101>(1.0f, x);
}

template <bool AL>
ASCA_DEV void store4(float* __restrict__ p, float4 x) {
    if constexpr (AL) *reinterpret_cast<float4*>(p) = x;
    else { p[0] = x.x; p[1] = x.y; p[2] = x.z; p[3] = x.w; }
}

ASCA_DEV float4 f4scale(float s, float4 x) { return make_float4(s * x.x, s * x.y, s * x.z, s * x.w); }
ASCA_DEV float4 f4add(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }

struct BArgs {
    const void *q, *k, *v, *d_o;   // f32 or bf16 rows
    const float *alpha, *beta, *u, *ckpt, *rec, *qn, *kn;
    float *gq, *gk, *gv, *ga, *gb;
    float* gsc;   // scratch of this call: per block the sums of the gate gradients (GS_SZ floats)
    long ldx, ldv, ldg, d;   // row strides of gq, gk; of gv; of ga, gb; of the inputs
    long x_vs, g_vs;         // between the column splits' partial gq, gk and ga, gb
    int B, T, H, nslots, NC;
    int vs;                  // column split (filled in by the kernel)
    int di, ldxi, ldvi, ldgi;   // the strides as 32-bit ones (the launcher checks they fit)
};

// Buffer resources over the unit's part of every array the block loops read,
// made once per kernel (after the unit rebase): a load's lane offset is then
// loop-invariant and the block's offset a uniform register.  Rows past the
// sequence end lie outside the row resources and load as 0.
struct BRes {
    Rsrc ck, rec, nq, nk, v, k, q, dO, u;
};

template <class D, bool BF>
ASCA_DEV BRes bres_make(const BArgs& A) {
    BRes r;
    r.ck = make_rsrc(A.ckpt, 4u * (unsigned)(A.nslots * D::DH2));
    r.rec = make_rsrc(A.rec, 4u * (unsigned)(A.NC * R_SZ));
    const unsigned rows = (BF ? 2u : 4u) * (unsigned)((A.T - 1) * A.di + D::DH);   // the unit's columns of rows t < T
    r.v = make_rsrc(A.v, rows);
    r.k = make_rsrc(A.k, rows);
    r.q = make_rsrc(A.q, rows);
    r.dO = make_rsrc(A.d_o, rows);
    r.u = make_rsrc(A.u, 4u * (unsigned)(A.NC * D::U_BLK));
    const unsigned nrm = 4u * (unsigned)((A.T - 1) * A.H + 1);
    r.nq = make_rsrc(A.qn ? A.qn : A.rec, A.qn ? nrm : 0u);
    r.nk = make_rsrc(A.kn ? A.kn : A.rec, A.kn ? nrm : 0u);
    return r;
}

template <bool BF>
struct BChainIn {
    RawRow<BF> v;     // V[16c + n][16vt + 4g ..]
    float4 tr, mr;    // T and M of the block (accumulator layout)
    float4 gm, bg, gc;  // gamma, beta gamma, Gamma[15][.] of steps 4g .. 4g + 3
    float g15, bn;    // gamma_15; beta of step n
};

template <bool BF, bool AL>
ASCA_DEV void bchain_load(BChainIn<BF>& ci, int c, const BArgs& A, const BRes& R, int vt, int lane) {
    const int n = lane & 15, g = lane >> 4;
    if constexpr (AL) {
        // v of rows past the sequence end: 0 (outside the resource; their dv is not stored)
        ci.v = row_ld<BF>(R.v, (unsigned)(n * A.di + 16 * vt + 4 * g), (unsigned)(c * C * A.di));
    } else {
        const int t = min(c * C + n, A.T - 1);
        ci.v = row_ld_any<BF>(A.v, (unsigned)(t * A.di + 16 * vt + 4 * g));
    }
    const unsigned sb = 4u * (unsigned)(c * R_SZ);
    ci.tr = buf_load4(R.rec, 16u * ((R_T >> 2) + lane), sb);
    ci.mr = buf_load4(R.rec, 16u * ((R_M >> 2) + lane), sb);
    ci.gm = buf_load4(R.rec, 16u * ((RV_GAM >> 2) + g), sb);
    ci.bg = buf_load4(R.rec, 16u * ((RV_BG >> 2) + g), sb);
    ci.gc = buf_load4(R.rec, 16u * ((RV_GC >> 2) + g), sb);
    ci.g15 = buf_load1(R.rec, 4u * (RV_GAM + 15), sb);
    ci.bn = buf_load1(R.rec, 4u * (RV_BET + n), sb);
}

// Returns Y[0], not finite where a dU or dO is not (they are in every row of T^T dU).
// MASKED: dU[m] and Y[m] from the steps t >= m alone (see any_bad).
template <class D, bool BF, bool AL, bool MASKED = false>
ASCA_DEV float bchain_step(f32x4 (&X)[D::NR], const BChainIn<BF>& ci, const float* __restrict__ sb,
                          float* __restrict__ ho, float* __restrict__ scr, int c, const BArgs& A, int w, int vt,
                          int lane) {
    using L = BL<D>;
    constexpr int NR = D::NR;
    const int n = lane & 15, g = lane >> 4;
    const bool live = c * C + n < A.T;
    const float bt = ci.bn;
    const float g15 = ci.g15;
    const float4 gm = ci.gm, bg = ci.bg, gc = ci.gc;
    float4 kc[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) kc[r] = *reinterpret_cast<const float4*>(sb + L::SB_K + n * D::RK + 16 * r + 4 * g);
    float dO[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) dO[j] = sb[L::SB_DO + (4 * g + j) * D::RV + 16 * w + n];
    constexpr int NA = NR == 4 ? 1 : NR < 4 ? NR : 4;  // accumulators, as in the forward
    f32x4 kx[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) kx[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r0 = 0; r0 < NR; r0 += NA)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int a = 0; a < NA; ++a)
                if (r0 + a < NR) kx[a] = mfma4(el(kc[r0 + a], j), X[r0 + a][j], kx[a]);
    f32x4 dU;
#pragma unroll
    for (int j = 0; j < 4; ++j) dU[j] = el(gc, j) * acc_sum(kx, j);
    f32x4 Y = {0.f, 0.f, 0.f, 0.f};
    if constexpr (!MASKED && D::FINE) {
        const f32x4 md = mfma_sum(ci.mr, dO);
        float du[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) du[j] = dU[j] += md[j];
        Y = dU + mfma_sum(ci.tr, du);
    } else if constexpr (!MASKED) {
#pragma unroll
        for (int j = 0; j < 4; ++j) dU = mfma4(el(ci.mr, j), dO[j], dU);
#pragma unroll
        for (int j = 0; j < 4; ++j) Y = mfma4(el(ci.tr, j), dU[j], Y);
    } else {
        // M[t][m], T[t][m] at 4 (16 (t / 4) + m) + t % 4 of their record tiles
        const float* rec = A.rec + (unsigned)(c * R_SZ);
#pragma unroll 1
        for (int t = 0; t < C; ++t) {
            const float x = sb[L::SB_DO + t * D::RV + 16 * w + n];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float y = fmaf(rec[R_M + 4 * (16 * (t >> 2) + 4 * g + j) + (t & 3)], x, dU[j]);
                dU[j] = t >= 4 * g + j ? y : dU[j];
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) scr[(4 * g + j) * OTP + n] = dU[j];
        if constexpr (D::FINE) Y = dU;  // T's diagonal
        wave_sync();
#pragma unroll 1
        for (int t = 0; t < C; ++t) {
            const float x = scr[t * OTP + n];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float y = fmaf(rec[R_T + 4 * (16 * (t >> 2) + 4 * g + j) + (t & 3)], x, Y[j]);
                Y[j] = t > 4 * g + j || (!D::FINE && t == 4 * g + j) ? y : Y[j];
            }
        }
        wave_sync();
    }
    // hand X (the gradient after this block) and Y over to the helpers
#pragma unroll
    for (int r = 0; r < NR; ++r)
        *reinterpret_cast<float4*>(ho + L::HO_DS + ((r * D::NV + w) * 64 + lane) * 4) = tile_t(X[r], scr, lane);
    const float4 y4 = tile_t(Y, scr, lane);  // Y[n][16w + 4g ..]
    *reinterpret_cast<float4*>(ho + L::HO_Y + (w * 64 + lane) * 4) = y4;
    if (live) store4<AL>(A.gv + (unsigned)((c * C + n) * A.ldvi + 16 * vt + 4 * g), f4scale(bt, y4));
    // the wave's shares of dO U^T and Y U^T, and of the row sums of Y o V
    const float4 do4 = *reinterpret_cast<const float4*>(sb + L::SB_DO + n * D::RV + 16 * w + 4 * g);
    const float4 u4 = *reinterpret_cast<const float4*>(sb + L::SB_U + n * D::RV + 16 * w + 4 * g);
    f32x4 pm = {0.f, 0.f, 0.f, 0.f}, pl = pm;
    if constexpr (D::FINE) {
        pm = mfma_sum(do4, u4);
        pl = mfma_sum(y4, u4);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            pm = mfma4(el(do4, j), el(u4, j), pm);
            pl = mfma4(el(y4, j), el(u4, j), pl);
        }
    }
    *reinterpret_cast<float4*>(ho + L::HO_DM + (w * 64 + lane) * 4) = make_float4(pm[0], pm[1], pm[2], pm[3]);
    *reinterpret_cast<float4*>(ho + L::HO_DL + (w * 64 + lane) * 4) = make_float4(pl[0], pl[1], pl[2], pl[3]);
    const float4 vv = live ? widen(ci.v) : make_float4(0.f, 0.f, 0.f, 0.f);
    float yv = y4.x * vv.x + y4.y * vv.y + y4.z * vv.z + y4.w * vv.w;
    yv = add_xor32(add_xor16(yv));
    if (lane < 16) ho[L::HO_YV + w * 16 + lane] = yv;
    // X <- gamma_15 X + Q^T (diag(gamma) dO) - K^T (diag(beta gamma) Y)
    float dOg[4], Yb[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        dOg[j] = el(gm, j) * dO[j];
        Yb[j] = -el(bg, j) * Y[j];
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        X[r] *= g15;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float qv = sb[L::SB_Q + (4 * g + j) * D::RK + 16 * r + n];
            const float kv = sb[L::SB_K + (4 * g + j) * D::RK + 16 * r + n];
            X[r] = mfma4(qv, dOg[j], X[r]);
            X[r] = mfma4(kv, Yb[j], X[r]);
        }
    }
    return Y[0];
}

// The step of block c again, with the masked products.
template <class D, bool BF, bool AL>
ASCA_DEV void bchain_again(f32x4 (&X)[D::NR], const float* __restrict__ sb, float* __restrict__ ho,
                           float* __restrict__ scr, int c, const BArgs& A, const BRes& R, int w, int vt, int lane) {
    using L = BL<D>;
    const int n = lane & 15, g = lane >> 4;
    BChainIn<BF> ci;
    bchain_load<BF, AL>(ci, c, A, R, vt, lane);
    // X before its update, from the tiles handed over
#pragma unroll
    for (int r = 0; r < D::NR; ++r)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            X[r][j] = ho[L::HO_DS + ((r * D::NV + w) * 64 + 16 * (n >> 2) + 4 * g + j) * 4 + (n & 3)];
    wave_sync();
    bchain_step<D, BF, AL, true>(X, ci, sb, ho, scr, c, A, w, vt, lane);
}

template <class D>
struct BHelpIn {
    float4 sk[D::KS][D::NV];  // checkpoint before block c & ~1: S[16kt + n][16vt + 4g ..], key tile kt, value tile vt
    float gam, gcn, bt;  // gamma, Gamma[15][.], beta of step 16c + n
    float4 bb;           // beta of steps 4g .. 4g + 3
    float4 gq;           // block c - 1 (odd c): Gamma'[15][4i + g], i = 0..3
    float g15p;          // block c - 1: gamma'_15
    float qn, kn;        // norms of row 16c + n (1 for the raw gradients)
    float4 gr;           // Gamma of the block (accumulator layout)
};

template <class D, bool FUSED>
ASCA_DEV void bhelp_load(BHelpIn<D>& hi, int c, const BArgs& A, const BRes& R, int hw, int lane) {
    const int n = lane & 15, g = lane >> 4;
    const unsigned sc = 4u * (unsigned)((c >> 1) * D::DH2);
#pragma unroll
    for (int s = 0; s < D::KS; ++s)
#pragma unroll
        for (int cc = 0; cc < D::NV; ++cc)
            hi.sk[s][cc] =
                buf_load4(R.ck, 16u * (((hw * D::KS + s) * D::NR + (D::VS > 1 ? A.vs * D::NV : 0) + cc) * 64 + lane), sc);
    const unsigned sb = 4u * (unsigned)(c * R_SZ);
    hi.gam = buf_load1(R.rec, 4u * (RV_GAM + n), sb);
    hi.gcn = buf_load1(R.rec, 4u * (RV_GC + n), sb);
    hi.bt = buf_load1(R.rec, 4u * (RV_BET + n), sb);
    hi.bb = buf_load4(R.rec, 16u * ((RV_BET >> 2) + g), sb);
    const unsigned sp = 4u * (unsigned)(max(c - 1, 0) * R_SZ);  // block c - 1 is whole for odd c
    hi.gq = make_float4(buf_load1(R.rec, 4u * (RV_GC + g), sp), buf_load1(R.rec, 4u * (RV_GC + 4 + g), sp),
                        buf_load1(R.rec, 4u * (RV_GC + 8 + g), sp), buf_load1(R.rec, 4u * (RV_GC + 12 + g), sp));
    hi.g15p = buf_load1(R.rec, 4u * (RV_GAM + 15), sp);
    if constexpr (FUSED) {
        // rows past the sequence end read row T - 1 (their norms must stay finite)
        const unsigned t = (unsigned)min(c * C + n, A.T - 1);
        hi.qn = buf_load1(R.nq, 4u * t * (unsigned)A.H, 0u);
        hi.kn = buf_load1(R.nk, 4u * t * (unsigned)A.H, 0u);
    } else {
        hi.qn = 1.0f;
        hi.kn = 1.0f;
    }
    hi.gr = buf_load4(R.rec, 16u * ((R_G >> 2) + lane), sb);
}

ASCA_DEV float rowsum16(float x) { return group_sum<16>(x); }

// What a helper carries from the products of a block to its epilogue: dq, dk as
// row pieces (lane (g, n): row n, keys 16kt + 4g .. + 3 of its key tiles), ready to store.
template <class D>
struct BCarry {
    f32x4 dq[D::KS], dk[D::KS];   // raw dq, dk
    float4 qr[D::KS], kr[D::KS];  // qhat, khat at the same places
    float rq, rk;   // 1 / |q|, 1 / |k| of row n
};

// The products of block c for the helper's keys (KS tiles of 16), computed
// transposed (keys as accumulator rows): lane (g, n) holds row n (step) and keys
// 16kt + 4g + r, so the per-step gate factors are the lane's own, the row sums
// over keys are in-register sums plus two lane swaps, and dq, dk leave without a
// transpose.
// Returns a value that is not finite where a dq or dk of the lane is not.
// MASKED: dq and dk from the terms of their own steps alone (see any_bad).
template <class D, bool MASKED = false>
ASCA_DEV float bhelp_products(BCarry<D>& cy, const BHelpIn<D>& hi, const float* __restrict__ sb,
                             const float* __restrict__ sbp, const float* __restrict__ ho, float* __restrict__ ep,
                             float* __restrict__ scr, int c, const BArgs& A, int hw, int lane) {
    using L = BL<D>;
    constexpr int KS = D::KS, NV = D::NV, RK = D::RK, RV = D::RV;
    const int n = lane & 15, g = lane >> 4;
    const float bt = hi.bt, gam = hi.gam, gcn = hi.gcn;
    const float4 bb = hi.bb;                    // beta of rows 4g .. 4g + 3
    const float G[4] = {hi.gr.x, hi.gr.y, hi.gr.z, hi.gr.w};
    // The forward stores the state before every other block.  An odd block's
    // state follows from the block before (staged in `sbp`, always whole):
    // S = gamma'_15 S' + K'^T diag(Gamma'[15][:]) U', here for the helper's
    // keys (rows) as the transposed tiles of the checkpoint layout.
    float4 sk[KS][NV];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int cc = 0; cc < NV; ++cc) sk[s][cc] = hi.sk[s][cc];
    if (c & 1) {
        const float g15 = hi.g15p;
        const float4 gq = hi.gq;  // Gamma'[15][4i + g], i = 0..3
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            float kg[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                kg[i] = el(gq, i) * sbp[L::SB_K + (4 * i + g) * RK + 16 * (hw * KS + s) + n];
#pragma unroll
            for (int cc = 0; cc < NV; ++cc) {
                f32x4 t4 = {g15 * sk[s][cc].x, g15 * sk[s][cc].y, g15 * sk[s][cc].z, g15 * sk[s][cc].w};
#pragma unroll
                for (int i = 0; i < 4; ++i) t4 = mfma4(sbp[L::SB_U + (4 * i + g) * RV + 16 * cc + n], kg[i], t4);
                sk[s][cc] = make_float4(t4[0], t4[1], t4[2], t4[3]);
            }
        }
    }
    // (dO S^T)^T, (Y S^T)^T, (U X^T)^T: keys x steps, over the block's value columns
    f32x4 F[KS], Zt[KS], Dx[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) F[s] = Zt[s] = Dx[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    float dss = 0.0f;
#pragma unroll
    for (int cc = 0; cc < NV; ++cc) {
        const float4 dO4 = *reinterpret_cast<const float4*>(sb + L::SB_DO + n * RV + 16 * cc + 4 * g);
        const float4 u4 = *reinterpret_cast<const float4*>(sb + L::SB_U + n * RV + 16 * cc + 4 * g);
        const float4 y4 = *reinterpret_cast<const float4*>(ho + L::HO_Y + (cc * 64 + lane) * 4);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const float4 x4 =
                *reinterpret_cast<const float4*>(ho + L::HO_DS + (((hw * KS + s) * NV + cc) * 64 + lane) * 4);
            // (a column split's value tiles apart: their sums are half of what is added)
            f32x4 f = {0.f, 0.f, 0.f, 0.f}, z = f, d = f;
            if constexpr (D::VS == 1) {
                f = F[s];
                z = Zt[s];
                d = Dx[s];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f = mfma4(el(sk[s][cc], j), el(dO4, j), f);
                z = mfma4(el(sk[s][cc], j), el(y4, j), z);
                d = mfma4(el(x4, j), el(u4, j), d);
                dss += el(x4, j) * el(sk[s][cc], j);
            }
            F[s] = D::VS == 1 ? f : F[s] + f;
            Zt[s] = D::VS == 1 ? z : Zt[s] + z;
            Dx[s] = D::VS == 1 ? d : Dx[s] + d;
        }
    }
    // dM = tril(dO U^T), dL = -strict_tril(Y U^T) from the chain waves' shares
    float4 pm = *reinterpret_cast<const float4*>(ho + L::HO_DM + lane * 4);
    float4 pl = *reinterpret_cast<const float4*>(ho + L::HO_DL + lane * 4);
#pragma unroll
    for (int w = 1; w < NV; ++w) {
        pm = f4add(pm, *reinterpret_cast<const float4*>(ho + L::HO_DM + (w * 64 + lane) * 4));
        pl = f4add(pl, *reinterpret_cast<const float4*>(ho + L::HO_DL + (w * 64 + lane) * 4));
    }
    f32x4 dM, dL, GdM, dA;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int t = 4 * g + j;
        dM[j] = n <= t ? el(pm, j) : 0.0f;
        dL[j] = n < t ? -el(pl, j) : 0.0f;
        GdM[j] = G[j] * dM[j];
        dA[j] = dL[j] * el(bb, j) * G[j];
    }
    float4 gdmt, dat;  // (Gamma o dM)[n][4g ..], dA[n][4g ..]
    tile_t2(GdM, dA, gdmt, dat, scr, lane);
    float rs[5];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const int k0 = 16 * (hw * KS + s);
        float kb[4], qb[4];  // K, Q[4g + j][k0 + n]
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            kb[j] = sb[L::SB_K + (4 * g + j) * RK + k0 + n];
            qb[j] = sb[L::SB_Q + (4 * g + j) * RK + k0 + n];
        }
        const float4 qr = *reinterpret_cast<const float4*>(sb + L::SB_Q + n * RK + k0 + 4 * g);
        const float4 kr = *reinterpret_cast<const float4*>(sb + L::SB_K + n * RK + k0 + 4 * g);
        // dq^T = gamma o F^T + K^T (Gamma o dM)^T,
        // dk^T = Gamma[15] o Dx^T - beta gamma o Zt^T + Q^T (Gamma o dM) + K^T (dA + dA^T)
        f32x4 dq, dk;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            dq[j] = gam * F[s][j];
            dk[j] = gcn * Dx[s][j] - bt * gam * Zt[s][j];
        }
        if constexpr (!MASKED && D::FINE) {
            const float gd[4] = {GdM[0], GdM[1], GdM[2], GdM[3]};
            const float as[4] = {dA[0] + dat.x, dA[1] + dat.y, dA[2] + dat.z, dA[3] + dat.w};
            const float gt[4] = {gdmt.x, gdmt.y, gdmt.z, gdmt.w};
            dq += mfma_sum(kb, gt);
            dk += mfma_sum(qb, gd) + mfma_sum(kb, as);
        } else if constexpr (!MASKED) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                dq = mfma4(kb[j], el(gdmt, j), dq);
                dk = mfma4(qb[j], GdM[j], dk);
                dk = mfma4(kb[j], dA[j] + el(dat, j), dk);
            }
        } else {  // (Gamma o dM and dA are in scr)
#pragma unroll 1
            for (int m = 0; m < C; ++m) {
                const float4 km = *reinterpret_cast<const float4*>(sb + L::SB_K + m * RK + k0 + 4 * g);
                const float4 qm = *reinterpret_cast<const float4*>(sb + L::SB_Q + m * RK + k0 + 4 * g);
                const float gnm = scr[n * OTP + m], gmn = scr[m * OTP + n];
                const float a = scr[(C + max(m, n)) * OTP + min(m, n)];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (m <= n) dq[j] = fmaf(el(km, j), gnm, dq[j]);
                    if (m >= n) dk[j] = fmaf(el(qm, j), gmn, dk[j]);
                    if (m != n) dk[j] = fmaf(el(km, j), a, dk[j]);
                }
            }
        }
        // row sums over the helper's keys: in-register, then over the four lanes of
        // row n (lane bits 4 and 5)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool first = s == 0 && j == 0;
            rs[EP_RQ] = first ? el(qr, j) * dq[j] : rs[EP_RQ] + el(qr, j) * dq[j];
            rs[EP_RK] = first ? el(kr, j) * dk[j] : rs[EP_RK] + el(kr, j) * dk[j];
            rs[EP_QF] = first ? el(qr, j) * F[s][j] : rs[EP_QF] + el(qr, j) * F[s][j];
            rs[EP_ZK] = first ? el(kr, j) * Zt[s][j] : rs[EP_ZK] + el(kr, j) * Zt[s][j];
            rs[EP_KD] = first ? el(kr, j) * Dx[s][j] : rs[EP_KD] + el(kr, j) * Dx[s][j];
        }
        cy.dq[s] = dq;
        cy.dk[s] = dk;
        cy.qr[s] = qr;
        cy.kr[s] = kr;
    }
    const float qkb = rs[EP_RQ] + rs[EP_RK];
#pragma unroll
    for (int e = 0; e < 5; ++e) rs[e] = add_xor32(add_xor16(rs[e]));
    float* gs = A.gsc + (unsigned)(c * GS_SZ);
    if (lane < 16) {
        ep[(hw * 2 + EP_RQ) * 16 + n] = rs[EP_RQ];
        ep[(hw * 2 + EP_RK) * 16 + n] = rs[EP_RK];
#pragma unroll
        for (int e = EP_QF; e <= EP_KD; ++e) gs[GS_ROW + (hw * 3 + e - EP_QF) * 16 + n] = rs[e];
    }
    dss = wave_sum(dss);
    if (lane == 0) gs[GS_DSS + hw] = dss;
    if (hw == 0) {
        if (lane < 16) {
            float yv = 0.0f;
#pragma unroll
            for (int w = 0; w < NV; ++w) yv += ho[L::HO_YV + w * 16 + lane];
            gs[GS_YV + lane] = yv;
        }
        *reinterpret_cast<float4*>(gs + GS_DM + 4 * lane) = make_float4(dM[0], dM[1], dM[2], dM[3]);
        *reinterpret_cast<float4*>(gs + GS_DL + 4 * lane) = make_float4(dL[0], dL[1], dL[2], dL[3]);
    }
    cy.rq = __builtin_amdgcn_rcpf(hi.qn);
    cy.rk = __builtin_amdgcn_rcpf(hi.kn);
    return qkb;
}

template <class D, bool FUSED, bool AL>
ASCA_DEV void bhelp_epilogue(const BCarry<D>& cy, const float* __restrict__ ep, int c, const BArgs& A, int hw,
                             int lane) {
    const int n = lane & 15, g = lane >> 4;
    float dotq = 0.0f, dotk = 0.0f;
    if constexpr (FUSED) {
        dotq = ep[EP_RQ * 16 + n];
        dotk = ep[EP_RK * 16 + n];
#pragma unroll
        for (int w = 1; w < D::NH; ++w) {
            dotq += ep[(w * 2 + EP_RQ) * 16 + n];
            dotk += ep[(w * 2 + EP_RK) * 16 + n];
        }
    }
#pragma unroll
    for (int s = 0; s < D::KS; ++s) {
        f32x4 dq = cy.dq[s], dk = cy.dk[s];
        if constexpr (FUSED) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                dq[j] = (dq[j] - el(cy.qr[s], j) * dotq) * cy.rq;
                dk[j] = (dk[j] - el(cy.kr[s], j) * dotk) * cy.rk;
            }
        }
        if (c * C + n < A.T) {
            const unsigned o = (unsigned)((c * C + n) * A.ldxi + 16 * (hw * D::KS + s) + 4 * g);
            store4<AL>(A.gq + o, make_float4(dq[0], dq[1], dq[2], dq[3]));
            store4<AL>(A.gk + o, make_float4(dk[0], dk[1], dk[2], dk[3]));
        }
    }
}

// Gate gradients of block c (dalpha, dbeta and their sigmoid backward), run by
// one wave from the sums the helpers left in the scratch (loaded with the
// block's record, one block ahead); lane t of each row is step t.
template <int NH>
struct BGateIn {
    float4 ar, bq, gr;  // K K^T, Q K^T, Gamma of the block (accumulator layout)
    float a, b;         // gates of step 16c + n (as loaded, for the sigmoid backward)
    float gam, bm;      // gamma, beta of step 16c + n (beta 0 past the sequence end)
    float4 bb;          // beta of steps 4g .. 4g + 3 (0 past the sequence end)
    float4 pm, pl;      // dM, dL (accumulator layout)
    float rw[3][NH];    // the helpers' row sums q.F, k.Zt, k.D of row n
    float ds[NH];       // the helpers' <X, S>
    float yv;           // row sum of Y o V of row n
};

template <bool FUSED, int NH>
ASCA_DEV void bgate_load(BGateIn<NH>& gi, int c, const BArgs& A, int lane) {
    const float4* rq = reinterpret_cast<const float4*>(A.rec + (unsigned)(c * R_SZ));
    gi.ar = rq[(R_A >> 2) + lane];
    gi.bq = rq[(R_BQ >> 2) + lane];
    gi.gr = rq[(R_G >> 2) + lane];
    if constexpr (FUSED) {  // (the raw gradients' callers may have no gates at hand)
        const int t = min(c * C + (lane & 15), A.T - 1);
        gi.a = A.alpha[(unsigned)(t * A.H)];
        gi.b = A.beta[(unsigned)(t * A.H)];
    }
    const int n = lane & 15;
    const float* rb = A.rec + (unsigned)(c * R_SZ);
    gi.gam = rb[RV_GAM + n];
    gi.bm = rb[RV_BET + n];
    gi.bb = rq[(RV_BET >> 2) + (lane >> 4)];
    const float* gs = A.gsc + (unsigned)(c * GS_SZ);
    gi.pm = *reinterpret_cast<const float4*>(gs + GS_DM + 4 * lane);
    gi.pl = *reinterpret_cast<const float4*>(gs + GS_DL + 4 * lane);
#pragma unroll
    for (int w = 0; w < NH; ++w) {
#pragma unroll
        for (int e = 0; e < 3; ++e) gi.rw[e][w] = gs[GS_ROW + (w * 3 + e) * 16 + n];
        gi.ds[w] = gs[GS_DSS + w];
    }
    gi.yv = gs[GS_YV + n];
}

// The gate gradients of NB blocks at once (block cs[i] from gin[i]): every
// phase runs over all NB blocks before the next, so their dependency chains
// interleave and the LDS transposes share their wave syncs.  scr holds NB
// areas of WSCR floats.  Blocks past the sequence end (clamped loads) store
// nothing: their rows lie outside the resources' range.
template <bool FUSED, bool CAUSAL, int NH, int NB>
ASCA_DEV void bgate_batch(const BGateIn<NH> (&gin)[NB], const int (&cs)[NB], float* __restrict__ scr,
                          const BArgs& A, Rsrc rga, Rsrc rgb, int lane) {
    const int n = lane & 15, g = lane >> 4;
    float szk[NB], dgam[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const BGateIn<NH>& gi = gin[i];
        float sqf = 0.f, dss = 0.f;
        szk[i] = 0.f;
#pragma unroll
        for (int w = 0; w < NH; ++w) {
            sqf += gi.rw[0][w];
            szk[i] += gi.rw[1][w];
            dss += gi.ds[w];
        }
        dgam[i] = -gi.bm * szk[i] + sqf + (n == C - 1 ? dss : 0.0f);
        scr[i * WSCR + SVO + 16 * g + n] = dgam[i];   // every lane: row n of copy g
    }
    wave_sync();
    float4 dg4[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) dg4[i] = *reinterpret_cast<const float4*>(scr + i * WSCR + SVO + 4 * g);
    wave_sync();
    // dGamma (strict lower part), row sums of dL o Gamma o A, the first term of dalpha
    f32x4 dgs[NB];
    float t1[NB], rb[NB][4];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const BGateIn<NH>& gi = gin[i];
        float skd = 0.f;
#pragma unroll
        for (int w = 0; w < NH; ++w) skd += gi.rw[2][w];
        t1[i] = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = 4 * g + j;
            const float dL = el(gi.pl, j), G = el(gi.gr, j);
            rb[i][j] = rowsum16(dL * G * el(gi.ar, j));
            dgs[i][j] = n < t ? el(gi.pm, j) * el(gi.bq, j) + dL * el(gi.bb, j) * el(gi.ar, j) +
                                    (t == C - 1 ? skd : 0.0f)
                              : 0.0f;
            t1[i] += G * el(dg4[i], j);
        }
        t1[i] = add_xor32(add_xor16(t1[i]));
    }
    // R = dGs Gamma'^T with Gamma'[m][i] = Gamma[m-1][i] (the row above, zero for
    // m = 0) on the matrix cores, then sum_t Gamma[t][m] R[t][m]
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        float* st = scr + i * WSCR;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            st[(4 * g + j) * OTP + n] = dgs[i][j];
            st[C * OTP + (4 * g + j) * OTP + n] = el(gin[i].gr, j);
        }
        *reinterpret_cast<float4*>(st + SVO + 64 + 4 * g) = make_float4(rb[i][0], rb[i][1], rb[i][2], rb[i][3]);
    }
    wave_sync();
    float dal[NB], dbe[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const float* st = scr + i * WSCR;
        const float4 dgst = *reinterpret_cast<const float4*>(st + n * OTP + 4 * g);       // dGs[n][4g ..]
        const float4 gt = *reinterpret_cast<const float4*>(st + C * OTP + n * OTP + 4 * g);  // Gamma[n][4g ..]
        const float gp[4] = {dpp_or<0x111>(0.0f, gt.x), dpp_or<0x111>(0.0f, gt.y), dpp_or<0x111>(0.0f, gt.z),
                             dpp_or<0x111>(0.0f, gt.w)};   // Gamma[n-1][4g ..]
        f32x4 R = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) R = mfma4(el(dgst, j), gp[j], R);
        float t2 = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) t2 += el(gin[i].gr, j) * R[j];
        t2 = add_xor32(add_xor16(t2));
        const float gprev = dpp_or<0x111>(1.0f, gin[i].gam);   // gamma_{n-1}
        dal[i] = gprev * t1[i] + t2;
        if constexpr (CAUSAL) {
            if (any_bad(dal[i])) {  // dalpha of step n from the rows t >= n and columns before n
                float s1 = 0.0f, s2 = 0.0f;
#pragma unroll 1
                for (int t = 0; t < C; ++t) {
                    const float G = st[C * OTP + t * OTP + n];
                    float r = 0.0f;
#pragma unroll 1
                    for (int m = 0; m < C - 1; ++m) {
                        const float x = fmaf(st[t * OTP + m], st[C * OTP + max(n - 1, 0) * OTP + m], r);
                        r = m < n ? x : r;
                    }
                    const float x1 = fmaf(G, st[SVO + t], s1), x2 = fmaf(G, r, s2);
                    s1 = t >= n ? x1 : s1;
                    s2 = t >= n ? x2 : s2;
                }
                dal[i] = fmaf(gprev, s1, s2);
            }
        }
        // dbeta of step n: Y.V - gamma Z'.K + sum_l dL Gamma A (row n's sum from lane (n/4, .))
        const float rbn = st[SVO + 64 + n];
        dbe[i] = gin[i].yv - gin[i].gam * szk[i] + rbn;
    }
    wave_sync();
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        // every lane stores (the four lanes of row n hold the same values); rows
        // past the sequence end fall outside the resources and are dropped
        const unsigned r = 4u * (unsigned)((cs[i] * C + n) * A.ldgi);
        if constexpr (FUSED) {
            const float a = gin[i].a, b = gin[i].b;
            dal[i] *= a * (1.0f - a);
            dbe[i] *= b * (1.0f - b);
        }
        buf_store1(rga, r, dal[i]);
        buf_store1(rgb, r, dbe[i]);
    }
}

// Staging of block c's rows of k, q, dO and u by W waves (this one the hw-th):
// 16-byte pieces, piece e = 64 (W j + hw) + lane of each matrix.
template <class D, bool BF, int W>
struct BStage {
    static constexpr int NK = (D::NR + W - 1) / W, NU = (D::NV + W - 1) / W;
    RawRow<BF> k[NK], q[NK], d[NU];
    float4 u[NU];
};

template <class D, bool BF, bool AL, int W>
ASCA_DEV void bstage_load(BStage<D, BF, W>& st, int c, const BArgs& A, const BRes& R, int hw, int lane) {
    const unsigned so = (unsigned)(c * C * A.di);
    const int v0 = D::VS > 1 ? A.vs * D::NV * 16 : 0;
#pragma unroll
    for (int j = 0; j < st.NK; ++j) {
        if (D::NR % W && W * j + hw >= D::NR) continue;   // uniform
        const int e = 64 * (W * j + hw) + lane, r = e / (4 * D::NR), col = 4 * (e % (4 * D::NR));
        if constexpr (AL) {
            // rows past the sequence end load as 0 (outside the row resources)
            const unsigned vo = (unsigned)(r * A.di + col);
            st.k[j] = row_ld<BF>(R.k, vo, so);
            st.q[j] = row_ld<BF>(R.q, vo, so);
        } else {
            const unsigned off = (unsigned)(min(c * C + r, A.T - 1) * A.di + col);
            st.k[j] = row_ld_any<BF>(A.k, off);
            st.q[j] = row_ld_any<BF>(A.q, off);
        }
    }
#pragma unroll
    for (int j = 0; j < st.NU; ++j) {
        if (D::NV % W && W * j + hw >= D::NV) continue;   // uniform
        const int e = 64 * (W * j + hw) + lane, r = e / (4 * D::NV), cq = e % (4 * D::NV);
        if constexpr (AL)
            st.d[j] = row_ld<BF>(R.dO, (unsigned)(r * A.di + v0 + 4 * cq), so);
        else
            st.d[j] = row_ld_any<BF>(A.d_o, (unsigned)(min(c * C + r, A.T - 1) * A.di + v0 + 4 * cq));
        // u in the forward's tile layout: the tile of columns v0 + 16 (cq / 4), row r, columns 4 (cq % 4) ..
        st.u[j] = buf_load4(R.u, 4u * (unsigned)((v0 / 16 + (cq >> 2)) * 256 + r * 16 + 4 * (cq & 3)),
                            4u * (unsigned)(c * D::U_BLK));
    }
}

// WHOLE: the caller knows block c is whole (every block but the last is).
template <bool WHOLE, class D, bool BF, int W>
ASCA_DEV void bstage_store(const BStage<D, BF, W>& st, int c, float* __restrict__ sb, int T, int hw, int lane) {
    using L = BL<D>;
    const bool full = WHOLE || (c + 1) * C <= T;   // uniform
    const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int j = 0; j < st.NK; ++j) {
        if (D::NR % W && W * j + hw >= D::NR) continue;
        const int e = 64 * (W * j + hw) + lane, r = e / (4 * D::NR), col = 4 * (e % (4 * D::NR));
        const bool live = full || c * C + r < T;
        *reinterpret_cast<float4*>(sb + L::SB_K + r * D::RK + col) = live ? widen(st.k[j]) : z;
        *reinterpret_cast<float4*>(sb + L::SB_Q + r * D::RK + col) = live ? widen(st.q[j]) : z;
    }
#pragma unroll
    for (int j = 0; j < st.NU; ++j) {
        if (D::NV % W && W * j + hw >= D::NV) continue;
        const int e = 64 * (W * j + hw) + lane, r = e / (4 * D::NV), col = 4 * (e % (4 * D::NV));
        const bool live = full || c * C + r < T;
        *reinterpret_cast<float4*>(sb + L::SB_DO + r * D::RV + col) = live ? widen(st.d[j]) : z;
        *reinterpret_cast<float4*>(sb + L::SB_U + r * D::RV + col) = live ? st.u[j] : z;
    }
}

// After the block loop: the gate gradients of every block, block c on wave
// c mod NWT, four blocks of a wave at a time; the loop's LDS is free by then
// (the block's final barrier) and gives each wave four scratch areas.
template <class D, bool FUSED>
ASCA_DEV void bgate_tail(const BArgs& A, float* __restrict__ lds, int w, int lane) {
    constexpr int NB = 4;
    __syncthreads();   // the scratch writes of every wave are visible, the loop's LDS is free
    float* scr = lds + w * NB * WSCR;
    // the unit's rows of dalpha, dbeta: row t at t * ldg
    const unsigned gbytes = 4u * (unsigned)((A.T - 1) * A.ldgi + 1);
    const Rsrc rga = make_rsrc(A.ga, gbytes), rgb = make_rsrc(A.gb, gbytes);
    for (int c0 = w; c0 < A.NC; c0 += D::NWT * NB) {
        BGateIn<D::NH> gin[NB];
        int cs[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            cs[i] = c0 + D::NWT * i;                // past NC: rows beyond T, stores dropped
            bgate_load<FUSED>(gin[i], min(cs[i], A.NC - 1), A, lane);
        }
        bgate_batch<FUSED, D::CAUSAL, D::NH, NB>(gin, cs, scr, A, rga, rgb, lane);
    }
}

template <class D, bool BF, bool FUSED, bool AL>
__global__ __launch_bounds__(D::NT) void ut_bwd_k(BArgs A) {
    using L = BL<D>;
    constexpr int NV = D::NV, NH = D::NH;
    static_assert(D::VS == 1 || !FUSED, "a column split's sums are partial");
    extern __shared__ float lds[];
    {
        const int units = A.B * A.H;
        A.vs = D::VS > 1 ? blockIdx.x / units : 0;
        const int unit = blockIdx.x - A.vs * units;  // h*B + b
        const int h = unit / A.B;
        const int b = unit - h * A.B;
        const long ubase = (long)b * A.T * A.d + (long)h * D::DH;
        const long gbase = (long)b * A.T * A.H + h;
        const long rowbase = (long)b * A.T;
        // every pointer rebased on the unit: the per-block offsets are 32-bit
        A.q = at_el<BF>(A.q, ubase); A.k = at_el<BF>(A.k, ubase); A.v = at_el<BF>(A.v, ubase);
        A.d_o = at_el<BF>(A.d_o, ubase);
        A.u += (long)unit * A.NC * D::U_BLK;
        A.alpha += gbase; A.beta += gbase;
        if (A.qn) { A.qn += gbase; A.kn += gbase; }
        A.ckpt += (long)unit * A.nslots * D::DH2;
        A.rec += (long)unit * A.NC * R_SZ;
        A.gsc += (long)blockIdx.x * A.NC * GS_SZ;
        A.gq += A.vs * A.x_vs + rowbase * A.ldx + (long)h * D::DH;
        A.gk += A.vs * A.x_vs + rowbase * A.ldx + (long)h * D::DH;
        A.gv += rowbase * A.ldv + (long)h * D::DH;
        A.ga += A.vs * A.g_vs + rowbase * A.ldg + h; A.gb += A.vs * A.g_vs + rowbase * A.ldg + h;
    }
    // the wave index, uniform in a scalar register (so are the block indices and
    // buffer offsets derived from it)
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int NC = A.NC;
    const BRes R = bres_make<D, BF>(A);
    float* scr = lds + L::B_SCR + w * WSCR;
    if (w >= NV) {
        // helper: step s runs the epilogue of block NC + 1 - s and the products
        // of block NC - s (the chain waves stage the rows).  Every global load is
        // made two steps ahead into buffer s & 1, unconditionally (clamped block
        // indices), and consumed at the start of its step, so no wait falls on a
        // recent memory operation.
        const int hw = w - NV;
        BHelpIn<D> hin[2];
        BCarry<D> cy;
        {
            BStage<D, BF, NH> st0;
            bstage_load<D, BF, AL, NH>(st0, NC - 1, A, R, hw, lane);
            bstage_store<false>(st0, NC - 1, lds + L::B_STG + ((NC - 1) % NSB) * L::SB_BUF, A.T, hw, lane);
        }
        bhelp_load<D, FUSED>(hin[1], NC - 1, A, R, hw, lane);
        bhelp_load<D, FUSED>(hin[0], max(NC - 2, 0), A, R, hw, lane);
        lds_barrier();
        lds_barrier();  // step 0: the chain's first block
        // steps 1 .. NC: the products of block cp = NC - s on every path (the
        // carried dq, dk are then never copied), the epilogue of cp + 1 from
        // step 2 on; step NC + 1: the epilogue of block 0
        auto step = [&](int s, BHelpIn<D>& hb) {
            const int cp = NC - s;
            if (s >= 2)
                bhelp_epilogue<D, FUSED, AL>(cy, lds + L::B_EP + ((cp + 1) & 1) * L::EP_SZ, cp + 1, A, hw, lane);
            auto products = [&](const BHelpIn<D>& in, auto Masked) {
                return bhelp_products<D, decltype(Masked)::value>(
                    cy, in, lds + L::B_STG + (cp % NSB) * L::SB_BUF, lds + L::B_STG + ((cp + NSB - 1) % NSB) * L::SB_BUF,
                    lds + L::B_HO + (cp & 1) * L::HO_SZ, lds + L::B_EP + (cp & 1) * L::EP_SZ, scr, cp, A, hw, lane);
            };
            const float qk = products(hb, std::false_type{});
            bhelp_load<D, FUSED>(hb, max(cp - 2, 0), A, R, hw, lane);
            if constexpr (D::CAUSAL) {
                if (any_bad(qk)) {
                    BHelpIn<D> h2;
                    bhelp_load<D, FUSED>(h2, cp, A, R, hw, lane);
                    products(h2, std::true_type{});
                }
            }
            lds_barrier();
        };
        for (int s = 1; s <= NC; s += 2) {
            step(s, hin[1]);
            if (s + 1 <= NC) step(s + 1, hin[0]);
        }
        bhelp_epilogue<D, FUSED, AL>(cy, lds + L::B_EP, 0, A, hw, lane);
        lds_barrier();
        bgate_tail<D, FUSED>(A, lds, w, lane);
        return;
    }
    // chain: step s runs block NC - 1 - s and stages the rows of the block after
    // (NC - 2 - s) into its buffer, which no wave reads in step s
    const int vt = (D::VS > 1 ? A.vs * NV : 0) + w;
    f32x4 X[D::NR];
#pragma unroll
    for (int r = 0; r < D::NR; ++r) X[r] = f32x4{0.f, 0.f, 0.f, 0.f};
    BChainIn<BF> cb[2];
    // rows staged two steps ahead (one at dh > 64, where two sets spill)
    constexpr int SETS = D::NR > 4 ? 1 : 2;
    BStage<D, BF, NV> sg[SETS];
    bchain_load<BF, AL>(cb[0], NC - 1, A, R, vt, lane);
    bchain_load<BF, AL>(cb[1], max(NC - 2, 0), A, R, vt, lane);
    bstage_load<D, BF, AL, NV>(sg[0], max(NC - 2, 0), A, R, w, lane);
    if constexpr (SETS == 2) bstage_load<D, BF, AL, NV>(sg[1], max(NC - 3, 0), A, R, w, lane);
    lds_barrier();
    for (int s = 0; s < NC; ++s) {
        const int c = NC - 1 - s;
        float y0;
        // the chain's inputs are loaded two steps ahead into buffer s & 1
        // (static indices: no register copies; X is updated on every path)
        if ((s & 1) == 0) {
            // block c - 1 < NC - 1 is whole (only the last block can be partial)
            if (c >= 1)
                bstage_store<true>(sg[0], c - 1, lds + L::B_STG + ((c - 1) % NSB) * L::SB_BUF, A.T, w, lane);
            y0 = bchain_step<D, BF, AL>(X, cb[0], lds + L::B_STG + (c % NSB) * L::SB_BUF,
                                        lds + L::B_HO + (c & 1) * L::HO_SZ, scr, c, A, w, vt, lane);
            bchain_load<BF, AL>(cb[0], max(c - 2, 0), A, R, vt, lane);
            bstage_load<D, BF, AL, NV>(sg[0], max(c - 1 - SETS, 0), A, R, w, lane);
        } else {
            // block c - 1 < NC - 1 is whole (only the last block can be partial)
            if (c >= 1)
                bstage_store<true>(sg[SETS - 1], c - 1, lds + L::B_STG + ((c - 1) % NSB) * L::SB_BUF, A.T, w, lane);
            y0 = bchain_step<D, BF, AL>(X, cb[1], lds + L::B_STG + (c % NSB) * L::SB_BUF,
                                        lds + L::B_HO + (c & 1) * L::HO_SZ, scr, c, A, w, vt, lane);
            bchain_load<BF, AL>(cb[1], max(c - 2, 0), A, R, vt, lane);
            bstage_load<D, BF, AL, NV>(sg[SETS - 1], max(c - 1 - SETS, 0), A, R, w, lane);
        }
        if constexpr (D::CAUSAL)
            if (any_bad(y0))
                bchain_again<D, BF, AL>(X, lds + L::B_STG + (c % NSB) * L::SB_BUF, lds + L::B_HO + (c & 1) * L::HO_SZ, scr,
                                        c, A, R, w, vt, lane);
        lds_barrier();
    }
    // the helpers' last two steps (products of block 0, then its epilogue)
    lds_barrier();
    lds_barrier();
    bgate_tail<D, FUSED>(A, lds, w, lane);
}

}  // namespace ut64

static bool ut_aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <class D, bool BF, bool AL>
static int launch_ut_fwd_t(const void* q, const void* k, const void* v, const float* alpha, const float* beta,
                           float* o, const DeltaWs& ws, int B, int T, int H, hipStream_t st) {
    if (int arc = allow_lds(reinterpret_cast<const void*>(&ut64::ut_fwd_k<D, BF, AL>), D::F_LDS)) return arc;
    int rc = pre_launch("ut_fwd");
    if (rc) return rc;
    hipLaunchKernelGGL((ut64::ut_fwd_k<D, BF, AL>), dim3(B * H * D::VS), dim3(D::NT), D::F_LDS, st, q, k, v, alpha,
                       beta, o, ws.sk, ws.ckpt, ws.rec, B, T, H, ws.nslots);
    return post_launch("ut_fwd");
}

// Floats of the backward's gate-sum scratch (ut64::BArgs::gsc).
inline size_t ut_bwd_scratch_floats(long blocks, int NC) { return (size_t)blocks * NC * ut64::GS_SZ; }

template <class D, bool BF, bool FUSED, bool AL>
static int launch_ut_bwd_t(const ut64::BArgs& a, hipStream_t st) {
    if (int arc = allow_lds(reinterpret_cast<const void*>(&ut64::ut_bwd_k<D, BF, FUSED, AL>), ut64::BL<D>::B_LDS))
        return arc;
    int rc = pre_launch("ut_bwd");
    if (rc) return rc;
    hipLaunchKernelGGL((ut64::ut_bwd_k<D, BF, FUSED, AL>), dim3(a.B * a.H * D::VS), dim3(D::NT), ut64::BL<D>::B_LDS,
                       st, a);
    return post_launch("ut_bwd");
}

// The head widths (key tiles NR): forward and backward splits.
template <int NR> struct UtDims;
template <> struct UtDims<1> { using F = ut64::Dim<1, 1, 1>; using B = ut64::Dim<1, 1, 1>; };
template <> struct UtDims<2> { using F = ut64::Dim<2, 2, 2>; using B = ut64::Dim<2, 2, 2>; };
template <> struct UtDims<3> { using F = ut64::Dim<3, 3, 3>; using B = ut64::Dim<3, 3, 3>; };
template <> struct UtDims<4> { using F = ut64::Dim<4, 4, 4>; using B = ut64::Dim<4, 4, 4>; };
template <> struct UtDims<6> { using F = ut64::Dim<6, 2, 2>; using B = ut64::Dim<6, 2, 3>; };
template <> struct UtDims<8> { using F = ut64::Dim<8, 2, 2>; using B = ut64::Dim<8, 2, 4>; };

// One head width's variants (the f32 dh = 64 forward and fused, aligned backward
// apart, which delta_ut64.hip launches).  Raw gradients where BF or the columns split.
template <int NR>
static int ut_fwd_variant(const void* q, const void* k, const void* v, bool bf, bool al, const float* alpha,
                          const float* beta, float* o, const DeltaWs& ws, int B, int T, int H, hipStream_t st) {
    using D = typename UtDims<NR>::F;
    if (bf)
        return al ? launch_ut_fwd_t<D, true, true>(q, k, v, alpha, beta, o, ws, B, T, H, st)
                  : launch_ut_fwd_t<D, true, false>(q, k, v, alpha, beta, o, ws, B, T, H, st);
    return al ? launch_ut_fwd_t<D, false, true>(q, k, v, alpha, beta, o, ws, B, T, H, st)
              : launch_ut_fwd_t<D, false, false>(q, k, v, alpha, beta, o, ws, B, T, H, st);
}
template <int NR>
static int ut_bwd_variant(const ut64::BArgs& a, bool bf, bool fused, bool al, hipStream_t st) {
    using D = typename UtDims<NR>::B;
    if (bf)
        return fused ? fail(ASCA_ERR_UNSUPPORTED, "ut_bwd: fused gradients of bf16 rows")
               : al  ? launch_ut_bwd_t<D, true, false, true>(a, st)
                     : launch_ut_bwd_t<D, true, false, false>(a, st);
    if constexpr (D::VS == 1) {
        if (fused) {
            if constexpr (NR != 4)
                if (al) return launch_ut_bwd_t<D, false, true, true>(a, st);
            return launch_ut_bwd_t<D, false, true, false>(a, st);
        }
    }
    return al ? launch_ut_bwd_t<D, false, false, true>(a, st) : launch_ut_bwd_t<D, false, false, false>(a, st);
}

int launch_ut_fwd_other(const void* q, const void* k, const void* v, bool bf, bool al, const float* alpha,
                        const float* beta, float* o, const DeltaWs& ws, int B, int T, int H, int dh, hipStream_t st);
int launch_ut_fwd_n(const void* q, const void* k, const void* v, bool bf, bool al, const float* alpha,
                    const float* beta, float* o, const DeltaWs& ws, int B, int T, int H, int dh, hipStream_t st);
int launch_ut_bwd_other(const ut64::BArgs& a, int dh, bool bf, bool fused, bool al, hipStream_t st);
int launch_ut_bwd_n(const ut64::BArgs& a, int dh, bool bf, bool fused, bool al, hipStream_t st);

}  // namespace asca

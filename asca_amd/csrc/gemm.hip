// f32 GEMM on the CDNA4 matrix cores, with the operand/epilogue variants the
// model needs:
//
//   C = alpha * op(A) op(B) (+ bias per column) (+ beta * C)
//
// where op(A) is A (M x K, row-major) or A^T (A stored K x M), op(B) is B
// (K x N) or B^T (B stored N x K) -- the reference's matmul_f32 / matmul_ta_f32
// / matmul_ld_f32 family (rust/kernels/asca.cu:14-141) and Mat::matmul /
// matmul_ta / matmul_t (rust/src/tensor.rs:91-201).  On top of that:
//   - storage-row indirection per operand (row gather) and on C (row scatter),
//     replacing gather_rows_f32 / scatter_rows_f32 round trips (asca.cu:576-594);
//   - grouped launches over expert buckets (CSR offsets on the device): either
//     M varies per group (expert forward GEMMs, dpre, dxn) or K varies per
//     group (expert weight gradients), one launch for all experts;
//   - fused epilogues: bias + SiLU writing both pre and hidden (HashMoe
//     forward, rust/src/model.rs:236-248), and the SiLU backward
//     dpre = acc * s (1 + pre (1 - s)) (model.rs:432-440);
//   - split-K with f32 partials and a deterministic reduction, for the
//     K = tokens weight-gradient products that have few output tiles.
//
// The products run on the bf16 matrix cores with every f32 split in three (see
// "f32 products on the bf16 matrix cores" below): block tiles of 128 x 256 and
// 128 x 128 staged in LDS (gemm_k) and 64 x 64 with the k range dealt to the
// block's waves (gemm_small_k); best_tile chooses.  The batched per-chunk
// products of the chunked delta rule (gemm_batched_k) use
// v_mfma_f32_16x16x4_f32 with k-tiles of 32 double-buffered in LDS.
#include <limits.h>

#include <mutex>
#include <type_traits>

#include "common.h"
#include "gemm.h"
#include "runtime.h"

namespace asca {

// gemm_batched_k's tiles: (64 WM) x (64 WN) with one 64 x 64 wave tile per wave.
// Each operand keeps its global layout in LDS: a k-contiguous tile is [mn][k]
// with a 36-float row stride, an mn-contiguous tile is [k][mn].  The MFMA k
// index is permuted inside every 16-k group (step s, lane l uses
// k = 4 (l / 16) + s) so every fragment read is one 16-byte ds_read: a [mn][k]
// read yields four k-steps of one 16-row tile, a [k][mn] read yields one k-step
// of four tiles whose rows are interleaved by 4.
constexpr int GM_BM = 128, GM_BN = 128, GM_BK = 32;
constexpr int GM_LDK = GM_BK + 4;  // [mn][k] tile row stride (floats)

// floats of one LDS operand tile with R mn-rows
template <bool KC, int R>
constexpr int tile_floats() { return KC ? R * GM_LDK : GM_BK * R; }

ASCA_DEV float silu_ref(float x) { return x / (1.0f + expf(-x)); }

// 4 consecutive floats from p, of which n (<= 0 .. >= 4) are valid; the rest 0.
template <bool VEC>
ASCA_DEV float4 ld4(const float* p, int n) {
    if (VEC && n >= 4) return *reinterpret_cast<const float4*>(p);
    float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
    if (n > 0) r.x = p[0];
    if (n > 1) r.y = p[1];
    if (n > 2) r.z = p[2];
    if (n > 3) r.w = p[3];
    return r;
}

ASCA_DEV long srow(const int* rows, long off, long i) { return rows ? (long)rows[off + i] : off + i; }

// Global -> registers for one operand tile (8 R / NT float4 per thread).
//   KC (k-contiguous, stored [mn][k]): R mn-rows x 32 k, 8 threads per row.
//   MC (mn-contiguous, stored [k][mn]): 32 k-rows x R mn, R/4 threads per row.
// `lim_mn`, `lim_k`: valid extents relative to the tile origin.
template <bool KC, bool VEC, int R, int NT>
ASCA_DEV void tile_load(float4 (&r)[8 * R / NT], const float* base, long ld, const int* rows, long row_off,
                        int mn0, int lim_mn, long k0, long lim_k, int tid) {
#pragma unroll
    for (int j = 0; j < 8 * R / NT; ++j) {
        const int sl = tid + NT * j;
        if constexpr (KC) {
            const int rr = sl >> 3;
            const int kk = 4 * (sl & 7);
            const bool ok = rr < lim_mn;
            const long sr = ok ? srow(rows, row_off, mn0 + rr) : 0;
            r[j] = ld4<VEC>(base + sr * ld + k0 + kk, ok ? (int)min(lim_k - kk, 4L) : 0);
        } else {
            const int kr = sl / (R / 4);
            const int mm = 4 * (sl % (R / 4));
            const bool ok = kr < lim_k;
            const long sr = ok ? srow(rows, row_off, k0 + kr) : 0;
            r[j] = ld4<VEC>(base + sr * ld + mn0 + mm, ok ? min(lim_mn - mm, 4) : 0);
        }
    }
}

template <bool KC, int R, int NT>
ASCA_DEV void tile_store(const float4 (&r)[8 * R / NT], float* t, int tid) {
#pragma unroll
    for (int j = 0; j < 8 * R / NT; ++j) {
        const int sl = tid + NT * j;
        if constexpr (KC)
            *reinterpret_cast<float4*>(t + (sl >> 3) * GM_LDK + 4 * (sl & 7)) = r[j];
        else
            *reinterpret_cast<float4*>(t + (sl / (R / 4)) * R + 4 * (sl % (R / 4))) = r[j];
    }
}

// Fragments of one 16-k group h for the wave's 64 mn-rows starting at w0:
// f[s][t] = operand value of MFMA k-step s for 16-row tile t.
template <bool KC, int R>
ASCA_DEV void frag_read(float (&f)[4][4], const float* t, int w0, int h, int lane) {
    if constexpr (KC) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const float4 v =
                *reinterpret_cast<const float4*>(t + (w0 + 16 * x + (lane & 15)) * GM_LDK + 16 * h + 4 * (lane >> 4));
            f[0][x] = v.x;
            f[1][x] = v.y;
            f[2][x] = v.z;
            f[3][x] = v.w;
        }
    } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float4 v =
                *reinterpret_cast<const float4*>(t + (16 * h + 4 * (lane >> 4) + s) * R + w0 + 4 * (lane & 15));
            f[s][0] = v.x;
            f[s][1] = v.y;
            f[s][2] = v.z;
            f[s][3] = v.w;
        }
    }
}

// ---------------------------------------------------------------------------
// f32 products on the bf16 matrix cores.
//
// Every operand value is split on its way into LDS into three bf16 values,
// x = x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x - x0), x2 = x - x0 - x1 (each
// rounded to nearest; a bf16 holds 8 bits, so the three hold all 24 of x and
// both subtractions are exact).  A product of two splits is six bf16 products
// (x2 y0, x0 y2, x1 y1, x1 y0, x0 y1, x0 y0), each exact in f32 and summed in
// the f32 accumulator; the three left out come to at most 2^-24 of x y (x1 y2 and x2
// y1 a half each), over many products to 6e-9 of their sum.  Six
// v_mfma_f32_16x16x32_bf16 take 96 cycles where eight
// v_mfma_f32_16x16x4_f32 take 256 (and those hold the SIMD's VALU besides),
// and a sum is rounded 6 times per 32 terms instead of 8 times.
//
// The bf16 MFMA rounds its sums down (towards minus infinity: mean error -2.6e-8
// of the rms at K = 512, where the f32 MFMA shows none), and a sum over many
// rows of such a product (a bias gradient over 16384 tokens) adds these up: its
// error was 3.7e-6 against 1.2e-6.  So odd rows of the large tiles are multiplied
// negated and negated back at the end, which makes every second row's error
// positive, and equal rows of A differ in their last bits between odd and even
// places.  The 64 x 64 tile negates every second wave's part of the k range instead,
// so that equal rows of A (a batch of sequences being decoded) give equal rows of C.
// In the large tiles that cost 3% (the sums negated every four k-tiles), signs by a row's
// values instead of its place 1 to 5% (routed FFN 777 -> 815 us).
//
// The bf16 MFMA takes subnormal inputs as zero, and x1 and x2 hold the bits of x down
// to 2^-23 of it: unscaled, operands below 2^-110 lost them (a product of rows at
// 2^-120 had an error of 3.5e-5, at 2^-128 9e-3).  So both operands are split as
// 2^24 x, where the smallest subnormal float is a normal bf16, and the sums are
// scaled back by 2^-48: the same bits where nothing under- or overflows.  The
// sign is part of the factor.  The multiplications cost 1 to 2%
// (16384x512x1536 forward and backward 418 -> 426 us, training step 14.00 -> 14.15 ms).
//
// A value that is not finite, or is 2^104 or more, or a sum of 2^80 or more
// leaves a non-finite sum wherever it enters: a wave that finds one among its sums
// computes its tile again with f32 products (f32_products), so infinities and
// NaN come out as the f32 products give them.
//
// LDS image of one operand tile (R rows x 32 k): three planes (x0, x1, x2) of
// [k / 8][slot][8 bf16], 16 bytes per (row, k / 8), so every fragment read is
// lane l reading slot l % 16 of k-group l / 16: one conflict-free ds_read_b128.
// The k-group stride is 32 bytes over a multiple of 256, which keeps the eight
// lanes of a write phase (two rows x four k-groups) on different banks.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
// global accesses of 8 and 16 bytes at 4-byte alignment (one instruction)
typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int SP_BK = 32;

ASCA_DEV f32x2 buf_load2(Rsrc r, unsigned voff, unsigned soff) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0);
    return f32x2{__uint_as_float(x[0]), __uint_as_float(x[1])};
}

// Elements c .. c + 3 of a run of n (> 0) valid floats, 0 past them: loads at
// clamped places and no branch, since a conditional load is waited for on its
// own.  at(i): element i.
template <class F>
ASCA_DEV f32x4 ld4_edge(int c, int n, F at) {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = at(min(c + e, n - 1));
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = c + e < n ? v[e] : 0.0f;
    return v;
}
template <int R>
constexpr int sp_kg() { return 16 * R + 32; }  // bytes of one k-group of a plane
template <int R>
constexpr int sp_plane() { return 4 * sp_kg<R>(); }
template <int R>
constexpr int sp_tile() { return 3 * sp_plane<R>(); }

ASCA_DEV unsigned pk_bf16(float a, float b) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{a, b}), bf16x2));
}
// the three bf16 parts of a and b, a in the low half of each word
ASCA_DEV void split2(float a, float b, unsigned& w0, unsigned& w1, unsigned& w2) {
    w0 = pk_bf16(a, b);
    a -= __uint_as_float(w0 << 16);
    b -= __uint_as_float(w0 & 0xffff0000u);
    w1 = pk_bf16(a, b);
    a -= __uint_as_float(w1 << 16);
    b -= __uint_as_float(w1 & 0xffff0000u);
    w2 = pk_bf16(a, b);
}

// The longest k range that is not split: one f32 MFMA, each product rounded once,
// where the six parts' sum of one product is 1.4 times as far off (2.5e-8 -> 3.4e-8, up to
// 2.7 units of 2^-24 instead of 1; from 4 products on it is the closer one).  Nor is
// anything staged: 16384 x 1536 x 4 33 -> 22 us, 27 with the f32 kernels.
constexpr long SP_F32_K = 4;
constexpr float SP_SCALE = 0x1p24f, SP_UNSCALE = 0x1p-48f;
// the factor of an operand's values: SP_SCALE, negative where `odd` is not zero
ASCA_DEV float sp_factor(int odd) { return odd ? -SP_SCALE : SP_SCALE; }

// A thread's share of one operand tile (R rows x 32 k on NT threads).
//   KC (k-contiguous, stored [mn][k]): items of 8 consecutive k of one row,
//     four threads to a row; slot = row.
//   MC (mn-contiguous, stored [k][mn]): 4 k x W columns; lanes 2i, 2i + 1 hold
//     the halves of one 8-k group.  Row 4 i + j of each 64 is slot 16 j + i, so
//     a wave's four 16-slot tiles interleave by 4 and the epilogue finds four
//     consecutive columns in one lane.
// Rows past the operand's extent repeat a valid one (KC) or read as 0 (MC);
// k past the range read as 0.
// Stored as SP_SCALE x; NEG: odd rows negated.
enum { LD_EDGE, LD_QUADS, LD_WHOLE };
template <bool KC, bool GATHER, bool NEG, int R, int NT>
struct SplitTile {
    static constexpr int NI = KC ? R * 4 / NT : 1, W = R * 8 / NT, NF = R * 32 / NT;
    const float* p[NI];
    long ld;
    int col, kofs;      // MC: column and k of the thread's piece within the tile
    int idx[4];         // GATHER (MC): storage rows of the next k-tile
    float x[NF];

    ASCA_DEV void init(const float* base, long ld_, const int* rows, long off, int mn0, int lim_mn, long K_lo,
                       long K_hi, int tid) {
        ld = ld_;
        if constexpr (KC) {
            kofs = 8 * (tid & 3);
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const int r = min((tid + NT * j) >> 2, lim_mn - 1);
                p[j] = base + srow(rows, off, mn0 + r) * ld + K_lo + kofs;
            }
        } else {
            const int lane = tid & 63, w = tid >> 6;
            constexpr int NB = R / (W == 4 ? 128 : 64);  // column blocks of a wave's width
            static_assert((NT / 64) == 4 * NB && (W == 2 || W == 4), "tile split");
            kofs = 8 * (w / NB) + 4 * (lane & 1);
            if constexpr (W == 4)
                col = 128 * (w % NB) + 4 * (lane >> 1);
            else
                col = 64 * (w % NB) + 4 * ((lane >> 1) & 15) + 2 * (lane >> 5);
            // a thread whose columns all lie past the extent repeats valid ones
            const int cc = col < lim_mn ? col : 0;
            p[0] = base + mn0 + cc + (GATHER ? 0 : (off + K_lo + kofs) * ld);
            if constexpr (GATHER) next_rows(rows, off, K_lo, K_hi);
        }
    }
    ASCA_DEV void next_rows(const int* rows, long off, long k0, long K_hi) {
#pragma unroll
        for (int e = 0; e < 4; ++e) idx[e] = rows[off + min(k0 + kofs + e, K_hi - 1)];
    }
    // Whether every thread's columns of the tile are all valid or all past the extent.
    ASCA_DEV static bool whole(int lim_mn) { return KC || lim_mn >= R || lim_mn % W == 0; }
    // k-tile at K_lo + k.  WHOLE: all of its k are valid and whole(lim_mn).  QUADS:
    // whole(lim_mn) and lim_k a multiple of 4, so that four k are valid or not together
    // (one by one, each element a load of its own: 16384 x 1536 x 48 41.5 us instead of
    // 37.9, its twin with B transposed 51 and 43.6; the f32 kernels took 37.5 and 46.6).
    template <int MODE>
    ASCA_DEV void load(long k, long lim_k, int lim_mn) {
        constexpr bool WHOLE = MODE == LD_WHOLE;
        if constexpr (MODE == LD_QUADS) {
            const int lk = (int)min(lim_k, (long)SP_BK);
            if constexpr (KC) {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const float* q = p[j] + k - kofs;
                    const f32x4u a = *reinterpret_cast<const f32x4u*>(q + min(kofs, lk - 4));
                    const f32x4u b = *reinterpret_cast<const f32x4u*>(q + min(kofs + 4, lk - 4));
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        x[8 * j + e] = kofs < lk ? a[e] : 0.0f;
                        x[8 * j + 4 + e] = kofs + 4 < lk ? b[e] : 0.0f;
                    }
                }
            } else {
                const int k0 = min(kofs, lk - 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float* q = GATHER ? p[0] + (long)idx[e] * ld : p[0] + (k + k0 - kofs + e) * ld;
                    if constexpr (W == 4) {
                        const f32x4u a = *reinterpret_cast<const f32x4u*>(q);
#pragma unroll
                        for (int c = 0; c < 4; ++c) x[4 * e + c] = kofs < lk ? a[c] : 0.0f;
                    } else {
                        const f32x2u a = *reinterpret_cast<const f32x2u*>(q);
                        x[2 * e] = kofs < lk ? a[0] : 0.0f;
                        x[2 * e + 1] = kofs < lk ? a[1] : 0.0f;
                    }
                }
            }
            return;
        }
        if constexpr (KC) {
            if constexpr (WHOLE) {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const f32x4u a = *reinterpret_cast<const f32x4u*>(p[j] + k);
                    const f32x4u b = *reinterpret_cast<const f32x4u*>(p[j] + k + 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        x[8 * j + e] = a[e];
                        x[8 * j + 4 + e] = b[e];
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const float* q = p[j] + k - kofs;
                    const int lk = (int)min(lim_k, (long)SP_BK);
                    const f32x4 a = ld4_edge(kofs, lk, [&](int i) { return q[i]; });
                    const f32x4 b = ld4_edge(kofs + 4, lk, [&](int i) { return q[i]; });
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        x[8 * j + e] = a[e];
                        x[8 * j + 4 + e] = b[e];
                    }
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if constexpr (!WHOLE) {
                    const int lk = (int)min(lim_k, (long)SP_BK), ke = min(kofs + e, lk - 1);
                    const float* q = GATHER ? p[0] + (long)idx[e] * ld : p[0] + (k + ke - kofs) * ld;
                    const int cc = col < lim_mn ? col : 0;
                    const f32x4 a = ld4_edge(col, lim_mn, [&](int i) { return q[i - cc]; });
#pragma unroll
                    for (int c = 0; c < W; ++c) x[W * e + c] = kofs + e < lim_k ? a[c] : 0.0f;
                    continue;
                }
                const float* q = GATHER ? p[0] + (long)idx[e] * ld : p[0] + (k + e) * ld;
                if constexpr (W == 4) {
                    const f32x4u a = *reinterpret_cast<const f32x4u*>(q);
#pragma unroll
                    for (int c = 0; c < 4; ++c) x[4 * e + c] = a[c];
                } else {
                    const f32x2u a = *reinterpret_cast<const f32x2u*>(q);
                    x[2 * e] = a[0];
                    x[2 * e + 1] = a[1];
                }
            }
        }
    }
    ASCA_DEV void store(char* t, int tid) const {
        if constexpr (KC) {
#pragma unroll
            for (int j = 0; j < NI; ++j) {
                const int it = tid + NT * j;
                char* d = t + (it & 3) * sp_kg<R>() + (it >> 2) * 16;
                static_assert(NT % 8 == 0, "a thread's rows share their parity");
                float y[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] = sp_factor(NEG ? tid & 4 : 0) * x[8 * j + e];
                uint4 w0, w1, w2;
                split2(y[0], y[1], w0.x, w1.x, w2.x);
                split2(y[2], y[3], w0.y, w1.y, w2.y);
                split2(y[4], y[5], w0.z, w1.z, w2.z);
                split2(y[6], y[7], w0.w, w1.w, w2.w);
                *reinterpret_cast<uint4*>(d) = w0;
                *reinterpret_cast<uint4*>(d + sp_plane<R>()) = w1;
                *reinterpret_cast<uint4*>(d + 2 * sp_plane<R>()) = w2;
            }
        } else {
            char* d = t + (kofs >> 3) * sp_kg<R>() + (kofs & 4) * 2 + ((col & ~63) + ((col >> 2) & 15)) * 16;
#pragma unroll
            for (int c = 0; c < W; ++c) {
                const int o = (W == 4 ? c : (col & 2) + c) * 256;
                constexpr float sg[2] = {SP_SCALE, NEG ? -SP_SCALE : SP_SCALE};
                const float f = sg[c & 1];
                uint2 w0, w1, w2;
                split2(f * x[c], f * x[W + c], w0.x, w1.x, w2.x);
                split2(f * x[2 * W + c], f * x[3 * W + c], w0.y, w1.y, w2.y);
                *reinterpret_cast<uint2*>(d + o) = w0;
                *reinterpret_cast<uint2*>(d + o + sp_plane<R>()) = w1;
                *reinterpret_cast<uint2*>(d + o + 2 * sp_plane<R>()) = w2;
            }
        }
    }
};

// acc (64 x 64 of one wave) += the k-tile in LDS
template <int RA, int RB>
ASCA_DEV void split_mma(f32x4 (&acc)[4][4], const char* As, const char* Bs, int wm, int wn, int lane) {
    const char* ap = As + (lane >> 4) * sp_kg<RA>() + (wm + (lane & 15)) * 16;
    const char* bp = Bs + (lane >> 4) * sp_kg<RB>() + (wn + (lane & 15)) * 16;
    bf16x8 a[3][4];
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) a[s][i] = *reinterpret_cast<const bf16x8*>(ap + s * sp_plane<RA>() + i * 256);
#pragma unroll
    for (int y = 0; y < 4; ++y) {
        bf16x8 b[3];
#pragma unroll
        for (int s = 0; s < 3; ++s) b[s] = *reinterpret_cast<const bf16x8*>(bp + s * sp_plane<RB>() + y * 256);
        constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int s = 0; s < 6; ++s)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                acc[i][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[PA[s]][i], b[PB[s]], acc[i][y], 0, 0, 0);
    }
}

// One operand element (row mn0 + r, k) for f32_products; 0 outside the product
template <bool KC>
ASCA_DEV float split_elem(const float* base, long ld, const int* rows, long off, int mn0, int r, int lim_mn, long k,
                          long K_hi) {
    if (r >= lim_mn || k >= K_hi) return 0.0f;
    return KC ? base[srow(rows, off, mn0 + r) * ld + k] : base[srow(rows, off, k) * ld + mn0 + r];
}

// The sums of the NX x NY 16 x 16 tiles from (x0, y0) of a wave's 64 x 64 as f32
// products straight from memory: for sums that the split leaves non-finite, and for a k
// range of at most SP_F32_K.  A product whose sums are all redone takes 4 to 6 times
// as long (16384 x 1536 x 512 142 -> 624 us, 220 with the f32 kernels; 64 x 1536 x 512
// 8.8 -> 39); only the waves that find one redo theirs (one NaN row of 16384: 190).
// Vector loads two steps ahead made that 1.7 times as fast and the finite products 2
// to 8% slower (registers).
// (CB: columns of an mn-contiguous B interleaved over so many tiles)
template <bool TA, bool TB, int CB, int NX, int NY>
ASCA_DEV void f32_products(f32x4 (&acc)[NX][NY], int x0, int y0, const float* A, const float* B, const GemmArgs& p,
                         long a_off, long b_off, int m0, int n0, int lim_m, int lim_n, long K_lo, long K_hi,
                         int lane) {
    const int i = lane & 15;
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (long k = K_lo; k < K_hi; k += 4) {
        const long kk = k + (lane >> 4);
        float a[NX], b[NY];
#pragma unroll
        for (int x = 0; x < NX; ++x)
            a[x] = split_elem<!TA>(A, p.lda, p.a_rows, a_off, m0, TA ? 4 * i + x0 + x : 16 * (x0 + x) + i, lim_m, kk,
                                   K_hi);
#pragma unroll
        for (int y = 0; y < NY; ++y)
            b[y] = split_elem<TB>(B, p.ldb, p.b_rows, b_off, n0, TB ? 16 * (y0 + y) + i : CB * i + y0 + y, lim_n, kk,
                                  K_hi);
#pragma unroll
        for (int x = 0; x < NX; ++x)
#pragma unroll
            for (int y = 0; y < NY; ++y)
                acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[x], b[y], acc[x][y], 0, 0, 0);
    }
}

// The sums scaled back; ODD: those of the rows that were multiplied negated (odd rows
// of the tile: row 16 x + 4 (lane / 16) + r, or 4 i + x of an mn-contiguous A)
// negated back.  Plus zero, so that a sum of zeros is not a negative one.
template <bool ODD, bool TA, int NX, int NY>
ASCA_DEV void split_unscale(f32x4 (&acc)[NX][NY]) {
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                acc[x][y][r] = fmaf(acc[x][y][r], ODD && ((TA ? x : r) & 1) ? -SP_UNSCALE : SP_UNSCALE, 0.0f);
}

// Any infinity or NaN among a wave's sums?
template <int NX, int NY>
ASCA_DEV bool split_bad(const f32x4 (&acc)[NX][NY]) {
    float z = 0.0f;
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y)
#pragma unroll
            for (int r = 0; r < 4; ++r) z = fmaf(acc[x][y][r], 0.0f, z);
    return __any(z != z);
}

// Main loop: a k-tile of 32 per step, loaded into registers two steps ahead,
// split and stored to LDS one step ahead.  DB: two LDS stages and one barrier
// per step (146 KB for 128 x 256, one block per CU); otherwise one stage and
// two barriers (49 KB for 128 x 128), the CU's other block filling the waits.
// Bound: power.  At 4096^3 the 128 x 256 tile runs 225 to 232 TFLOP/s (f32 products on
// the same shape: 139), 1350 TFLOP/s of bf16 products, and 258 on operands of
// zeros; a plain bf16 product of torch runs 1130 there.  16384x1536x512
// 208 -> 143 us, its input gradient 210 -> 124, its weight gradient 218 -> 133.
template <bool TA, bool TB, int GATHER, int WM, int WN, bool DB>
ASCA_DEV void split_mainloop(f32x4 (&acc)[4][4], const float* A, const float* B, const GemmArgs& p, long a_off,
                             long b_off, int m0, int n0, int lim_m, int lim_n, long K_lo, long K_hi, int tid,
                             int wm, int wn) {
    constexpr int NT = 64 * WM * WN, RA = 64 * WM, RB = 64 * WN, ST = sp_tile<RA>() + sp_tile<RB>();
    extern __shared__ float4 lds4[];
    char* lds = reinterpret_cast<char*>(lds4);
    const int lane = tid & 63;
    SplitTile<!TA, GATHER == 1, true, RA, NT> ta;
    SplitTile<TB, GATHER == 2, false, RB, NT> tb;
    ta.init(A, p.lda, p.a_rows, a_off, m0, lim_m, K_lo, K_hi, tid);
    tb.init(B, p.ldb, p.b_rows, b_off, n0, lim_n, K_lo, K_hi, tid);
    const long nk = (K_hi - K_lo + SP_BK - 1) / SP_BK;  // > 0
    const bool whole = ta.whole(lim_m) && tb.whole(lim_n);
    const long nw = whole ? (K_hi - K_lo) / SP_BK : 0;  // k-tiles that load without checks
    const bool quads = whole && (K_hi - K_lo) % 4 == 0;
    auto load_as = [&](long kt, auto Mode) {
        constexpr int mode = decltype(Mode)::value;
        const long k = kt * SP_BK, lim_k = K_hi - K_lo - k;
        ta.template load<mode>(k, lim_k, lim_m);
        tb.template load<mode>(k, lim_k, lim_n);
        const long kn = K_lo + min(kt + 1, nk - 1) * SP_BK;  // the storage rows of the k-tile after it
        if constexpr (GATHER == 1) ta.next_rows(p.a_rows, a_off, kn, K_hi);
        if constexpr (GATHER == 2) tb.next_rows(p.b_rows, b_off, kn, K_hi);
    };
    auto load = [&](long kt) {
        if (kt < nw)
            load_as(kt, std::integral_constant<int, LD_WHOLE>{});
        else if (kt < nk && quads)
            load_as(kt, std::integral_constant<int, LD_QUADS>{});
        else if (kt < nk)
            load_as(kt, std::integral_constant<int, LD_EDGE>{});
    };
    load(0);
    ta.store(lds, tid);
    tb.store(lds + sp_tile<RA>(), tid);
    load(1);
    lds_barrier();
    long t = 0;
    // Step t: k-tile t multiplied from its stage, t + 1 split and stored, t + 2
    // loaded.  The steps whose loads need no checks run in a loop of their own:
    // without branches the splits and the products of a step interleave.
    auto step = [&](auto Whole) {
        char* cur = lds + (DB && (t & 1) ? ST : 0);
        char* nxt = lds + (DB && !(t & 1) ? ST : 0);
        split_mma<RA, RB>(acc, cur, cur + sp_tile<RA>(), wm, wn, lane);
        if constexpr (!DB) lds_barrier();
        ta.store(nxt, tid);  // (past the last k-tile: not read)
        tb.store(nxt + sp_tile<RA>(), tid);
        if constexpr (decltype(Whole)::value)
            load_as(t + 2, std::integral_constant<int, LD_WHOLE>{});
        else
            load(t + 2);
        if constexpr (DB && decltype(Whole)::value) {
            // order of the step's instructions: fragment reads ahead of their
            // products, splits and stores spread between the last 72 products
            // (left alone the compiler puts all splits first, the matrix cores
            // idle: 4096^3 641 -> 620 us)
            __builtin_amdgcn_sched_group_barrier(0x100, 15, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 12, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 12, 0);
#pragma unroll
            for (int q = 0; q < 9; ++q) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
                }
                if (q == 1 || q == 4) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
                __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
            }
        }
        lds_barrier();
    };
    for (; t + 2 < nw; ++t) step(std::true_type{});
    for (; t < nk; ++t) step(std::false_type{});
    split_unscale<true, TA>(acc);
    if (split_bad(acc))
        f32_products<TA, TB, 4>(acc, 0, 0, A, B, p, a_off, b_off, m0 + wm, n0 + wn, lim_m - wm, lim_n - wn, K_lo, K_hi, lane);
}

// The tile, group and K range of a block.
template <bool TA, bool TB, int BM, int BN>
struct BlockTile {
    int m0, n0, lim_m, lim_n, Mg;
    long K_lo, K_hi, goff_g, a_off, b_off;
    const float *A, *B, *bias, *resid;
    float* C;
    // Row tiles of all groups (gmode 1): 64 groups at a time, a wave's lanes count
    // their tiles (one group after another, each bound read is waited for).
    ASCA_DEV static int row_tiles(const GemmArgs& p) {
        int n = 0;
        const int lane = threadIdx.x & 63;
        for (int g = lane; g < p.ngroups; g += 64) n += (p.goff[g + 1] - p.goff[g] + BM - 1) / BM;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) n += __shfl_xor(n, o);
        return __builtin_amdgcn_readfirstlane(n);
    }
    ASCA_DEV static int total(const GemmArgs& p) {
        return p.tiles_n * (p.gmode == 1 ? row_tiles(p) : p.gmode == 0 ? p.tiles_m : p.tiles_m * p.ngroups);
    }
    // Block b of n -> tile, XCD-aware: hardware places block i on XCD i % 8, so
    // give each XCD a contiguous run of tiles (neighbours share operand rows).
    ASCA_DEV static int of_block(int b, int n) {
        const int x = b & 7;
        return x * (n >> 3) + min(x, n & 7) + (b >> 3);
    }
    // The block's tile; false: a surplus block (a grouped grid is an upper bound).
    ASCA_DEV bool init(const GemmArgs& p) {
        const int n = p.gmode == 1 ? total(p) : (int)gridDim.x;
        if ((int)blockIdx.x >= n) return false;
        init(p, of_block(blockIdx.x, n));
        return true;
    }
    // Tile L (below total()).
    ASCA_DEV void init(const GemmArgs& p, int L) {
        int g = 0, tm, tn = L % p.tiles_n;
        Mg = p.M;
        K_lo = 0;
        K_hi = p.K;
        goff_g = 0;
        if (p.gmode == 1) {
            int mt = L / p.tiles_n;
            const int lane = threadIdx.x & 63;
            for (; g < p.ngroups; g += 64) {
                const int gl = min(g + lane, p.ngroups - 1);
                const int nt = g + lane < p.ngroups ? (p.goff[gl + 1] - p.goff[gl] + BM - 1) / BM : 0;
                int upto = nt;  // tiles of groups g .. g + lane
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int x = __shfl_up(upto, o);
                    if (lane >= o) upto += x;
                }
                const unsigned long long past = __ballot(upto > mt);
                if (past) {
                    const int l = __builtin_ctzll(past);
                    g += l;
                    mt -= __builtin_amdgcn_readlane(upto - nt, l);
                    break;
                }
                mt -= __builtin_amdgcn_readlane(upto, 63);
            }
            g = __builtin_amdgcn_readfirstlane(g);
            mt = __builtin_amdgcn_readfirstlane(mt);
            tm = mt;
            goff_g = p.goff[g];
            Mg = p.goff[g + 1] - p.goff[g];
        } else if (p.gmode == 2) {
            const int r = L / p.tiles_n;
            tm = r % p.tiles_m;
            g = r / p.tiles_m;
            goff_g = p.goff[g];
            K_hi = p.goff[g + 1] - p.goff[g];
        } else if (p.gmode == 3) {
            const int r = L / p.tiles_n;
            tm = r % p.tiles_m;
            g = r / p.tiles_m;
        } else {
            tm = L / p.tiles_n;
            K_lo = (long)blockIdx.y * p.k_per_split;
            K_hi = min((long)p.K, K_lo + p.k_per_split);
        }
        m0 = tm * BM;
        n0 = tn * BN;
        lim_m = Mg - m0;
        lim_n = p.N - n0;
        A = p.A + g * p.a_gs;
        B = p.B + g * p.b_gs;
        C = p.C + g * p.c_gs + (long)blockIdx.y * p.c_split_stride;
        bias = p.bias ? p.bias + g * p.bias_gs : nullptr;
        resid = p.resid ? p.resid + g * p.r_gs : nullptr;
        a_off = ((p.gmode == 1 && !TA) || (p.gmode == 2 && TA)) ? goff_g : 0;
        b_off = (p.gmode == 2 && !TB) ? goff_g : 0;
    }
};

template <int N>
ASCA_DEV void store_row(float* d, const float (&o)[N]) {
    if constexpr (N == 4)
        *reinterpret_cast<f32x4u*>(d) = f32x4u{o[0], o[1], o[2], o[3]};
    else if constexpr (N == 2)
        *reinterpret_cast<f32x2u*>(d) = f32x2u{o[0], o[1]};
    else
        d[0] = o[0];
}

// C of the NX x NY 16 x 16 tiles from (x0, y0) of the wave's 64 x 64 at (m0, n0).
template <bool TA, bool TB, int EPI, int CB, int NX, int NY, class T>
ASCA_DEV void gemm_epilogue(const f32x4 (&acc)[NX][NY], int x0, int y0, int m0, int n0, const T& t, const GemmArgs& p,
                            int lane) {
    constexpr bool A_KC = !TA, B_KC = TB;
    float* const C = t.C;
    const float *const bias = t.bias, *const resid = t.resid;
    const int Mg = t.Mg;
    const long goff_g = t.goff_g;
    // result register r of tile (x, y) sits at tile row 4 (lane / 16) + r,
    // tile column lane % 16.  Element y of a lane's row is column nc0 + NS y.
    // Every load the epilogue needs is unconditional (indices clamped into the
    // operand) and issued ahead of its use: the bias once per thread, the scatter
    // indices, residual, C and pre of four rows at a time.  A load under a
    // per-element condition is waited for on its own, one latency per element.
    constexpr int NS = B_KC ? 16 : 1;
    const int nc0 = B_KC ? n0 + 16 * y0 + (lane & 15) : n0 + CB * (lane & 15) + y0;
    const int nmax = p.N - 1;
    float bv[NY];
    if (bias) {
#pragma unroll
        for (int y = 0; y < NY; ++y) bv[y] = bias[min(nc0 + NS * y, nmax)];
    }
    const bool add_c = EPI == EPI_STORE && p.beta != 0.0f;
#pragma unroll
    for (int x = 0; x < NX; ++x) {
        long srt[4], crow[4];
        bool rok[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int tr = 4 * (lane >> 4) + r;
            const int m = m0 + (A_KC ? 16 * (x0 + x) + tr : 4 * tr + x0 + x);
            rok[r] = m < Mg;
            srt[r] = (p.gmode == 1 ? goff_g : 0) + min(m, Mg - 1);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) crow[r] = p.c_rows ? (long)p.c_rows[srt[r]] : srt[r];
        float lr[4][NY], lc[4][NY], la[4][NY];
        if constexpr (EPI == EPI_STORE) {
            if (resid) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int y = 0; y < NY; ++y) lr[r][y] = resid[crow[r] * p.ld_resid + min(nc0 + NS * y, nmax)];
            }
            if (add_c) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int y = 0; y < NY; ++y) lc[r][y] = C[crow[r] * p.ldc + min(nc0 + NS * y, nmax)];
            }
        } else if constexpr (EPI == EPI_SILU_BWD) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int y = 0; y < NY; ++y) la[r][y] = p.aux[srt[r] * p.ld_aux + min(nc0 + NS * y, nmax)];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (!rok[r]) continue;
            float* Cr = C + crow[r] * p.ldc;
            float o[NY], hb[NY];
#pragma unroll
            for (int y = 0; y < NY; ++y) {
                float a = p.alpha * acc[x][y][r];
                if (bias) a += bv[y];
                if constexpr (EPI == EPI_STORE) {
                    if (add_c) a += p.beta * lc[r][y];
                    if (resid) a += lr[r][y];
                } else if constexpr (EPI == EPI_SILU) {
                    hb[y] = silu_ref(a);
                } else {
                    const float pr = la[r][y];
                    const float sg = 1.0f / (1.0f + expf(-pr));
                    a = acc[x][y][r] * (sg * (1.0f + pr * (1.0f - sg)));
                }
                o[y] = a;
            }
            if constexpr (!B_KC) {
                // columns nc0 .. nc0 + NY - 1 of one row
                if (nc0 >= p.N) continue;
                const int cnt = min(p.N - nc0, NY);
                const long ao = srt[r] * p.ld_aux + nc0;
                if (cnt == NY) {
                    store_row<NY>(Cr + nc0, o);
                    if constexpr (EPI == EPI_SILU) store_row<NY>(p.aux_out + ao, hb);
                } else {
#pragma unroll
                    for (int y = 0; y < NY; ++y)
                        if (y < cnt) {
                            Cr[nc0 + y] = o[y];
                            if constexpr (EPI == EPI_SILU) p.aux_out[ao + y] = hb[y];
                        }
                }
            } else {
#pragma unroll
                for (int y = 0; y < NY; ++y) {
                    const int n = nc0 + 16 * y;
                    if (n >= p.N) continue;
                    Cr[n] = o[y];
                    if constexpr (EPI == EPI_SILU) p.aux_out[srt[r] * p.ld_aux + n] = hb[y];
                }
            }
        }
    }
}

// Block tile (64 WM) x (64 WN) on WM x WN waves; a wave owns 64 x 64.  FEW: the k
// range can be at most SP_F32_K.
template <bool TA, bool TB, int EPI, int GATHER, int WM, int WN, bool DB, bool FEW, class T>
ASCA_DEV void gemm_tile(const T& t, const GemmArgs& p) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = (w / WN) * 64, wn = (w % WN) * 64;
    f32x4 acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (FEW && t.K_hi - t.K_lo <= SP_F32_K)
        f32_products<TA, TB, 4>(acc, 0, 0, t.A, t.B, p, t.a_off, t.b_off, t.m0 + wm, t.n0 + wn, t.lim_m - wm,
                                t.lim_n - wn, t.K_lo, t.K_hi, lane);
    else if (t.K_hi > t.K_lo)
        split_mainloop<TA, TB, GATHER, WM, WN, DB>(acc, t.A, t.B, p, t.a_off, t.b_off, t.m0, t.n0, t.lim_m, t.lim_n,
                                                   t.K_lo, t.K_hi, tid, wm, wn);
    gemm_epilogue<TA, TB, EPI, 4>(acc, 0, 0, t.m0 + wm, t.n0 + wn, t, p, lane);
}

template <bool TA, bool TB, int EPI, int GATHER>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_k(GemmArgs p) {
    BlockTile<TA, TB, 128, 128> t;
    if (!t.init(p)) return;
    gemm_tile<TA, TB, EPI, GATHER, 2, 2, false, true>(t, p);
}

// Products too small to fill the chip with the tiles above: one 64 x 64 tile
// per block, the k-tiles dealt to its NW waves, whose sums are added through
// LDS at the end (in wave order).  Nothing is staged: a wave loads its
// fragments from memory (k-contiguous operands 8 k of one row per lane,
// mn-contiguous ones 8 k of four columns) and splits them in registers, so
// the loop has no barrier and a wave's next k-tile loads behind its products.
// Loads are buffer loads (32-bit lane offsets, the k-tile's offset in a scalar
// register: 64-bit addresses would take the registers the fragments need), so
// an operand's rows must lie within 4 GB (small_fits).
// NTL 16-row tiles (mn-contiguous: row NTL i + j is row i of tile j).
template <bool KC, bool GATHER, int NTL>
struct FragTile {
    const float* base;           // KC: k = K_lo of row 0; MC: k = K_lo of the tile's first column
    unsigned vo[KC ? NTL : 1];   // lane's byte offsets: KC: row 16 x + i at its k; MC: its k and column NTL i
    long ld;
    int kofs, col;
    f32x4 x[KC ? 2 * NTL : 8];   // KC: [2 x + half]; MC: [k], NTL columns
    ASCA_DEV void init(const float* b, long ld_, const int* rows, long off, int mn0, int lim_mn, long K_lo, int lane) {
        ld = ld_;
        kofs = 8 * (lane >> 4);
        col = NTL * (lane & 15);
        if constexpr (KC) {
            base = b + (rows ? 0 : (off + mn0) * ld) + K_lo;
#pragma unroll
            for (int j = 0; j < NTL; ++j) {
                const int r = min(16 * j + (lane & 15), lim_mn - 1);
                vo[j] = (unsigned)(((rows ? rows[off + mn0 + r] : r) * ld + kofs) * 4);
            }
        } else {
            base = b + mn0 + (GATHER ? 0 : (off + K_lo) * ld);
            vo[0] = (unsigned)(((GATHER ? 0 : kofs * ld) + (col < lim_mn ? col : 0)) * 4);
        }
    }
    ASCA_DEV static bool whole(int lim_mn) { return KC || lim_mn >= 16 * NTL || lim_mn % NTL == 0; }
    static ASCA_DEV f32x4 ld4(Rsrc r, unsigned vo, unsigned so) {
        const float4 v = buf_load4(r, vo, so);
        return f32x4{v.x, v.y, v.z, v.w};
    }
    // k-tile at K_lo + k; WHOLE: no k past the range, whole(lim_mn)
    template <bool WHOLE>
    ASCA_DEV void load(const int* rows, long off, long K_lo, long k, long lim_k, int lim_mn) {
        const int lk = (int)min(lim_k, (long)SP_BK);
        if constexpr (KC) {
            const Rsrc r = make_rsrc(base + k, ~0u);
#pragma unroll
            for (int j = 0; j < NTL; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if constexpr (WHOLE) {
                        x[2 * j + h] = ld4(r, vo[j], 16 * h);
                    } else {
                        const unsigned v = vo[j] - 4 * kofs;
                        x[2 * j + h] = ld4_edge(kofs + 4 * h, lk, [&](int i) { return buf_load1(r, v + 4 * i, 0); });
                    }
                }
        } else {
            const Rsrc r = make_rsrc(base + (GATHER ? 0 : k * ld), ~0u);
            const unsigned l4 = (unsigned)(4 * ld);
            unsigned v[8], so[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int ke = WHOLE ? kofs + e : min(kofs + e, lk - 1);
                v[e] = GATHER ? vo[0] + rows[off + K_lo + k + ke] * l4 : WHOLE ? vo[0] : vo[0] + (ke - kofs) * l4;
                so[e] = GATHER || !WHOLE ? 0 : e * l4;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if constexpr (WHOLE) {
                    if constexpr (NTL == 4) {
                        x[e] = ld4(r, v[e], so[e]);
                    } else if constexpr (NTL == 2) {
                        const f32x2 u = buf_load2(r, v[e], so[e]);
                        x[e][0] = u[0];
                        x[e][1] = u[1];
                    } else {
                        x[e][0] = buf_load1(r, v[e], so[e]);
                    }
                } else {
                    const unsigned c0 = v[e] - 4 * (col < lim_mn ? col : 0);
#pragma unroll
                    for (int c = 0; c < NTL; ++c) x[e][c] = buf_load1(r, c0 + 4 * min(col + c, lim_mn - 1), 0);
#pragma unroll
                    for (int c = 0; c < NTL; ++c) x[e][c] = kofs + e < lk && col + c < lim_mn ? x[e][c] : 0.0f;
                }
            }
        }
    }
    // the three bf16 fragments of f times 16-row tile j
    ASCA_DEV void frag(int j, bf16x8 (&out)[3], float f) const {
        typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
        u32x4 w[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float a = KC ? x[2 * j + e / 2][2 * (e & 1)] : x[2 * e][j];
            float b = KC ? x[2 * j + e / 2][2 * (e & 1) + 1] : x[2 * e + 1][j];
            a *= f;
            b *= f;
            unsigned w0, w1, w2;
            split2(a, b, w0, w1, w2);
            w[0][e] = w0;
            w[1][e] = w1;
            w[2][e] = w2;
        }
#pragma unroll
        for (int s = 0; s < 3; ++s) out[s] = __builtin_bit_cast(bf16x8, w[s]);
    }
};

// NX x NY tiles of 16 x 16 per block: 4 x 4, or fewer columns or rows where
// those leave CUs idle (decode: few rows, the weights streamed once).
constexpr int SM_NW = 8;  // waves of a small-product block
template <bool TA, bool TB, int EPI, int GATHER, int NX, int NY, class T>
ASCA_DEV void small_tile(const T& t, const GemmArgs& p) {
    static_assert(!TA || NX == 4, "tile rows of A^T");
    extern __shared__ float4 lds4[];
    f32x4* const part = reinterpret_cast<f32x4*>(lds4);  // [wave][tile][lane]
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    f32x4 acc[NX][NY];
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bool few = t.K_hi - t.K_lo <= SP_F32_K;
    const long nk = few ? 0 : (t.K_hi - t.K_lo + SP_BK - 1) / SP_BK;
    if (w < nk) {
        FragTile<!TA, GATHER == 1, NX> fa;
        FragTile<TB, GATHER == 2, NY> fb;
        fa.init(t.A, p.lda, p.a_rows, t.a_off, t.m0, t.lim_m, t.K_lo, lane);
        fb.init(t.B, p.ldb, p.b_rows, t.b_off, t.n0, t.lim_n, t.K_lo, lane);
        const bool whole = fa.whole(t.lim_m) && fb.whole(t.lim_n);
        auto load_a = [&](long kt) {
            const long k = kt * SP_BK, lim_k = t.K_hi - t.K_lo - k;
            if (whole && lim_k >= SP_BK)
                fa.template load<true>(p.a_rows, t.a_off, t.K_lo, k, lim_k, t.lim_m);
            else
                fa.template load<false>(p.a_rows, t.a_off, t.K_lo, k, lim_k, t.lim_m);
        };
        auto load_b = [&](long kt) {
            const long k = kt * SP_BK, lim_k = t.K_hi - t.K_lo - k;
            if (whole && lim_k >= SP_BK)
                fb.template load<true>(p.b_rows, t.b_off, t.K_lo, k, lim_k, t.lim_n);
            else
                fb.template load<false>(p.b_rows, t.b_off, t.K_lo, k, lim_k, t.lim_n);
        };
        load_a(w);
        load_b(w);
#pragma unroll 1
        for (long kt = w;;) {
            bf16x8 a[NX][3];
#pragma unroll
            for (int x = 0; x < NX; ++x) fa.frag(x, a[x], sp_factor(w & 1));
            kt += SM_NW;
            if (kt < nk) load_a(kt);
            // one column tile at a time: its fragments are split beside the
            // products of the one before (all at once, the registers spill)
#pragma unroll
            for (int y = 0; y < NY; ++y) {
                bf16x8 b[3];
                fb.frag(y, b, SP_SCALE);
                constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
                for (int s = 0; s < 6; ++s)
#pragma unroll
                    for (int x = 0; x < NX; ++x)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[x][PA[s]], b[PB[s]], acc[x][y], 0, 0, 0);
                if (y < NY - 1) __builtin_amdgcn_sched_barrier(0);
            }
            if (kt < nk) load_b(kt);
            if (kt >= nk) break;
        }
    }
    constexpr int TL = NX * NY, PW = TL > SM_NW ? TL / SM_NW : 1;  // tiles; tiles a wave adds up
    static_assert(NY % PW == 0 && TL <= SM_NW * PW, "sums per wave");
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y) part[(w * TL + NY * x + y) * 64 + lane] = acc[x][y];
    lds_barrier();
    // wave w adds up and stores tiles PW w .. PW w + PW - 1
    if (PW * w >= TL) return;
    const int x0 = PW * w / NY, y0 = PW * w % NY;
    f32x4 sum[1][PW];
#pragma unroll
    for (int y = 0; y < PW; ++y) {
        sum[0][y] = part[(NY * x0 + y0 + y) * 64 + lane];
#pragma unroll
        for (int v = 1; v < SM_NW; ++v) {
            const f32x4 pv = part[(v * TL + NY * x0 + y0 + y) * 64 + lane];
            sum[0][y] = v & 1 ? sum[0][y] - pv : sum[0][y] + pv;  // (sp_factor(w & 1))
        }
    }
    split_unscale<false, TA>(sum);
    if (few || split_bad(sum))
        f32_products<TA, TB, NY>(sum, x0, y0, t.A, t.B, p, t.a_off, t.b_off, t.m0, t.n0, t.lim_m, t.lim_n, t.K_lo, t.K_hi,
                               lane);
    gemm_epilogue<TA, TB, EPI, NY>(sum, x0, y0, t.m0, t.n0, t, p, lane);
}

template <bool TA, bool TB, int EPI, int GATHER, int NX, int NY>
__global__ __launch_bounds__(64 * SM_NW) __attribute__((amdgpu_waves_per_eu(NX == 1 ? 4 : 2))) void gemm_small_k(
    GemmArgs p) {
    BlockTile<TA, TB, 16 * NX, 16 * NY> t;
    if (!t.init(p)) return;
    small_tile<TA, TB, EPI, GATHER, NX, NY>(t, p);
}

// 128 x 256 tiles on 8 waves, one block per CU.  Where the tiles leave a last
// round that is nearly empty (at most p.tail_max of them beyond whole rounds of
// p.cus, a number that a grouped launch knows only on the device), the last
// p.tail_blocks blocks take those as 64 x 64 tiles, which all CUs share:
// 17408 x 1024 x 512 (544 tiles, 32 past two rounds) 125 -> 108 us, its twin of
// 16 groups (the routed FFN) alike, 17000 x 512 x 512 74 -> 55 us, 10900 x 1532 x
// 240 74 -> 63 us; whole rounds as before (16384 x 1536 x 512 144 us).
template <bool TA, bool TB, int EPI, int GATHER>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_wide_k(GemmArgs p) {
    BlockTile<TA, TB, 128, 256> t;
    const int n = t.total(p), rem = n % p.cus;
    const int cut = p.tail_blocks && rem <= p.tail_max ? n - rem : n;
    const int first = gridDim.x - p.tail_blocks;  // blocks of whole tiles
    if ((int)blockIdx.x < first) {
        if ((int)blockIdx.x >= cut) return;
        t.init(p, t.of_block(blockIdx.x, cut));
        // (few k: groups of a grouped K; best_tile keeps other products of so few off this tile)
        gemm_tile<TA, TB, EPI, GATHER, 2, 4, true, TA && !TB>(t, p);
        return;
    }
    for (int i = blockIdx.x - first; i < 8 * (n - cut); i += p.tail_blocks) {
        t.init(p, cut + (i >> 3));
        const int dm = 64 * ((i >> 2) & 1), dn = 64 * (i & 3);
        t.m0 += dm;
        t.n0 += dn;
        t.lim_m -= dm;
        t.lim_n -= dn;
        if (t.lim_m <= 0 || t.lim_n <= 0) continue;  // uniform
        small_tile<TA, TB, EPI, GATHER, 4, 4>(t, p);
        lds_barrier();  // the sums are read before the next tile's are written
    }
}

// Persistent batched products (gmode 3, plain epilogue): a block walks work
// items (batch g, tile tm, tn) with a stride of gridDim.x and the k-tile
// pipeline runs across item boundaries, so the first k-tile of the next item
// loads while the last one of the current item is multiplied.  The per-chunk
// products of the chunked delta rule are small (K = 64 or 128), and as one
// block per product each paid its whole load latency up front.
template <bool TA, bool TB, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) __attribute__((amdgpu_waves_per_eu(1, 2))) void gemm_batched_k(
    GemmArgs p) {
    constexpr int NT = 64 * WM * WN, BM = 64 * WM, BN = 64 * WN;
    constexpr bool A_KC = !TA, B_KC = TB;
    constexpr int A_F = tile_floats<A_KC, BM>();
    constexpr int B_F = tile_floats<B_KC, BN>();
    extern __shared__ float4 lds4[];
    float* lds = reinterpret_cast<float*>(lds4);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wm = (w / WN) * 64, wn = (w % WN) * 64;
    const int per = p.tiles_m * p.tiles_n;
    const long items = (long)p.ngroups * per;
    const int nk = (p.K + GM_BK - 1) / GM_BK;  // the host guarantees K > 0
    long item = blockIdx.x;
    if (item >= items) return;

    long g = item / per;
    int m0 = (int)(item % per) / p.tiles_n * BM, n0 = (int)(item % per) % p.tiles_n * BN;
    const float* A = p.A + g * p.a_gs;
    const float* B = p.B + g * p.b_gs;
    float4 ra[8 * BM / NT], rb[8 * BN / NT];
    tile_load<A_KC, true, BM, NT>(ra, A, p.lda, nullptr, 0, m0, p.M - m0, 0, p.K, tid);
    tile_load<B_KC, true, BN, NT>(rb, B, p.ldb, nullptr, 0, n0, p.N - n0, 0, p.K, tid);
    tile_store<A_KC, BM, NT>(ra, lds, tid);
    tile_store<B_KC, BN, NT>(rb, lds + A_F, tid);
    __syncthreads();
    int it = 0;  // k-iterations so far (LDS buffer parity)
    for (;;) {
        const long next = item + gridDim.x;
        const bool has_next = next < items;
        const long gn = has_next ? next / per : g;
        const int rn = has_next ? (int)(next % per) : 0;
        const int m0n = rn / p.tiles_n * BM, n0n = rn % p.tiles_n * BN;
        const float* An = p.A + gn * p.a_gs;
        const float* Bn = p.B + gn * p.b_gs;
        f32x4 acc[4][4];
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int kt = 0; kt < nk; ++kt, ++it) {
            const float* As = lds + (it & 1) * (A_F + B_F);
            const float* Bs = As + A_F;
            const bool more = kt + 1 < nk || has_next;
            if (kt + 1 < nk) {
                const long k0 = (long)(kt + 1) * GM_BK;
                tile_load<A_KC, true, BM, NT>(ra, A, p.lda, nullptr, 0, m0, p.M - m0, k0, p.K - k0, tid);
                tile_load<B_KC, true, BN, NT>(rb, B, p.ldb, nullptr, 0, n0, p.N - n0, k0, p.K - k0, tid);
            } else if (has_next) {
                tile_load<A_KC, true, BM, NT>(ra, An, p.lda, nullptr, 0, m0n, p.M - m0n, 0, p.K, tid);
                tile_load<B_KC, true, BN, NT>(rb, Bn, p.ldb, nullptr, 0, n0n, p.N - n0n, 0, p.K, tid);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float fa[4][4], fb[4][4];
                frag_read<A_KC, BM>(fa, As, wm, h, lane);
                frag_read<B_KC, BN>(fb, Bs, wn, h, lane);
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int x = 0; x < 4; ++x)
#pragma unroll
                        for (int y = 0; y < 4; ++y)
                            acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[s][x], fb[s][y], acc[x][y], 0, 0, 0);
            }
            if (more) {
                float* Ns = lds + ((it + 1) & 1) * (A_F + B_F);
                tile_store<A_KC, BM, NT>(ra, Ns, tid);
                tile_store<B_KC, BN, NT>(rb, Ns + A_F, tid);
            }
            __syncthreads();
        }
        // epilogue of this item: C = alpha acc + bias + beta C + resid
        float* C = p.C + g * p.c_gs;
        const float* bias = p.bias ? p.bias + g * p.bias_gs : nullptr;
        const float* resid = p.resid ? p.resid + g * p.r_gs : nullptr;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int tr = 4 * (lane >> 4) + r;
                const int m = m0 + wm + (A_KC ? 16 * x + tr : 4 * tr + x);
                if (m >= p.M) continue;
                float* Cr = C + (long)m * p.ldc;
                const float* Rr = resid ? resid + (long)m * p.ld_resid : nullptr;
                if constexpr (!B_KC) {
                    const int n = n0 + wn + 4 * (lane & 15);
                    if (n >= p.N) continue;
                    float o[4];
#pragma unroll
                    for (int y = 0; y < 4; ++y) {
                        float a = p.alpha * acc[x][y][r];
                        if (n + y < p.N) {
                            if (bias) a += bias[n + y];
                            if (p.beta != 0.0f) a += p.beta * Cr[n + y];
                            if (Rr) a += Rr[n + y];
                        }
                        o[y] = a;
                    }
                    if (n + 3 < p.N) {
                        *reinterpret_cast<float4*>(Cr + n) = make_float4(o[0], o[1], o[2], o[3]);
                    } else {
#pragma unroll
                        for (int y = 0; y < 4; ++y)
                            if (n + y < p.N) Cr[n + y] = o[y];
                    }
                } else {
#pragma unroll
                    for (int y = 0; y < 4; ++y) {
                        const int n = n0 + wn + 16 * y + (lane & 15);
                        if (n >= p.N) continue;
                        float a = p.alpha * acc[x][y][r];
                        if (bias) a += bias[n];
                        if (p.beta != 0.0f) a += p.beta * Cr[n];
                        if (Rr) a += Rr[n];
                        Cr[n] = a;
                    }
                }
            }
        }
        if (!has_next) break;
        item = next;
        g = gn;
        m0 = m0n;
        n0 = n0n;
        A = An;
        B = Bn;
    }
}

// Split-K reduction: C = alpha * sum_s part[s] + bias + beta * C, summed in the
// order of s.  Bound by reading the partials once: RD_U of a thread's loads are
// in flight (one after another they were waited for one by one).  VEC: four
// columns a thread, where rows and pointers allow 16-byte access (32 splits of
// 512 x 256: 9.5 -> 5.5 us; ten of 512 x 1536: 7.5 us, 4.2 TB/s).
constexpr int RD_U = 8;
template <bool VEC>
__global__ __launch_bounds__(256) void splitk_reduce_k(const float* __restrict__ part, int splits, long MN, int N,
                                                       float* __restrict__ C, long ldc, float alpha, float beta,
                                                       const float* __restrict__ bias) {
    constexpr int V = VEC ? 4 : 1;
    using T = float __attribute__((ext_vector_type(V)));
    const long stride = (long)gridDim.x * blockDim.x;
    for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < MN / V; e += stride) {
        const long i = e * V;
        T s = 0.0f;
        for (int k = 0; k < splits; k += RD_U) {
            T x[RD_U];
#pragma unroll
            for (int u = 0; u < RD_U; ++u) x[u] = *reinterpret_cast<const T*>(part + min(k + u, splits - 1) * MN + i);
            __builtin_amdgcn_sched_barrier(0);  // the loads go out together
#pragma unroll
            for (int u = 0; u < RD_U; ++u)
                if (k + u < splits) s += x[u];  // uniform
        }
        const long r = i / N;
        const int c = (int)(i - r * N);
        T a = alpha * s;
        if (bias) {
            const T b = *reinterpret_cast<const T*>(bias + c);
            a += b;
        }
        T* cp = reinterpret_cast<T*>(C + r * ldc + c);
        if (beta != 0.0f) a += beta * *cp;
        *cp = a;
    }
}

// Column sums, optionally per group of rows: out[g*N + c] (+)= sum over the
// rows of group g of X[r][c] (bias gradients: colsum_raw of
// rust/src/cuda/mod.rs:642-669 and the per-expert db1 of model.rs:432-440).
// Pass 1: a block sums 64 columns over one row slice, its four waves taking
// every fourth row with four independent accumulators; pass 2 sums the slices.
// Every sum has a fixed order, so results are deterministic.  Both passes are
// short and wait for memory: a lane has CS_U loads in flight (rows past the end
// read the last row and add 0), which covers most of a slice in one round trip:
// 17408 grouped rows of 1024 10.4 -> 8 to 12 us and 7.0 -> 4.7 us for the second
// pass, 1000 x 1000 5.3 + 4.1 -> 4.4 + 3.5 us.
constexpr int CS_U = 16;
constexpr int CS_SLICE = 128;  // target rows per slice
__global__ __launch_bounds__(256) void colsum_part_k(const float* __restrict__ X, long rows, int N, long ldx,
                                                     const int* __restrict__ goff, float* __restrict__ part,
                                                     int nslices) {
    // grid: (ceil(N / 64), nslices, groups)
    __shared__ float red[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane;
    const int g = blockIdx.z;
    long lo = 0, hi = rows;
    if (goff) {
        lo = goff[g];
        hi = goff[g + 1];
    }
    const long per = (hi - lo + nslices - 1) / nslices;
    const long a = lo + (long)blockIdx.y * per;
    const long b = min(hi, a + per);
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
    if (c < N) {
        for (long r = a + w; r < b; r += 4 * CS_U) {
            float x[CS_U];
#pragma unroll
            for (int u = 0; u < CS_U; ++u) x[u] = X[min(r + 4 * u, b - 1) * ldx + c];
            __builtin_amdgcn_sched_barrier(0);  // the loads go out together
#pragma unroll
            for (int u = 0; u < CS_U; u += 4) {
                s0 += r + 4 * u < b ? x[u] : 0.0f;
                s1 += r + 4 * u + 4 < b ? x[u + 1] : 0.0f;
                s2 += r + 4 * u + 8 < b ? x[u + 2] : 0.0f;
                s3 += r + 4 * u + 12 < b ? x[u + 3] : 0.0f;
            }
        }
    }
    red[w][lane] = (s0 + s1) + (s2 + s3);
    __syncthreads();
    if (w == 0 && c < N)
        part[((long)g * nslices + blockIdx.y) * N + c] = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

__global__ __launch_bounds__(256) void colsum_fin_k(const float* __restrict__ part, int nslices, int N,
                                                    float* __restrict__ out, int accumulate) {
    // grid: (ceil(N / 64), groups)
    __shared__ float red[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane;
    const long g = blockIdx.y;
    float s = 0.0f;
    if (c < N)
        for (int k = w; k < nslices; k += 4 * CS_U) {
            float x[CS_U];
#pragma unroll
            for (int u = 0; u < CS_U; ++u) x[u] = part[(g * nslices + min(k + 4 * u, nslices - 1)) * N + c];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < CS_U; ++u) s += k + 4 * u < nslices ? x[u] : 0.0f;
        }
    red[w][lane] = s;
    __syncthreads();
    if (w == 0 && c < N) {
        const float t = (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
        const long o = g * N + c;
        out[o] = accumulate ? out[o] + t : t;
    }
}

// ---------------------------------------------------------------- host side

static int ws_check(const Ws& ws, size_t floats, const char* name) {
    if (floats == 0) return ASCA_OK;
    if (!ws.p || ws.floats < floats)
        return fail(ASCA_ERR_INVALID, "%s: workspace of %zu floats, %zu needed", name, ws.floats, floats);
    return ASCA_OK;
}

template <bool TA, bool TB, int EPI, int GATHER>
static int launch_gemm_t(const GemmArgs& a, dim3 grid, hipStream_t st) {
    constexpr size_t lds = 2 * (size_t)sp_tile<128>();
    if (int arc = allow_lds(reinterpret_cast<const void*>(&gemm_k<TA, TB, EPI, GATHER>), lds)) return arc;
    hipLaunchKernelGGL((gemm_k<TA, TB, EPI, GATHER>), grid, dim3(256), lds, st, a);
    return ASCA_OK;
}
template <bool TA, bool TB, int EPI, int GATHER>
static int launch_wide_t(const GemmArgs& a, dim3 grid, hipStream_t st) {
    constexpr size_t lds = 2 * (size_t)(sp_tile<128>() + sp_tile<256>());
    static_assert(lds >= (size_t)SM_NW * 64 * 64 * sizeof(float), "the 64 x 64 tiles' sums fit");
    if (int arc = allow_lds(reinterpret_cast<const void*>(&gemm_wide_k<TA, TB, EPI, GATHER>), lds)) return arc;
    hipLaunchKernelGGL((gemm_wide_k<TA, TB, EPI, GATHER>), grid, dim3(512), lds, st, a);
    return ASCA_OK;
}

template <bool TA, bool TB, int EPI, int GATHER, int NX, int NY>
static int launch_small_t(const GemmArgs& a, dim3 grid, hipStream_t st) {
    constexpr size_t lds = (size_t)SM_NW * 256 * NX * NY * sizeof(float);
    if (int arc = allow_lds(reinterpret_cast<const void*>(&gemm_small_k<TA, TB, EPI, GATHER, NX, NY>), lds)) return arc;
    hipLaunchKernelGGL((gemm_small_k<TA, TB, EPI, GATHER, NX, NY>), grid, dim3(64 * SM_NW), lds, st, a);
    return ASCA_OK;
}

// Which tile a product takes: the one whose time on the device this model puts
// lowest.  Measured on MI355X, per k-tile of 32 (steps of them), a CU at a time:
//   WIDE  (128 x 256, one block per CU)  2.5 us    (4096^3: 225 TFLOP/s against 195 with 128 x 128)
//   T128  (128 x 128)                    1.75 us alone on its CU, 2.8 us for two blocks side by side
//   SMALL (64 x 64, k-tiles over 8 waves) 3.5 us for eight k-tiles
// and 4-7 us of first loads, sums and stores per round of blocks (the first
// round's 3 us of a small tile overlap the launch).  Products
// that fill the chip with the large tiles take those (a 64 x 64 tile splits
// each value for 64 products instead of 128 or 256); where those leave CUs idle
// the small tile wins: 1000x1000x320 22 -> 9.5 us, 64x1536x512 30 -> 11 us,
// 1000x320x1000 55 -> 19 us.
enum Tile { T_SMALL, T_128, T_WIDE };
// The most tiles beyond whole rounds that WIDE does as 64 x 64 tiles: while those
// take less time than another round (32 of 256 at K = 512: 14 us against 45; a
// tile is eight of them, so 96 are three rounds of 14 us).
static long tail_max(long steps) {
    const long cus = cu_count() > 0 ? cu_count() : 256;
    const double small = 3.5 * (double)((steps + 7) / 8) + 7.0;
    return (long)((2.5 * (double)steps + 5.0) / small) * cus / 8;
}
static double tile_us(Tile t, long tiles, long steps, bool tail) {
    const long cus = cu_count() > 0 ? cu_count() : 256;
    const double s = (double)steps;
    if (t == T_SMALL) return (double)((tiles + cus - 1) / cus) * (3.5 * (double)((steps + 7) / 8) + 7.0) - 4.0;
    if (t == T_WIDE) {
        const long rem = tiles % cus;
        const double round = 2.5 * s + 5.0;
        const double last = rem == 0 ? 0.0 : tail && rem <= tail_max(steps) ? tile_us(T_SMALL, 8 * rem, steps, false) + 4.0 : round;
        return (double)(tiles / cus) * round + last;
    }
    const long full = tiles / (2 * cus), rem = tiles % (2 * cus);
    return (double)full * (2.8 * s + 4.0) + (rem == 0 ? 0.0 : rem <= cus ? 1.75 * s + 5.0 : 2.8 * s + 4.0);
}
// tiles of an M x N product (rows in `groups` buckets of about M / groups when grouped)
static long tile_count(Tile t, long M, long N, int groups) {
    const long bm = t == T_SMALL ? 64 : 128, bn = t == T_SMALL ? 64 : t == T_WIDE ? 256 : 128;
    const long tn = (N + bn - 1) / bn;
    if (groups <= 0) return (M + bm - 1) / bm * tn;
    return (groups * ((M / groups + bm - 1) / bm) + (groups + 1) / 2) * tn;
}
static Tile best_tile(long M, long N, int groups, long mult, long steps, bool small_ok, bool whole_k, double* us) {
    Tile best = T_WIDE;
    // (one K range: the splits' blocks are not tiles of one launch dimension)
    const bool tail = small_ok && whole_k;
    double t = tile_us(T_WIDE, mult * tile_count(T_WIDE, M, N, groups), steps, tail);
    if (steps <= 1) t = 1e30;  // (SP_F32_K; and the first loads of two blocks per CU overlap)
    for (Tile c : {T_128, T_SMALL}) {
        if (c == T_SMALL && !small_ok) continue;
        const double u = tile_us(c, mult * tile_count(c, M, N, groups), steps, false);
        if (u < t) {
            t = u;
            best = c;
        }
    }
    if (us) *us = t;
    return best;
}
// Shape of the small tile, in 16 x 16 tiles: one row tile where the rows (of a
// group on average) do not pass 16 -- a 64-row tile would split and multiply
// mostly padding -- and fewer columns per block while the blocks fill less than
// half of the CUs.  One token for 64 sequences of the 8-layer d = 512 model (16 experts)
// 834 -> 676 us: its projections 15.8 -> 9.9 us each, its expert products 25.6 ->
// 15.0.  Sixteen waves per block instead of eight were slower (the 64 x 16 tile spills).
static void small_shape(long M, long N, int groups, long mult, int& nx, int& ny) {
    const long cus = cu_count() > 0 ? cu_count() : 256;
    const long rows = groups > 0 ? M / groups : M;
    if (rows <= 16) {
        nx = 1;
        return;
    }
    const long tm = mult * (groups > 0 ? groups : 1) * ((rows + 63) / 64);
    if (2 * tm * ((N + 63) / 64) <= cus) ny = 2;
    if (2 * tm * ((N + 31) / 32) <= cus) ny = 1;
}
template <bool TA, bool TB, int EPI, int GATHER>
static int launch_small(const GemmArgs& a, int nx, int ny, dim3 grid, hipStream_t st) {
    if constexpr (!TA) {
        if (nx == 1) return launch_small_t<TA, TB, EPI, GATHER, 1, 4>(a, grid, st);
        if (ny == 2) return launch_small_t<TA, TB, EPI, GATHER, 4, 2>(a, grid, st);
        if (ny == 1) return launch_small_t<TA, TB, EPI, GATHER, 4, 1>(a, grid, st);
    }
    return launch_small_t<TA, TB, EPI, GATHER, 4, 4>(a, grid, st);
}
// The small tile addresses an operand tile with 32-bit byte offsets: 64 rows
// (or 32 k-rows) of the leading dimension, or all `rows` of a gathered operand.
static bool small_fits(long ld, long rows) { return ld <= (1L << 22) && rows <= (1L << 30) / ld; }

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <bool TA, bool TB, int WM, int WN>
static int launch_batched_t(const GemmArgs& a, long items, hipStream_t st) {
    constexpr size_t lds =
        2 * (size_t)(tile_floats<!TA, 64 * WM>() + tile_floats<TB, 64 * WN>()) * sizeof(float);
    if (int arc = allow_lds(reinterpret_cast<const void*>(&gemm_batched_k<TA, TB, WM, WN>), lds)) return arc;
    // two resident blocks per CU, each walking items with a grid stride
    const long cap = 2L * (cu_count() > 0 ? cu_count() : 256);
    const unsigned grid = (unsigned)(items < cap ? items : cap);
    hipLaunchKernelGGL((gemm_batched_k<TA, TB, WM, WN>), dim3(grid), dim3(64 * WM * WN), lds, st, a);
    return ASCA_OK;
}

// Validates and launches one (possibly grouped) GEMM.  `m_total`: for gmode 1,
// the total rows over all groups (bounds the grid).
int gemm_launch(int ta, int tb, int epi, GemmArgs a, long m_total, hipStream_t st, const char* name) {
    if (a.M < 0 || a.N < 0 || a.K < 0) return fail(ASCA_ERR_INVALID, "%s: negative shape", name);
    if (a.gmode == 1 && ta) return fail(ASCA_ERR_INVALID, "%s: grouped rows need a non-transposed A", name);
    if (a.resid && (epi != EPI_STORE || a.k_per_split > 0))
        return fail(ASCA_ERR_UNSUPPORTED, "%s: residual input needs the plain epilogue without split-K", name);
    if (a.gmode == 2 && (!ta || tb)) return fail(ASCA_ERR_INVALID, "%s: grouped K needs A^T and B", name);
    if (epi == EPI_SILU && (ta || tb)) return fail(ASCA_ERR_UNSUPPORTED, "%s: SiLU epilogue is NN only", name);
    if (epi == EPI_SILU_BWD && (ta || !tb)) return fail(ASCA_ERR_UNSUPPORTED, "%s: SiLU-bwd epilogue is NT only", name);
    if (a.gmode == 3 && (a.a_rows || a.b_rows || a.c_rows || epi != EPI_STORE))
        return fail(ASCA_ERR_UNSUPPORTED, "%s: batched products take no row indirection or fused epilogue", name);
    const bool vec = (a.lda % 4 == 0) && (a.ldb % 4 == 0) && (a.ldc % 4 == 0) && (a.ld_aux % 4 == 0) &&
                     aligned16(a.A) && aligned16(a.B) && aligned16(a.C) && (!a.aux || aligned16(a.aux)) &&
                     (!a.aux_out || aligned16(a.aux_out)) && (a.a_gs % 4 == 0) && (a.b_gs % 4 == 0) &&
                     (a.c_gs % 4 == 0) && (a.c_split_stride % 4 == 0);
    // batched per-chunk products with at most 64 rows use 64 x 128 tiles
    const int wm = (a.gmode == 3 && vec && a.K > 0 && a.M <= 64) ? 1 : 2;
    const bool batched = a.gmode == 3 && vec && a.K > 0;
    const long splits = a.gmode == 0 && a.k_per_split > 0 ? (a.K + a.k_per_split - 1) / a.k_per_split : 1;
    if (a.gmode != 0 || a.k_per_split <= 0) a.k_per_split = a.K;
    // rows the gathered operands' indices can reach (grouped K: m_total rows in all)
    const long grows = a.gmode == 0 && (a.a_rows || a.b_rows) ? LONG_MAX : m_total;
    const bool small_ok = small_fits(max(a.lda, 1L), a.a_rows ? grows : 64) &&
                          small_fits(max(a.ldb, 1L), a.b_rows ? grows : 64);
    const long k_each = a.gmode == 2 ? m_total / max(a.ngroups, 1) : a.k_per_split;
    const Tile tile = best_tile(a.gmode == 1 ? m_total : a.M, a.N, a.gmode == 1 ? a.ngroups : 0,
                                a.gmode >= 2 ? a.ngroups : splits, (k_each + SP_BK - 1) / SP_BK, small_ok, splits == 1, nullptr);
    // the small tile's rows and columns (16 nx x 16 ny)
    int nx = 4, ny = 4;
    if (tile == T_SMALL && !ta) small_shape(a.gmode == 1 ? m_total : a.M, a.N, a.gmode == 1 ? a.ngroups : 0,
                                            a.gmode == 3 ? a.ngroups : splits, nx, ny);
    const int bm = tile == T_SMALL ? 16 * nx : GM_BM;
    const int bn = batched ? 128 : tile == T_SMALL ? 16 * ny : tile == T_WIDE ? 256 : 128;
    a.tiles_n = (a.N + bn - 1) / bn;
    a.tiles_m = batched ? (a.M + 64 * wm - 1) / (64 * wm) : (a.M + bm - 1) / bm;
    long blocks;
    if (a.gmode == 1)
        blocks = ((m_total + bm - 1) / bm + a.ngroups) * a.tiles_n;
    else if (a.gmode == 2 || a.gmode == 3)
        blocks = (long)a.ngroups * a.tiles_m * a.tiles_n;
    else
        blocks = (long)a.tiles_m * a.tiles_n;
    if (blocks == 0 || a.N == 0) return ASCA_OK;
    if (blocks > 0x7fffffffL) return fail(ASCA_ERR_INVALID, "%s: grid too large", name);
    int rc = pre_launch(name);
    if (rc) return rc;
    if (tile == T_WIDE && !batched) {
        a.cus = cu_count() > 0 ? cu_count() : 256;
        a.tail_max = splits == 1 && small_ok ? (int)tail_max((k_each + SP_BK - 1) / SP_BK) : 0;
        const long rem = blocks % a.cus;
        a.tail_blocks = a.tail_max == 0 ? 0 : a.gmode == 1 ? a.cus : rem <= a.tail_max ? (int)min((long)a.cus, 8 * rem) : 0;
        blocks += a.tail_blocks;
    }
    const dim3 grid((unsigned)blocks, (unsigned)splits);
    // operand whose K rows are gathered (mn-contiguous operands; k-contiguous ones gather rows in any variant)
    const int gather = ta && a.a_rows ? 1 : !tb && a.b_rows ? 2 : 0;
    if (gather && (!ta || tb || epi != EPI_STORE || (a.a_rows && a.b_rows)))
        return fail(ASCA_ERR_UNSUPPORTED, "%s: one gathered operand, of A^T B", name);
#define ASCA_GEMM_CASE(TA_, TB_, EPI_, G_)                                              \
    if (ta == TA_ && tb == TB_ && epi == EPI_ && gather == G_)                          \
        rc = tile == T_SMALL  ? launch_small<TA_, TB_, EPI_, G_>(a, nx, ny, grid, st)   \
             : tile == T_WIDE ? launch_wide_t<TA_, TB_, EPI_, G_>(a, grid, st)          \
                              : launch_gemm_t<TA_, TB_, EPI_, G_>(a, grid, st);         \
    else
#define ASCA_GEMM_BATCHED(TA_, TB_)                                                                     \
    if (ta == TA_ && tb == TB_)                                                                         \
        rc = wm == 1 ? launch_batched_t<TA_, TB_, 1, 2>(a, blocks, st)                                  \
                     : launch_batched_t<TA_, TB_, 2, 2>(a, blocks, st);                                 \
    else
    if (batched) {
        ASCA_GEMM_BATCHED(0, 0)
        ASCA_GEMM_BATCHED(1, 0)
        ASCA_GEMM_BATCHED(0, 1)
        ASCA_GEMM_BATCHED(1, 1)
        rc = fail(ASCA_ERR_UNSUPPORTED, "%s: no kernel for this variant", name);
        if (rc) return rc;
        return post_launch(name);
    }
#undef ASCA_GEMM_BATCHED
    ASCA_GEMM_CASE(0, 0, EPI_STORE, 0)
    ASCA_GEMM_CASE(1, 0, EPI_STORE, 0)
    ASCA_GEMM_CASE(1, 0, EPI_STORE, 1)
    ASCA_GEMM_CASE(1, 0, EPI_STORE, 2)
    ASCA_GEMM_CASE(0, 1, EPI_STORE, 0)
    ASCA_GEMM_CASE(1, 1, EPI_STORE, 0)
    ASCA_GEMM_CASE(0, 0, EPI_SILU, 0)
    ASCA_GEMM_CASE(0, 1, EPI_SILU_BWD, 0)
    rc = fail(ASCA_ERR_UNSUPPORTED, "%s: no kernel for this variant", name);
#undef ASCA_GEMM_CASE
    if (rc) return rc;
    return post_launch(name);
}

GemmArgs gemm_args() {
    GemmArgs a{};
    a.alpha = 1.0f;
    a.beta = 0.0f;
    return a;
}

// Slices of a column sum: about CS_SLICE rows each (twice as many per group:
// group sizes vary).
static int colsum_slices(long rows, int G, bool grouped) {
    const long avg = grouped ? (2 * rows) / G + 1 : rows;
    const int ns = (int)min((avg + CS_SLICE - 1) / CS_SLICE, 1024L);
    return ns < 1 ? 1 : ns;
}

size_t colsum_ws_floats(long rows, int N, bool grouped, int ngroups) {
    const int G = grouped ? ngroups : 1;
    if (N <= 0 || G <= 0) return 0;
    return (size_t)G * colsum_slices(rows, G, grouped) * N;
}

// Column sums of X (rows x N, ld ldx), per group when goff is given.
int colsum_launch(const float* X, long rows, int N, long ldx, const int* goff, int ngroups, float* out,
                  int accumulate, Ws ws, hipStream_t st) {
    if (N == 0) return ASCA_OK;
    const int G = goff ? ngroups : 1;
    if (G == 0) return ASCA_OK;
    const int cb = (N + 63) / 64;
    const int ns = colsum_slices(rows, G, goff != nullptr);
    int rc = ws_check(ws, (size_t)G * ns * N, "colsum");
    if (rc) return rc;
    float* const part = ws.p;
    rc = pre_launch("colsum");
    if (rc) return rc;
    hipLaunchKernelGGL(colsum_part_k, dim3(cb, ns, G), dim3(256), 0, st, X, rows, N, ldx, goff, part, ns);
    rc = post_launch("colsum");
    if (rc) return rc;
    rc = pre_launch("colsum_fin");
    if (rc) return rc;
    hipLaunchKernelGGL(colsum_fin_k, dim3(cb, G), dim3(256), 0, st, part, ns, N, out, accumulate);
    return post_launch("colsum_fin");
}

// ---------------------------------------------------------------------------
// Skinny products with n <= 16 output columns (the gate projection, n = 2H):
// the 16-wide MFMA output tile matches them, where a 128-wide block tile of
// the general kernel would multiply mostly padding.
//
// Forward Y (T x n) = X (T x K) W (K x n) + b: one block per 16 rows, a quarter
// of K to each of its four waves (a wave's loads and its chain of products are
// the time of a decode step's few rows; the sums meet in LDS: 64 rows of K = 512
// 8.7 -> 3.7 us, 16384 rows 12.0 -> 9.7).  Lane
// (i = l % 16, q = l / 16) supplies A = X[row i][16 j + 4 q + e] from one
// 16-byte load per 16-k group j (e = 0..3 are four MFMA k-steps: the k index
// is permuted inside each group of 16, which the sum does not see) and keeps
// the matching B = W[16 j + 4 q + e][i] for its whole K in registers.
template <int KT>  // K = 64 KT
__global__ __launch_bounds__(256) void skinny_fwd_k(const float* __restrict__ X, long ldx, const float* __restrict__ W,
                                                    const float* __restrict__ b, float* __restrict__ Y, long T, int n) {
    __shared__ f32x4 part[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long r0 = (long)blockIdx.x * 16;
    const int i = lane & 15, q = lane >> 4;
    const int ic = min(i, n - 1), k0 = 16 * KT * w + 4 * q;
    float wb[4 * KT];
#pragma unroll
    for (int j = 0; j < KT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = W[(long)(k0 + 16 * j + e) * n + ic];
            wb[4 * j + e] = i < n ? v : 0.0f;
        }
    const float* xr = X + min(r0 + i, T - 1) * ldx + k0;
    float4 xv[KT];
#pragma unroll
    for (int j = 0; j < KT; ++j) xv[j] = *reinterpret_cast<const float4*>(xr + 16 * j);
    // every load above is in flight before the first product (the scheduler
    // would otherwise interleave them with the products, one wait each)
    __builtin_amdgcn_sched_barrier(0);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < KT; ++j) {
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[j].x, wb[4 * j + 0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[j].y, wb[4 * j + 1], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[j].z, wb[4 * j + 2], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[j].w, wb[4 * j + 3], acc, 0, 0, 0);
    }
    part[w][lane] = acc;
    __syncthreads();
    if (w) return;
    acc = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    const float bi = b ? b[ic] : 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const long row = r0 + 4 * q + r;
        if (i < n && row < T) Y[row * n + i] = acc[r] + bi;
    }
}

// Weight gradient G (K x n) = X^T D and bias gradient db = column sums of D,
// over T rows.  Block (64 columns of X, chunk s) reduces rows s*SK_T .. +SK_T
// into a 64 x 16 partial of G, its four waves a quarter of the rows each: per
// MFMA k-step the four lane groups q take rows t = 4 m + q, lane (i, q) supplies
// X[t][64 it + 4 i .. + 3] (16 bytes; the four columns go to four output tiles)
// and D[t][i].  The kernel is the reading of X, so a wave has all its loads in
// flight and rows are read 256 bytes at a time.  Blocks of it = 0 also sum D for
// db.  Partials go to part[s][K + 1][16] (row K: db) and skinny_reduce_k adds
// them in a fixed order.  16384 x 512: 75 us with a wave per 16 columns (64 bytes
// of a row, each 128-byte line read by two XCDs), 28 us beside the backward's
// products.
constexpr int SK_T = 256;  // rows per block
__global__ __launch_bounds__(256) void skinny_wgrad_k(const float* __restrict__ X, long ldx,
                                                      const float* __restrict__ D, long T, int K, int n,
                                                      float* __restrict__ part) {
    __shared__ float4 red[4][16 * 16];  // [wave][column of X, output column / 4]
    __shared__ float red_db[4][16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int it = blockIdx.x % (K / 64);
    const long s = blockIdx.x / (K / 64);
    const int i = lane & 15, q = lane >> 4;
    const int ic = min(i, n - 1);
    const long t0 = s * SK_T + w * (SK_T / 4) + q;
    f32x4 acc[4] = {};
    float dsum = 0.0f;
    constexpr int NM = SK_T / 16;
    float4 av[NM];
    float bv[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        const long t = min(t0 + 4 * m, T - 1);
        av[m] = *reinterpret_cast<const float4*>(X + t * ldx + 64 * it + 4 * i);
        bv[m] = D[t * n + ic];
    }
    __builtin_amdgcn_sched_barrier(0);  // the loads go out together
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        const bool in = t0 + 4 * m < T;
        const float b = in && i < n ? bv[m] : 0.0f;
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? av[m].x : 0.0f, b, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? av[m].y : 0.0f, b, acc[1], 0, 0, 0);
        acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? av[m].z : 0.0f, b, acc[2], 0, 0, 0);
        acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? av[m].w : 0.0f, b, acc[3], 0, 0, 0);
        dsum += b;
    }
    float* const mine = reinterpret_cast<float*>(red[w]);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) mine[(16 * q + 4 * r + u) * 16 + i] = acc[u][r];
    if (it == 0) {
        dsum += __shfl_xor(dsum, 16);
        dsum += __shfl_xor(dsum, 32);
        if (q == 0) red_db[w][i] = dsum;
    }
    __syncthreads();
    float* const ps = part + s * (long)(K + 1) * 16;
    const float4 a = red[0][threadIdx.x], b = red[1][threadIdx.x], c = red[2][threadIdx.x], d = red[3][threadIdx.x];
    reinterpret_cast<float4*>(ps + 64 * it * 16)[threadIdx.x] =
        make_float4((a.x + b.x) + (c.x + d.x), (a.y + b.y) + (c.y + d.y), (a.z + b.z) + (c.z + d.z),
                    (a.w + b.w) + (c.w + d.w));
    if (it == 0 && threadIdx.x < 16) {
        const int j = threadIdx.x;
        ps[K * 16 + j] = (red_db[0][j] + red_db[1][j]) + (red_db[2][j] + red_db[3][j]);
    }
}

// One wave per output row of the (K + 1) x n result: lane (c = l % 16,
// g = l / 16) adds chunks g, g + 4, ... (independent loads, all in flight),
// then the four lane groups are added (a fixed order).
__global__ __launch_bounds__(256) void skinny_reduce_k(const float* __restrict__ part, long nch, int K, int n,
                                                       float* __restrict__ G, float* __restrict__ db) {
    const int lane = threadIdx.x & 63;
    const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row > K) return;  // whole wave
    const int c = lane & 15, g = lane >> 4;
    float acc = 0.0f;
    for (long s = g; s < nch; s += 4 * CS_U) {
        float x[CS_U];
#pragma unroll
        for (int u = 0; u < CS_U; ++u) x[u] = part[(min(s + 4 * u, nch - 1) * (K + 1) + row) * 16 + c];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < CS_U; ++u) acc += s + 4 * u < nch ? x[u] : 0.0f;
    }
    acc += __shfl_xor(acc, 16);
    acc += __shfl_xor(acc, 32);
    if (g == 0 && c < n) {
        if (row < K)
            G[row * n + c] = acc;
        else if (db)
            db[c] = acc;
    }
}

static bool skinny_ok(const float* X, long ldx, int K, int n) {
    return n >= 1 && n <= 16 && (K == 128 || K == 256 || K == 512) && ldx % 4 == 0 &&
           (reinterpret_cast<uintptr_t>(X) & 15) == 0;
}

int skinny_fwd_launch(const float* X, long ldx, const float* W, const float* b, float* Y, long T, int K, int n,
                      hipStream_t st) {
    if (T <= 0 || n <= 0) return ASCA_OK;
    if (!skinny_ok(X, ldx, K, n)) {
        GemmArgs a = gemm_args();
        a.A = X;
        a.lda = ldx;
        a.B = W;
        a.ldb = n;
        a.C = Y;
        a.ldc = n;
        a.M = (int)T;
        a.N = n;
        a.K = K;
        a.bias = b;
        return gemm_launch(0, 0, EPI_STORE, a, T, st, "skinny_fwd");
    }
    int rc = pre_launch("skinny_fwd");
    if (rc) return rc;
    const dim3 grid((unsigned)((T + 15) / 16));
    if (K == 512)
        hipLaunchKernelGGL(skinny_fwd_k<8>, grid, dim3(256), 0, st, X, ldx, W, b, Y, T, n);
    else if (K == 256)
        hipLaunchKernelGGL(skinny_fwd_k<4>, grid, dim3(256), 0, st, X, ldx, W, b, Y, T, n);
    else
        hipLaunchKernelGGL(skinny_fwd_k<2>, grid, dim3(256), 0, st, X, ldx, W, b, Y, T, n);
    return post_launch("skinny_fwd");
}

size_t skinny_wgrad_ws_floats(long T, int K, int n) {
    if (n <= 0 || K <= 0) return 0;
    const size_t fallback = max(gemm_ws_floats(K, n, (int)min(T, 0x7fffffffL)), colsum_ws_floats(T, n, false, 0));
    const long nch = (max(T, 0L) + SK_T - 1) / SK_T;
    return max(fallback, (size_t)nch * (K + 1) * 16);
}

int skinny_wgrad_launch(const float* X, long ldx, const float* D, float* G, float* db, long T, int K, int n,
                        Ws ws, hipStream_t st) {
    if (n <= 0 || K <= 0) return ASCA_OK;
    if (T <= 0 || !skinny_ok(X, ldx, K, n)) {
        int rc = gemm_run(1, 0, K, n, (int)T, 1.0f, X, ldx, D, n, 0.0f, G, n, nullptr, ws, st);
        if (rc || !db) return rc;
        return colsum_launch(D, T, n, n, nullptr, 0, db, 0, ws, st);
    }
    const long nch = (T + SK_T - 1) / SK_T;
    int rc = ws_check(ws, (size_t)nch * (K + 1) * 16, "skinny_wgrad");
    if (rc) return rc;
    float* const part = ws.p;
    if ((rc = pre_launch("skinny_wgrad"))) return rc;
    hipLaunchKernelGGL(skinny_wgrad_k, dim3((unsigned)(K / 64 * nch)), dim3(256), 0, st, X, ldx, D, T, K, n,
                       part);
    if ((rc = post_launch("skinny_wgrad"))) return rc;
    if ((rc = pre_launch("skinny_reduce"))) return rc;
    hipLaunchKernelGGL(skinny_reduce_k, dim3((unsigned)((K + 1 + 3) / 4)), dim3(256), 0, st, part, nch, K, n, G, db);
    return post_launch("skinny_reduce");
}

// Split-K decision of a plain product: split K when the output has too few
// tiles to fill the chip, into as many K ranges as keep the grid within one
// round of two blocks per CU (rounding up would give 512x1536x16384 eleven
// splits, 528 blocks: a second round of 16).
// Returns the split count and the K range per split.
static int gemm_splits(int M, int N, int K, long* kps_out) {
    const long tiles = (long)((M + GM_BM - 1) / GM_BM) * ((N + GM_BN - 1) / GM_BN);
    const int cus = cu_count() > 0 ? cu_count() : 256;
    int splits = 1;
    if (tiles < cus && K >= 1024) {
        splits = (int)min((long)K / 512, (2L * cus) / tiles);
        if (splits < 1) splits = 1;
    }
    long kps = K;
    if (splits > 1) {
        kps = ((K + splits - 1) / splits + GM_BK - 1) / GM_BK * GM_BK;
        splits = (int)((K + kps - 1) / kps);
    }
    *kps_out = kps;
    return splits;
}

size_t gemm_ws_floats(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    long kps = 0;
    const int splits = gemm_splits(M, N, K, &kps);
    return splits > 1 ? (size_t)splits * M * N : 0;
}

int gemm_check(int trans_a, int trans_b, int M, int N, int K, const float* A, long lda, const float* B, long ldb,
               const float* C, long ldc) {
    if (M < 0 || N < 0 || K < 0) return fail(ASCA_ERR_INVALID, "asca_gemm: negative shape");
    if (M == 0 || N == 0) return ASCA_OK;
    if (!C || (K > 0 && (!A || !B))) return fail(ASCA_ERR_INVALID, "asca_gemm: null pointer");
    const long a_cols = trans_a ? M : K, b_cols = trans_b ? K : N;
    if (lda < a_cols || ldb < b_cols || ldc < N) return fail(ASCA_ERR_INVALID, "asca_gemm: leading dimension too small");
    return ASCA_OK;
}

// C = alpha op(A) op(B) + beta C (+ bias), split-K partials in ws.
int gemm_run(int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A, long lda, const float* B,
             long ldb, float beta, float* C, long ldc, const float* bias, Ws ws, hipStream_t st) {
    if (M == 0 || N == 0) return ASCA_OK;
    GemmArgs a = gemm_args();
    a.A = A;
    a.B = B;
    a.C = C;
    a.lda = lda;
    a.ldb = ldb;
    a.ldc = ldc;
    a.M = M;
    a.N = N;
    a.K = K;
    a.alpha = alpha;
    a.beta = beta;
    a.bias = bias;
    long kps = 0;
    int splits = K > 0 ? gemm_splits(M, N, K, &kps) : 1;
    if (splits > 1) {
        // one pass over K where that is no slower than the partials and their sum
        double one, cut;
        const bool fits = small_fits(max(lda, 1L), 64) && small_fits(max(ldb, 1L), 64);
        best_tile(M, N, 0, 1, (K + SP_BK - 1) / SP_BK, fits, true, &one);
        best_tile(M, N, 0, splits, (kps + SP_BK - 1) / SP_BK, fits, false, &cut);
        if (one <= cut + 5.0 + 1e-6 * splits * M * N) splits = 1;
    }
    if (splits == 1) return gemm_launch(trans_a, trans_b, EPI_STORE, a, M, st, "gemm");
    const long MN = (long)M * N;
    int rc = ws_check(ws, (size_t)splits * MN, "gemm split-K");
    if (rc) return rc;
    float* const part = ws.p;
    GemmArgs s = a;
    s.C = part;
    s.ldc = N;
    s.alpha = 1.0f;
    s.beta = 0.0f;
    s.bias = nullptr;
    s.k_per_split = kps;
    s.c_split_stride = MN;
    rc = gemm_launch(trans_a, trans_b, EPI_STORE, s, M, st, "gemm_splitk");
    if (rc) return rc;
    rc = pre_launch("splitk_reduce");
    if (rc) return rc;
    const int cus = cu_count() > 0 ? cu_count() : 256;
    const bool vec = N % 4 == 0 && ldc % 4 == 0 &&
                     ((reinterpret_cast<uintptr_t>(part) | reinterpret_cast<uintptr_t>(C) |
                       reinterpret_cast<uintptr_t>(bias)) & 15) == 0;
    const long blocks = min((MN / (vec ? 4 : 1) + 255) / 256, 4L * cus * 8);
    if (vec)
        hipLaunchKernelGGL(splitk_reduce_k<true>, dim3((unsigned)blocks), dim3(256), 0, st, part, splits, MN, N, C, ldc,
                           alpha, beta, bias);
    else
        hipLaunchKernelGGL(splitk_reduce_k<false>, dim3((unsigned)blocks), dim3(256), 0, st, part, splits, MN, N, C,
                           ldc, alpha, beta, bias);
    return post_launch("splitk_reduce");
}

// Scratch of asca_gemm_noalloc, the entry point for callers that cannot
// allocate: a static device array of SCRATCH_FLOATS floats (32 MiB), which
// every device the library runs on holds until the process ends.  Its size is
// the most split-K partials can take on gfx950 (256 CUs): gemm_splits keeps
// splits * tiles <= 2 * CUs and a tile covers at most GM_BM x GM_BN outputs,
// so splits * M * N <= 2 * 256 * GM_BM * GM_BN floats; the size check in
// asca_gemm_noalloc stays as a guard.  In host code `scratch` names a
// host-side stand-in, never the device memory: its device address comes from
// hipGetSymbolAddress, once per device at asca_init (with that device
// current), and only that address is used.
constexpr size_t SCRATCH_FLOATS = (size_t)2 * 256 * GM_BM * GM_BN;
static __device__ __align__(256) float scratch[SCRATCH_FLOATS];
static float* g_scratch_dev[64] = {};

int noalloc_scratch_init(int device) {
    if (device < 0 || device >= 64) return fail(ASCA_ERR_INVALID, "device %d out of range", device);
    if (g_scratch_dev[device]) return ASCA_OK;
    void* p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        return fail(ASCA_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", device, hipGetErrorString(e));
    g_scratch_dev[device] = reinterpret_cast<float*>(p);
    return ASCA_OK;
}

}  // namespace asca

using namespace asca;

extern "C" {

int asca_gemm_ws_bytes(int trans_a, int trans_b, int M, int N, int K, size_t* bytes) {
    (void)trans_a;
    (void)trans_b;
    if (!bytes) return fail(ASCA_ERR_INVALID, "null output pointer");
    if (M < 0 || N < 0 || K < 0) return fail(ASCA_ERR_INVALID, "asca_gemm_ws_bytes: negative shape");
    *bytes = gemm_ws_floats(M, N, K) * sizeof(float);
    return ASCA_OK;
}

int asca_gemm_ws(int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A, long lda, const float* B,
                 long ldb, float beta, float* C, long ldc, const float* bias, void* ws, size_t ws_bytes,
                 void* stream) {
    int rc = gemm_check(trans_a, trans_b, M, N, K, A, lda, B, ldb, C, ldc);
    if (rc || M == 0 || N == 0) return rc;
    return gemm_run(trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, bias,
                    Ws{reinterpret_cast<float*>(ws), ws_bytes / sizeof(float)}, as_stream(stream));
}

// The reference's matmul takes no workspace: split-K partials come from the
// stream-ordered allocator on the call's stream and go back to it behind the
// reduction, so calls on different streams never share them.
int asca_gemm(int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A, long lda, const float* B,
              long ldb, float beta, float* C, long ldc, const float* bias, void* stream) {
    int rc = gemm_check(trans_a, trans_b, M, N, K, A, lda, B, ldb, C, ldc);
    if (rc || M == 0 || N == 0) return rc;
    const hipStream_t st = as_stream(stream);
    const size_t need = gemm_ws_floats(M, N, K);
    StreamScratch sc;
    if ((rc = sc.get(need, st))) return rc;
    rc = gemm_run(trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, bias, sc.ws, st);
    const int rf = sc.release(st);
    return rc ? rc : rf;
}

// asca_gemm whose split-K partials live in the static scratch: allocates
// nothing.  Calls that overlap on one device share that scratch and race.
int asca_gemm_noalloc(int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A, long lda,
                      const float* B, long ldb, float beta, float* C, long ldc, const float* bias, void* stream) {
    int rc = gemm_check(trans_a, trans_b, M, N, K, A, lda, B, ldb, C, ldc);
    if (rc || M == 0 || N == 0) return rc;
    if ((rc = ensure_device())) return rc;
    const size_t need = gemm_ws_floats(M, N, K);
    if (need > SCRATCH_FLOATS)
        return fail(ASCA_ERR_INVALID,
                    "asca_gemm_noalloc: the split-K partials of %dx%dx%d need %zu bytes, the static scratch holds "
                    "%zu (use asca_gemm_ws)",
                    M, N, K, need * sizeof(float), SCRATCH_FLOATS * sizeof(float));
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64 || !g_scratch_dev[dev])
        return fail(ASCA_ERR_NOT_INIT, "asca_gemm_noalloc: no static scratch address for device %d", dev);
    return gemm_run(trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, bias,
                    Ws{g_scratch_dev[dev], SCRATCH_FLOATS}, as_stream(stream));
}

int asca_colsum_ws_bytes(long rows, int cols, size_t* bytes) {
    if (!bytes) return fail(ASCA_ERR_INVALID, "null output pointer");
    if (rows < 0 || cols < 0) return fail(ASCA_ERR_INVALID, "asca_colsum_ws_bytes: negative shape");
    *bytes = colsum_ws_floats(rows, cols, false, 0) * sizeof(float);
    return ASCA_OK;
}

int asca_colsum_ws(const float* X, long rows, int cols, float* out, int accumulate, void* ws, size_t ws_bytes,
                   void* stream) {
    if (rows < 0 || cols < 0) return fail(ASCA_ERR_INVALID, "asca_colsum: negative shape");
    if (cols == 0) return ASCA_OK;
    if (!out || (rows > 0 && !X)) return fail(ASCA_ERR_INVALID, "asca_colsum: null pointer");
    return colsum_launch(X, rows, cols, cols, nullptr, 0, out, accumulate,
                         Ws{reinterpret_cast<float*>(ws), ws_bytes / sizeof(float)}, as_stream(stream));
}

int asca_colsum(const float* X, long rows, int cols, float* out, int accumulate, void* stream) {
    if (rows < 0 || cols < 0) return fail(ASCA_ERR_INVALID, "asca_colsum: negative shape");
    if (cols == 0) return ASCA_OK;
    if (!out || (rows > 0 && !X)) return fail(ASCA_ERR_INVALID, "asca_colsum: null pointer");
    const hipStream_t st = as_stream(stream);
    StreamScratch sc;
    int rc = sc.get(colsum_ws_floats(rows, cols, false, 0), st);
    if (rc) return rc;
    rc = colsum_launch(X, rows, cols, cols, nullptr, 0, out, accumulate, sc.ws, st);
    const int rf = sc.release(st);
    return rc ? rc : rf;
}

}  // extern "C"

// mm_kq_impl.h — products of several Q8_K activation columns with K-quant weights (Q4_K, Q5_K,
// Q6_K) on the matrix cores: prompts, multi-token steps and the routed experts of both. One
// translation unit per weight type (k_mm_q4_k.hip, ...) instantiates it; k_mm_kq.hip holds the
// dispatch.
//
// ggml-cpu's q4_K / q5_K / q6_K x q8_K dots (the oracle's oracle_vec_dot_q{4,5,6}_K_q8_K) keep eight
// float accumulators per output, one per element index mod 8: for every 256-element super-block,
// aux32[l] = sum over the 32 elements e = 8k + l of sc[sub-block of e] * q[e] * q8[e] (an exact
// integer), sums[l] += (d_w * d_x) * aux32[l]; Q4_K and Q5_K subtract their mins as
// sumf -= (dmin_w * d_x) * sum_j bsums[j] * m[j / 2]; the output is sumf + sums[0] + ... + sums[7].
//
// A wave takes 16 weight rows and NT tiles of 16 columns over the whole of K, so
// the nine running sums of its outputs stay in registers and are added in ggml's order. One
// v_mfma_f32_16x16x32_f16 per slice l gives aux32[l] of a tile: the activations come in a form
// (q8k_act::x16) whose slices are f16 runs in MFMA operand order, and each lane decodes its own
// share of a weight row (row lane % 16, the elements 64 q .. 64 q + 63 of the super-block with
// q = lane / 16, which are k = 8q .. 8q + 7 of every slice) in registers: no weight goes through
// LDS and a decoded operand serves all NT tiles. sc * q is exact in f16 for Q4_K (at most 945) and
// Q5_K (1953); Q6_K's sc * (q - 32) is split as sc * (q % 16) + sc * 16 (q / 16 - 2), both exact,
// in two accumulating MFMAs. Every product and partial sum is an integer of at most 2^24, so the
// MFMA sums are exact in any order. The mins term is one v_mfma_f32_16x16x16_f16 of the mins (each
// repeated for its two 16-element halves) against the 16 bsums.
//
// The activations of the workgroup's columns go through LDS a super-block at a time, in two buffers,
// the next one's loads in flight while the current one is used (mm_kq_kernel), or all of K at once
// where the columns are few (mm_kq_res_kernel); with few tiles K is split over the waves instead
// (mm_kq_split_kernel).
//
// What bounds it: the VALU (per 16 x 16 tile and super-block 80 operations for the nine sums, and
// about 120 to decode the weights, shared by the NT tiles) together with the matrix cores. Counted over 512
// columns of Q4_K: the vector instructions fill 60% of the SIMDs' time in 64 x 64 tiles and 51% in 64 x 48
// ones, the matrix instructions 16% and 14%; the rest waits at the barriers and, for small grids, on CUs
// with two workgroups beside CUs with one. Routed 64 x 32 tiles stand at 34-38%, workgroups with
// resident columns at 62%. Measured (us, with the activation's quantization) against the kernels it
// replaced: a prompt's gate and up
// projections (Q4_K, K = 2560, 2 x 9728 rows, 512 columns) 200 -> 152, its down projection (K =
// 9728, 2560 rows) 100 -> 94; 16 columns 120 -> 17.7 (K = 9728, 2560 rows), 63 columns of Q6_K 510 ->
// 50; the routed experts of a 384-token prompt (128 experts of 768, top 8) 3138 -> 260, of a 16-token
// step 104 -> 79.
#pragma once

#include "kernels.h"
#include "gemv_ops.h"

#include "ggml.h"

#include <type_traits>

namespace mm_kq_detail {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));   // (arrays of HIP's uint4 copied whole stay in scratch)

struct mm_kargs {
    gemv_launch L;
    int row_begin[GEMV_MAX_MATS + 1];            // in rows of the grid, every matrix on a workgroup boundary
    int n_rt, n_ct;                              // row tiles, column tiles (or items) of the grid
    expert_groups g;                             // g.cols set: column tile i is item i
};

__device__ __forceinline__ uint32_t and_or(uint32_t v, uint32_t mask, uint32_t bits) { return (v & mask) | bits; }
__device__ __forceinline__ __half2 h2(uint32_t v) { return __builtin_bit_cast(__half2, v); }
__device__ __forceinline__ uint32_t u2(__half2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ __half2 h2_of(int v) { return __half2half2(__int2half_rn(v)); }
// byte b of x and of y, zero-extended to the halves of a dword
template <int B>
__device__ __forceinline__ uint32_t byte_pair(uint32_t x, uint32_t y) {
    return __builtin_amdgcn_perm(y, x, 0x0c000c00u | (uint32_t) B | ((uint32_t) (4 + B) << 16));
}

// One lane's share of a weight row (wrow: where its first super-block's pieces are) and of one
// super-block of it (wlane: the raw bytes; wprep: its scales as f16 pairs, and slice<l>, the MFMA
// operand of slice l).
template <int TYPE> struct wlane;

// (uniform bases of the wave's first row, 32-bit lane offsets from them)
template <int TYPE>
struct wrow {
    static constexpr int BYTES = TYPE == GGML_TYPE_Q4_K ? Q4_K_BYTES : Q5_K_BYTES;
    const uint8_t * base;
    uint32_t h, a;
    __device__ __forceinline__ void at(const gemv_mat & m, int64_t erow, int first, int row, int nsb, int q) {
        base = m.w + (erow + first) * nsb * BYTES;
        h = (uint32_t) (row - first) * (uint32_t) (nsb * BYTES);
        a = h + (TYPE == GGML_TYPE_Q4_K ? 16 : 48) + 32 * q;
    }
};
template <>
struct wrow<GGML_TYPE_Q6_K> {
    const uint8_t * bl, * bh, * bs, * bd;
    uint32_t ql, qh, sc, d;
    __device__ __forceinline__ void at(const gemv_mat & m, int64_t erow, int first, int row, int nsb, int q) {
        const int64_t b = (erow + first) * nsb;
        const uint32_t o = (uint32_t) (row - first) * (uint32_t) nsb;
        bl = m.w + b * 128;
        bh = m.wqh + b * 64;
        bs = (const uint8_t *) m.wsc + b * 16;
        bd = (const uint8_t *) (m.wd + b);
        ql = o * 128 + 64 * (q / 2);
        qh = o * 64 + 32 * (q / 2);
        sc = o * 16 + 4 * q;
        d = o * 2;
    }
};

template <>
struct wlane<GGML_TYPE_Q4_K> {
    uint4 h, a, b;
    __device__ __forceinline__ void load(const wrow<GGML_TYPE_Q4_K> & w, int sb) {
        const uint8_t * p = w.base + (int64_t) sb * Q4_K_BYTES;
        h = *(const uint4 *) (p + w.h);
        a = *(const uint4 *) (p + w.a);
        b = *(const uint4 *) (p + w.a + 16);
    }
};
template <>
struct wlane<GGML_TYPE_Q5_K> {
    uint4 h, a, b, f0, f1;      // f: the fifth bits
    __device__ __forceinline__ void load(const wrow<GGML_TYPE_Q5_K> & w, int sb) {
        const uint8_t * p = w.base + (int64_t) sb * Q5_K_BYTES;
        h = *(const uint4 *) (p + w.h);
        f0 = *(const uint4 *) (p + w.h + 16);
        f1 = *(const uint4 *) (p + w.h + 32);
        a = *(const uint4 *) (p + w.a);
        b = *(const uint4 *) (p + w.a + 16);
    }
};
template <>
struct wlane<GGML_TYPE_Q6_K> {
    uint4 a, b, c, d, f0, f1;   // low bits of runs A and B (32 bytes each), the half's high bits
    uint32_t sc;                // the lane's four scales
    __half dw;
    __device__ __forceinline__ void load(const wrow<GGML_TYPE_Q6_K> & w, int sb) {
        const uint4 * ql = (const uint4 *) (w.bl + (int64_t) sb * 128 + w.ql);
        const uint4 * qh = (const uint4 *) (w.bh + (int64_t) sb * 64 + w.qh);
        a = ql[0]; b = ql[1]; c = ql[2]; d = ql[3];
        f0 = qh[0]; f1 = qh[1];
        sc = *(const uint32_t *) (w.bs + (int64_t) sb * 16 + w.sc);
        dw = *(const __half *) (w.bd + (int64_t) sb * 2 + w.d);
    }
};

template <int TYPE> struct wprep;

// Q4_K / Q5_K: the lane's sub-blocks 2q (low nibbles) and 2q + 1 (high nibbles, kept as 16 n). A
// nibble n placed under the f16 exponent of 1024 is 1024 + n, and one fused multiply-add
// (1024 + n) * sc - 1024 sc gives n * sc exactly (1024 * 63 is below f16's largest value).
template <int TYPE>
struct wprep_q45 {
    __half2 sa, ca, sb, cb;
    float dw, dm;
    f16x4 mins;
    uint32_t w[8];
    __device__ __forceinline__ void prep45(const uint4 & h, const uint4 & a, const uint4 & b, int q) {
        dw = __half2float(__ushort_as_half((unsigned short) (h.x & 0xffff)));
        dm = __half2float(__ushort_as_half((unsigned short) (h.x >> 16)));
        // the 6-bit scales and mins of sub-blocks 2q, 2q + 1, two bytes at a time
        const int sh = 16 * (q & 1);
        const uint32_t s0 = h.y >> sh, s1 = h.z >> sh, s2 = h.w >> sh;
        const bool up = q >= 2;
        const uint32_t sc = up ? (s2 & 0x0f0fu) | ((s0 & 0xc0c0u) >> 2) : s0 & 0x3f3fu;
        const uint32_t mn = up ? ((s2 >> 4) & 0x0f0fu) | ((s1 & 0xc0c0u) >> 2) : s1 & 0x3f3fu;
        sa = h2_of((int) (sc & 0xff));
        sb = h2_of((int) (sc >> 8));
        ca = __hmul2(sa, __float2half2_rn(-1024.0f));
        cb = __hmul2(sb, __float2half2_rn(-64.0f));
        sb = __hmul2(sb, __float2half2_rn(0.0625f));
        const _Float16 ma = (_Float16) (float) (mn & 0xff), mb = (_Float16) (float) (mn >> 8);
        mins = f16x4{ ma, ma, mb, mb };
        w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
        w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
    }
};

template <>
struct wprep<GGML_TYPE_Q4_K> : wprep_q45<GGML_TYPE_Q4_K> {
    static constexpr bool MINS = true, SPLIT = false;
    __device__ __forceinline__ void prep(const wlane<GGML_TYPE_Q4_K> & r, int q) { prep45(r.h, r.a, r.b, q); }
    // slice l: bytes l, l + 8, l + 16, l + 24 of the pair's 32
    template <int L>
    __device__ __forceinline__ f16x8 slice(f16x8 &) const {
        constexpr int B = L % 4, D = L / 4;
        const uint32_t p = byte_pair<B>(w[D], w[D + 2]), r = byte_pair<B>(w[D + 4], w[D + 6]);
        const uint32_t lo0 = and_or(p, 0x000f000fu, 0x64006400u), hi0 = and_or(p, 0x00f000f0u, 0x64006400u);
        const uint32_t lo1 = and_or(r, 0x000f000fu, 0x64006400u), hi1 = and_or(r, 0x00f000f0u, 0x64006400u);
        return __builtin_bit_cast(f16x8, make_uint4(u2(__hfma2(h2(lo0), sa, ca)), u2(__hfma2(h2(lo1), sa, ca)),
                                                    u2(__hfma2(h2(hi0), sb, cb)), u2(__hfma2(h2(hi1), sb, cb))));
    }
};

template <>
struct wprep<GGML_TYPE_Q5_K> : wprep_q45<GGML_TYPE_Q5_K> {
    static constexpr bool MINS = true, SPLIT = false;
    uint32_t f[8];      // the fifth bits of the lane's two sub-blocks at bits 0 and 1 of each byte
    __device__ __forceinline__ void prep(const wlane<GGML_TYPE_Q5_K> & r, int q) {
        prep45(r.h, r.a, r.b, q);
        const uint32_t v[8] = { r.f0.x, r.f0.y, r.f0.z, r.f0.w, r.f1.x, r.f1.y, r.f1.z, r.f1.w };
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] = (v[i] >> (2 * q)) & 0x03030303u;
    }
    template <int L>
    __device__ __forceinline__ f16x8 slice(f16x8 &) const {
        constexpr int B = L % 4, D = L / 4;
        const uint32_t p = byte_pair<B>(w[D], w[D + 2]), r = byte_pair<B>(w[D + 4], w[D + 6]);
        const uint32_t fp = byte_pair<B>(f[D], f[D + 2]), fr = byte_pair<B>(f[D + 4], f[D + 6]);
        // bit 4 of a low quant (n + 16 b), bit 8 of a high one (16 (n + 16 b))
        const uint32_t lo0 = and_or(p, 0x000f000fu, and_or(fp << 4, 0x00100010u, 0x64006400u));
        const uint32_t hi0 = and_or(p, 0x00f000f0u, and_or(fp << 7, 0x01000100u, 0x64006400u));
        const uint32_t lo1 = and_or(r, 0x000f000fu, and_or(fr << 4, 0x00100010u, 0x64006400u));
        const uint32_t hi1 = and_or(r, 0x00f000f0u, and_or(fr << 7, 0x01000100u, 0x64006400u));
        return __builtin_bit_cast(f16x8, make_uint4(u2(__hfma2(h2(lo0), sa, ca)), u2(__hfma2(h2(lo1), sa, ca)),
                                                    u2(__hfma2(h2(hi0), sb, cb)), u2(__hfma2(h2(hi1), sb, cb))));
    }
};

// Q6_K: the lane's 64 elements are runs A and B of 32 (groups g and g + 1 of half q / 2, g = 2 (q & 1)):
// nibble q & 1 of ql bytes 0..31 (A) and 32..63 (B), bits 2g, 2g + 1 (A) and 2g + 2, 2g + 3 (B) of
// the half's qh bytes; each 16 elements have their own scale.
template <>
struct wprep<GGML_TYPE_Q6_K> {
    static constexpr bool MINS = false, SPLIT = true;
    float dw, dm;
    f16x4 mins;
    __half2 s[4];
    uint32_t wa[8], wb[8], f[8];
    __device__ __forceinline__ void prep(const wlane<GGML_TYPE_Q6_K> & r, int q) {
        dw = __half2float(r.dw);
#pragma unroll
        for (int i = 0; i < 4; i++) s[i] = h2_of((int) (int8_t) (r.sc >> (8 * i)));
        const int sh = 4 * (q & 1);
        const uint32_t va[8] = { r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w };
        const uint32_t vb[8] = { r.c.x, r.c.y, r.c.z, r.c.w, r.d.x, r.d.y, r.d.z, r.d.w };
        const uint32_t vf[8] = { r.f0.x, r.f0.y, r.f0.z, r.f0.w, r.f1.x, r.f1.y, r.f1.z, r.f1.w };
#pragma unroll
        for (int i = 0; i < 8; i++) {
            wa[i] = va[i] >> sh;
            wb[i] = vb[i] >> sh;
            f[i] = vf[i] >> sh;
        }
    }
    // sc * (q % 16), returned, and sc * (16 (q / 16) - 32), in hi
    template <int L>
    __device__ __forceinline__ f16x8 slice(f16x8 & hi) const {
        constexpr int B = L % 4, D = L / 4;
        const __half2 b0 = __float2half2_rn(-1024.0f), b1 = __float2half2_rn(-1056.0f);
        const uint32_t n[4] = { byte_pair<B>(wa[D], wa[D + 2]), byte_pair<B>(wa[D + 4], wa[D + 6]),
                                byte_pair<B>(wb[D], wb[D + 2]), byte_pair<B>(wb[D + 4], wb[D + 6]) };
        const uint32_t f0 = byte_pair<B>(f[D], f[D + 2]), f1 = byte_pair<B>(f[D + 4], f[D + 6]);
        const uint32_t t[4] = { f0 << 4, f1 << 4, f0 << 2, f1 << 2 };
        uint32_t lo[4], up[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            lo[i] = u2(__hmul2(__hadd2(h2(and_or(n[i], 0x000f000fu, 0x64006400u)), b0), s[i]));
            up[i] = u2(__hmul2(__hadd2(h2(and_or(t[i], 0x00300030u, 0x64006400u)), b1), s[i]));
        }
        hi = __builtin_bit_cast(f16x8, make_uint4(up[0], up[1], up[2], up[3]));
        return __builtin_bit_cast(f16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
    }
};

// the running sums of a wave's outputs for one matrix: lane (c, q) holds row c, columns 16 t + 4 q + r
template <int NT>
struct macc {
    float mins[NT][4], sums[NT][8][4];
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                mins[t][r] = 0.0f;
#pragma unroll
                for (int l = 0; l < 8; l++) sums[t][l][r] = 0.0f;
            }
    }
};

// Step I of a super-block's products: slice I / H against TP column tiles (H = NT / TP groups of
// them). The next step's operands are read from LDS and this step's MFMAs issued before the previous
// step's sums, whose VALU work covers both latencies; the scheduling barriers keep that order (left
// alone, the compiler saves registers by waiting for each). Tile t's operand of slice l is at
// xp + t * TS + l * LS.
template <int TYPE, int NT, int TP, int TS, int LS, int I>
__device__ __forceinline__ void steps(const wprep<TYPE> & w, const uint8_t * xp, const float (&dd)[NT][4], const f16x8 (&x)[TP],
                                      const f32x4 (&prev)[TP], f16x8 lo, f16x8 hi, macc<NT> & acc) {
    constexpr int H = NT / TP, N = 8 * H, L = I / H, T0 = I % H * TP;
    f32x4 d[TP];
    f16x8 xn[TP];
    if constexpr (I < N) {
        if constexpr (I + 1 < N) {
#pragma unroll
            for (int t = 0; t < TP; t++) xn[t] = *(const f16x8 *) (xp + ((I + 1) % H * TP + t) * TS + (I + 1) / H * LS);
        }
        if constexpr (T0 == 0) lo = w.template slice<L>(hi);
#pragma unroll
        for (int t = 0; t < TP; t++) {
            d[t] = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
            if constexpr (wprep<TYPE>::SPLIT) d[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[t], hi, d[t], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < TP; t++) d[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[t], lo, d[t], 0, 0, 0);
    }
    if constexpr (I > 0) {
        constexpr int PL = (I - 1) / H, PT = (I - 1) % H * TP;
#pragma unroll
        for (int t = 0; t < TP; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc.sums[PT + t][PL][r] = acc.sums[PT + t][PL][r] + dd[PT + t][r] * prev[t][r];
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (I < N) steps<TYPE, NT, TP, TS, LS, I + 1>(w, xp, dd, xn, d, lo, hi, acc);
}

// One super-block: raw the weights, xp the lane's operand of slice 0 of tile 0, bp its share of that
// tile's sums, dp the scales of its four output columns
template <int TYPE, int NT, int TS, int LS>
__device__ __forceinline__ void superblock(const wlane<TYPE> & raw, int q, const uint8_t * xp, const uint8_t * bp,
                                           const uint8_t * const (&dp)[4], macc<NT> & acc) {
    constexpr int TP = NT == 4 && TYPE != GGML_TYPE_Q6_K ? 2 : 1;
    // the LDS reads of the scales, the sums and the first operands, covered by the decoding of the scales
    float dx[NT][4];
    f16x4 bs[NT];
    f16x8 x[TP];
#pragma unroll
    for (int t = 0; t < NT; t++) {
#pragma unroll
        for (int r = 0; r < 4; r++) dx[t][r] = *(const float *) (dp[r] + t * TS);
        if constexpr (wprep<TYPE>::MINS) bs[t] = *(const f16x4 *) (bp + t * TS);
    }
#pragma unroll
    for (int t = 0; t < TP; t++) x[t] = *(const f16x8 *) (xp + t * TS);
    wprep<TYPE> w;
    w.prep(raw, q);
    __builtin_amdgcn_sched_barrier(0);
    float dd[NT][4];
    f32x4 v[NT];
    if constexpr (wprep<TYPE>::MINS) {
#pragma unroll
        for (int t = 0; t < NT; t++) v[t] = __builtin_amdgcn_mfma_f32_16x16x16f16(bs[t], w.mins, f32x4{ 0.0f, 0.0f, 0.0f, 0.0f }, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            dd[t][r] = w.dw * dx[t][r];
            if constexpr (wprep<TYPE>::MINS) acc.mins[t][r] = acc.mins[t][r] - (w.dm * dx[t][r]) * v[t][r];
        }
    __builtin_amdgcn_sched_barrier(0);
    const f32x4 none[TP] = {};
    steps<TYPE, NT, TP, TS, LS, 0>(w, xp, dd, x, none, f16x8{}, f16x8{}, acc);
}

// the eight scaled slices of one super-block of a tile to out[0], out[WAVE], ...
template <int TYPE, int L>
__device__ __forceinline__ void split_slices(const wprep<TYPE> & w, const f16x8 (&x)[8], const float (&dd)[4], f32x4 * out) {
    if constexpr (L < 8) {
        f16x8 hi;
        const f16x8 lo = w.template slice<L>(hi);
        f32x4 s = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
        if constexpr (wprep<TYPE>::SPLIT) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[L], hi, s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f32_16x16x32_f16(x[L], lo, s, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; r++) s[r] = dd[r] * s[r];
        out[L * WAVE] = s;
        split_slices<TYPE, L + 1>(w, x, dd, out);
    }
}

// A workgroup's place in the grid. Dense: consecutive workgroups of one XCD take the column tiles of
// one row tile, which share its weights in that XCD's L2. Grouped: item by item as dispatched, so
// that the items in use (the first ones) spread over all XCDs.
struct mm_tile {
    int rt, first, ncols, mi;     // row tile, first column (list position when grouped) and count, matrix
    int64_t erow;
};
template <int COLS, int BM>
__device__ __forceinline__ bool tile_of(const mm_kargs & A, mm_tile & T) {
    const gemv_launch & L = A.L;
    int ct;
    T.erow = 0;
    if (A.g.cols) {
        ct = blockIdx.x / A.n_rt;
        T.rt = blockIdx.x - ct * A.n_rt;
        if (ct >= *A.g.n_items) return false;
        const int32_t * item = A.g.items + 3 * ct;
        T.erow = (int64_t) __builtin_amdgcn_readfirstlane(item[0]) * L.expert_rows;
        T.first = __builtin_amdgcn_readfirstlane(item[1]);
        T.ncols = __builtin_amdgcn_readfirstlane(item[2]);
    } else {
        const int n = A.n_rt * A.n_ct, xcd = blockIdx.x % 8, per = n / 8, rem = n % 8;
        const int t = xcd * per + min(xcd, rem) + blockIdx.x / 8;
        T.rt = t / A.n_ct;
        ct = t - T.rt * A.n_ct;
        T.first = ct * COLS;
        T.ncols = min(COLS, L.ncols - T.first);
    }
    T.mi = 0;
#pragma unroll
    for (int i = 1; i < GEMV_MAX_MATS; i++) if (i < L.n_mats && T.rt * BM >= A.row_begin[i]) T.mi = i;
    return true;
}
// the activation column of column j of the tile
__device__ __forceinline__ int x_column(const mm_kargs & A, const mm_tile & T, int j) {
    if (!A.g.cols) return T.first + j;
    const int gc = A.g.cols[T.first + j], tok = gc / A.L.n_slots;
    return tok * A.L.x_cols + (gc - tok * A.L.n_slots) % A.L.x_cols;
}

// the outputs of a wave: row, columns c0 + 16 t + 4 q + r of the tile
template <int NT>
__device__ __forceinline__ void store_out(const mm_kargs & A, const mm_tile & T, int row, int c0, int q, const macc<NT> & acc) {
    const gemv_mat & m = A.L.m[T.mi];
    if (row >= m.n_rows) return;
    // the columns and the residuals: every load before the first store
    int col[NT][4];
    float add[NT][4];
#pragma unroll
    for (int i = 0; i < NT; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = T.first + min(c0 + 16 * i + 4 * q + r, T.ncols - 1);
            col[i][r] = A.g.cols ? A.g.cols[j] : j;
            add[i][r] = 0.0f;
        }
    const bool res = m.add;
    if (res) {
#pragma unroll
        for (int i = 0; i < NT; i++)
#pragma unroll
            for (int r = 0; r < 4; r++) add[i][r] = m.add[col[i][r] * m.add_stride + row];
    }
#pragma unroll
    for (int i = 0; i < NT; i++) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float v = acc.mins[i][r];
#pragma unroll
            for (int l = 0; l < 8; l++) v = v + acc.sums[i][l][r];
            if (res) v = v + add[i][r];
            if (c0 + 16 * i + 4 * q + r < T.ncols) m.y[col[i][r] * m.y_stride + row] = v;
        }
    }
}

// 16 bytes per lane from base + off straight into LDS: lane i's land at dst + 16 i (base, dst uniform)
template <typename OFF>
__device__ __forceinline__ void to_lds(const uint8_t * base, OFF off, uint8_t * dst) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *) (base + off),
                                     (__attribute__((address_space(3))) void *) dst, 16, 0, 0);
}

// the shapes that a grouped launch may take (mm_shape_of)
constexpr bool mm_groups(int wr, int wc, int nt) { return wr == 4 && wc == 1 && nt <= 2; }

// WR x WC waves: WR groups of 16 rows, WC groups of 16 NT columns. Two LDS buffers of one super-block
// of the workgroup's column groups, filled by direct global -> LDS loads (a group's super-block is
// nine 1 KB pieces); separate objects, so that the compiler sees that reading one does not wait for
// the loads into the other.
template <int TYPE, int WR, int WC, int NT>
__global__ __launch_bounds__(64 * WR * WC, 2) void mm_kq_kernel(const mm_kargs A_) {
    const mm_kargs & A = kernargs_prefetched(A_);
    const gemv_launch & L = A.L;
    constexpr int WAVES = WR * WC, COLS = 16 * NT * WC, BM = 16 * WR, G = NT * WC;
    constexpr int WPG = WAVES % G == 0 ? WAVES / G : 0;          // waves per column group (0: not whole)
    constexpr bool GROUPS = mm_groups(WR, WC, NT);
    static_assert(!GROUPS || WPG > 0, "a grouped launch's waves read the columns of one group");
    __shared__ __align__(16) uint8_t s_x0[G * X16_BYTES];
    __shared__ __align__(16) uint8_t s_x1[G * X16_BYTES];
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x / WAVE);
    const int c = lane % 16, q = lane / 16, nsb = L.K / 256;
    mm_tile T;
    if (!tile_of<COLS, BM>(A, T)) return;
    const int r0 = T.rt * BM - A.row_begin[T.mi] + 16 * (wave % WR);

    // this wave's pieces: those of one column group, or every WAVES-th of all. Grouped, each lane
    // reads its own column's units (columns past the end repeat the last one), at 64-bit offsets: the
    // x16 form of a large routed batch passes 4 GiB. Dense, a group's pieces are contiguous (groups
    // past the end repeat the last one)
    const int64_t gstride = (int64_t) nsb * X16_BYTES;
    const int ng = (T.first + T.ncols + 15) / 16 - T.first / 16;
    const uint8_t * xbase = (const uint8_t *) L.xq;
    std::conditional_t<GROUPS, int64_t, uint32_t> xoff = lane * 16;
    if (GROUPS && A.g.cols) {
        const int xc = x_column(A, T, min(16 * (wave / (WPG ? WPG : 1)) + c, T.ncols - 1));
        xoff = (xc / 16) * gstride + (xc % 16) * 16 + q * 256;
    } else {
        xbase += (T.first / 16) * gstride;
    }
    auto fetch = [&](uint8_t * buf, int sb) {
        const uint8_t * src = xbase + (int64_t) sb * X16_BYTES;
        if constexpr (WPG > 0) {
            const int g = wave / WPG;
            if (!GROUPS || !A.g.cols) src += min(g, ng - 1) * gstride;
#pragma unroll
            for (int i = 0; i < (X16_PIECES + WPG - 1) / WPG; i++) {
                const int j = wave % WPG + i * WPG;
                if ((i + 1) * WPG <= X16_PIECES || j < X16_PIECES) to_lds(src + j * 1024, xoff, buf + g * X16_BYTES + j * 1024);
            }
        } else {
#pragma unroll
            for (int i = 0; i < (G * X16_PIECES + WAVES - 1) / WAVES; i++) {
                const int p = wave + i * WAVES, g = p / X16_PIECES, j = p - g * X16_PIECES;
                if ((i + 1) * WAVES <= G * X16_PIECES || p < G * X16_PIECES) {
                    to_lds(src + min(g, ng - 1) * gstride + j * 1024, xoff, buf + p * 1024);
                }
            }
        }
    };
    fetch(s_x0, 0);
    wrow<TYPE> wr;
    wlane<TYPE> raw[2];
    wr.at(L.m[T.mi], T.erow, min(r0, L.m[T.mi].n_rows - 1), min(r0 + c, L.m[T.mi].n_rows - 1), nsb, q);
    raw[0].load(wr, 0);
    macc<NT> acc;
    acc.zero();
    const int c0 = 16 * NT * (wave / WR), tile0 = (c0 / 16) * X16_BYTES;
    const int xo = tile0 + lane * 16, bo = tile0 + X16_SUMS + (q / 2) * 256 + c * 16 + (q % 2) * 8, dofs = tile0 + X16_D + 64 * q;

    // the loads of every wave of a super-block are complete when all have passed the barrier
    auto arrived = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    arrived();
    auto step = [&](const uint8_t * cur, uint8_t * nxt, wlane<TYPE> & now, wlane<TYPE> & then, int sb) {
        const int s1 = min(sb + 1, nsb - 1);
        fetch(nxt, s1);
        then.load(wr, s1);
        const uint8_t * d = cur + dofs;
        superblock<TYPE, NT, X16_BYTES, 1024>(now, q, cur + xo, cur + bo, { d, d + 16, d + 32, d + 48 }, acc);
        arrived();
    };
    for (int sb = 0; sb < nsb; sb += 2) {
        step(s_x0, s_x1, raw[0], raw[1], sb);
        if (sb + 1 < nsb) step(s_x1, s_x0, raw[1], raw[0], sb + 1);
    }
    store_out<NT>(A, T, r0 + c, c0, q, acc);
}

// The same with all of K of at most NC columns staged at once (four waves of 16 rows): after one
// barrier the waves run on their own, with their weights PF super-blocks ahead. LDS: [super-block]
// [unit][NC columns][16 bytes].
template <int TYPE, int NC>
__global__ __launch_bounds__(256, 2) void mm_kq_res_kernel(const mm_kargs A_) {
    const mm_kargs & A = kernargs_prefetched(A_);
    const gemv_launch & L = A.L;
    constexpr int PF = 3, SB = X16_USED * NC * 16;
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int s_xcol[NC];
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int c = lane % 16, q = lane / 16, nsb = L.K / 256;
    mm_tile T;
    if (!tile_of<NC, 64>(A, T)) return;
    const int r0 = T.rt * 64 - A.row_begin[T.mi] + 16 * wave;
    wrow<TYPE> wr;
    wlane<TYPE> raw[PF];
    wr.at(L.m[T.mi], T.erow, min(r0, L.m[T.mi].n_rows - 1), min(r0 + c, L.m[T.mi].n_rows - 1), nsb, q);
#pragma unroll
    for (int p = 0; p < PF; p++) raw[p].load(wr, min(p, nsb - 1));
    if (tid < NC) s_xcol[tid] = x_column(A, T, min(tid, T.ncols - 1));
    __syncthreads();
    // piece p: column p % NC, unit, super-block
    u32x4 * sx = (u32x4 *) smem;
    const int total = nsb * X16_USED * NC;
    for (int p0 = tid; p0 < total; p0 += 4 * 256) {
        u32x4 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int p = min(p0 + 256 * k, total - 1), u = p / NC, sb = u / X16_USED, xc = s_xcol[p % NC];
            v[k] = *(const u32x4 *) ((const uint8_t *) L.xq + ((int64_t) (xc / 16) * nsb + sb) * X16_BYTES + (u - sb * X16_USED) * 256 + (xc % 16) * 16);
        }
#pragma unroll
        for (int k = 0; k < 4; k++) if (p0 + 256 * k < total) sx[p0 + 256 * k] = v[k];
    }
    macc<1> acc;
    acc.zero();
    const int cc = c % NC;                             // lanes past NC columns repeat them; unused
    const uint8_t * xp = smem + q * (NC * 16) + cc * 16, * bp = smem + (32 + q / 2) * (NC * 16) + cc * 16 + (q % 2) * 8;
    const uint8_t * dp = smem + 34 * (NC * 16);
    __syncthreads();
    for (int sb = 0; sb < nsb; sb += PF) {
#pragma unroll
        for (int p = 0; p < PF; p++) {
            if (sb + p < nsb) {
                const uint8_t * d = dp + (sb + p) * SB;
                superblock<TYPE, 1, 0, NC * 64>(raw[p], q, xp + (sb + p) * SB, bp + (sb + p) * SB,
                                                { d + (4 * q) % NC * 16, d + (4 * q + 1) % NC * 16, d + (4 * q + 2) % NC * 16,
                                                  d + (4 * q + 3) % NC * 16 }, acc);
                raw[p].load(wr, min(sb + p + PF, nsb - 1));
            }
        }
    }
    store_out<1>(A, T, r0 + c, 0, q, acc);
}

// Few rows and columns: a workgroup of SPLIT waves takes 16 rows x 16 columns, wave w the super-blocks
// w, w + SPLIT, ... A chunk of SPLIT super-blocks: every wave forms its super-block's eight scaled
// slices and its mins term of the tile and leaves them in LDS, then wave w adds slice w's terms of
// the chunk to its running sums in super-block order (wave 0 the mins too): ggml's order. The
// operands come straight from memory: a slice's is 1 KB in lane order.
constexpr int SPLIT = 8;
template <int TYPE>
__global__ __launch_bounds__(64 * SPLIT, 4) void mm_kq_split_kernel(const mm_kargs A_) {
    const mm_kargs & A = kernargs_prefetched(A_);
    const gemv_launch & L = A.L;
    constexpr bool MINS = wprep<TYPE>::MINS;
    __shared__ __align__(16) f32x4 s_t[SPLIT][9][WAVE];
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x / WAVE);
    const int c = lane % 16, q = lane / 16, nsb = L.K / 256;
    mm_tile T;
    tile_of<16, 16>(A, T);
    const int n_rows = L.m[T.mi].n_rows, r0 = T.rt * 16 - A.row_begin[T.mi];
    wrow<TYPE> wr;
    wr.at(L.m[T.mi], 0, r0, min(r0 + c, n_rows - 1), nsb, q);
    const uint8_t * xg = (const uint8_t *) L.xq + (int64_t) (T.first / 16) * nsb * X16_BYTES;
    wlane<TYPE> raw;
    f16x8 x[8];
    f16x4 bs;
    float dx[4];
    auto load = [&](int sb) {
        const uint8_t * p = xg + (int64_t) sb * X16_BYTES;
        raw.load(wr, sb);
#pragma unroll
        for (int r = 0; r < 4; r++) dx[r] = *(const float *) (p + (uint32_t) (X16_D + 64 * q + 16 * r));
        if constexpr (MINS) bs = *(const f16x4 *) (p + (uint32_t) (X16_SUMS + (q / 2) * 256 + c * 16 + (q % 2) * 8));
#pragma unroll
        for (int l = 0; l < 8; l++) x[l] = *(const f16x8 *) (p + (uint32_t) (lane * 16 + l * 1024));
    };
    load(min(wave, nsb - 1));
    f32x4 sum = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f }, sumf = sum;
    for (int s0 = 0; s0 < nsb; s0 += SPLIT) {
        if (s0 + wave < nsb) {
            wprep<TYPE> w;
            w.prep(raw, q);
            float dd[4];
#pragma unroll
            for (int r = 0; r < 4; r++) dd[r] = w.dw * dx[r];
            if constexpr (MINS) {
                const f32x4 v = __builtin_amdgcn_mfma_f32_16x16x16f16(bs, w.mins, f32x4{ 0.0f, 0.0f, 0.0f, 0.0f }, 0, 0, 0);
                f32x4 t;
#pragma unroll
                for (int r = 0; r < 4; r++) t[r] = (w.dm * dx[r]) * v[r];
                s_t[wave][8][lane] = t;
            }
            split_slices<TYPE, 0>(w, x, dd, &s_t[wave][0][lane]);
        }
        load(min(s0 + SPLIT + wave, nsb - 1));
        __syncthreads();
        const int n = min(SPLIT, nsb - s0);
        for (int i = 0; i < n; i++) {
            const f32x4 t = s_t[i][wave][lane];
#pragma unroll
            for (int r = 0; r < 4; r++) sum[r] = sum[r] + t[r];
        }
        if (MINS && wave == 0) {
            for (int i = 0; i < n; i++) {
                const f32x4 t = s_t[i][8][lane];
#pragma unroll
                for (int r = 0; r < 4; r++) sumf[r] = sumf[r] - t[r];
            }
        }
        __syncthreads();
    }
    // the tile's chains, one output per thread of the first four waves
    s_t[0][wave][lane] = sum;
    if (wave == 0) s_t[0][8][lane] = sumf;
    __syncthreads();
    const int t = threadIdx.x;
    if (t >= 256) return;
    const int row = r0 + t % 16, j = t / 16;                  // lane (row, j / 4), component j % 4
    if (row >= n_rows || j >= T.ncols) return;
    const float * ch = (const float *) &s_t[0][0][t % 16 + 16 * (j / 4)] + j % 4;
    float v = ch[8 * WAVE * 4];
#pragma unroll
    for (int l = 0; l < 8; l++) v = v + ch[l * WAVE * 4];
    const gemv_mat & m = L.m[T.mi];
    const int64_t col = T.first + j;
    if (m.add) v = v + m.add[col * m.add_stride + row];
    m.y[col * m.y_stride + row] = v;
}

// the grid's rows, every matrix on a workgroup boundary, and its column tiles
inline void mm_grid(mm_kargs & a, const gemv_launch & L, const expert_groups * G, int bm, int cols) {
    a.L = L;
    int r = 0;
    for (int i = 0; i < L.n_mats; i++) {
        a.row_begin[i] = r;
        r += (L.m[i].n_rows + bm - 1) / bm * bm;
    }
    for (int i = L.n_mats; i <= GEMV_MAX_MATS; i++) a.row_begin[i] = r;
    a.n_rt = r / bm;
    a.n_ct = G ? G->max_items : (L.ncols + cols - 1) / cols;
    if (G) a.g = *G;
    if ((int64_t) a.n_rt * a.n_ct > INT32_MAX) HIP_ABORT("mm_kq: %d x %d tiles", a.n_rt, a.n_ct);
}

template <int TYPE, int WR, int WC, int NT>
void mm_launch(const gemv_launch & L, const expert_groups * G, hipStream_t st) {
    if (G && !mm_groups(WR, WC, NT)) HIP_ABORT("mm_kq: a %d x %d tile takes no expert groups", 16 * WR, 16 * NT * WC);
    mm_kargs a{};
    mm_grid(a, L, G, 16 * WR, 16 * NT * WC);
    launch(mm_kq_kernel<TYPE, WR, WC, NT>, dim3((unsigned) (a.n_rt * a.n_ct)), dim3(64 * WR * WC), 0, st, a);
}

template <int TYPE, int NC>
void mm_launch_res(const gemv_launch & L, const expert_groups * G, hipStream_t st) {
    mm_kargs a{};
    mm_grid(a, L, G, 64, NC);
    static bool attr = false;
    if (!attr) {
        HIP_CHECK(hipFuncSetAttribute((const void *) mm_kq_res_kernel<TYPE, NC>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int) MM_RES_MAX_LDS));
        attr = true;
    }
    launch(mm_kq_res_kernel<TYPE, NC>, dim3((unsigned) (a.n_rt * a.n_ct)), dim3(256), mm_res_lds(L.K, NC), st, a);
}

template <int TYPE>
void mm_launch_split(const gemv_launch & L, hipStream_t st) {
    mm_kargs a{};
    mm_grid(a, L, nullptr, 16, 16);
    launch(mm_kq_split_kernel<TYPE>, dim3((unsigned) (a.n_rt * a.n_ct)), dim3(64 * SPLIT), 0, st, a);
}

template <int TYPE>
void mm_dispatch(mm_shape s, const gemv_launch & L, const expert_groups * G, hipStream_t st) {
    switch (s) {
        case MM_64x64: mm_launch<TYPE, 4, 1, 4>(L, G, st); break;
        case MM_64x48: mm_launch<TYPE, 4, 1, 3>(L, G, st); break;
        case MM_32x64: mm_launch<TYPE, 2, 2, 2>(L, G, st); break;
        case MM_64x32: mm_launch<TYPE, 4, 1, 2>(L, G, st); break;
        case MM_64x16: mm_launch<TYPE, 4, 1, 1>(L, G, st); break;
        case MM_16x16: mm_launch<TYPE, 1, 1, 1>(L, G, st); break;
        case MM_SPLIT: mm_launch_split<TYPE>(L, st); break;
        case MM_RES2: mm_launch_res<TYPE, 2>(L, G, st); break;
        case MM_RES4: mm_launch_res<TYPE, 4>(L, G, st); break;
        case MM_RES8: mm_launch_res<TYPE, 8>(L, G, st); break;
        case MM_RES16: mm_launch_res<TYPE, 16>(L, G, st); break;
    }
}

} // namespace mm_kq_detail

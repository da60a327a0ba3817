// k_mm_q.hip — Q4_0 / Q8_0 weights times a few activation columns on the matrix cores: multi-token
// decode steps, prompts too short for the GEMM, and the columns of a mul_mat_id grouped by expert. Mostly 4
// to 63 columns (MM_Q_MIN_COLS, GEMM_MIN_COLS); 2 and 3 where the rows are too long for the vector kernel's
// LDS, 64 and more where the GEMM's outputs are not 16-byte aligned.
//
// Per (row, column) the arithmetic is the GEMV's: exact integer block dots, the terms (sumi * d_w) * d_x
// (Q4_0) and sumi * (d_w * d_x) (Q8_0), added in block order, so the result is the CPU reference's float.
//
// A workgroup owns 16 rows x 16 columns of one matrix (SwiGLU: of gate and of up, 4 waves each). Its 4
// waves take turns over K: in a phase of 16 blocks, wave s forms the terms of blocks 4 s .. 4 s + 3 and
// stores them to LDS, and after a barrier thread (row, column) adds the phase's 16 terms in order. A
// lane loads whole blocks, 4 consecutive ones of a row or column by 4 lanes, and 4 x 4 transposes over
// the lane groups (v_permlane32_swap, v_permlane16_swap) turn them into MFMA operands: lane (c, q) of
// v_mfma_i32_16x16x32_i8 holds dwords q and q + 4 of a block's 32 values, in both operands (the order
// of the values inside a block does not matter to its integer dot). Nothing but the terms passes
// through LDS, two phases of loads are in flight, and K split over the waves gives a 3072-row matrix
// 768 waves. Launches with tiles enough (MQ_WAVE_MIN_TILES) give each tile to one wave instead.
//
// Wide launches are bound by what a block costs a wave (18 vector instructions on its 4 x 64 terms, the
// scattered 16-byte pieces of 16 rows and columns), narrow ones by the memory latency of K / 512 phases.
// Measured (us a product with the activation's quantization; before: gemv_mc_kernel, integer dots on the
// vector ALU): Q4_0 3072 x 8192 by 4 / 16 / 37 columns 13.5 / 41.7 / 96 -> 12.9 / 15.2 / 23 (the last on the
// GEMM); 8192 x 3072 by 4 / 16 / 37 19.6 / 43.3 / 101 -> 17.5 / 17.6 / 30; Q8_0 8192 x 3072 by 16 / 63 42.7 / 148 -> 18.7 / 39.
// MFMA lane layout: A[i][k], B[k][j] at lane i (j) + 16 (k / 8), D[i][j] in register i % 4 of lane j + 16 (i / 4).
#include "kernels.h"
#include "gemv_ops.h"

#include "ggml.h"

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int MQ_TILE = 16;            // rows, and columns, of a workgroup
constexpr int MQ_WAVES = 4;            // waves per chain of terms
constexpr int MQ_PHASE = 4 * MQ_WAVES; // blocks per phase
constexpr int MQ_STRIDE = MQ_PHASE + 4;   // floats per (row, column) of a phase's terms: 20, so that 16-byte accesses spread over the banks

struct mm_q_args {
    gemv_kargs a;
    int n_ct;                // column tiles
    expert_groups g;         // g.cols set: column tile blockIdx.y is item blockIdx.y
};

// v[j] of lane group q = dword j of block q  ->  v[j] of lane group q = dword q of block j
__device__ __forceinline__ void transpose4(u32x4 & v) {
    const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false));
    const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false));
    const u32x2 c = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false));
    const u32x2 d = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false));
    v = u32x4{ c[0], c[1], d[0], d[1] };
}

// where lane (c, q) reads: rows r0 + c and r0 + 4 q .. (scales) of m from row erow, past the end the last row; weights at a
// uniform base and 32-bit offsets. One column's values and scales.
template <int TYPE>
struct q_source {
    static constexpr int QS = TYPE == GGML_TYPE_Q4_0 ? Q4_0_QS : Q8_0_QS;
    const uint8_t * wb, * db;
    uint32_t wo, dwo[4];
    const int8_t * xp;
    const float * xd;
    __device__ __forceinline__ q_source(const gemv_mat & m, int64_t erow, int r0, int nb, const int8_t * xq, const float * xd_, int c, int q)
        : wb(m.w + erow * nb * QS), db((const uint8_t *) m.wd + erow * nb * 2),
          wo((uint32_t) (min(r0 + c, m.n_rows - 1) * nb + q) * QS), xp(xq + q * 32), xd(xd_) {
#pragma unroll
        for (int r = 0; r < 4; r++) dwo[r] = (uint32_t) (min(r0 + 4 * q + r, m.n_rows - 1) * nb) * 2;
    }
};
// four consecutive blocks of 16 rows and 16 columns: lane (c, q) loads block q of row c and of column c, the
// scales of rows 4 q .. 4 q + 3 and of column c
template <int TYPE>
struct q_stage {
    static constexpr int QS = q_source<TYPE>::QS;
    u32x4 w[2], x[2];
    u32x2 dw[4];
    f32x4 dx;
    __device__ __forceinline__ void load(const q_source<TYPE> & S, int b) {
#pragma unroll
        for (int k = 0; k < QS / 16; k++) w[k] = *(const u32x4 *) (S.wb + (S.wo + (uint32_t) (b * QS + 16 * k)));
        x[0] = *(const u32x4 *) (S.xp + b * 32);
        x[1] = *(const u32x4 *) (S.xp + b * 32 + 16);
        dx = *(const f32x4 *) (S.xd + b);
#pragma unroll
        for (int r = 0; r < 4; r++) dw[r] = *(const u32x2 *) (S.db + (S.dwo[r] + (uint32_t) b * 2));
    }
    __device__ __forceinline__ void unpack() {
        transpose4(x[0]);
        transpose4(x[1]);
        transpose4(w[0]);
        if constexpr (TYPE == GGML_TYPE_Q4_0) {
            // 16 (nibble - 8) as int8: the nibble's top bit inverted, in the byte's upper half
            const u32x4 v = w[0] ^ 0x88888888u;
            w[0] = (v << 4) & 0xf0f0f0f0u;
            w[1] = v & 0xf0f0f0f0u;
        } else {
            transpose4(w[1]);
        }
    }
    // block j's terms of rows 4 q .. 4 q + 3 and column c
    __device__ __forceinline__ f32x4 terms(int j) const {
        const long a = __builtin_bit_cast(long, u32x2{ w[0][j], w[1][j] });
        const long b = __builtin_bit_cast(long, u32x2{ x[0][j], x[1][j] });
        const i32x4 si = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, i32x4{ 0, 0, 0, 0 }, 0, 0, 0);
        // Q4_0's dots come 16 times as large: a power of two, taken out of d_x (every float between is
        // exact or rounds the same)
        const float d = TYPE == GGML_TYPE_Q4_0 ? dx[j] * 0.0625f : dx[j];
        f32x4 t;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float s = __half2float(__ushort_as_half((unsigned short) (dw[r][j / 2] >> (16 * (j % 2)))));
            t[r] = TYPE == GGML_TYPE_Q4_0 ? ((float) si[r] * s) * d : (float) si[r] * (s * d);
        }
        return t;
    }
};

// the row and first column of a dense launch's workgroup: the column tiles of a row tile on one XCD, whose
// L2 then serves the weights again
__device__ __forceinline__ void tile_of(const mm_q_args & A, int & rt, int & first) {
    const unsigned blocks = gridDim.x;
    const unsigned id = blocks % 8 == 0 ? (blockIdx.x % 8) * (blocks / 8) + blockIdx.x / 8 : blockIdx.x;
    rt = (int) (id / (unsigned) A.n_ct);
    first = (int) (id % (unsigned) A.n_ct) * MQ_TILE;
}

// step(i, i % 3) for i = 0 .. n - 1, the second a compile-time constant. Whole threes without a branch
// inside: where branches meet, the compiler waits for every load in flight.
template <typename F>
__device__ __forceinline__ void in_threes(int n, F step) {
    int i = 0;
    for (; i + 3 <= n; i += 3) {
        step(i, std::integral_constant<int, 0>{});
        step(i + 1, std::integral_constant<int, 1>{});
        step(i + 2, std::integral_constant<int, 2>{});
    }
    if (i < n) step(i, std::integral_constant<int, 0>{});
    if (i + 1 < n) step(i + 1, std::integral_constant<int, 1>{});
}

// One wave per 16 rows x 16 columns (SwiGLU: one for gate, one for up), all of K in order: the sums stay in
// registers, no LDS and no barrier.
template <int TYPE, bool SWIGLU>
__global__ __launch_bounds__(64 * (SWIGLU ? 2 : 1), 4) void mm_q_wave_kernel(const mm_q_args A) {
    prefetch_kernargs<sizeof(mm_q_args)>();
    __shared__ __align__(16) f32x4 s_up[SWIGLU ? WAVE : 1];
    const gemv_launch & L = A.a.L;
    const int K = L.K, nb = K / 32, n_quads = nb / 4;
    const int lane = threadIdx.x % WAVE, ch = SWIGLU ? __builtin_amdgcn_readfirstlane((int) threadIdx.x / WAVE) : 0;
    const int c = lane % 16, q = lane / 16;
    int rt, first;
    tile_of(A, rt, first);
    const int mi = SWIGLU ? ch : find_mat(A.a, rt * MQ_TILE);
    const gemv_mat & m = L.m[mi];
    const int r0 = rt * MQ_TILE - (SWIGLU ? 0 : A.a.row_begin[mi]);
    const int64_t col = min(first + c, L.ncols - 1);
    const q_source<TYPE> src(m, 0, r0, nb, L.xq + col * K, L.xd + col * nb, c, q);
    q_stage<TYPE> S[3];
    auto load = [&](q_stage<TYPE> & T, int i) { T.load(src, 4 * min(i, n_quads - 1)); };
    f32x4 acc = { 0.0f, 0.0f, 0.0f, 0.0f };
    load(S[0], 0);
    __builtin_amdgcn_sched_barrier(0);           // in order: what a step waits for is counted from the last load
    load(S[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    in_threes(n_quads, [&](int i, auto u) {
        load(S[(u + 2) % 3], i + 2);
        __builtin_amdgcn_sched_barrier(0);
        S[u].unpack();
#pragma unroll
        for (int j = 0; j < 4; j++) acc += S[u].terms(j);
        __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (SWIGLU) {
        // act = silu(gate) * up (two roundings, as the silu and mul ops)
        if (ch == 1) s_up[lane] = acc;
        __syncthreads();
        if (ch == 1) return;
        const f32x4 up = s_up[lane];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float sl = acc[r] / (1.0f + exp_cr(-acc[r]));
            acc[r] = sl * up[r];
        }
    }
    if (first + c >= L.ncols) return;
    float * y = m.y + col * m.y_stride + r0 + 4 * q;
    const float * ad = !SWIGLU && m.add ? m.add + col * m.add_stride + r0 + 4 * q : nullptr;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        if (r0 + 4 * q + r < m.n_rows) y[r] = ad ? acc[r] + ad[r] : acc[r];
    }
}

template <int TYPE, bool SWIGLU>
__global__ __launch_bounds__(256 * (SWIGLU ? 2 : 1), 4) void mm_q_kernel(const mm_q_args A) {
    prefetch_kernargs<sizeof(mm_q_args)>();
    constexpr int NCH = SWIGLU ? 2 : 1;
    __shared__ __align__(16) float s_terms[2][NCH][MQ_TILE * MQ_TILE * MQ_STRIDE];
    const gemv_launch & L = A.a.L;
    const int K = L.K, nb = K / 32;
    const int t = threadIdx.x, lane = t % WAVE, wave = __builtin_amdgcn_readfirstlane(t / WAVE);
    const int c = lane % 16, q = lane / 16;
    const int ch = SWIGLU ? wave / MQ_WAVES : 0, s = wave % MQ_WAVES;

    // the workgroup's rows and columns
    int rt, first = 0, n = 0;
    int64_t erow = 0;
    if (A.g.cols) {
        if ((int) blockIdx.y >= *A.g.n_items) return;
        const int32_t * item = A.g.items + 3 * blockIdx.y;
        rt = blockIdx.x;
        erow = (int64_t) item[0] * L.expert_rows;
        first = item[1];
        n = item[2];
    } else {
        tile_of(A, rt, first);
        n = min(MQ_TILE, L.ncols - first);
    }
    const int mi = SWIGLU ? ch : find_mat(A.a, rt * MQ_TILE);
    const gemv_mat & m = L.m[mi];
    const int r0 = rt * MQ_TILE - (SWIGLU ? 0 : A.a.row_begin[mi]);       // first row in the matrix
    auto column_of = [&](int k) { return A.g.cols ? A.g.cols[first + k] : first + k; };

    const int col = column_of(min(c, n - 1));
    const int64_t xcol = L.ids ? (int64_t) (col / L.n_slots) * L.x_cols + (col % L.n_slots) % L.x_cols : col;
    const q_source<TYPE> src(m, erow, r0, nb, L.xq + xcol * K, L.xd + xcol * nb, c, q);
    const int n_quads = nb / 4, n_phases = (nb + MQ_PHASE - 1) / MQ_PHASE;
    auto load = [&](q_stage<TYPE> & T, int ph) { T.load(src, 4 * min(ph * MQ_WAVES + s, n_quads - 1)); };   // past the end: loaded, not added

    // thread (row, column) of the sums: element e = 16 row + column
    const int e = t % 256;
    float acc = 0.0f;
    auto step = [&](q_stage<TYPE> & T, int ph) {
        T.unpack();
        f32x4 term[4];                           // [block]: rows 4 q .. 4 q + 3, column c
#pragma unroll
        for (int j = 0; j < 4; j++) term[j] = T.terms(j);
        float * out = s_terms[ph & 1][ch] + (64 * q + c) * MQ_STRIDE + 4 * s;
#pragma unroll
        for (int r = 0; r < 4; r++) *(f32x4 *) (out + 16 * r * MQ_STRIDE) = f32x4{ term[0][r], term[1][r], term[2][r], term[3][r] };
    };
    auto add = [&](int ph) {
        const float * in = s_terms[ph & 1][ch] + e * MQ_STRIDE;
        f32x4 v[MQ_WAVES];
#pragma unroll
        for (int k = 0; k < MQ_WAVES; k++) v[k] = *(const f32x4 *) (in + 4 * k);
        const int left = n_quads - ph * MQ_WAVES;
#pragma unroll
        for (int k = 0; k < MQ_WAVES; k++) {
            if (k < left) {
#pragma unroll
                for (int j = 0; j < 4; j++) acc += v[k][j];
            }
        }
    };
    // One barrier per phase: phase ph's terms go to the buffer that phase ph - 2 used, whose sums every
    // wave had read before the barrier of phase ph - 1. Past the last phase a stage is loaded
    // (clamped) but not stepped.
    q_stage<TYPE> S[3];
    load(S[0], 0);
    __builtin_amdgcn_sched_barrier(0);           // in order: what a step waits for is counted from the last load
    load(S[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    in_threes(n_phases, [&](int ph, auto u) {
        load(S[(u + 2) % 3], ph + 2);
        __builtin_amdgcn_sched_barrier(0);
        step(S[u], ph);
        __syncthreads();
        add(ph);
    });

    const int row = e / 16, k = e % 16;
    if constexpr (SWIGLU) {
        // act = silu(gate) * up (two roundings, as the silu and mul ops); the up sums through LDS
        __syncthreads();
        float * s_up = s_terms[0][0];
        if (ch == 1) s_up[e] = acc;
        __syncthreads();
        if (ch == 0 && k < n && r0 + row < m.n_rows) {
            const float sl = acc / (1.0f + exp_cr(-acc));
            m.y[(int64_t) column_of(k) * m.y_stride + r0 + row] = sl * s_up[e];
        }
    } else if (k < n && r0 + row < m.n_rows) {
        const int64_t cc = column_of(k);
        float v = acc;
        if (m.add) v = v + m.add[cc * m.add_stride + r0 + row];
        m.y[cc * m.y_stride + r0 + row] = v;
    }
}

template <int TYPE>
void launch_mm_q_type(const mm_q_args & A, bool wave, dim3 grid, hipStream_t st) {
    if (A.a.L.swiglu) {
        if (wave) launch((mm_q_wave_kernel<TYPE, true>), grid, dim3(128), 0, st, A);
        else launch((mm_q_kernel<TYPE, true>), grid, dim3(512), 0, st, A);
    } else {
        if (wave) launch((mm_q_wave_kernel<TYPE, false>), grid, dim3(64), 0, st, A);
        else launch((mm_q_kernel<TYPE, false>), grid, dim3(256), 0, st, A);
    }
}

// More dense tiles than this give the chip enough waves without K split over them, and then the terms need
// no way through LDS (us with the activation's quantization, split / whole K per wave; Q4_0): 3072 x
// 32064 by 8 columns (2004 tiles) 34.9 / 28.8; 3072 x 8192 by 32 (1024) 24.6 / 21.0; 4096 x 4096 by 48 (768)
// 21.0 / 20.1; 3072 x 8192 by 8 (512) 13.8 / 14.9; 8192 x 3072 by 16 (192) 17.6 / 27.2. An expert's items are few and
// split.
constexpr int MQ_WAVE_MIN_TILES = 512;

} // namespace

bool mm_q_supported(int type, int64_t K, int64_t n_rows) {
    return (type == GGML_TYPE_Q4_0 || type == GGML_TYPE_Q8_0) && K > 0 && K % 128 == 0 && n_rows * K <= INT32_MAX;
}

void launch_mm_q(const gemv_launch & L, const expert_groups * G, hipStream_t st) {
    if (!mm_q_supported(L.type, L.K, L.m[0].n_rows) || L.norm.x || !L.xq || !L.xd || L.ncols < 1) HIP_ABORT("mm_q: unsupported launch (type %d, K=%d)", L.type, L.K);
    if (L.swiglu && (L.n_mats != 2 || L.m[0].n_rows != L.m[1].n_rows)) HIP_ABORT("mm_q: swiglu needs two equal matrices");
    if (G && (!L.ids || L.n_slots < 1 || L.x_cols < 1 || L.n_experts < 1 || G->nc > MQ_TILE)) HIP_ABORT("mm_q: bad mul_mat_id geometry");
    uintptr_t align = (uintptr_t) L.xq | (uintptr_t) L.xd;
    mm_q_args A{};
    A.a.L = L;
    A.a.rows_per_block = MQ_TILE;
    int r = 0;
    for (int i = 0; i < L.n_mats; i++) {
        align |= (uintptr_t) L.m[i].w | ((uintptr_t) L.m[i].wd << 1);
        if ((int64_t) L.m[i].n_rows * L.K > INT32_MAX) HIP_ABORT("mm_q: %d rows of %d", L.m[i].n_rows, L.K);
        A.a.row_begin[i] = r;
        if (!L.swiglu || i == 0) r += (L.m[i].n_rows + MQ_TILE - 1) / MQ_TILE * MQ_TILE;
    }
    if (align % 16) HIP_ABORT("mm_q: operands must be 16-byte aligned (weight scales 8)");
    for (int i = L.n_mats; i <= GEMV_MAX_MATS; i++) A.a.row_begin[i] = r;
    A.a.total_rows = r;
    A.n_ct = (L.ncols + MQ_TILE - 1) / MQ_TILE;
    dim3 grid((unsigned) (r / MQ_TILE));
    const bool wave = !G && (int64_t) grid.x * (L.swiglu ? 2 : 1) * A.n_ct > MQ_WAVE_MIN_TILES;
    if (G) {
        A.g = *G;
        grid.y = (unsigned) G->max_items;
    } else {
        grid.x *= (unsigned) A.n_ct;
    }
    if (L.type == GGML_TYPE_Q4_0) launch_mm_q_type<GGML_TYPE_Q4_0>(A, wave, grid, st);
    else launch_mm_q_type<GGML_TYPE_Q8_0>(A, wave, grid, st);
}

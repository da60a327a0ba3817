// k_gemm.hip — the prefill GEMM: Q4_0 / Q8_0 weights times Q8_0-quantized activation columns on
// the matrix cores.
//
// ggml-cpu computes every output of a quantized mul_mat as a float sum over the weight row's
// 32-element blocks, in block order, of an exact integer block dot scaled by the two fp16 block
// scales: Q8_0 sumf += sumi * (d_w * d_x), Q4_0 sumf += (sumi * d_w) * d_x. The integer quants are
// staged as int8 (Q4_0 nibbles as nibble - 8), so one v_mfma_i32_16x16x32_i8 yields the exact
// block dots of a tile of 16 weight rows x 16 activation columns, and the kernel adds the scaled
// terms (the block dot converted to float, exactly: it is below 2^24 in magnitude) to f32
// accumulators in block order: every output is the same float as the GEMV's and the CPU
// reference's. The per-term float work (a conversion, two multiplies, one add) runs on the VALU
// and bounds the kernel, not the MFMA rate.
//
// Tiling: a workgroup is 2 x 2 waves; a wave owns WTM x WTN MFMA tiles. Each pipeline stage moves
// KB blocks of the workgroup's weight rows and activation columns from global memory (16-byte
// loads, consecutive threads on consecutive bytes) into LDS as int8 rows (Q4_0 unpacked on the
// way) and the fp16 weight scales as floats; the next stage's loads are in flight while the
// current stage is reduced, with one barrier per stage. In a tile, lane l reads weight row l%16
// and activation column l%16, k-slice 8(l/16)..8(l/16)+7 of the block (one 8-byte LDS read each;
// rows are 8 bytes longer than their blocks, so the 16 rows of a read fall on distinct banks), and
// receives the results of rows 4(l/16)..4(l/16)+3 of column l%16. Workgroups are numbered so that
// the column tiles of one row tile run on one XCD and share its L2.
#include "kernels.h"
#include "gemv_ops.h"

#include "ggml.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

namespace {

// one Q4_0 block's 16 bytes -> its 32 weights as int8 of value nibble - 8 (low nibbles are elements
// 0-15, high 16-31), 8 bytes per store: per byte n in 0..15, ((n | 0x80) - 8) ^ 0x80 = n - 8 with no
// borrow between bytes
__device__ __forceinline__ void store_q4x32_i8(int8_t * dst, const uint4 & a) {
    const uint32_t w[4] = { a.x, a.y, a.z, a.w };
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        lo[k] = (((w[k] & 0x0F0F0F0Fu) | 0x80808080u) - 0x08080808u) ^ 0x80808080u;
        hi[k] = ((((w[k] >> 4) & 0x0F0F0F0Fu) | 0x80808080u) - 0x08080808u) ^ 0x80808080u;
    }
    uint2 * d = (uint2 *) dst;
    d[0] = make_uint2(lo[0], lo[1]); d[1] = make_uint2(lo[2], lo[3]);
    d[2] = make_uint2(hi[0], hi[1]); d[3] = make_uint2(hi[2], hi[3]);
}

// 32 int8 (two 16-byte loads) to an 8-byte aligned LDS row
__device__ __forceinline__ void store_i8x32_raw(int8_t * dst, const uint4 & a, const uint4 & b) {
    uint2 * d = (uint2 *) dst;
    d[0] = make_uint2(a.x, a.y); d[1] = make_uint2(a.z, a.w);
    d[2] = make_uint2(b.x, b.y); d[3] = make_uint2(b.z, b.w);
}

template <int TYPE, int WTM, int WTN, int KB>
struct gemm_cfg {
    static constexpr int QB = TYPE == GGML_TYPE_Q4_0 ? Q4_0_QS : Q8_0_QS;
    static constexpr int BM = 32 * WTM, BN = 32 * WTN;
    static constexpr int ROW = KB * 32 + 8;                               // int8 per LDS row (8-byte pad)
    static constexpr int UA = (BM * KB + 255) / 256, UB = (BN * KB + 255) / 256;   // staged blocks per thread
    static constexpr int A_BYTES = BM * ROW, B_BYTES = BN * ROW;
    static constexpr size_t LDS = 2 * ((size_t) (A_BYTES + B_BYTES) + (size_t) KB * (BM + BN) * 4);
};

template <int TYPE, int WTM, int WTN, int KB>
__global__ __launch_bounds__(256, WTM == 1 ? 4 : 1) void gemm_q_kernel(const gemm_launch G) {
    prefetch_kernargs<sizeof(gemm_launch)>();
    using C = gemm_cfg<TYPE, WTM, WTN, KB>;
    constexpr int QB = C::QB, BM = C::BM, BN = C::BN, ROW = C::ROW;
    extern __shared__ __align__(16) uint8_t g_lds[];
    int8_t * sA = (int8_t *) g_lds;                           // [2][BM][ROW]
    int8_t * sB = sA + 2 * C::A_BYTES;                        // [2][BN][ROW]
    float * sdw = (float *) (sB + 2 * C::B_BYTES);            // [2][KB][BM]
    float * sdx = sdw + 2 * KB * BM;                          // [2][KB][BN]

    const int64_t M = G.n_rows, N = G.ncols, K = G.K, nb = K / 32;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    const int q = lane / 16, c = lane % 16;

    const int64_t n_ct = (N + BN - 1) / BN, tiles = ((M + BM - 1) / BM) * n_ct;
    int64_t t = blockIdx.x;
    if (tiles % 8 == 0) t = (int64_t) (blockIdx.x % 8) * (tiles / 8) + blockIdx.x / 8;
    const int64_t m0 = (t / n_ct) * BM, n0 = (t % n_ct) * BN;
    const int wr = (wave / 2) * 16 * WTM, wc = (wave % 2) * 16 * WTN;   // wave's tile origin in the workgroup tile

    // staging: unit u = (row or column, block of the stage); rows / columns past the end repeat the last one
    uint4 ra[C::UA][2], rb[C::UB][2];
    __half rd[C::UA];
    float rx[C::UB];
    auto load = [&](int64_t b0) {
#pragma unroll
        for (int k = 0; k < C::UA; k++) {
            const int u = tid + 256 * k;
            if (u < BM * KB) {
                const int64_t row = min(m0 + u / KB, M - 1);
                const int64_t blk = row * nb + b0 + u % KB;
                const uint4 * p = (const uint4 *) (G.w + blk * QB);
                ra[k][0] = p[0];
                if constexpr (QB == 32) ra[k][1] = p[1];
                rd[k] = G.wd[blk];
            }
        }
#pragma unroll
        for (int k = 0; k < C::UB; k++) {
            const int u = tid + 256 * k;
            if (u < BN * KB) {
                const int64_t col = min(n0 + u / KB, N - 1);
                const uint4 * p = (const uint4 *) (G.xq + col * K + (b0 + u % KB) * 32);
                rb[k][0] = p[0];
                rb[k][1] = p[1];
                rx[k] = G.xd[col * nb + b0 + u % KB];
            }
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int k = 0; k < C::UA; k++) {
            const int u = tid + 256 * k;
            if (u < BM * KB) {
                const int r = u / KB, kb = u % KB;
                int8_t * dst = sA + buf * C::A_BYTES + r * ROW + kb * 32;
                if constexpr (QB == 32) store_i8x32_raw(dst, ra[k][0], ra[k][1]);
                else store_q4x32_i8(dst, ra[k][0]);
                sdw[(buf * KB + kb) * BM + r] = __half2float(rd[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < C::UB; k++) {
            const int u = tid + 256 * k;
            if (u < BN * KB) {
                const int cc = u / KB, kb = u % KB;
                store_i8x32_raw(sB + buf * C::B_BYTES + cc * ROW + kb * 32, rb[k][0], rb[k][1]);
                sdx[(buf * KB + kb) * BN + cc] = rx[k];
            }
        }
    };

    float acc[WTM][WTN][4];
#pragma unroll
    for (int i = 0; i < WTM; i++)
#pragma unroll
        for (int j = 0; j < WTN; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[i][j][r] = 0.0f;

    // Stage s's loads are issued before stage s - 1's dots and stored to LDS at the top of
    // iteration s, so the previous stage's MFMAs and epilogue cover their latency (stored at the end
    // of the iteration, the compiler would move the stores and their wait ahead of the epilogue).
    // One barrier per stage: a stage's stores go to the buffer that the stage before last read, and
    // every wave passed the last barrier after that.
    const int64_t n_stages = nb / KB;
    load(0);
    for (int64_t s = 0; s < n_stages; s++) {
        const int buf = (int) (s & 1);
        store(buf);
        __syncthreads();
        if (s + 1 < n_stages) load((s + 1) * KB);
        const int8_t * A = sA + buf * C::A_BYTES;
        const int8_t * B = sB + buf * C::B_BYTES;
#pragma unroll
        for (int kb = 0; kb < KB; kb++) {
            long a[WTM], b[WTN];
            f32x4 dw[WTM];
            float dx[WTN];
#pragma unroll
            for (int i = 0; i < WTM; i++) {
                a[i] = *(const long *) (A + (wr + 16 * i + c) * ROW + kb * 32 + 8 * q);
                dw[i] = *(const f32x4 *) (sdw + (buf * KB + kb) * BM + wr + 16 * i + 4 * q);
            }
#pragma unroll
            for (int j = 0; j < WTN; j++) {
                b[j] = *(const long *) (B + (wc + 16 * j + c) * ROW + kb * 32 + 8 * q);
                dx[j] = sdx[(buf * KB + kb) * BN + wc + 16 * j + c];
            }
#pragma unroll
            for (int i = 0; i < WTM; i++)
#pragma unroll
                for (int j = 0; j < WTN; j++) {
                    const i32x4 si = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[i], b[j], i32x4{ 0, 0, 0, 0 }, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float sv = (float) si[r];
                        if constexpr (TYPE == GGML_TYPE_Q8_0) {
                            const float dd = dw[i][r] * dx[j];
                            acc[i][j][r] += sv * dd;
                        } else {
                            acc[i][j][r] += (sv * dw[i][r]) * dx[j];
                        }
                    }
                }
        }
    }

#pragma unroll
    for (int j = 0; j < WTN; j++) {
        const int64_t col = n0 + wc + 16 * j + c;
        if (col >= N) continue;
#pragma unroll
        for (int i = 0; i < WTM; i++) {
            const int64_t r0 = m0 + wr + 16 * i + 4 * q;
            if (r0 >= M) continue;
            float v[4] = { acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3] };
            if (G.add) {
                const float * ap = G.add + col * G.add_stride + r0;
                for (int r = 0; r < 4; r++) if (r0 + r < M) v[r] = v[r] + ap[r];
            }
            float * yp = G.y + col * G.y_stride + r0;
            if (r0 + 3 < M) {
                *(float4 *) yp = make_float4(v[0], v[1], v[2], v[3]);
            } else {
                for (int r = 0; r < 4; r++) if (r0 + r < M) yp[r] = v[r];
            }
        }
    }
}

template <int TYPE, int WTM, int WTN, int KB>
void launch_gemm_t(const gemm_launch & G, hipStream_t st) {
    using C = gemm_cfg<TYPE, WTM, WTN, KB>;
    static bool attr = false;
    if (!attr && C::LDS > 65536) {
        HIP_CHECK(hipFuncSetAttribute((const void *) gemm_q_kernel<TYPE, WTM, WTN, KB>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int) C::LDS));
    }
    attr = true;
    const int64_t tiles = ((G.n_rows + C::BM - 1) / C::BM) * ((G.ncols + C::BN - 1) / C::BN);
    launch(gemm_q_kernel<TYPE, WTM, WTN, KB>, dim3((unsigned) tiles), dim3(256), C::LDS, st, G);
}

int64_t n_tiles(const gemm_launch & G, int bm, int bn) { return ((G.n_rows + bm - 1) / bm) * ((G.ncols + bn - 1) / bn); }

// The workgroup tile of a launch. Q4_0 / Q8_0: the largest tile that still gives every CU two
// workgroups (Q4_0) or four (Q8_0, whose staging moves twice the weight bytes per block; measured:
// Phi-3 prefill 26.1 -> 24.9 ms, while Q4_0 is slower with the smaller tiles).
enum gemm_tile { TILE_4x4x2, TILE_2x4x2, TILE_1x2x4 };

gemm_tile tile_of(const gemm_launch & G) {
    const int64_t target = G.type == GGML_TYPE_Q8_0 ? 1024 : 512;
    if (n_tiles(G, 128, 128) >= target) return TILE_4x4x2;
    if (n_tiles(G, 64, 128) >= target) return TILE_2x4x2;
    return TILE_1x2x4;
}

template <int TYPE>
void launch_gemm_type(const gemm_launch & G, hipStream_t st) {
    switch (tile_of(G)) {
        case TILE_4x4x2: launch_gemm_t<TYPE, 4, 4, 2>(G, st); break;
        case TILE_2x4x2: launch_gemm_t<TYPE, 2, 4, 2>(G, st); break;
        default: launch_gemm_t<TYPE, 1, 2, 4>(G, st); break;
    }
}

} // namespace

const char * gemm_tile_name(const gemm_launch & G) {
    switch (tile_of(G)) {
        case TILE_4x4x2: return "4x4x2";
        case TILE_2x4x2: return "2x4x2";
        default: return "1x2x4";
    }
}

bool gemm_supported(int type, int64_t K, int64_t n_rows) {
    return (type == GGML_TYPE_Q4_0 || type == GGML_TYPE_Q8_0) && K > 0 && K % 128 == 0 && n_rows > 0;
}

void launch_gemm(const gemm_launch & G, hipStream_t st) {
    if (!gemm_supported(G.type, G.K, G.n_rows) || G.ncols <= 0) {
        HIP_ABORT("gemm: unsupported geometry (type %d, K %lld, rows %lld, cols %lld)", G.type, (long long) G.K,
                  (long long) G.n_rows, (long long) G.ncols);
    }
    const uintptr_t align = (uintptr_t) G.y | (uintptr_t) G.add | (uintptr_t) G.w | (uintptr_t) G.xq;
    if (align % 16 || G.y_stride % 4 || (G.add && G.add_stride % 4)) {
        HIP_ABORT("gemm: operands must be 16-byte aligned with strides of whole float4s");
    }
    if (G.type == GGML_TYPE_Q4_0) launch_gemm_type<GGML_TYPE_Q4_0>(G, st);
    else launch_gemm_type<GGML_TYPE_Q8_0>(G, st);
}

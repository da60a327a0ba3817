// k_q8k.hip — activations of several columns quantized to Q8_K in the x16 form that the multi-column
// K-quant products read (q8k_act::x16): a float matrix, or silu(gate) * up of two.
//
// A workgroup of 16 waves takes one super-block of 16 columns, a wave per column (four elements per
// lane, 16-byte loads), and builds the group's x16 block in LDS, so that its 9 KB go out as whole
// lines. The maximum of a super-block is a DPP reduction and a ballot instead of six rounds of
// shuffles of three values; the launch is bound by its loads and stores. Measured,
// 9728 elements x 512 columns: silu(gate) * up 34 -> 13 us against one workgroup per super-block and
// column (swiglu_kernel, which also wrote the floats that no one reads).
#include "kernels.h"

template <bool SWIGLU>
__global__ __launch_bounds__(1024) void q8k_x16_kernel(const float * __restrict__ a, int64_t a_stride, const float * __restrict__ b,
                                                       int64_t b_stride, float * __restrict__ y, int64_t y_stride, int nsb, int ncols,
                                                       q8k_act out) {
    __shared__ __align__(16) uint8_t s_x[X16_USED * 256];
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE, sb = blockIdx.x, c0 = blockIdx.y * 16;
    const int64_t col = min(c0 + w, ncols - 1);            // waves past the last column repeat it, unstored
    const float4 x = *(const float4 *) (a + col * a_stride + sb * 256 + 4 * lane);
    float v[4] = { x.x, x.y, x.z, x.w };
    if constexpr (SWIGLU) {
        const float4 u4 = *(const float4 *) (b + col * b_stride + sb * 256 + 4 * lane);
        const float u[4] = { u4.x, u4.y, u4.z, u4.w };
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float s = v[j] / (1.0f + exp_cr(-v[j]));
            v[j] = s * u[j];
        }
        if (y && c0 + w < ncols) *(float4 *) (y + col * y_stride + sb * 256 + 4 * lane) = make_float4(v[0], v[1], v[2], v[3]);
    }
    // the value of largest magnitude, the first one on ties
    float ax = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) ax = fmaxf(ax, fabsf(v[j]));
    const float m = wave_max(ax);
    int q[4] = { 0, 0, 0, 0 };
    float d = 0.0f;
    if (m > 0.0f) {
        const int first = __builtin_ctzll(__ballot(ax == m));
        const float mine = fabsf(v[0]) == m ? v[0] : fabsf(v[1]) == m ? v[1] : fabsf(v[2]) == m ? v[2] : v[3];
        const float iscale = -127.f / lane_f(mine, first);
#pragma unroll
        for (int j = 0; j < 4; j++) q[j] = min(round_half_even(iscale * v[j]), 127);
        d = 1 / iscale;
    }
    int sum = (q[0] + q[1]) + (q[2] + q[3]);
    sum += dpp_i<0xB1>(sum);
    sum += dpp_i<0x4E>(sum);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int e = 4 * lane + j;
        *(__half *) (s_x + (e % 8 * 4 + e / 64) * 256 + w * 16 + e / 8 % 8 * 2) = __int2half_rn(q[j]);
    }
    if (lane % 4 == 0) *(__half *) (s_x + X16_SUMS + lane / 32 * 256 + w * 16 + lane / 4 % 8 * 2) = __int2half_rn(sum);
    if (lane == 0) *(float *) (s_x + X16_D + w * 16) = d;
    __syncthreads();
    const int t = threadIdx.x;
    if (t < X16_USED * 16 && c0 + t % 16 < ncols) {
        *(uint4 *) (out.x16 + ((int64_t) blockIdx.y * nsb + sb) * X16_BYTES + t * 16) = *(const uint4 *) (s_x + t * 16);
    }
}

bool q8k_x16_ok(const float * a, int64_t a_stride, const float * b, int64_t b_stride, const float * y, int64_t y_stride) {
    return ((uintptr_t) a | (uintptr_t) b | (uintptr_t) y) % 16 == 0 && (a_stride | b_stride | y_stride) % 4 == 0;
}

// up null: gate itself; y (optional): the values as floats. K a multiple of 256, columns 16-byte aligned
void launch_q8k_x16(const float * gate, int64_t g_stride, const float * up, int64_t u_stride, float * y, int64_t y_stride, int64_t K,
                    int64_t ncols, q8k_act out, hipStream_t st) {
    if (!out.x16 || K % 256 || !q8k_x16_ok(gate, g_stride, up, u_stride, y, y_stride)) HIP_ABORT("q8k_x16: unsupported operands");
    const dim3 grid((unsigned) (K / 256), (unsigned) ((ncols + 15) / 16));
    if (up) launch(q8k_x16_kernel<true>, grid, dim3(1024), 0, st, gate, g_stride, up, u_stride, y, y_stride, (int) (K / 256), (int) ncols, out);
    else launch(q8k_x16_kernel<false>, grid, dim3(1024), 0, st, gate, g_stride, up, u_stride, y, y_stride, (int) (K / 256), (int) ncols, out);
}

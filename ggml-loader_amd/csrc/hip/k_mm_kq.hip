// k_mm_kq.hip — workgroup shapes of the multi-column K-quant products (mm_kq_impl.h) and their entry
// point.
#include "kernels.h"

#include "ggml.h"

#include <algorithm>

mm_shape mm_shape_of(const gemv_launch & L, const expert_groups * G) {
    // An expert's items: up to 32 columns; few of them stay in LDS for all of K
    if (G) {
        if (G->nc > 16) return MM_64x32;
        if (mm_res_lds(L.K, G->nc) > MM_RES_MAX_LDS) return MM_64x16;
        return G->nc <= 2 ? MM_RES2 : G->nc <= 4 ? MM_RES4 : G->nc <= 8 ? MM_RES8 : MM_RES16;
    }
    int64_t rows = 0;
    for (int i = 0; i < L.n_mats; i++) rows += (L.m[i].n_rows + 63) / 64;
    auto tiles = [&](int cols) { return rows * ((L.ncols + cols - 1) / cols); };
    // 64 columns and more. The 64 x 64 tile decodes the weights least often; below one per CU the 32 x
    // 64 one (each wave a quarter of the columns) doubles the waves, and between one and two per CU,
    // where some CUs would run two tiles and others one, 64 x 48 ones even that out while they too are at
    // most two per CU. Measured, 64x64 / 64x48, us with the quantization launch (rows x K by columns):
    // Q4_K 288 tiles of 64 x 64 (4608 x 2560 by 256) 31.2 / 28.0, 320 (2560 x 9728 by 512) 97.8 / 85.3, 352
    // (2816 x 2560 by 512) 33.7 / 30.5; past two 64 x 48 per CU, 384 (6144 x 2560 by 256) 31.8 / 42.4, 448
    // (3584 x 2560 by 512) 34.2 / 44.5; Q5_K 320 112 / 99, 384 54 / 74; Q6_K 320 179 / 141, 384 54 / 63. At one per
    // CU exactly there is nothing to even out: 4096 x 2560 by 256 Q4_K 25.2 / 27.9, Q5_K 28.4 / 31.2; Q6_K, whose 64 x
    // 64 tile spills registers, 46.1 / 42.7.
    if (L.ncols >= 64) {
        if (tiles(64) < 256) return MM_32x64;
        const bool uneven = tiles(64) > 256 || L.type == GGML_TYPE_Q6_K;
        return uneven && tiles(64) < 512 && tiles(48) <= 512 ? MM_64x48 : MM_64x64;
    }
    // Below 64 columns, 16 per tile. With a 64-row workgroup for every CU its four waves share the
    // staged columns. With fewer, one-wave workgroups spread over all CUs; where those are too few to
    // keep the weights streaming, K is split over eight waves: while all its workgroups (two per CU)
    // run at once, or for long rows. Measured (us with the quantization launch, 64x16 / 16x16 / split):
    // Q4_K K = 2560, 9728 rows, 16 columns 14.2 / 14.2 / 16.5; Q6_K 22.2 / 19.4 / 26.4; Q4_K K = 9728,
    // 2560 rows, 16 columns - / 32.2 / 17.7, 37 columns 33.8 / 33.2 / 24.0; Q6_K 63 columns 64.1 / 52 / 50.4;
    // Q4_K K = 4096, 2048 rows, 16 columns - / 19 / 11.4.
    if (tiles(16) >= 256) return MM_64x16;
    return tiles(16) <= 128 || L.K >= 4096 ? MM_SPLIT : MM_16x16;
}

const char * mm_shape_name(mm_shape s) {
    switch (s) {
        case MM_64x64: return "64x64";
        case MM_32x64: return "32x64";
        case MM_64x48: return "64x48";
        case MM_64x32: return "64x32";
        case MM_64x16: return "64x16";
        case MM_16x16: return "16x16";
        case MM_SPLIT: return "split";
        default: return "res";
    }
}

void launch_mm_kq(const gemv_launch & L, const expert_groups * G, hipStream_t st) {
    if (!is_kquant(L.type) || L.K < 256 || L.K % 256 || L.ncols < 1 || !L.xq || L.n_mats < 1 || L.n_mats > GEMV_MAX_MATS ||
        L.swiglu || ((uintptr_t) L.xq) % 16) {
        HIP_ABORT("mm_kq: unsupported launch (type %d, K=%d, %d columns)", L.type, L.K, L.ncols);
    }
    if (G && (!L.ids || L.n_slots < 1 || L.x_cols < 1 || L.n_experts < 1)) HIP_ABORT("mm_kq: bad mul_mat_id geometry");
    for (int i = 0; i < L.n_mats; i++) {
        if (L.m[i].n_rows < 1 || ((uintptr_t) L.m[i].w) % 16 ||
            (L.type == GGML_TYPE_Q6_K && (((uintptr_t) L.m[i].wqh) % 16 || ((uintptr_t) L.m[i].wsc) % 4))) HIP_ABORT("mm_kq: misaligned weights");
    }
    const mm_shape s = mm_shape_of(L, G);
    switch (L.type) {
        case GGML_TYPE_Q4_K: mm_dispatch_q4_k(s, L, G, st); break;
        case GGML_TYPE_Q5_K: mm_dispatch_q5_k(s, L, G, st); break;
        default: mm_dispatch_q6_k(s, L, G, st); break;
    }
}

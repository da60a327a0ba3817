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
    // staged columns. With fewer, one-wave workgroups spread over all CUs; and K is split over eight waves
    // while all those workgroups (two per CU) run at once: 128 tiles of 64 rows. Past that the split costs its LDS
    // exchange for nothing, except over Q6_K's long rows. Measured, 64x16 / 16x16 / split, us with the
    // quantization launch (rows x K by columns):
    // up to 128 tiles: Q4_K 2048 x 2560 by 16 (32) 12.4 / 12.3 / 8.9, 4096 x 4096 by 16 (64) 17.1 / 16.3 / 10.4, 2560 x 9728
    // by 37 (120) 31.6 / 32.3 / 23.0, 8192 x 2560 by 16 (128) 12.5 / 12.6 / 12.0; Q5_K 128 14.8 / 14.0 / 13.9; Q6_K 128 20.1 / 18.3 / 18.3;
    // past it: 2560 rows by 60 (160), K = 4096 Q4_K 17.7 / 17.1 / 18.9, Q5_K 21.5 / 19.4 / 22.4, Q6_K 27.4 / 25.2 / 27.7;
    // K = 6144 23.5 / 22.7 / 23.9, 29.1 / 26.0 / 29.8, 41.0 / 34.2 / 34.9; K = 8192 29.4 / 28.3 / 29.5, 36.7 / 32.5 / 35.6,
    // 50.6 / 44.2 / 43.3; K = 14336 47.5 / 45.1 / 45.7, 59.8 / 52.3 / 56.9, 88.4 / 71.5 / 65.9.
    if (tiles(16) >= 256) return MM_64x16;
    return tiles(16) <= 128 || (L.type == GGML_TYPE_Q6_K && L.K >= 8192) ? MM_SPLIT : MM_16x16;
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

// k_mm_q5_k.hip — Q5_K instantiations of the multi-column product (mm_kq_impl.h)
#include "mm_kq_impl.h"

void mm_dispatch_q5_k(mm_shape s, const gemv_launch & L, const expert_groups * G, hipStream_t st) {
    mm_kq_detail::mm_dispatch<GGML_TYPE_Q5_K>(s, L, G, st);
}

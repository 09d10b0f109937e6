/*
 * tl_decode_rag_q8.hip — the instances of the decode kernel for batches of sessions of
 * unequal lengths (attn_decode_ring_kernel_rag, tl_decode_kernels.h; design in
 * tl_decode.hip): Q8_0 cache, without RoPE.  Their own translation unit so the kernel
 * instances build in parallel.
 */
#include "tl_decode_kernels.h"

template <int D>
static DecKernel pick_rag(int G) {
    constexpr int NT = 64 * TL_RING_WAVES;
    switch (G) {
#define TL_CASE(g)                                                                              \
    case g: {                                                                                   \
        constexpr bool mf = tl_decode_matrix_tile(D, g, true);                                  \
        return {(const void *)attn_decode_ring_kernel_rag<D, g, false, true, mf>, 4096, NT};   \
    }
        TL_CASE(1) TL_CASE(2) TL_CASE(3) TL_CASE(4)
        TL_CASE(5) TL_CASE(6) TL_CASE(7) TL_CASE(8)
#undef TL_CASE
    default:
        return {nullptr, 0, 0};
    }
}

DecKernel tl_pick_decode_rag_q8(int D, int G) {
    switch (D) {
    case 64: return pick_rag<64>(G);
    case 128: return pick_rag<128>(G);
    case 256: return pick_rag<256>(G);
    default: return {nullptr, 0, 0};
    }
}

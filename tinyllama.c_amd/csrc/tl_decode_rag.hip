/*
 * tl_decode_rag.hip — the instances of the decode kernel for batches of sessions of
 * unequal lengths (attn_decode_ring_kernel_rag, tl_decode_kernels.h; design in
 * tl_decode.hip): f16 cache.  Their own translation unit so the kernel
 * instances build in parallel.
 */
#include "tl_decode_kernels.h"

template <int D>
static DecKernel pick_rag(int G, bool rope) {
    constexpr int NT = 64 * TL_RING_WAVES;
    switch (G) {
#define TL_CASE(g)                                                                              \
    case g: {                                                                                   \
        constexpr bool mf = tl_decode_matrix_tile(D, g, false);                                 \
        if (rope) return {(const void *)attn_decode_ring_kernel_rag<D, g, true, false, mf>, 4096, NT}; \
        return {(const void *)attn_decode_ring_kernel_rag<D, g, false, false, mf>, 4096, NT};   \
    }
        TL_CASE(1) TL_CASE(2) TL_CASE(3) TL_CASE(4)
        TL_CASE(5) TL_CASE(6) TL_CASE(7) TL_CASE(8)
#undef TL_CASE
    default:
        return {nullptr, 0, 0};
    }
}

DecKernel tl_pick_decode_rag(int D, int G, bool rope) {
    switch (D) {
    case 64: return pick_rag<64>(G, rope);
    case 128: return pick_rag<128>(G, rope);
    case 256: return pick_rag<256>(G, rope);
    default: return {nullptr, 0, 0};
    }
}

/*
 * tl_prefill.hip — chunked-prefill attention on MFMA (gfx950).
 *
 * Math of op_attn (reference src/backend/cpu/cpu_op.c:1011-1062) for a batch
 * of n rows at positions pos..pos+n-1: row i attends to keys
 * [start_i, pos+i] (causal, start_i = pos+i+1-window when windowed) through
 * the slot table; out = softmax(q.K^T * scale) V.
 *
 * Work decomposition:
 *   A kv-head's work is a list of tasks (32 query rows, one q-head of the GQA
 *   group); a workgroup owns W consecutive tasks, one per wave, and one split of
 *   the key range, so every K/V tile staged in LDS serves W*32 query rows and
 *   every wave has work at any gqa.  W and the split count: plan() below.
 *   Per tile of BN keys (64 at head_dim <= 128, 32 at 256):
 *     S^T[key][row] = K . Q^T      v_mfma_f32_32x32x16_f16 per 32-key block,
 *                                  A = K rows from LDS, B = Q (registers, f16,
 *                                  pre-scaled by scale*log2 e); each lane ends
 *                                  up owning one query row and 16 keys of the
 *                                  block, so the row max / sum need one shuffle
 *                                  between the two half-waves.
 *     online softmax in f32 (exp2); mask arithmetic only on tiles that cross
 *                                  the causal diagonal, the window edge or the
 *                                  range end.  Each row's reference mu moves
 *                                  only when a tile's max passes it by more
 *                                  than 2^8 (then O and the sum are rescaled);
 *                                  -mu seeds the QK accumulators, so S - mu
 *                                  leaves the MFMA as is.  P^T is packed to
 *                                  f16 straight from the accumulator
 *                                  registers; the row sum is a dot2 of the
 *                                  packed P with (1, 1).
 *     O^T[d][row] += V^T . P^T     v_mfma_f32_32x32x16_f16 per 16 keys,
 *                                  A = V^T read from the row-major V tile with
 *                                  ds_read_b64_tr_b16 (a 4x16 -> 16x4 transpose
 *                                  per 16-lane group), B = P^T.  The MFMA's
 *                                  reduction index k is mapped to the keys each
 *                                  lane already holds, so P^T never goes
 *                                  through LDS and V is stored as loaded.
 *   K/V tiles are double-buffered in LDS (one barrier per tile): the next
 *   tile's rows are loaded into registers while the current one is computed
 *   and written to the other buffer afterwards.  Key splits (when the grid
 *   would not fill the chip) write partial (O, max, sum) rows that
 *   attn_merge_kernel combines.
 */
#include "tl_prefill_kernels.h"

TL_PREFILL_PICKER(tl_prefill_fn, false)

/* ------------------------------------------------------------------------ */
/* RoPE of a prefill batch                                                   */
/* ------------------------------------------------------------------------ */

/* Before the attention launch of a batch with RoPE: q rotated, scaled to log2
 * units and rounded to f16 as the kernel's MFMA operand, K rotated and
 * appended, V appended (f16 or Q8_0: the append kernels' conversions).  One
 * workgroup per row: a row's (cos, sin) pairs are formed once for all its
 * heads, while the row's loads are in flight.  The f16 q goes where the
 * attention output will be (the first half of each head's D floats of dst),
 * so nothing is allocated; the attention launch reads it before that output
 * is written.  dst may be q: the D/8 lanes of one head are of one wave, and
 * every read of the head is before its stores (the wave barrier).
 *
 * Bound by latency: one round trip for the row beside one sincosf, then the
 * stores.  Rotated inside the attention launch instead, every key split and
 * kv-head repeated the rotation before its first tile (us per OP_ATTN, with
 * powf + sincosf per lane and element / with a table per workgroup / here):
 * 333 rows from position 0 at 28/4/128 NEOX 77.9 / 28.6 / 23.7; 512 rows at
 * 8/4/256 NEOX over a 1024-key window 131 / 49.0 / 37.1; 512 rows at 32/8/128
 * over 4K keys of a Q8_0 cache (which always had an append launch) 84.7 /
 * 67.0 / 62.6; 512 rows at 32/8/128 over 32K keys 312 / 290 / 294. */
template <int D, bool Q8>
__global__ __launch_bounds__(256) void attn_rope_prep_kernel(const PrepParams p) {
    constexpr int VPR = D / 8, U = 4;
    __shared__ float2 s_tab[D / 2];
    const u32 tid = threadIdx.x, pairs = p.rope.rdim >> 1;
    const u32 items = (p.n_head + 2 * p.n_kv) * VPR;
    const bool part = p.rope.neox && rope_aligned8(p.rope.rdim, 1);
    const float th = tid < pairs ? rope_theta(tid, p.rope.rdim, p.rope.theta) : 0.f;
    for (u32 row = blockIdx.x; row < p.n; row += gridDim.x) {
        const u32 key = p.pos + row;
        const u32 ph = p.ring ? key % p.ring : (p.slots ? p.slots[key] : key);
        for (u32 i0 = 0; i0 < items; i0 += 256 * U) {
            /* item = 8 elements of one head: the q heads, then K, then V */
            float x[U][8], y[U][8];
            auto src_of = [&](u32 i) -> const float * {
                const u32 hd = i / VPR;
                if (hd < p.n_head) return p.q + (u64)row * p.q_stride + (u64)hd * D;
                const bool kk = hd < p.n_head + p.n_kv;
                return (kk ? p.k : p.v) + (u64)row * p.kv_stride +
                       (u64)(hd - p.n_head - (kk ? 0u : p.n_kv)) * D;
            };
#pragma unroll
            for (int u = 0; u < U; u++) {
                const u32 i = i0 + u * 256 + tid, e0 = (i % VPR) * 8;
                if (i < items) {
                    const float *hrow = src_of(i);
                    const float4 a = *(const float4 *)(hrow + e0), b = *(const float4 *)(hrow + e0 + 4);
                    x[u][0] = a.x; x[u][1] = a.y; x[u][2] = a.z; x[u][3] = a.w;
                    x[u][4] = b.x; x[u][5] = b.y; x[u][6] = b.z; x[u][7] = b.w;
                    if (part && e0 < p.rope.rdim) {
                        const u32 o = rope_partner(e0, p.rope.rdim);
                        const float4 c = *(const float4 *)(hrow + o), d = *(const float4 *)(hrow + o + 4);
                        y[u][0] = c.x; y[u][1] = c.y; y[u][2] = c.z; y[u][3] = c.w;
                        y[u][4] = d.x; y[u][5] = d.y; y[u][6] = d.z; y[u][7] = d.w;
                    }
                }
            }
            if (i0 == 0) {
                if (row != blockIdx.x) __syncthreads();   /* the previous row's readers */
                if (tid < pairs) {
                    float c, s;
                    sincosf((float)key * th, &s, &c);
                    s_tab[tid] = make_float2(c, s);
                }
                __syncthreads();
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const u32 i = i0 + u * 256 + tid, e0 = (i % VPR) * 8, hd = i / VPR;
                if (i >= items) continue;
                if (hd < p.n_head + p.n_kv) {
                    if (rope_aligned8(p.rope.rdim, p.rope.neox))
                        rope8_tab(x[u], y[u], e0, p.rope.rdim, p.rope.neox, s_tab);
                    else
                        rope8_tab_any(x[u], src_of(i), e0, p.rope.rdim, s_tab);
                }
                /* in place (dst = q) the stores below replace elements that other
                 * lanes of the head rotate with (read above, or just now for a
                 * half that is no multiple of 8): no lane stores before all of
                 * them have read, also where lanes past rope_dim read nothing */
                __builtin_amdgcn_wave_barrier();
                if (hd < p.n_head) {
                    const float sc = p.scale_log2;
                    u16 *o = (u16 *)(p.dst + (u64)row * p.q_stride + (u64)hd * D) + e0;
                    *(uint4 *)o = make_uint4(pack2(x[u][0] * sc, x[u][1] * sc), pack2(x[u][2] * sc, x[u][3] * sc),
                                             pack2(x[u][4] * sc, x[u][5] * sc), pack2(x[u][6] * sc, x[u][7] * sc));
                    continue;
                }
                const bool kk = hd < p.n_head + p.n_kv;
                const u64 prow = (u64)(hd - p.n_head - (kk ? 0u : p.n_kv)) * p.cap + ph;
                u16 *c = kk ? p.kc : p.vc;
                if constexpr (Q8) {
                    /* the 4 lanes of a 32-value block are an aligned group */
                    const float d = group_max<4>(amax8(x[u])) / 127.0f;
                    if (ph >= p.cap) continue;
                    *(uint2 *)((uint8_t *)c + prow * D + e0) = q8_pack8(x[u], d > 0.0f ? 1.0f / d : 0.0f);
                    if ((e0 & 31) == 0) (kk ? p.ks : p.vs)[prow * (D / 32) + e0 / 32] = (u16)f32_to_f16_bits(d);
                } else {
                    if (ph >= p.cap) continue;
                    *(uint4 *)(c + prow * D + e0) =
                        make_uint4(pack_f16x2(x[u][0], x[u][1]), pack_f16x2(x[u][2], x[u][3]),
                                   pack_f16x2(x[u][4], x[u][5]), pack_f16x2(x[u][6], x[u][7]));
                }
            }
        }
    }
}

static const void *prep_fn(u32 D, bool q8) {
    switch (D) {
    case 64: return q8 ? (const void *)attn_rope_prep_kernel<64, true> : (const void *)attn_rope_prep_kernel<64, false>;
    case 128: return q8 ? (const void *)attn_rope_prep_kernel<128, true> : (const void *)attn_rope_prep_kernel<128, false>;
    case 256: return q8 ? (const void *)attn_rope_prep_kernel<256, true> : (const void *)attn_rope_prep_kernel<256, false>;
    default: return nullptr;
    }
}

static int launch_rope_prep(const LayerView &L, const tl_attn_args *a, const RopeCfg &rope, float scale_log2,
                            hipStream_t st) {
    PrepParams p;
    memset(&p, 0, sizeof(p));
    p.q = a->q;
    p.k = a->k;
    p.v = a->v;
    p.dst = a->dst;
    p.kc = (u16 *)L.k;
    p.vc = (u16 *)L.v;
    p.ks = (u16 *)L.ks;
    p.vs = (u16 *)L.vs;
    p.slots = a->slots;
    p.cap = L.cap;
    p.ring = L.ring;
    p.pos = a->pos;
    p.n = a->n;
    p.n_head = a->n_head;
    p.n_kv = L.n_kv_head;
    p.q_stride = a->q_stride;
    p.kv_stride = a->kv_stride;
    p.scale_log2 = scale_log2;
    p.rope = rope;
    const void *fn = prep_fn(L.head_dim, L.q8);
    if (!fn) return tl_fail(TL_EINVAL, "prefill: head_dim %u", L.head_dim);
    void *args[] = {(void *)&p};
    HIP_TRY(hipLaunchKernel(fn, dim3(a->n < 2048 ? a->n : 2048), dim3(256), args, 0, st));
    return TL_OK;
}

/* ------------------------------------------------------------------------ */

bool tl_prefill_supported(const LayerView &L, const tl_attn_args *a) {
    if (tl_tune(TL_TUNE_NO_PREFILL) == 1) return false;
    const u32 G = a->n_head / L.n_kv_head;
    return (L.head_dim == 64 || L.head_dim == 128 || L.head_dim == 256) && G >= 1 && G <= 8;
}

/* The prefill kernel for batches of more than TL_DEC_FOLD_MAX_ROWS rows, and for
 * those of at least TL_PREFILL_MIN_ROWS whose rows x visible keys x heads x
 * head_dim exceed a bound; smaller ones run on the decode kernel, whose matrix
 * tile folds the rows into its columns; a quantized key is dearer there.  The
 * bound is the same with RoPE, so that a fused call takes the kernel, and gives
 * the bits, of the rotation and the plain call; with it the prefill side would
 * win earlier, because the decode side needs a rotating append launch first
 * (28/4/128 NEOX, 32 rows over 500 keys 18.7 / 17.5).  Measured, us per OP_ATTN,
 * decode / prefill kernel (32/8/128 unless said): f16, 17 rows over 4K keys 19.9
 * / 20.2, 8K 26.9 / 22.6; 32 rows 2K 17.7 / 19.6, 4K 23.3 / 22.5; 64 rows 1K
 * 17.6 / 19.5, 2K 23.2 / 22.5, 4K 33.6 / 24.5; 32/8/64, 32 rows 4K 15.1 / 17.1,
 * 8K 20.3 / 20.5, 16K 29.4 / 23.7; 8/4/256, 32 rows 2K 21.5 / 22.7, 4K 29.9 /
 * 26.5.  Q8_0, 32 rows 1K 17.1 / 21.4, 2K 22.9 / 23.2, 4K 31.0 / 27.0; 8/4/256
 * 2K 24.8 / 24.8.  One q-head per kv-head (where the line lies at more rows x
 * keys), just below and just above it: 8/8/128, 17 rows 22K 29.2 / 28.0, 24K
 * 31.0 / 29.2; 64 rows 5.8K 19.8 / 19.6, 6.4K 20.4 / 20.0; Q8_0, 32 rows 7.2K
 * 22.4 / 23.5, 8K 23.4 / 23.8; 32/32/128, 64 rows 1.4K 19.8 / 18.8, 1.6K 20.9 /
 * 18.5.  Few heads: 4/4/64, 32 rows 46K 24.2 / 26.3, 51K 25.2 / 27.3, 17 rows 55K
 * 26.2 / 27.8, 87K 42.0 / 34.8; Q8_0, 64 rows 14K 21.1 / 23.3, 16K 21.6 / 23.7;
 * 1/1/64, 64 rows 103K 19.3 / 32.5, 17 rows 221K 26.8 / 41.1 — but 349K 246 /
 * 50: past TL_DEC_FOLD_MAX_KEYS the chunks of a slot table make more splits than
 * a folded group merges (16 columns x 128), and each row reads the keys again.
 * Up to TL_DEC_MAX_NEW rows the decode launch appends them itself and the line
 * lies higher at head_dim <= 128: 16 rows, decode / prefill kernel, 32/8/128 over
 * 6.1K keys 17.5 / 19.7, 10.4K 22.3 / 23.2, 13.4K 26.0 / 25.1; 28/4/128 7K 18.0 /
 * 20.3, 11.9K 24.2 / 23.3; 32/8/64 12.2K 14.2 / 19.4, 20.8K 20.2 / 23.4; Q8_0, 32/8/128
 * 3.8K 18.0 / 21.3, 6.5K 23.2 / 25.5, 28/4/128 7.4K 24.8 / 24.6; 8/4/256 6.1K 22.9 /
 * 22.4. */
#define TL_DEC_FOLD_MAX_KEYS (TL_DEC_MAX_CHUNK * 2048u / 16u)
static u64 prefill_min_work(const LayerView &L) {
    const bool wide = L.head_dim == 256;
    if (L.q8) return wide ? 180000000u : 250000000u;
    return wide ? 200000000u : 400000000u;
}

bool tl_use_prefill(const LayerView &L, const tl_attn_args *a) {
    if (a->n < TL_PREFILL_MIN_ROWS || !tl_prefill_supported(L, a)) return false;
    if (tl_tune(TL_TUNE_NO_PREFILL) == 2) return true;
    const u64 keys = (u64)a->pos + a->n;
    const u64 vis = (a->window && keys > a->window) ? a->window : keys;
    u64 most = prefill_min_work(L);
    if (a->n <= TL_DEC_MAX_NEW && L.head_dim <= 128) most += most / 5 * 3;
    return a->n > TL_DEC_FOLD_MAX_ROWS || vis > TL_DEC_FOLD_MAX_KEYS ||
           (u64)a->n * vis * a->n_head * L.head_dim > most;
}

/* workgroups of W tasks per kv-head; GN = tasks of a 32-row block */
static u32 task_blocks(u32 n, u32 GN, u32 W) { return (GN * ((n + 31) / 32) + W - 1) / W; }
static u32 tasks_per_block(u32 D, u32 G) { return D == 256 ? G * pf_parts<256>() : G; }

/* us per tile (64 keys; 32 at head_dim 256) of a workgroup of w waves: the
 * slope of long runs with one workgroup per CU (f16 at head_dim 128 1.70 / 1.55
 * for 8 / 4 waves, at 64 1.1 / 0.9; Q8_0 1.87 / 2.03 and 1.12 / 1.26: there the
 * workgroup's threads dequantize the tile, so half of them take longer), then
 * moved to where the plan's choices cost least over 260 shapes (65 to 1024 rows,
 * 0 to 14K keys, 1 to 32 heads, both caches), each timed at both widths and up
 * to 16 split counts: the choices are 1.4% from the best ones on average (4.1%
 * with one Q8_0 cost for all and a merge that costs the same for any count), 7%
 * for one shape in 20.  At 256 (slopes 1.39 / 1.5, Q8_0 1.63 / 1.9) and for 4
 * waves over a Q8_0 cache short runs count for more than the slope. */
static float tile_us(u32 D, u32 w, bool q8) {
    if (q8) return D == 64 ? (w == 8 ? 1.12f : 1.45f) : D == 128 ? (w == 8 ? 1.90f : 2.10f)
                                                                 : (w == 8 ? 2.06f : 1.90f);
    return D == 64 ? (w == 8 ? 1.10f : 0.94f) : D == 128 ? (w == 8 ? 1.70f : 1.55f)
                                                         : (w == 8 ? 1.39f : 1.33f);
}

/* Waves per workgroup (W) and key splits of a launch, by a cost in us: the
 * tiles of one workgroup's share of the keys, plus, with splits, the merge
 * launch: 3.5 us, 0.11 for each split (a thread folds them in turn; 65 rows at
 * 1/1/64 over 12K keys: 32 splits 16.4, 189 splits 28.8) and the partials' way
 * through memory (~6 TB/s; 2048 rows at 12/4/64 from position 0, 8 waves: 1
 * split 50.4, 2 splits 38.0).  At most one workgroup per CU counts: a partial
 * second round doubles the time (512 rows at 28/4/128 over 16K keys: 4 splits
 * 148 us, 5 splits 221).
 * 8 waves read and stage each key for twice the rows at nearly the same speed
 * and win where they fill the chip; 4 waves start ~3 us sooner (half the rows
 * to append and stage) and win below that.  Measured, W = 8 / 4, best split
 * counts (us): 512
 * rows from position 0 at 32/8/128 27.1 / 23.3, 333 at 28/4/128 23.4 / 18.3,
 * 512 at 32/8/64 20.5 / 16.0; 333 rows over 1K keys at 32/8/64 21.4 / 19.7;
 * 100 over 2K 18.7 / 16.6; 512 rows over 4.6K keys at 32/8/128 58.9 / 62.2,
 * at 32/8/64 39.3 / 40.0; 70 rows over 20K at 28/4/128 52.3 / 53.7; Q8_0, 512
 * rows from position 0 at 32/8/64 20.4 / 19.2, at 32/8/128 29.1 / 28.4, at
 * 8/4/256 30.8 / 28.9; 333 over 800 keys at 32/8/128 29.7 / 33.8; 200 over 12K
 * at 4/4/64 25.7 / 24.9. */
static void plan(const LayerView &L, const tl_attn_args *a, u32 G, u32 cus, u32 &W, u32 &ns) {
    const u32 D = L.head_dim, bn = D <= 128 ? 64 : 32, GN = tasks_per_block(D, G);
    const float part_us = 0.11f + (float)a->n * a->n_head * D * 4.f * 2.f / 6.1e6f;   /* per split */
    float best = 0.f;
    u32 wide = 0;                              /* workgroups with 8 waves */
    W = 0;
    for (u32 w = 8; w >= 4; w -= 4) {
        const float tile = tile_us(D, w, L.q8), start = w == 8 && D <= 128 ? 3.f : 0.f;
        const u32 base = task_blocks(a->n, GN, w) * L.n_kv_head;
        if (base > cus && W) break;
        /* no more workgroups with 4 waves: the other 4 at least stage the tiles
         * (at head_dim 256: 17 rows over 8K keys at 8/4/256, 8 / 4 waves 26.4 /
         * 27.5, Q8_0 28.2 / 30.3) */
        if (W && D > 128 && base == wide) break;
        wide = base;
        const u32 rows = ((w - 1) / GN + 1) * 32;
        u32 span = a->pos + a->n;              /* most keys any workgroup sees */
        if (a->window && span > (u64)a->window + rows) span = a->window + rows;
        const u32 most = base < cus ? cus / base : 1u;
        for (u32 k = 1; k <= most; k++) {
            const u32 tiles = ((span + k - 1) / k + bn - 1) / bn;
            const float t = tiles * tile + start + (k > 1 ? 3.5f + k * part_us : 0.f);
            if (!W || t < best) {
                best = t;
                W = w;
                ns = k;
            }
            if (tiles == 1) break;
        }
    }
}

int tl_launch_prefill(const LayerView &L, const tl_attn_args *a, const RopeCfg &rope,
                      hipStream_t st, bool append, const AppendParams *own) {
    const bool rope_on = rope.rdim != 0;
    if (append && L.q8 && !rope_on)
        return tl_fail(TL_EINVAL, "prefill: no fused append into a Q8_0 cache");
    const u32 D = L.head_dim, G = a->n_head / L.n_kv_head;
    if (L.q8 && (!L.ks || !L.vs)) return tl_fail(TL_EINVAL, "prefill: a Q8_0 cache needs scales");
    PrefParams p;
    memset(&p, 0, sizeof(p));
    p.k = (const u16 *)L.k;
    p.v = (const u16 *)L.v;
    p.ks = L.ks;
    p.vs = L.vs;
    p.slots = a->slots;
    p.cap = L.cap;
    p.ring = L.ring;
    p.q = a->q;
    p.dst = a->dst;
    p.q_stride = a->q_stride;
    p.pos = a->pos;
    p.n = a->n;
    p.n_head = a->n_head;
    p.n_kv = L.n_kv_head;
    p.window = a->window;
    p.scale_log2 = a->scale * 1.4426950408889634f;
    if (rope_on) {
        if (!append) return tl_fail(TL_EINVAL, "prefill: RoPE without the batch's K/V rows");
        append = false;      /* the pre-launch below writes them */
        p.q = nullptr;
    }

    p.gqa = G;
    int cus = 256;
    {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
            cus = n;
    }
    u32 W, ns;
    plan(L, a, G, (u32)cus, W, ns);
    const u32 base = task_blocks(a->n, tasks_per_block(D, G), W) * L.n_kv_head;
    if (const u32 t = tl_tune(TL_TUNE_PREFILL_SPLITS)) ns = t;
    if (const size_t fixed = tl_workspace_fixed_acc()) {
        /* no-allocation call: as many key splits as the fixed region holds */
        const size_t per_split = (size_t)a->n * a->n_head * D;
        if ((size_t)ns * per_split > fixed) ns = (u32)(fixed / per_split);
        if (ns < 1) ns = 1;
    }
    p.n_split = ns;
    const u32 blocks = base * ns;
    if (append && own && blocks > (u32)cus) {
        /* workgroups of the fused append wait for units that other workgroups
         * write, so all of them have to run at once: one per CU is sure to.
         * With more, a writer may not start before a waiter ends, every such
         * wait runs into its bound and the waiter writes all the rows itself
         * (us per OP_ATTN from position 0, fused / separate: 3072 rows at
         * 32/8/128, 384 workgroups, 1147 / 113; 4096 rows at 32/8/64, 512
         * workgroups, 1264 / 113; where all run at once fusing is the faster:
         * 4096 rows at 8/8/128 86 / 88, 3072 rows at 4/1/128 39.8 / 43.4) */
        const int rc = tl_launch_append(*own, 1, st);
        if (rc) return rc;
        append = false;
    }
    const size_t units = (size_t)L.n_kv_head * ((a->n + TL_PF_ROWS - 1) / TL_PF_ROWS);
    if (ns > 1 || append) {
        TlWorkspace *w;
        size_t parts = ns > 1 ? (size_t)a->n * a->n_head * ns : 0;
        /* fused append: launch counter and unit flags past the decode
         * merge's counters */
        int rc = tl_workspace_get(st, parts * D, parts,
                                  append ? TL_MERGE_CNT_WORDS + TL_PF_CTR_WORDS + units : 0, &w);
        if (rc) return rc;
        if (ns > 1) {
            p.ws_acc = w->acc;
            p.ws_ml = (float2 *)w->ml;
        }
        if (append) {
            p.kin = a->k;
            p.vin = a->v;
            p.kv_stride = a->kv_stride;
            p.ctr = w->cnt + TL_MERGE_CNT_WORDS;
            p.flags = p.ctr + TL_PF_CTR_WORDS;
            const u32 polls = tl_tune(TL_TUNE_PREFILL_APPEND_POLLS);
            p.polls = polls ? polls - 1 : 4096;
        }
    }
    const void *fn = L.q8 ? tl_prefill_fn_q8((int)D, (int)W) : tl_prefill_fn((int)D, (int)W);
    if (!fn) return tl_fail(TL_EINVAL, "prefill: head_dim %u gqa %u", D, G);
    if (rope_on) {
        const int rc = launch_rope_prep(L, a, rope, p.scale_log2, st);
        if (rc) return rc;
    }
    void *args[] = {(void *)&p};
    HIP_TRY(hipLaunchKernel(fn, dim3(blocks), dim3(64 * W), args, 0, st));
    if (ns == 1) return TL_OK;
    /* combine the key splits (same partial layout as the decode kernel) */
    DecParams mp;
    memset(&mp, 0, sizeof(mp));
    mp.seq[0].dst = a->dst;
    mp.rows_per_seq = a->n;
    mp.n_kv = L.n_kv_head;
    mp.n_head = a->n_head;
    mp.q_stride = a->q_stride;
    mp.n_split = ns;
    mp.ws_acc = p.ws_acc;
    mp.ws_ml = p.ws_ml;
    return tl_launch_merge(mp, a->n, D, st);
}

/* ------------------------------------------------------------------------ */

/* MFMA ceiling probe: every wave runs `iters` rounds of 4 independent
 * v_mfma_f32_32x32x16_f16 chains on register operands (no memory traffic),
 * then folds its accumulators into one word of `sink` so nothing is dead. */
__global__ __launch_bounds__(256) void mfma_probe_kernel(u64 iters, float *sink) {
    const int tid = threadIdx.x;
    half8_t a, b;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        a[i] = (_Float16)((float)((tid + i) & 7) * 0.125f);
        b[i] = (_Float16)((float)((tid * 3 + i) & 7) * 0.0625f);
    }
    floatx16_t c[4] = {};
    for (u64 it = 0; it < iters; it++) {
#pragma unroll
        for (int j = 0; j < 4; j++) c[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c[j], 0, 0, 0);
    }
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) s += c[j][e];
    sink[(u64)blockIdx.x * blockDim.x + tid] = s;
}

extern "C" int tl_probe_mfma(uint64_t iters, uint32_t blocks, float *sink, void *stream) {
    if (!sink || blocks == 0 || iters == 0) return tl_fail(TL_EINVAL, "probe: bad arguments");
    hipLaunchKernelGGL(mfma_probe_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, (u64)iters,
                       sink);
    HIP_TRY(hipGetLastError());
    return TL_OK;
}

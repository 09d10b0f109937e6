"""Decode launches whose sessions differ in length (split counts by length),
and the ways a group's splits are merged, at the sizes where each begins.

References: the same sessions decoded one by one (pinned against the oracle
in test_gpu_kv.py) — split boundaries differ, and each split rounds its
probabilities to f16 against its own reference, so outputs agree to f16
rounding of P (3e-4, as split counts do there) — and, for the merges, the same
partials merged by the separate launch, equal up to the order of an f32 sum
of at most 64 non-negative weights (64 * 2^-24, times |out| <= 5)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    import tlkv
    tlkv.check(tlkv.lib().tl_init(0))
    return torch


def _layer(T, q8, cap, n_kv, hd, g, ring=0):
    import tlkv
    L = (tlkv.LayerQ8 if q8 else tlkv.Layer)(cap, n_kv, hd, ring=ring)
    k, v = (T.randn((cap, n_kv * hd), generator=g, device="cuda") for _ in range(2))
    fn = tlkv.lib().tl_kv_append_q8 if q8 else tlkv.lib().tl_kv_append
    no_ring = type(L.desc).from_buffer_copy(L.desc)
    no_ring.ring = 0
    tlkv.check(fn(no_ring, tlkv.ptr(k), tlkv.ptr(v), n_kv * hd, None, 0, cap, None))
    T.cuda.synchronize()
    return L


def _planes(L):
    return [getattr(L, x) for x in ("k", "v", "ks", "vs") if hasattr(L, x)]


RAGGED = [
    # n_head, n_kv, hd, positions, window, ring, q8, rope
    (28, 4, 128, [8000, 0, 511, 130, 2047, 128, 1, 4000], 0, False, False, True),
    (32, 8, 64, [3000, 17, 0], 0, False, False, False),
    (8, 8, 128, [900, 64, 63, 65, 700] * 3 + [5000], 0, False, False, True),
    (8, 4, 256, [6000, 40, 1500], 1024, True, False, False),
    (32, 4, 128, [9000, 300], 0, False, True, False),
    (8, 8, 64, [70, 5000, 1000], 2000, False, True, False),
]


@pytest.mark.parametrize("slots", [False, True])
@pytest.mark.parametrize("case", RAGGED)
def test_batch_of_unequal_sessions(T, case, slots):
    import tlkv
    n_head, n_kv, hd, lens, window, ring, q8, rope = case
    if ring and slots:
        pytest.skip("ring layers take no slot table")
    lib = tlkv.lib()
    g = T.Generator(device="cuda")
    g.manual_seed(len(lens) + hd)
    Seq = tlkv.DecodeSeqQ8 if q8 else tlkv.DecodeSeq
    rp = tlkv.RopeParams(hd, 1e4, 1)
    scale, keep, seqs, refs = hd ** -0.5, [], [], []
    for pos in lens:
        cap = window if ring else pos + 1
        L = _layer(T, q8, cap, n_kv, hd, g, ring=cap if ring else 0)
        twin = type(L)(cap, n_kv, hd, ring=cap if ring else 0)
        for a, b in zip(_planes(twin), _planes(L)):
            a.copy_(b)
        sl = T.randperm(cap, generator=g, device="cuda").to(T.int32) if slots else None
        q, k, v = (T.randn((1, h * hd), generator=g, device="cuda") for h in (n_head, n_kv, n_kv))
        out, ref = T.zeros_like(q), T.zeros_like(q)
        seqs.append(Seq(L.desc, None if sl is None else sl.data_ptr(), pos, 0, q.data_ptr(),
                        k.data_ptr(), v.data_ptr(), out.data_ptr()))
        a = tlkv.attn_args(q, k, v, ref, sl, pos, 1, n_head, hd, n_kv, window, scale)
        if rope:
            tlkv.check(lib.tl_attn_rope(twin.desc, a, rp, None))
        else:
            tlkv.check((lib.tl_attn_q8 if q8 else lib.tl_attn)(twin.desc, a, None))
        T.cuda.synchronize()
        keep.append((L, twin, sl, q, k, v, a))
        refs.append((out, ref))
    arr = (Seq * len(lens))(*seqs)
    for _ in range(3):      # merge state left clean for the next launch; same bits each time
        if rope:
            tlkv.check(lib.tl_attn_decode_batch_rope(arr, len(lens), n_head, window, scale, rp, None))
        else:
            fn = lib.tl_attn_decode_batch_q8 if q8 else lib.tl_attn_decode_batch
            tlkv.check(fn(arr, len(lens), n_head, window, scale, None))
        T.cuda.synchronize()
        for pos, (out, ref), (L, twin, *_r) in zip(lens, refs, keep):
            assert (out - ref).abs().max().item() < 3e-4, pos
            for a, b in zip(_planes(L), _planes(twin)):
                assert T.equal(a, b), pos


# n_head, n_kv, hd, keys, keys per split: split counts at the edges of a trip
# (8), of two trips (16, 17) and of a wave (64, 65), where the group's last
# workgroup merges; and both sides of the count from which every split merges a
# slice: at least 24, an output float4 in 16 per split, and with at most 128
# float4s a second trip of the last workgroup, else 72 KB of partials: 24 for 7
# or 8 heads at head_dim 128, 33 for 4, 32 for 8 heads at 256, 33 for 2, and
# never (65, 257: more than the 64 it is limited to) for 4 or 1 at 64
MERGES = [(32, 8, 128, 64 * n, 64) for n in (2, 8, 9, 16, 17, 23, 24, 32)] + [
    (7, 1, 128, 64 * 64, 64), (7, 1, 128, 64 * 65, 64), (8, 1, 256, 64 * 40, 64),
    (1, 1, 64, 128 * 33, 128), (4, 1, 128, 64 * 200, 64), (8, 4, 256, 32 * 39, 32)] + [
    (7, 1, 128, 64 * 23, 64), (7, 1, 128, 64 * 24, 64), (16, 2, 128, 64 * 24, 64),
    (16, 4, 128, 64 * 32, 64), (16, 4, 128, 64 * 33, 64), (8, 1, 256, 64 * 31, 64),
    (8, 1, 256, 64 * 32, 64), (4, 2, 256, 32 * 32, 32), (4, 2, 256, 32 * 33, 32),
    (8, 2, 64, 128 * 64, 128)]


def _merge_runs(T, case, wgs=0):
    """The partials of one launch merged by the separate launch, then as the
    plan has it, by each group's last workgroup, and with no waits."""
    import tlkv
    n_head, n_kv, hd, keys, per = case
    lib = tlkv.lib()
    g = T.Generator(device="cuda")
    g.manual_seed(keys)
    L = _layer(T, False, keys, n_kv, hd, g)
    q = T.randn((1, n_head * hd), generator=g, device="cuda")

    def run(**tune):
        out = T.full_like(q, float("nan"))
        a = tlkv.attn_args(q, None, None, out, None, keys - 1, 1, n_head, hd, n_kv, 0)
        with tlkv.tuning(tlkv.TUNE_DECODE_MIN_KEYS, per), tlkv.tuning(tlkv.TUNE_DECODE_WGS, wgs), \
             tlkv.tuning(tlkv.TUNE_DECODE_MERGE_KERNEL, tune.get("kernel", 0)), \
             tlkv.tuning(tlkv.TUNE_DECODE_SINGLE_MERGE, tune.get("single", 0)), \
             tlkv.tuning(tlkv.TUNE_DECODE_MERGE_POLLS, tune.get("polls", 0)):
            for _ in range(2):
                tlkv.check(lib.tl_attn_noappend(L.desc, a, None))
        T.cuda.synchronize()
        return out

    return run(kernel=1), (run(), run(single=1), run(polls=1))


@pytest.mark.parametrize("case", MERGES)
def test_split_merge_paths_agree(T, case):
    want, gots = _merge_runs(T, case)
    for got in gots:
        assert (got - want).abs().max().item() < 64 * 2.0 ** -24 * 5


# more splits than a wave has lanes, where the last workgroup's merge depends on
# the columns: shared by 16, 2 and 1 threads per column, shares from LDS (from 97
# splits on at head_dim 64), more than the 256 splits whose pairs are read at
# once; and two trips of few columns, where slices begin (33 splits of 7 heads,
# 49 of 5 at head_dim 64)
MANY = [(1, 1, 64, 128 * n, 128) for n in (65, 75, 224)] + [
    (7, 1, 64, 128 * n, 128) for n in (32, 33, 65, 96, 97)] + [
    (5, 1, 64, 128 * 48, 128), (5, 1, 64, 128 * 49, 128), (4, 2, 64, 128 * 128, 128),
    (1, 1, 128, 64 * 256, 64), (2, 1, 256, 32 * 200, 32), (4, 1, 256, 32 * 100, 32),
    (8, 1, 256, 32 * 100, 32), (7, 1, 128, 64 * 235, 64),
    (4, 1, 128, 64 * 256, 64), (4, 1, 128, 64 * 257, 64), (4, 1, 128, 64 * 500, 64),
    (1, 1, 64, 128 * 400, 128), (4, 1, 64, 128 * 300, 128)]


@pytest.mark.parametrize("case", MANY)
def test_many_splits_merged_alike(T, case):
    """As above, the f32 sums over up to 500 splits."""
    n_split = case[3] // case[4]
    want, gots = _merge_runs(T, case, 1024)
    for got in gots:
        assert (got - want).abs().max().item() < max(64, n_split) * 2.0 ** -24 * 5


def test_unequal_sessions_share_cache_lines(T):
    """Rows of 64 bytes (Q8_0 at head_dim 64) lie two to a cache line, their
    scales 32 to one: through permuted slot tables a group's splits share
    lines, so the plan for unequal lengths keeps a group on one L2, as the
    plan with 240 workgroups (10 equal splits of 24 groups) does.  Measured
    0.96 of the latter's time; 1.16 with the splits spread over the L2s."""
    import tlkv
    lib, g, keep = tlkv.lib(), T.Generator(device="cuda"), []
    g.manual_seed(1)
    n_head, n_kv, hd, lens = 32, 8, 64, [15000, 20000, 17321]

    def batch():
        seqs = []
        for pos in lens:
            L = tlkv.LayerQ8(pos + 1, n_kv, hd)
            sl = T.randperm(pos + 1, generator=g, device="cuda").to(T.int32)
            q, k, v = (T.randn((1, h * hd), generator=g, device="cuda") for h in (n_head, n_kv, n_kv))
            out = T.zeros_like(q)
            keep.append((L, sl, q, k, v, out))
            seqs.append(tlkv.DecodeSeqQ8(L.desc, sl.data_ptr(), pos, 0, q.data_ptr(), k.data_ptr(),
                                         v.data_ptr(), out.data_ptr()))
        return (tlkv.DecodeSeqQ8 * len(lens))(*seqs)

    arrs, times = [batch() for _ in range(8)], {0: [], 240: []}
    for _ in range(8):
        for wgs, t in times.items():     # in turn, so drift of the clocks meets both
            with tlkv.tuning(tlkv.TUNE_DECODE_WGS, wgs):
                e0, e1 = (T.cuda.Event(enable_timing=True) for _ in range(2))
                e0.record()
                for arr in arrs * 3:
                    tlkv.check(lib.tl_attn_decode_batch_q8(arr, len(lens), n_head, 0, hd ** -0.5,
                                                           tlkv.stream_handle()))
                e1.record()
                T.cuda.synchronize()
                t.append(e0.elapsed_time(e1))
    assert min(times[0]) < 1.08 * min(times[240]), times

"""The work that programs have the library do, as cases that can be timed and
checked: decode steps of one session and of several, draft rows, chunked
prefill, requests through a session with its prefix cache, and prefix forks.

A case is a dict of plain values.  `prepare` makes the caches, slot tables and
activations that a program holds before the call, `run` is one pass through
the C ABI (include/tlkv.h, include/tl_session.h) as such a program makes it,
`exact` the same results in 64 bits from plain torch.

Attention cases are a walk over `layers` layers (each with its own cache, as a
model's), one entry-point call per layer, with the argument blocks laid out
once.  Their outputs are every layer's attention rows and the whole caches
that the call appended to.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

for _p in (os.path.join(os.getcwd(), "tinyllama.c_amd"),):
    if _p not in sys.path:
        sys.path.insert(0, _p)
import tlkv  # noqa: E402

DEV = "cuda"

# (n_head, n_kv, head_dim, theta, neox): the shapes of the benchmark's configs
SHAPES = {
    "1b": (32, 8, 64, 5e5, 0),        # Llama-3.2-1B-shaped
    "8b": (32, 8, 128, 5e5, 0),       # Llama-3-8B-shaped
    "qwen": (28, 4, 128, 1e6, 1),     # Qwen2.5-7B-shaped (gqa 7)
    "gemma": (8, 4, 256, 1e4, 1),     # Gemma-3-4B-shaped
    "mha": (8, 8, 128, 5e5, 0),       # one query head per kv head
}


def _attn(name, kind, shape, pos, n=1, layers=1, n_seq=1, pos_min=0, q8=False, rope=True, window=0,
          ring=False, slots="permuted"):
    return dict(name=name, kind=kind, shape=shape, pos=pos, n=n, layers=layers, n_seq=n_seq,
                pos_min=pos_min, q8=q8, rope=rope, window=window, ring=ring, slots=slots)


def listed():
    return [
        # chat on a small model: a whole step's 16 layer calls, each ~1.5 MB (latency and launches)
        _attn("decode-1b", "decode", "1b", 701, layers=16),
        # the long-context decode of the headline metric: Q/K already rotated, identity slot table
        _attn("decode-8b-32k", "decode", "8b", 32781, layers=4, rope=False, slots="identity"),
        # the same model with the quantized cache at a middling depth
        _attn("decode-8b-q8", "decode", "8b", 12001, layers=4, q8=True),
        # a server's decode step: 8 sessions of ragged lengths in one launch per layer
        _attn("batch-qwen", "batch", "qwen", 8192, layers=4, n_seq=8, pos_min=512),
        # speculative decoding: 5 draft tokens verified at once
        _attn("draft-qwen", "decode", "qwen", 4099, n=5, layers=4),
        # sliding-window layers of a hybrid model, two sessions, ring caches
        _attn("batch-gemma-ring", "batch", "gemma", 16385, layers=5, n_seq=2, pos_min=9001,
              window=1024, ring=True, slots="none"),
        # a short first prompt (ragged row count)
        _attn("prefill-qwen-first", "prefill", "qwen", 0, n=333),
        # the last full chunk of a 32K prompt
        _attn("prefill-8b-deep", "prefill", "8b", 32256, n=512),
        # a chunk into the quantized cache
        _attn("prefill-8b-q8", "prefill", "8b", 4096, n=512, q8=True),
        # a chunk on a sliding-window layer with a ring cache
        _attn("prefill-gemma-ring", "prefill", "gemma", 8192, n=512, window=1024, ring=True,
              slots="none"),
        # a request whose system prompt is cached: prefix match, slot upload, 16 layers
        dict(name="session-1b", kind="session", shape="1b", prefix=700, suffix=333, layers=16,
             ctx=4096, ubatch=512, q8=False),
        # a cached prefix forked into another session's pool, every layer in one call
        dict(name="fork-qwen", kind="copy", shape="qwen", rows=1500, layers=28, cap=4608, q8=False),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "batch", "prefill", "prefill", "prefill", "session", "copy"])
    if kind == "session":
        shape = rng.choice(["1b", "qwen"])
        return dict(kind=kind, shape=shape, prefix=_log_int(rng, 16, 2000),
                    suffix=rng.choice([1, _log_int(rng, 2, 700)]), layers=16 if shape == "1b" else 8,
                    ctx=4096, ubatch=512, q8=rng.random() < 0.25)
    if kind == "copy":
        return dict(kind=kind, shape=rng.choice(["1b", "qwen"]), rows=_log_int(rng, 16, 4096),
                    layers=rng.choice([16, 28]), cap=4608, q8=rng.random() < 0.3)
    shape = rng.choice(list(SHAPES))
    pos = _log_int(rng, 16, 32000)
    c = _attn("", kind, shape, pos, q8=rng.random() < 0.3, rope=rng.random() < 0.7,
              slots=rng.choice(["none", "identity", "permuted"]))
    del c["name"]
    if kind == "decode":
        c.update(layers=4, n=1 if rng.random() < 0.6 else rng.randint(2, 15))
    elif kind == "batch":
        c.update(layers=4, n_seq=rng.randint(2, 16))
        c["pos"] = min(pos, 100000 // c["n_seq"])
        c["pos_min"] = _log_int(rng, 8, c["pos"])
        c["rope"] = c["rope"] and not c["q8"]    # the quantized batch takes rotated rows
    else:
        c.update(n=_log_int(rng, 17, 512), pos=rng.choice([0, pos]))
    if rng.random() < (0.5 if shape == "gemma" else 0.15):
        c["window"] = _log_int(rng, 64, 4096)
        if rng.random() < 0.6:
            c.update(ring=True, slots="none")
    return c


# ---- attention -----------------------------------------------------------------


def _positions(c):
    """Each session's position (batch: ragged, spread geometrically from pos_min to pos)."""
    m = c["n_seq"]
    if m == 1:
        return [c["pos"]]
    lo, hi = max(c["pos_min"], 1), c["pos"]
    p = [int(round(lo * (hi / lo) ** (i / (m - 1)))) for i in range(m)]
    return p[::2] + p[1::2]      # long and short sessions side by side


def _cap(c):
    n_keys = max(_positions(c)) + c["n"]
    return c["window"] + c["n"] - 1 if c["ring"] else (n_keys + 63) // 64 * 64


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _quantize(x):
    """Q8_0 blocks of f32/f64 x[..., D]: int8 values and binary16 scales."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1) / 127
    q = torch.round(b * torch.where(d > 0, 1 / d, torch.zeros_like(d))[..., None])
    return q.to(torch.int8).reshape(x.shape), d.to(torch.float16)


def _fresh_layer(c, g):
    """One layer's pools for every session ([n_seq][n_kv][cap][D]) and its activations."""
    H, KV, D, _, _ = SHAPES[c["shape"]]
    m, n, cap = c["n_seq"], c["n"], _cap(c)
    s = {}
    for x in "kv":
        if c["q8"]:
            pool = torch.empty((m, KV, cap, D), dtype=torch.int8, device=DEV)
            scale = torch.empty((m, KV, cap, D // 32), dtype=torch.float16, device=DEV)
            for i in range(m):
                pool[i], scale[i] = _quantize(torch.randn((KV, cap, D), generator=g, device=DEV))
            s[x], s[x + "s"] = pool, scale.view(torch.int16)
        else:
            s[x] = torch.randn((m, KV, cap, D), generator=g, device=DEV, dtype=torch.float16)
    s["q"] = torch.randn((m, n, H * D), generator=g, device=DEV)
    s["kin"] = torch.randn((m, n, KV * D), generator=g, device=DEV)
    s["vin"] = torch.randn((m, n, KV * D), generator=g, device=DEV)
    s["dst"] = torch.empty_like(s["q"])
    return s


def _slot_tables(c, g):
    cap = _cap(c)
    if c["slots"] == "none":
        return None
    if c["slots"] == "identity":
        t = torch.arange(cap, device=DEV).repeat(c["n_seq"], 1)
    else:
        t = torch.stack([torch.randperm(cap, generator=g, device=DEV) for _ in range(c["n_seq"])])
    return t.to(torch.int32).contiguous()


def _inputs(c, seed):
    g = _gen(seed)
    return _slot_tables(c, g), [_fresh_layer(c, g) for _ in range(c["layers"])]


def _lib():
    L = tlkv.lib()
    if not getattr(_lib, "ready", False):
        tlkv.check(L.tl_init(0))
        _lib.ready = True
    return L


def _prepare_attn(c, seed):
    H, KV, D, theta, neox = SHAPES[c["shape"]]
    L, cap, n, q8 = _lib(), _cap(c), c["n"], c["q8"]
    slots, layers = _inputs(c, seed)
    pos, ring, scale = _positions(c), cap if c["ring"] else 0, 1.0 / math.sqrt(D)
    stream = tlkv.stream_handle()
    rope = tlkv.RopeParams(D, theta, neox)

    def desc(s, i):
        if q8:
            return tlkv.KvLayerQ8(s["k"][i].data_ptr(), s["v"][i].data_ptr(), s["ks"][i].data_ptr(),
                                  s["vs"][i].data_ptr(), cap, KV, D, ring)
        return tlkv.KvLayer(s["k"][i].data_ptr(), s["v"][i].data_ptr(), cap, KV, D, ring)

    calls = []
    for s in layers:
        if c["kind"] == "batch":
            Seq = tlkv.DecodeSeqQ8 if q8 else tlkv.DecodeSeq
            seqs = (Seq * c["n_seq"])(*[
                Seq(desc(s, i), None if slots is None else slots[i].data_ptr(), pos[i], 0,
                    s["q"][i].data_ptr(), s["kin"][i].data_ptr(), s["vin"][i].data_ptr(),
                    s["dst"][i].data_ptr()) for i in range(c["n_seq"])])
            args = [seqs, c["n_seq"], H, c["window"], scale]
            fn = L.tl_attn_decode_batch_q8 if q8 else L.tl_attn_decode_batch
            if c["rope"]:
                fn = L.tl_attn_decode_batch_rope
                args.append(ctypes.byref(rope))
        else:
            a = tlkv.attn_args(s["q"], s["kin"], s["vin"], s["dst"], slots, pos[0], n, H, D, KV,
                               c["window"])
            d = desc(s, 0)
            args = [ctypes.byref(d), ctypes.byref(a)]
            if c["rope"]:
                fn = L.tl_attn_rope_q8 if q8 else L.tl_attn_rope
                args.append(ctypes.byref(rope))
            else:
                fn = L.tl_attn_q8 if q8 else L.tl_attn
        calls.append((fn, args + [stream]))
    out = [{x: s[x] for x in ("dst", "k", "v", "ks", "vs") if x in s} for s in layers]
    return dict(run=_run_calls, calls=calls, out=out, keep=(slots, layers, rope))


def _run_calls(st):
    for fn, args in st["calls"]:
        tlkv.check(fn(*args))
    return st["out"]


def _rotate(x, pos, D, theta, neox):
    """RoPE of x[n, heads, D] (64 bits) at positions pos.."""
    n = x.shape[0]
    i = torch.arange(D // 2, device=x.device, dtype=torch.float64)
    ang = (pos + torch.arange(n, device=x.device, dtype=torch.float64))[:, None] * theta ** (-2 * i / D)
    co, si = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    a, b = (x[..., : D // 2], x[..., D // 2:]) if neox else (x[..., 0::2], x[..., 1::2])
    ra, rb = a * co - b * si, a * si + b * co
    return torch.cat([ra, rb], -1) if neox else torch.stack([ra, rb], -1).reshape(x.shape)


def _attend(q, K, V, first, window):
    """q[n, H, D] at positions first + len(K[0]) - n .. over K, V[KV, keys, D] whose first key has
    position `first`; 64 bits, head by head."""
    n, H, D = q.shape
    KV, keys, _ = K.shape
    last = torch.arange(keys - n, keys, device=q.device)[:, None]
    at = torch.arange(keys, device=q.device)[None, :]
    hide = at > last
    if window:
        hide = hide | (at <= last - window)
    out = torch.empty_like(q)
    for h in range(H):
        s = (q[:, h] @ K[h * KV // H].T) / math.sqrt(D)
        out[:, h] = torch.softmax(s.masked_fill(hide, float("-inf")), -1) @ V[h * KV // H]
    return out


def _exact_attn(c, seed):
    H, KV, D, theta, neox = SHAPES[c["shape"]]
    slots, layers = _inputs(c, seed)
    n, cap, out = c["n"], _cap(c), []
    for s in layers:
        dst = torch.empty(s["q"].shape, dtype=torch.float64, device=DEV)
        pools = {x: s[x].double() for x in "kv"} if not c["q8"] else {}
        for i, pos in enumerate(_positions(c)):
            q = s["q"][i].double().reshape(n, H, D)
            new = {"k": s["kin"][i].double().reshape(n, KV, D), "v": s["vin"][i].double().reshape(n, KV, D)}
            if c["rope"]:
                q, new["k"] = _rotate(q, pos, D, theta, neox), _rotate(new["k"], pos, D, theta, neox)
            first = max(0, pos + 1 - c["window"]) if c["window"] else 0
            p = torch.arange(first, pos + n, device=DEV)
            rows = p % cap if c["ring"] else (p if slots is None else slots[i].long()[p])
            kv = {}
            for x in "kv":
                w = new[x].permute(1, 0, 2)
                if c["q8"]:
                    qv, d = _quantize(w)
                    w = (qv.double().reshape(KV, n, -1, 32) * d.double()[..., None]).reshape(KV, n, D)
                    old = (s[x][i][:, rows].double().reshape(KV, len(p), -1, 32) *
                           s[x + "s"].view(torch.float16)[i][:, rows].double()[..., None])
                    kv[x] = old.reshape(KV, len(p), D)
                else:
                    w = w.to(torch.float16).double()
                    kv[x] = pools[x][i][:, rows]
                    pools[x][i][:, rows[len(p) - n:]] = w
                kv[x] = torch.cat([kv[x][:, : len(p) - n], w], 1)
            dst[i] = _attend(q, kv["k"], kv["v"], first, c["window"]).reshape(n, H * D)
        held = ("k", "v", "ks", "vs") if c["q8"] else ()     # whole numbers: no 64-bit value
        out.append(dict(dst=dst, **pools, **{x: None for x in held}))
    return out


# ---- session ---------------------------------------------------------------------


def _session_rows(c, seed):
    H, KV, D, _, _ = SHAPES[c["shape"]]
    g, rows = _gen(seed), []
    n = c["prefix"] + c["suffix"]
    for _ in range(c["layers"]):
        rows.append({x: torch.randn((n, w * D), generator=g, device=DEV)
                     for x, w in (("q", H), ("k", KV), ("v", KV))})
    return rows


def _prepare_session(c, seed):
    H, KV, D, _, _ = SHAPES[c["shape"]]
    _lib()
    rows, p = _session_rows(c, seed), c["prefix"]
    s = tlkv.Session(c["layers"], H, KV, D, c["ctx"], c["ubatch"], kv_q8=c["q8"],
                     stream=tlkv.stream_handle())
    prefix = np.random.RandomState(int(seed) % (1 << 31)).randint(0, 30000, p).astype(np.uint32)
    head = {x: [r[x][:p] for r in rows] for x in "qkv"}
    tail = {x: [r[x][p:] for r in rows] for x in "qkv"}
    out = [torch.empty_like(x) for x in tail["q"]]
    s.kv_prepare(prefix)
    s.execute(prefix, head["q"], head["k"], head["v"], [torch.empty_like(x) for x in head["q"]],
              H * D, KV * D)
    torch.cuda.synchronize()
    return dict(run=_run_session, s=s, prefix=prefix, suffix=c["suffix"], next=30000, tail=tail,
                out=out, strides=(H * D, KV * D))


def _run_session(st):
    """A new request: the cached system prompt, then tokens that no request had before."""
    n = st["suffix"]
    tokens = np.concatenate([st["prefix"], np.arange(st["next"], st["next"] + n, dtype=np.uint32)])
    st["next"] += n
    _, at = st["s"].kv_prepare(tokens)
    st["s"].execute(tokens[at:], st["tail"]["q"], st["tail"]["k"], st["tail"]["v"], st["out"],
                    *st["strides"])
    return st["out"]


def _exact_session(c, seed):
    H, KV, D, _, _ = SHAPES[c["shape"]]
    out = []
    for r in _session_rows(c, seed):
        kv = []
        for x in "kv":
            w = r[x].reshape(-1, KV, D).permute(1, 0, 2)
            if c["q8"]:
                qv, d = _quantize(w.float())
                w = (qv.double().reshape(KV, -1, D // 32, 32) * d.double()[..., None]).reshape(w.shape)
            else:
                w = w.to(torch.float16).double()
            kv.append(w)
        q = r["q"][c["prefix"]:].double().reshape(-1, H, D)
        out.append(_attend(q, kv[0], kv[1], 0, 0).reshape(-1, H * D))
    return out


# ---- fork ------------------------------------------------------------------------


def _prepare_copy(c, seed):
    _, KV, D, _, _ = SHAPES[c["shape"]]
    L, g, n, cap = _lib(), _gen(seed), c["rows"], c["cap"]
    pools = []
    for side in range(2):
        side_pools = []
        for _ in range(c["layers"]):
            shape = (2, KV, cap, D)
            if side:
                kv = torch.zeros(shape, dtype=torch.int8 if c["q8"] else torch.float16, device=DEV)
            elif c["q8"]:
                kv = torch.randint(-127, 128, shape, generator=g, device=DEV, dtype=torch.int8)
            else:
                kv = torch.randn(shape, generator=g, device=DEV, dtype=torch.float16)
            t = {"kv": kv}
            if c["q8"]:
                sc = (2, KV, cap, D // 32)
                t["scales"] = (torch.zeros(sc, dtype=torch.int16, device=DEV) if side else
                               torch.randint(0, 15000, sc, generator=g, device=DEV, dtype=torch.int16))
            side_pools.append(t)
        pools.append(side_pools)

    def descs(side_pools):
        if c["q8"]:
            return (tlkv.KvLayerQ8 * len(side_pools))(*[
                tlkv.KvLayerQ8(t["kv"][0].data_ptr(), t["kv"][1].data_ptr(),
                               t["scales"][0].data_ptr(), t["scales"][1].data_ptr(), cap, KV, D, 0)
                for t in side_pools])
        return (tlkv.KvLayer * len(side_pools))(*[
            tlkv.KvLayer(t["kv"][0].data_ptr(), t["kv"][1].data_ptr(), cap, KV, D, 0)
            for t in side_pools])

    # the donor's rows as its requests left them, the receiver's as eviction freed them: runs of
    # neighbouring slots in places all over the pool
    def runs():
        blocks = torch.randperm((cap + 31) // 32, generator=g, device=DEV)
        at = (blocks[:, None] * 32 + torch.arange(32, device=DEV)).reshape(-1)
        return at[at < cap][:n].to(torch.int32).contiguous()

    src, dst = runs(), runs()
    fn = L.tl_kv_copy_between_q8 if c["q8"] else L.tl_kv_copy_between
    args = [descs(pools[1]), descs(pools[0]), c["layers"], tlkv.ptr(src), tlkv.ptr(dst), n,
            tlkv.stream_handle()]
    return dict(run=_run_calls, calls=[(fn, args)], out=pools[1], keep=(pools, src, dst))


# ---- the interface ---------------------------------------------------------------


def prepare(case, seed):
    kind = case["kind"]
    return (_prepare_session if kind == "session" else
            _prepare_copy if kind == "copy" else _prepare_attn)(case, seed)


def run(state):
    return state["run"](state)


def _visible(pos, n, window):
    """Keys seen by all rows together, and keys read (each once)."""
    seen = [min(pos + i + 1, window) if window else pos + i + 1 for i in range(n)]
    first = max(0, pos + 1 - window) if window else 0
    return sum(seen), pos + n - first


def work(case):
    H, KV, D, _, _ = SHAPES[case["shape"]]
    row = 2 * KV * (D + D // 16 if case["q8"] else 2 * D)       # K + V bytes of one cached token
    if case["kind"] == "copy":
        return dict(bytes=case["layers"] * case["rows"] * 2 * row + 8 * case["rows"], flops=0)
    if case["kind"] == "session":
        spans = [(case["prefix"], case["suffix"])]
        window, slots = 0, 4
    else:
        spans = [(p, case["n"]) for p in _positions(case)]
        window, slots = case["window"], 0 if case["slots"] == "none" else 4
    by = fl = 0
    for pos, n in spans:
        seen, keys = _visible(pos, n, window)
        by += (keys - n) * (row + slots) + n * (row + 2 * KV * D * 4 + 2 * H * D * 4)
        fl += 4 * H * D * seen
    return dict(bytes=case["layers"] * by, flops=case["layers"] * fl)


def tolerance(case):
    if case["kind"] == "copy":
        return "exact"
    # f16 caches, queries and probabilities: 2.2e-4 to 4.4e-4 from 64 bits where measured
    return {"rel": 2e-3, "max": 0.02}


def exact(case, seed):
    if case["kind"] == "copy":
        return None
    return _exact_session(case, seed) if case["kind"] == "session" else _exact_attn(case, seed)

"""The work this library is used for, as measurable cases: decode steps over shared KV fragments (through the operators,
through HogwildCache and as a captured graph), prompt chunks, the paged operators and merging segments.

A case is a dict of plain values.  A pass is what one step of a program does over `layers` decoder layers, every layer
with K/V of its own (so the caches hold what they hold in a real step, not the one layer that was just read).  Fragment
lengths are a text, "prompt,segment,segment,...", oldest first as worker 0 sees them; with cur = True the last W of them
are the workers' current-step fragments.  Data is N(0, 1) in the storage type, as in the benchmark's workloads.
"""
import math

import torch

from inference_lib_amd import attention as ops
from inference_lib_amd import cache as hc
from inference_lib_amd.cases import DTYPES, locations_for, rope_tables

DEV = "cuda"
HEADS = [(8, 2, 64), (28, 4, 128), (40, 8, 128), (32, 8, 128), (64, 8, 128), (16, 8, 256)]     # (Hq, Hkv, D)
ROPE_BASE = 1e6
MAX_KV_BYTES = 1.1e9         # K/V of all layers of one state
MAX_FLOPS = 4.0e11           # of one pass


def listed():
    return [
        # The smallest call: one fp32 layer with two workers, a 256-token prompt and 64-token segments.  Latency and launches.
        dict(name="fused_small_f32", kind="fused", dtype="f32", W=2, S=1, Hq=8, Hkv=2, D=64, lens="256,64,64", cur=False, layers=1),
        # A whole eager decode step through HogwildCache (append, inputs, attention; 12 layers): two workers, GQA 7.
        dict(name="step_cache_bf16", kind="step", dtype="bf16", W=2, S=1, Hq=28, Hkv=4, D=128, lens="2048,1024,1024", cur=False, layers=12),
        # The benchmark's headline: four workers, shared prompt, finished segments and ragged current-step fragments.
        dict(name="fused_headline_bf16", kind="fused", dtype="bf16", W=4, S=1, Hq=40, Hkv=8, D=128,
             lens="4096,2048,2048,2048,2048,41,16,110,73", cur=True, layers=16),
        # The same step as serving runs it: lengths in device memory, append + attention of all layers in one replayed graph.
        dict(name="graph_headline_bf16", kind="graph", dtype="bf16", W=4, S=1, Hq=40, Hkv=8, D=128,
             lens="4096,2048,2048,2048,2048,41,16,110,73", cur=True, layers=16),
        # Long context: eight workers behind a 16 K prompt, ragged segments, one-token current steps.
        dict(name="fused_long_bf16", kind="fused", dtype="bf16", W=8, S=1, Hq=32, Hkv=8, D=128,
             lens="16384,1899,1689,3322,1668,3001,969,2305,790,1,1,1,1,1,1,1,1", cur=True, layers=8),
        # Several new tokens per worker (speculative or chunked decoding): 128 query rows per kv head, fp16.
        dict(name="fused_multitoken_f16", kind="fused", dtype="f16", W=4, S=4, Hq=64, Hkv=8, D=128,
             lens="8192,2048,2048,2048,2048", cur=False, layers=8),
        # Reading a prompt: one worker brings 1024 tokens on top of 4096 that are already cached.
        dict(name="prefill_chunk_bf16", kind="fused", dtype="bf16", W=1, S=1024, Hq=40, Hkv=8, D=128, lens="4096,1024", cur=False, layers=2),
        # Decode at head dimension 256.
        dict(name="fused_d256_bf16", kind="fused", dtype="bf16", W=4, S=1, Hq=16, Hkv=8, D=256,
             lens="4096,2048,2048,2048,2048,100,79,112,62", cur=True, layers=8),
        # The two-operator path (rotation, then attention on rotated queries) at head dimension 64.
        dict(name="rope_sdpa_f16", kind="split", dtype="f16", W=3, S=2, Hq=8, Hkv=2, D=64, lens="1500,333,700,41", cur=False, layers=12),
        # Paged decode: append one token to four sequences of about 12.5 K tokens, then attend.
        dict(name="paged_decode_bf16", kind="paged", dtype="bf16", q_tokens="1,1,1,1", Hq=40, Hkv=8, D=128, lens="12528,12528,12528,12528",
             block=16, packed=False, layers=4),
        # Packed queries of different length over paged sequences: decoding, drafts and prompt chunks in one batch.
        dict(name="paged_packed_bf16", kind="paged", dtype="bf16", q_tokens="1,8,32,64", Hq=40, Hkv=8, D=128, lens="12528,12528,12528,12528",
             block=16, packed=True, layers=4),
        # Two workers' finished segments merged into the shared one (keys rotated further), 16 layers.
        dict(name="merge_bf16", kind="merge", dtype="bf16", W=2, S=1, Hq=40, Hkv=8, D=128, lens="2048,1000,777", cur=False, layers=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fused", "fused", "multi", "prefill", "prefill", "step", "graph", "split", "paged", "packed", "merge"])
    Hq, Hkv, D = rng.choice(HEADS)
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16"])
    if kind in ("fused", "step") and rng.random() < 0.15:
        dtype = "f32"
    if kind in ("paged", "packed"):
        W = rng.randint(1, 8)
        lens = [_log(rng, 200, 12528) for _ in range(W)]
        qt = [1] * W if kind == "paged" else [min(_log(rng, 1, 128), n) for n in lens]
        c = dict(kind="paged", dtype=dtype, q_tokens=",".join(map(str, qt)), Hq=Hq, Hkv=Hkv, D=D, lens=",".join(map(str, lens)),
                 block=rng.choice([16, 32, 64]), packed=kind == "packed", layers=rng.randint(1, 8))
    else:
        W = rng.randint(2, 8) if kind != "prefill" else rng.choice([1, 1, 2])
        S = 1
        if kind in ("multi", "split"):
            S = rng.randint(2, 8)
        elif kind == "prefill":
            S = _log(rng, 48, min(1500, 4080 // Hkv * 16 // (Hq // Hkv) // W))
        prompt = _log(rng, 64, 16384 if kind != "prefill" else 8192)
        seg = [max(S, _log(rng, 16, 4096)) if kind != "prefill" else S for _ in range(W)]
        cur = kind in ("fused", "graph") and rng.random() < 0.5
        lens = [prompt] + seg + ([max(S, _log(rng, 1, 128)) for _ in range(W)] if cur else [])
        c = dict(kind={"multi": "fused", "prefill": "fused"}.get(kind, kind), dtype=dtype, W=W, S=S, Hq=Hq, Hkv=Hkv, D=D,
                 lens=",".join(map(str, lens)), cur=cur, layers=rng.randint(1, 12))
    one = work(dict(c, layers=1))
    c["layers"] = max(1, min(c["layers"], int(MAX_KV_BYTES / one["bytes"]), int(MAX_FLOPS / max(one["flops"], 1))))
    return c


def _ints(text):
    return [int(x) for x in text.split(",")]


def _orders(W, cur):
    """Fragment 0 = prompt, 1..W = segments, then the current-step fragments: worker w sees the prompt, the others, its own."""
    out = []
    for w in range(W):
        o = [0] + [1 + x for x in range(W) if x != w] + [1 + w]
        if cur:
            o += [1 + W + x for x in range(W) if x != w] + [1 + W + w]
        out.append(o)
    return out


def work(case):
    sz = torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
    Hq, Hkv, D, lens, layers = case["Hq"], case["Hkv"], case["D"], _ints(case["lens"]), case["layers"]
    kv_row = 2 * Hkv * D * sz                              # one token's K and V
    if case["kind"] == "paged":
        qt = _ints(case["q_tokens"])
        q_rows = sum(qt) * Hq * D * sz
        pairs = sum(q * (n - q) + q * (q + 1) // 2 for q, n in zip(qt, lens))
        new = sum(qt) * kv_row                             # read as states, written to the cache (and read back by the attention)
        return {"bytes": float(layers * (sum(lens) * kv_row + 2 * q_rows + 2 * new)), "flops": float(layers * 4 * D * Hq * pairs)}
    W, S = case["W"], case["S"]
    if case["kind"] == "merge":
        return {"bytes": float(layers * 2 * sum(lens[1:]) * kv_row), "flops": float(layers * 3 * sum(lens[1:]) * Hkv * D)}
    loc = locations_for(_orders(W, case["cur"]), lens, S)
    pairs = sum(int((loc[f] + 1).clamp(0, n).sum()) for f, n in enumerate(lens))
    seen = sum(min(n, max(0, int(loc[f].max()) + 1)) for f, n in enumerate(lens))
    q_rows = W * S * Hq * D * sz
    total = layers * (seen * kv_row + q_rows * (2 + len(lens)))     # K/V, queries, result, the rotated queries of every fragment
    if case["kind"] == "split":
        total += layers * q_rows * len(lens)                        # the rotated queries are read back
    if case["kind"] in ("step", "graph"):
        total += layers * 2 * W * S * kv_row                        # the new tokens: read as states, written to the segments
    total += 2 * len(lens) * W * S * D * 4                          # cos / sin
    return {"bytes": float(total), "flops": float(layers * 4 * D * Hq * pairs)}


def tolerance(case):
    """About four times what the operators differ by from the same computation in float64 on the stored inputs."""
    if case["kind"] == "merge":                # one rounding more or less of a rotated key
        return {"bf16": {"rel": 1e-2, "max": 4e-2}, "f16": {"rel": 2e-3, "max": 8e-3}}[case["dtype"]]
    return {"bf16": {"rel": 1e-2, "max": 8e-2}, "f16": {"rel": 1.5e-3, "max": 1.2e-2}, "f32": {"rel": 1e-5, "max": 1e-4}}[case["dtype"]]


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(gen, td, *shape):
    return torch.randn(shape, generator=gen, dtype=td, device=DEV)


def _inv_freq(D):
    return (ROPE_BASE ** (-torch.arange(D // 2, dtype=torch.float64) * 2.0 / D)).to(torch.float32).to(DEV)


def prepare(case, seed):
    return {"fused": _prepare_ops, "split": _prepare_ops, "step": _prepare_cache, "graph": _prepare_cache, "paged": _prepare_paged,
            "merge": _prepare_merge}[case["kind"]](case, seed)


def run(state):
    return {"fused": _run_fused, "split": _run_split, "step": _run_step, "graph": _run_graph, "paged": _run_paged,
            "merge": _run_merge}[state["kind"]](state)


# ---- the operators on fragments ---------------------------------------------------------------------------------------
def _prepare_ops(case, seed):
    td, g = DTYPES[case["dtype"]], _gen(seed)
    W, S, Hq, Hkv, D, lens, layers = (case[k] for k in ("W", "S", "Hq", "Hkv", "D", "lens", "layers"))
    lens = _ints(lens)
    loc = locations_for(_orders(W, case["cur"]), lens, S)
    cos, sin = rope_tables(loc, D, ROPE_BASE)
    ks = [_randn(g, td, layers, Hkv, n, D) for n in lens]
    vs = [_randn(g, td, layers, Hkv, n, D) for n in lens]
    return {"kind": case["kind"], "scale": D ** -0.5, "q": list(_randn(g, td, layers, W, Hq, S, D)),
            "keys": [[k[i] for k in ks] for i in range(layers)], "values": [[v[i] for v in vs] for i in range(layers)],
            "loc": loc.to(DEV), "cos": cos.to(DEV), "sin": sin.to(DEV), "frag": torch.tensor(lens, dtype=torch.int32, device=DEV),
            "out": torch.empty((layers, W, Hq, S, D), dtype=td, device=DEV),
            "rq": torch.empty((len(lens), W, Hq, S, D), dtype=td, device=DEV)}


def _run_fused(s):
    out = s["out"]
    for q, k, v, o in zip(s["q"], s["keys"], s["values"], out):
        ops.hogwild_fused(q, s["loc"], k, v, s["scale"], s["frag"], s["cos"], s["sin"], rotated_queries=s["rq"], out=o)
    return out, s["rq"]


def _run_split(s):
    out = s["out"]
    for q, k, v, o in zip(s["q"], s["keys"], s["values"], out):
        ops.hogwild_rope(q, s["cos"], s["sin"], out=s["rq"])
        ops.hogwild_sdpa(s["rq"], s["loc"], k, v, s["scale"], s["frag"], out=o)
    return out, s["rq"]


# ---- a decode step through HogwildCache -------------------------------------------------------------------------------
def _prepare_cache(case, seed):
    td, g = DTYPES[case["dtype"]], _gen(seed)
    W, S, Hq, Hkv, D, layers = (case[k] for k in ("W", "S", "Hq", "Hkv", "D", "layers"))
    lens = _ints(case["lens"])
    segments = []
    for n in lens:
        seg = hc.SegmentCache(layers, Hkv, D, n + 256, dtype=td, device=DEV)
        for i in range(layers):
            seg.k[i][:, :n].copy_(_randn(g, td, Hkv, n, D))
            seg.v[i][:, :n].copy_(_randn(g, td, Hkv, n, D))
        seg.lengths = [n] * layers
        segments.append(seg)
    cache = hc.HogwildCache([[segments[f] for f in order] for order in _orders(W, case["cur"])], inv_freq=_inv_freq(D))
    own = [order[-1] for order in _orders(W, case["cur"])]
    pos = torch.tensor([[[lens[f] + i for i in range(S)] for f in own]], dtype=torch.int32)          # [1, W, S]
    cos, sin = (t[0].to(td).to(DEV) for t in rope_tables(pos, D, ROPE_BASE))
    # projections come as [W, S, heads, D] and are used transposed
    s = {"kind": case["kind"], "scale": D ** -0.5, "cache": cache, "segments": segments, "lens": lens, "cos": cos, "sin": sin,
         "q": [x.transpose(1, 2) for x in _randn(g, td, layers, W, S, Hq, D)],
         "k": [x.transpose(1, 2) for x in _randn(g, td, layers, W, S, Hkv, D)],
         "v": [x.transpose(1, 2) for x in _randn(g, td, layers, W, S, Hkv, D)],
         "out": torch.empty((layers, W, Hq, S, D), dtype=td, device=DEV)}
    if case["kind"] == "graph":
        cache.use_device_lengths(headroom=128, new_tokens=S)        # may move the segments into larger buffers
    # the new rows of all workers, of as many layers as the number of outputs allows (the attention results depend on all)
    s["written"] = [b[i][:, lens[f]:lens[f] + S] for i in range(min(layers, 24 // W)) for f in own for b in (segments[f].k, segments[f].v)]
    if case["kind"] == "step":
        return s
    s["start"] = torch.tensor([lens[f] for f in _orders(W, case["cur"])[0]], dtype=torch.int32, device=DEV)   # in worker 0's order
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        s["frags"] = _layers_of_a_step(s).frags              # the current lengths: a device tensor in this mode
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        _layers_of_a_step(s)
    return s


def _layers_of_a_step(s):
    cache = s["cache"]
    for i, (q, k, v, o) in enumerate(zip(s["q"], s["k"], s["v"], s["out"])):
        cs = cache.update_fused(k, v, s["cos"], s["sin"], i)
        rq = cache.get_queries_buffer(q, layer_idx=i)
        ops.hogwild_fused(q, cs.loc, cs.keys, cs.values, s["scale"], cs.frags, cs.cos, cs.sin, rotated_queries=rq, out=o,
                          device_lengths=cache.device_lengths)
    return cs


def _run_step(s):
    for seg, n in zip(s["segments"], s["lens"]):             # the step is taken back, as a rejected draft is
        seg.lengths = [n] * len(seg.lengths)
    cs = _layers_of_a_step(s)
    return s["out"], cs.loc, cs.cos, cs.sin, s["written"]


def _run_graph(s):
    s["frags"].copy_(s["start"])
    s["graph"].replay()
    return s["out"], s["frags"], s["written"]


# ---- the paged operators ----------------------------------------------------------------------------------------------
def _prepare_paged(case, seed):
    td, g = DTYPES[case["dtype"]], _gen(seed)
    Hq, Hkv, D, layers, bs = (case[k] for k in ("Hq", "Hkv", "D", "layers", "block"))
    lens, qt = _ints(case["lens"]), _ints(case["q_tokens"])          # lengths with the new tokens
    W, T = len(lens), sum(qt)
    per = [-(-n // bs) for n in lens]
    ids = torch.randperm(sum(per), generator=g, device=DEV).to(torch.int32).cpu()
    table = torch.zeros((W, max(per)), dtype=torch.int32)
    at = 0
    for w, n in enumerate(per):
        table[w, :n] = ids[at:at + n]
        at += n
    pos = torch.cat([torch.arange(n - q, n, dtype=torch.int32) for q, n in zip(qt, lens)])
    s = {"kind": "paged", "packed": case["packed"], "scale": D ** -0.5, "table": table.to(DEV),
         "kc": _randn(g, td, layers, sum(per), Hkv, bs, D), "vc": _randn(g, td, layers, sum(per), Hkv, bs, D)}
    if case["packed"]:
        cu = [sum(qt[:w]) for w in range(W + 1)]
        s.update(q=list(_randn(g, td, layers, 1, T, Hq, D)), loc=pos[None].to(DEV), frag=torch.tensor([lens], dtype=torch.int32, device=DEV),
                 cu=torch.tensor(cu, dtype=torch.int32, device=DEV), out=torch.empty((layers, T, Hq, D), dtype=td, device=DEV))
    else:                                                            # the longest sequence bounds the fragment, its location every other
        s.update(q=list(_randn(g, td, layers, 1, W, Hq, 1, D)), loc=pos.reshape(1, W, 1).to(DEV),
                 frag=torch.tensor([max(lens)], dtype=torch.int32, device=DEV), out=torch.empty((layers, W, Hq, 1, D), dtype=td, device=DEV),
                 k=[x.transpose(1, 2) for x in _randn(g, td, layers, W, 1, Hkv, D)], v=[x.transpose(1, 2) for x in _randn(g, td, layers, W, 1, Hkv, D)],
                 before=torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV))
    return s


def _run_paged(s):
    out = s["out"]
    for i, (q, kc, vc, o) in enumerate(zip(s["q"], s["kc"], s["vc"], out)):
        if s["packed"]:
            ops.hogwild_varlen_paged_sdpa(q, s["loc"], s["frag"], kc, vc, s["table"], s["cu"], None, s["scale"], out=o)
        else:
            ops.copy_to_blocks(s["k"][i], s["v"][i], kc, vc, s["table"], s["before"])
            ops.hogwild_paged_sdpa(q, s["loc"], s["frag"], kc, vc, s["table"], s["scale"], out=o)
    return out if s["packed"] else (out, s["kc"], s["vc"])


# ---- merging segments -------------------------------------------------------------------------------------------------
def _prepare_merge(case, seed):
    td, g = DTYPES[case["dtype"]], _gen(seed)
    Hkv, D, layers, lens = case["Hkv"], case["D"], case["layers"], _ints(case["lens"])
    total = sum(lens)
    segments = []
    for f, n in enumerate(lens):
        seg = hc.SegmentCache(layers, Hkv, D, total if f == 0 else n, dtype=td, device=DEV)
        for i in range(layers):
            seg.k[i][:, :n].copy_(_randn(g, td, Hkv, n, D))
            seg.v[i][:, :n].copy_(_randn(g, td, Hkv, n, D))
        seg.lengths = [n] * layers
        segments.append(seg)
    target = segments[0]
    return {"kind": "merge", "target": target, "sources": segments[1:], "n": lens[0], "inv": _inv_freq(D),
            "written": [b[i][:, lens[0]:] for i in range(layers) for b in (target.k, target.v)]}


def _run_merge(s):
    target = s["target"]
    target.lengths = [s["n"]] * len(target.lengths)          # merged anew in every pass
    for source in s["sources"]:
        hc.merge_caches(target, source, inv_freq=s["inv"])
    return s["written"]

"""Performance cases of the grouped multi-LoRA apply: what a serving program
has this framework do, from one small eager call to a whole prefill chunk.

A case is one forward step of a few layers: the step's routing table
(build_seg_bounds) and then every layer's LoRA calls on it.  Its fields:

  kind      which entry points the layers call (see _LAYERS below)
  graph     True: the step is captured once in a HIP graph and replayed, as a
            decode loop does; False: eager calls, as for prefill chunks, whose
            token count changes from step to step
  tokens    tokens in the step
  adapters  resident adapters; rank 0: the adapters' ranks are mixed
  route     how tokens are routed to adapters (see _route)
  hidden    input width; q, kv: the widths of a packed q/k/v layer's slices
            (kv 0: one slice); inter: the MLP width of the store kinds
  bias      V1 ops only: with a LoRA bias per slice
  dtype     of activations and weights

Calls update y in place, so a state passed to run() again adds the deltas
again, as the calls are defined to.
"""
import math

import torch

from adapterslotsplusplus_amd import WarpPipeConfig, WarpPipeEngine

_RANKS = (8, 16, 32, 64)
_DT = {"fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    """The measured cases, smallest first."""
    return [
        # One eager projection for a handful of requests: host time and launches.
        dict(name="eager_small", kind="o", graph=False, tokens=3, adapters=2, rank=16, route="uniform", hidden=4096,
             q=4096, kv=0, inter=0, layers=1, bias=False, dtype="fp16"),
        # A small captured decode batch (the reference's CPU-sized shape).
        dict(name="decode_64", kind="o", graph=True, tokens=64, adapters=4, rank=16, route="uniform", hidden=4096,
             q=4096, kv=0, inter=0, layers=8, bias=False, dtype="fp16"),
        # Captured decode through V1's separate shrink and expand ops (layers
        # whose buffer is exchanged between the two), with biases.
        dict(name="v1_split_decode", kind="v1", graph=True, tokens=48, adapters=8, rank=32, route="uniform",
             hidden=4096, q=4096, kv=1024, inter=0, layers=4, bias=True, dtype="bf16"),
        # The benchmark's decode batch: packed q/k/v over one A, and o.
        dict(name="decode_256", kind="qkv_o", graph=True, tokens=256, adapters=64, rank=32, route="zipf", hidden=4096,
             q=4096, kv=4096, inter=0, layers=4, bias=False, dtype="bf16"),
        # A draft model's step: 32 tenants of 4 tokens, one A per slice.
        dict(name="draft_128", kind="nslice", graph=True, tokens=128, adapters=32, rank=32, route="tenants",
             hidden=2048, q=2048, kv=2048, inter=0, layers=8, bias=False, dtype="bf16"),
        # Registered adapters of mixed ranks on an MLP (gate, up, down).
        dict(name="store_decode_512", kind="store", graph=True, tokens=512, adapters=128, rank=0, route="zipf",
             hidden=5120, q=0, kv=0, inter=13824, layers=1, bias=False, dtype="bf16"),
        # A large captured decode batch, every token its own request.
        dict(name="decode_1024", kind="nslice", graph=True, tokens=1024, adapters=64, rank=16, route="zipf",
             hidden=4096, q=4096, kv=1024, inter=0, layers=3, bias=False, dtype="bf16"),
        # A ragged prompt on a small model of odd widths.
        dict(name="prefill_ragged", kind="nslice", graph=False, tokens=777, adapters=5, rank=8, route="segments",
             hidden=1544, q=1100, kv=516, inter=0, layers=2, bias=False, dtype="fp16"),
        # V1's separate ops on a prompt.
        dict(name="v1_split_prefill", kind="v1", graph=False, tokens=1000, adapters=6, rank=32, route="segments",
             hidden=4096, q=4096, kv=1024, inter=0, layers=2, bias=False, dtype="bf16"),
        # A chunked-prefill step: prompt chunks, decode tokens and requests of
        # the base model side by side.
        dict(name="chunked_2048", kind="nslice", graph=False, tokens=2048, adapters=16, rank=16, route="requests",
             hidden=4096, q=4096, kv=1024, inter=0, layers=3, bias=False, dtype="bf16"),
        # A prompt through the store at mixed ranks.
        dict(name="store_prefill_3000", kind="store_one", graph=False, tokens=3000, adapters=24, rank=0,
             route="segments", hidden=5120, q=0, kv=0, inter=13824, layers=1, bias=False, dtype="bf16"),
        # The benchmark's prefill chunk.
        dict(name="prefill_8192", kind="qkv_o", graph=False, tokens=8192, adapters=16, rank=64, route="segments",
             hidden=4096, q=4096, kv=4096, inter=0, layers=1, bias=False, dtype="fp16"),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step`, uniform over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    """One more case of the listed ones' ranges."""
    while True:
        kind = rng.choice(("o", "qkv_o", "nslice", "nslice", "v1", "store", "store_one"))
        graph = rng.random() < 0.5
        tokens = _log(rng, 1, 1024) if graph else _log(rng, 3, 8192)
        if tokens > 3 and rng.random() < 0.5:
            tokens -= 1 - tokens % 2  # odd counts are as common as round ones
        store = kind.startswith("store")
        hidden = _log(rng, 512, 8192, 8)
        q = 0 if store else rng.choice((hidden, _log(rng, 256, 8192, 4)))
        # q feeds the o projection, whose input width is a multiple of 8.
        q -= q % 8 if kind == "qkv_o" or kind == "nslice" else 0
        kv = 0 if store or kind == "o" else rng.choice((q, max(64, q // 4 // 4 * 4)))
        case = dict(kind=kind, graph=graph, tokens=tokens, adapters=_log(rng, 1, 128),
                    rank=0 if store else rng.choice(_RANKS),
                    route=rng.choice(("zipf", "uniform", "tenants") if graph else ("segments", "requests", "zipf")),
                    hidden=hidden, q=q, kv=kv, inter=_log(rng, 1024, 14336, 8) if store else 0,
                    layers=rng.choice((1, 2, 4)), bias=kind == "v1" and rng.random() < 0.5,
                    dtype=rng.choice(("fp16", "bf16")))
        if work(case)["bytes"] <= 6e8:
            return case


# ------------------------------------------------------------------ inputs --

def _cpu(seed):
    return torch.Generator().manual_seed(int(seed) & 0x7FFFFFFF)


def _route(case, seed):
    """[tokens] int64 adapter ids (-1: the base model), on the CPU.

    zipf      every token its own request, adapter popularity 1 / rank^1.1
    uniform   every token its own request, adapters equally likely
    tenants   equal runs, one per adapter, in a random order
    segments  one run per adapter, lengths lognormal(6, 1)
    requests  half of the step in prompt chunks, half in decode tokens; one
              request in ten has no adapter
    """
    g = _cpu(seed)
    T, n = case["tokens"], case["adapters"]
    kind = case["route"]
    p = torch.arange(1, n + 1, dtype=torch.float64).pow(-1.1)

    def popular(k):
        return torch.multinomial(p, k, replacement=True, generator=g)

    if kind == "zipf":
        return popular(T)
    if kind == "uniform":
        return torch.randint(0, n, (T,), generator=g)
    order = torch.randperm(n, generator=g)
    if kind == "tenants":
        return order.repeat_interleave(-(-T // n))[:T]
    if kind == "segments":
        w = torch.exp(6.0 + torch.randn(n, generator=g, dtype=torch.float64))
        ends = (w.cumsum(0) / w.sum() * T).round().to(torch.int64)
        return torch.searchsorted(ends, torch.arange(T), right=True).clamp_(max=n - 1)[:T].apply_(lambda i: int(order[i]))
    chunks, left = [], T // 2
    while left > 0:
        k = min(left, int(torch.exp(5.0 + torch.randn((), generator=g)).item()) + 1)
        chunks.append(popular(1).expand(k) if torch.rand((), generator=g) > 0.1 else torch.full((k,), -1))
        left -= k
    tail = popular(T - T // 2)
    tail[torch.rand(tail.numel(), generator=g) < 0.1] = -1
    return torch.cat(chunks + [tail])


def _ranks(case, seed):
    if case["rank"]:
        return [case["rank"]] * case["adapters"]
    pick = torch.randint(0, 4, (case["adapters"],), generator=_cpu(seed + 7919))
    return [_RANKS[int(i)] for i in pick]


def _calls(case):
    """(input width, [slice widths], one A per slice) of each call of a layer."""
    h, q, kv, m = case["hidden"], case["q"], case["kv"], case["inter"]
    slices = [q, kv, kv] if kv else [q]
    if case["kind"] == "o":
        return [(h, [q], False)]
    if case["kind"] == "v1":
        return [(h, slices, True)]
    if case["kind"] in ("qkv_o", "nslice"):
        return [(h, slices, case["kind"] == "nslice"), (q - q % 8, [h], False)]
    return [(h, [m], False), (h, [m], False), (m, [h], False)]  # gate, up, down


_SCALE = 0.5


def _tensors(case, seed):
    """The step's routing, and for each call its x, y, weights and biases."""
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev).manual_seed(int(seed) & 0x7FFFFFFF)
    dt = _DT[case["dtype"]]

    def rn(*shape, std=1.0):
        return torch.randn(*shape, generator=g, device=dev, dtype=torch.float32).mul_(std).to(dt)

    ids = _route(case, seed)
    ranks = _ranks(case, seed)
    T, L = case["tokens"], case["adapters"]
    calls = []
    for _ in range(case["layers"]):
        for d, outs, per_slice in _calls(case):
            c = dict(d=d, outs=outs, x=rn(T, d), y=rn(T, sum(outs)), offs=[sum(outs[:i]) for i in range(len(outs))])
            if case["kind"].startswith("store"):
                c["A"] = [rn(r, d, std=0.02) for r in ranks]
                c["B"] = [rn(outs[0], r, std=0.02) for r in ranks]
            else:
                r = case["rank"]
                c["wa"] = [rn(L, 1, r, d, std=0.02) for _ in (outs if per_slice else [0])]
                c["wb"] = [rn(L, 1, o, r, std=0.02) for o in outs]
                c["bias"] = [rn(L, 1, o) for o in outs] if case["bias"] else None
            calls.append(c)
    return ids, ranks, calls


def _alpha(r):
    return 16.0 / r


# --------------------------------------------------------------- the passes --

def prepare(case, seed):
    """Weights, activations and routing on the GPU, the engine with its
    registered adapters, and (graph cases) the captured step."""
    ids, ranks, calls = _tensors(case, seed)
    dev = calls[0]["x"].device
    store = case["kind"].startswith("store")
    L = case["adapters"]
    cfg = WarpPipeConfig(layer_stride=L, max_adapter_ids=L * len(calls)) if store else WarpPipeConfig()
    engine = WarpPipeEngine(cfg)
    if store:
        engine.set_max_adapters(L * len(calls))
        for k, c in enumerate(calls):
            for i, (A, B) in enumerate(zip(c["A"], c["B"])):
                engine.register_adapter(i, A, B, _alpha(ranks[i]), rank=ranks[i], layer=k)
    if case["kind"] == "v1":
        for c in calls:
            c["h"] = torch.empty(len(c["outs"]), case["tokens"], case["rank"], dtype=torch.float32, device=dev)
    s = dict(case=case, engine=engine, ids=ids.to(dev), calls=calls, graph=None)
    if case["graph"]:
        y0 = [c["y"].clone() for c in calls]
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _step(s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            s["out"] = _step(s)
        for c, y in zip(calls, y0):
            c["y"].copy_(y)
        s["graph"] = graph
    return s


def _step(s):
    engine, case = s["engine"], s["case"]
    T, kind = case["tokens"], case["kind"]
    if not engine.build_seg_bounds(s["ids"]):
        raise RuntimeError("build_seg_bounds refused the step")
    out = []
    for k, c in enumerate(s["calls"]):
        y, x = c["y"], c["x"]
        if kind == "store":
            h = engine.shrink(x, c["d"], 0, T, layer=k)
            engine.expand(h, y, c["outs"][0], 0, layer=k)
            out += [h, y]
            continue
        if kind == "store_one":
            engine.shrink_expand(x, y, c["outs"][0], 0, layer=k)
            out.append(y)
            continue
        if kind == "v1":
            c["h"].zero_()
            ok = engine.lora_shrink(c["h"], x, c["wa"], _SCALE) and engine.lora_expand(
                y, c["h"], c["wb"], c["outs"], 0, True, c["bias"])
            out.append(c["h"])
        elif len(c["wa"]) > 1:
            ok = engine.add_lora_packed_nslice(y, x, c["wa"], c["wb"], _SCALE, c["outs"])
        elif len(c["wb"]) > 1:
            ok = engine.add_lora_slices(y, x, c["wa"][0], c["wb"], _SCALE, c["offs"])
        else:
            ok = engine.add_lora_packed(y, x, c["wa"][0], c["wb"][0], _SCALE)
        if not ok:
            raise RuntimeError("the engine has no kernel for the call")
        out.append(y)
    return out


def run(state):
    """One step: every call's y (and the H that the shrink calls return)."""
    if state["graph"] is None:
        return _step(state)
    state["graph"].replay()
    return state["out"]


def exact(case, seed):
    """What run() returns on these inputs, in 64 bits and with no rounding of
    H in between."""
    ids, ranks, calls = _tensors(case, seed)
    store = case["kind"].startswith("store")
    dev = calls[0]["x"].device
    ids = ids.to(dev)
    rows = [(i, t) for i, t in ((i, (ids == i).nonzero()[:, 0]) for i in range(case["adapters"])) if t.numel()]
    out = []
    for c in calls:
        y, n = c["y"].double(), len(c["outs"])
        width = 64 if store else case["rank"]
        h = torch.zeros(n, case["tokens"], width, dtype=torch.float64, device=dev)
        for i, t in rows:
            x = c["x"][t].double()
            for j, o in enumerate(c["outs"]):
                if store:
                    A, B, scale = c["A"][i], c["B"][i], _alpha(ranks[i])
                else:
                    A, B, scale = c["wa"][j if len(c["wa"]) > 1 else 0][i, 0], c["wb"][j][i, 0], _SCALE
                hv = scale * (x @ A.double().t().contiguous())
                h[j, t, :hv.size(1)] = hv
                d = hv @ B.double().t().contiguous()
                if not store and c["bias"] is not None:
                    d = d + c["bias"][j][i, 0].double()
                y[t, c["offs"][j]:c["offs"][j] + o] += d
        if case["kind"] == "v1":
            out.append(h)
        elif case["kind"] == "store":
            out.append(h[0])
        out.append(y)
    return out


def work(case):
    """Each call reads x, the touched adapters' A and B, and y, and writes y;
    calls that hand H over write and read it."""
    ids, ranks = _route(case, 0), _ranks(case, 0)
    T, kind = case["tokens"], case["kind"]
    count = torch.bincount(ids[ids >= 0], minlength=case["adapters"]).tolist()
    touched = sum(r for r, k in zip(ranks, count) if k)  # rank rows of the touched adapters
    rows = sum(r * k for r, k in zip(ranks, count))      # rank rows over all tokens
    routed = sum(count)
    nbytes = flops = 0
    for d, outs, per_slice in _calls(case):
        o, n_a = sum(outs), len(outs) if per_slice else 1
        nbytes += 2 * routed * d + 4 * routed * o + 2 * touched * (d * n_a + o)
        flops += 2 * rows * (d * n_a + o)
        if kind == "v1":
            nbytes += 2 * 4 * rows * len(outs)
        elif kind == "store":
            nbytes += 2 * 2 * rows
    return {"bytes": case["layers"] * nbytes + 8 * T, "flops": case["layers"] * flops}


def tolerance(case):
    """y and H are rounded to the activations' type; that rounding is the error
    seen against 64 bits (bf16 1.7e-3, fp16 2.2e-4), and the largest single
    difference is one or two steps of the type."""
    return {"rel": 7e-3, "max": 0.03} if case["dtype"] == "bf16" else {"rel": 9e-4, "max": 4e-3}

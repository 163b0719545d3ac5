"""The measured cases of this framework: what a streaming TTS engine built on it has the GPU do, call by call.

The engine's slow stack has 14 query / 2 KV heads of 64 dims, 24 layers and a KV cache of up to 2048 (here also
4096) positions per slot; a tick serves 1 to 192 slots. Its fast stack runs a two-token pass and then one-token
passes over a 10-position cache. An admission copies a voice's prefix K/V into its slots and runs a packed causal
prefill. A frame of the vocoder is 4 rows per slot through a channels-last convolution decoder. Widths the
checkpoint would give are the benchmark's: hidden 896, MLP 4864, a decoder of 1024 -> 1536 channels with strides
8, 8, 4, 2.

The engine captures its tick, its fast-AR passes and its vocoder frame as HIP graphs at start-up and replays them,
with inputs written into fixed buffers; a case of those kinds captures in prepare() and replays in run(). An
admission has other sizes each time: its cases call the operators eagerly. Lengths are spread evenly over their
range and given to the slots in an order drawn from the seed, so a case's work does not depend on the seed.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import __graft_entry__  # noqa: E402

BF16, F16, I32 = torch.bfloat16, torch.float16, torch.int32
NQ, NKV, HD = 14, 2, 64
W = (NQ + 2 * NKV) * HD
HIDDEN, INTER = 896, 4864
EPS = 1e-6
BASE = 10000.0


def _a8():
    __graft_entry__.ensure_built()
    return __graft_entry__.load_package()


def _module(name):
    import importlib
    return importlib.import_module(_a8().__name__ + "." + name)


def listed():
    return [
        # One caller alone: the attention of 24 layers for one row, a fresh conversation (385 keys). Every launch is
        # latency.
        {"name": "attend_1", "kind": "attend", "slots": 1, "cache": 512, "shortest": 385, "longest": 385, "layers": 24},
        # An ordinary load: 64 slots at whatever lengths their utterances have reached, in a 4096-position cache.
        {"name": "attend_64_ragged", "kind": "attend", "slots": 64, "cache": 4096, "shortest": 128, "longest": 2048,
         "layers": 24},
        # The peak load as it occurs: 192 slots, each somewhere in its utterance after a 300-position voice prefix.
        {"name": "attend_192_ragged", "kind": "attend", "slots": 192, "cache": 2048, "shortest": 300, "longest": 2048,
         "layers": 8},
        # The peak load at its worst: every one of 192 slots at 2048 keys.
        {"name": "attend_192_full", "kind": "attend", "slots": 192, "cache": 2048, "shortest": 2048, "longest": 2048,
         "layers": 8},
        # The fast AR of a peak-load tick: a two-token pass, then 8 one-token passes, 4 layers each.
        {"name": "fast_ar_192", "kind": "fast_ar", "slots": 192, "passes": 9, "layers": 4},
        # The attention of a full admission: 64 requests of 40 to 400 text tokens after a 300-position voice prefix.
        {"name": "prefill_64", "kind": "prefill", "requests": 64, "shortest": 40, "longest": 400, "prefix": 300,
         "layers": 4},
        # The same admission's voice prefixes: 4 voices into 16 slots each, all 24 layers' K and V.
        {"name": "prefix_copy_64", "kind": "prefix_copy", "slots": 64, "voices": 4, "prefix": 300, "cache": 704,
         "layers": 24},
        # The slow AR's decode step (attention, projections, norms, MLP), some layers of it, at a small load ...
        {"name": "slow_step_16", "kind": "slow_step", "slots": 16, "cache": 2048, "shortest": 300, "longest": 1400,
         "layers": 8},
        # ... and at the peak load.
        {"name": "slow_step_192", "kind": "slow_step", "slots": 192, "cache": 2048, "shortest": 2048, "longest": 2048,
         "layers": 4},
        # The slow AR's layers over an ordinary admission of 16 requests.
        {"name": "slow_prefill_16", "kind": "slow_prefill", "requests": 16, "shortest": 40, "longest": 400,
         "prefix": 300, "layers": 2},
        # A vocoder frame for a few callers, where the first audio's delay counts, ...
        {"name": "vocoder_8", "kind": "vocoder", "rows": 8, "frame": 4},
        # ... and for the peak load.
        {"name": "vocoder_192", "kind": "vocoder", "rows": 192, "frame": 4},
    ]


def _between(rng, lo, hi):
    """A whole number spread over [lo, hi] in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["attend", "attend", "attend", "fast_ar", "prefill", "prefix_copy", "slow_step", "slow_step",
                       "slow_prefill", "vocoder"])
    if kind in ("attend", "slow_step"):
        cache = rng.choice([512, 1024, 2048, 4096]) if kind == "attend" else rng.choice([1024, 2048])
        slots = _between(rng, 1, 192 if cache <= 2048 else 96)
        longest = _between(rng, 96, min(cache, 2048))
        shortest = rng.choice([longest, rng.randint(min(64, longest), longest)])
        return {"kind": kind, "slots": slots, "cache": cache, "shortest": shortest, "longest": longest,
                "layers": (24 if slots <= 64 else 8) if kind == "attend" else rng.choice([2, 3, 4])}
    if kind == "fast_ar":
        return {"kind": kind, "slots": _between(rng, 1, 192), "passes": rng.randint(4, 9), "layers": rng.choice([2, 4])}
    if kind in ("prefill", "slow_prefill"):
        shortest = rng.randint(20, 120)
        return {"kind": kind, "requests": _between(rng, 1, 64 if kind == "prefill" else 24), "shortest": shortest,
                "longest": rng.randint(shortest, 400), "prefix": rng.choice([0, rng.randint(100, 300), 300]),
                "layers": rng.choice([2, 4]) if kind == "prefill" else rng.choice([1, 2])}
    if kind == "prefix_copy":
        voices = rng.randint(1, 4)
        return {"kind": kind, "slots": voices * _between(rng, 1, 16), "voices": voices,
                "prefix": rng.randint(100, 300), "cache": rng.choice([704, 1024]), "layers": 24}
    frame = rng.choice([4, 4, 4, 8])
    return {"kind": kind, "rows": _between(rng, 1, 704 // frame), "frame": frame}


# ---------------------------------------------------------------- inputs

def _spread(count, lo, hi):
    """`count` whole numbers evenly spread over [lo, hi]."""
    return [lo + (hi - lo) * i // max(1, count - 1) if count > 1 else (lo + hi + 1) // 2 for i in range(count)]


def _lengths(count, lo, hi, seed):
    v = _spread(count, lo, hi)
    order = torch.randperm(count, generator=torch.Generator().manual_seed(int(seed) * 7919 + 11)).tolist()
    return [v[i] for i in order]


class _Draws:
    """Seeded inputs on the GPU: activations ~ N(0, 1), biases ~ N(0, 0.02^2), projections ~ N(0, 1 / fan-in)."""

    def __init__(self, seed):
        self.dev = torch.device("cuda:0")
        self.g = torch.Generator(device=self.dev).manual_seed(int(seed))

    def randn(self, *shape, std=1.0, mean=0.0, dt=BF16):
        return (torch.randn(*shape, generator=self.g, device=self.dev) * std + mean).to(dt)

    def fill(self, t):
        t.normal_(generator=self.g)

    def ints(self, values):
        return torch.tensor(values, dtype=I32, device=self.dev)


def _capture(fn):
    """The engine's capture: two warm-up calls on a side stream, then one graph."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()
        fn()
    torch.cuda.current_stream().wait_stream(s)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn()
    return g


def _slow_weights(d, layers):
    def lin(n, k):
        return d.randn(n, k, std=k ** -0.5)

    return [dict(wqkv=lin(W, HIDDEN), bqkv=d.randn(W, std=0.02), wo=lin(HIDDEN, NQ * HD), w13=lin(2 * INTER, HIDDEN),
                 w2=lin(HIDDEN, INTER), ln1=d.randn(HIDDEN, std=0.05, mean=1.0),
                 ln2=d.randn(HIDDEN, std=0.05, mean=1.0)) for _ in range(layers)], d.randn(HIDDEN, std=0.05, mean=1.0)


_tuned = {}  # row count -> the GEMM dispatch a program tunes once, at its start


def _dispatch(weights, rows):
    if rows not in _tuned:
        mm = _a8().GemmDispatch()
        mm.tune([L[k] for L in weights for k in ("wqkv", "wo", "w13", "w2")], [rows], gated=[L["w13"] for L in weights],
                large_m=0)
        _tuned[rows] = mm
    return _tuned[rows]


VOC_IN, VOC_CH, VOC_RATES, VOC_K, VOC_DILS = 1024, 1536, (8, 8, 4, 2), 7, (1, 3, 9)


def _voc_weights(d):
    """The decoder's weights in their modules' layouts (Conv1d [out, in, k], ConvTranspose1d [in, out, 2 stride]).
    Gains below one in the units' second convs and the transposed convs keep the activations of order one through
    the whole decoder, as a trained decoder's are (at unit gain they grow by 3 a block, and the snakes' sines of
    large fp16 arguments would turn the waveform into noise)."""
    def conv(co, ci, k, gain=1.0):
        return (d.randn(co, ci, k, std=gain * (ci * k) ** -0.5, dt=torch.float32),
                d.randn(co, std=0.02, dt=torch.float32))

    def alpha(c):
        return 0.5 + torch.rand(c, generator=d.g, device=d.dev)

    w = {"conv_in": conv(VOC_CH, VOC_IN, VOC_K), "blocks": []}
    c = VOC_CH
    for s in VOC_RATES:
        tw = d.randn(c, c // 2, 2 * s, std=0.6 * (2 * c) ** -0.5, dt=torch.float32)
        tb = d.randn(c // 2, std=0.02, dt=torch.float32)
        a0 = alpha(c)
        c //= 2
        units = []
        for dil in VOC_DILS:
            w1, b1 = conv(c, c, VOC_K)
            w2, b2 = conv(c, c, 1, 0.3)
            units.append((alpha(c), w1, b1, dil, alpha(c), w2, b2))
        w["blocks"].append((a0, tw, tb, s, units))
    wf, bf = conv(1, c, VOC_K, 0.3)
    w["final"] = (alpha(c), wf, bf)
    return w


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def _prepare_attend(case, seed):
    a8, d, b, S, n = _a8(), _Draws(seed), case["slots"], case["cache"], case["layers"]
    lens_h = _lengths(b, case["shortest"], case["longest"], seed)
    st = a8.AttnStack(n, NQ, NKV, HD, BASE, max_rows=max(16 * b, 8192), cache_rows=b + 1, cache_len=S, max_pos=S,
                      dev=d.dev)
    d.fill(st.kc_all)
    d.fill(st.vc_all)
    lens, slot = d.ints(lens_h), torch.arange(b, dtype=I32, device=d.dev)
    pos = lens - 1
    qkv = [d.randn(b, W) for _ in range(n)]
    bias = [d.randn(W, std=0.02) for _ in range(n)]
    q = torch.empty(b, NQ, HD, dtype=BF16, device=d.dev)
    outs = [torch.empty(b, NQ, HD, dtype=BF16, device=d.dev) for _ in range(n)]
    nsplit = a8.ref_nsplit(b, NKV)
    g = _capture(lambda: st.forward(qkv, bias, pos, slot, lens, nsplit=nsplit, rowmap=False, q=q, outs=outs, fuse=True))
    return {"graph": g, "out": (outs, st.kc_all, st.vc_all), "keep": (st, lens, pos, slot, qkv, bias, q),
            "lens_h": lens_h}


def _fast_passes(d, b, passes):
    r = list(range(2 * b))
    got = [(d.ints([i % 2 for i in r]), d.ints([i // 2 for i in r]), d.ints([i % 2 + 1 for i in r]), True, 2 * b)]
    ar = torch.arange(b, dtype=I32, device=d.dev)
    for p in range(2, passes + 1):
        got.append((torch.full((b,), p, dtype=I32, device=d.dev), ar,
                    torch.full((b,), p + 1, dtype=I32, device=d.dev), False, b))
    return got


def _prepare_fast_ar(case, seed):
    a8, d, b, n = _a8(), _Draws(seed), case["slots"], case["layers"]
    st = a8.AttnStack(n, NQ, NKV, HD, BASE, max_rows=max(2 * b, 16), cache_rows=b, cache_len=case["passes"] + 1,
                      max_pos=16, dev=d.dev, nsplit_max=1)
    passes = _fast_passes(d, b, case["passes"])
    qkvs = [[d.randn(nr, W) for _ in range(n)] for (_, _, _, _, nr) in passes]
    bias = [d.randn(W, std=0.02) for _ in range(n)]
    q = torch.empty(2 * b, NQ, HD, dtype=BF16, device=d.dev)
    outs = [[torch.empty(nr, NQ, HD, dtype=BF16, device=d.dev) for _ in range(n)] for (_, _, _, _, nr) in passes]

    def all_passes():
        for (pos, slot, lens, rmap, nr), qkv, o in zip(passes, qkvs, outs):
            st.forward(qkv, bias, pos, slot, lens, nsplit=1, rowmap=rmap, q=q[:nr], outs=o, fuse=not rmap)

    g = _capture(all_passes)
    return {"graph": g, "out": (outs, st.kc_all, st.vc_all), "keep": (st, passes, qkvs, bias, q)}


def _packed(d, case, seed):
    """(token counts, rows, positions, slots) of an admission packed in request order."""
    ns = _lengths(case["requests"], case["shortest"], case["longest"], seed)
    pos = d.ints([case["prefix"] + j for n in ns for j in range(n)])
    slot = d.ints([i for i, n in enumerate(ns) for _ in range(n)])
    return ns, sum(ns), pos, slot


def _plan(a8, ns, case, dev):
    r0s = [sum(ns[:i]) for i in range(len(ns))]
    return a8.PrefillPlan(r0s, ns, list(range(len(ns))), [case["prefix"]] * len(ns), dev)


def _prepare_prefill(case, seed):
    a8, d, n = _a8(), _Draws(seed), case["layers"]
    ns, R, pos, slot = _packed(d, case, seed)
    S = 704
    st = a8.AttnStack(n, NQ, NKV, HD, BASE, max_rows=8192, cache_rows=len(ns) + 1, cache_len=S, max_pos=S, dev=d.dev)
    d.fill(st.kc_all)
    d.fill(st.vc_all)
    return {"call": "prefill", "st": st, "plan": _plan(a8, ns, case, d.dev), "pos": pos, "slot": slot,
            "qkv": [d.randn(R, W) for _ in range(n)], "bias": [d.randn(W, std=0.02) for _ in range(n)],
            "q": torch.empty(R, NQ, HD, dtype=BF16, device=d.dev),
            "outs": [torch.empty(R, NQ, HD, dtype=BF16, device=d.dev) for _ in range(n)], "ns": ns}


def _prepare_prefix_copy(case, seed):
    a8, d, n, v, p = _a8(), _Draws(seed), case["layers"], case["voices"], case["prefix"]
    kc = torch.zeros(n, case["slots"] + 1, NKV, case["cache"], HD, dtype=BF16, device=d.dev)
    vc = torch.zeros_like(kc)
    order = torch.randperm(case["slots"], generator=torch.Generator().manual_seed(int(seed))).tolist()
    each = case["slots"] // v
    return {"call": "prefix_copy", "a8": a8, "kc": kc, "vc": vc,
            "k": [d.randn(n, NKV, p, HD) for _ in range(v)], "v": [d.randn(n, NKV, p, HD) for _ in range(v)],
            "slots": [d.ints(sorted(order[j * each:(j + 1) * each])) for j in range(v)]}


def _slow_stack(case, seed, cache_rows, S, rows):
    a8, d, n = _a8(), _Draws(seed), case["layers"]
    layers, norm = _slow_weights(d, n)
    st = a8.SlowStack(layers, norm, NQ, NKV, HD, EPS, BASE, max_rows=max(16 * cache_rows, 8192), cache_rows=cache_rows,
                      cache_len=S, max_pos=S, dev=d.dev, mm=_dispatch(layers, rows))
    st.fuse_norm = True
    d.fill(st.kc_all)
    d.fill(st.vc_all)
    embed = d.randn(4096, HIDDEN)
    return a8, d, st, layers, norm, embed


def _prepare_slow_step(case, seed):
    b, S = case["slots"], case["cache"]
    a8, d, st, layers, norm, embed = _slow_stack(case, seed, b + 1, S, b)
    lens_h = _lengths(b, case["shortest"], case["longest"], seed)
    lens, slot = d.ints(lens_h), torch.arange(b, dtype=I32, device=d.dev)
    pos = lens - 1
    tokens = torch.randint(0, embed.shape[0], (b,), generator=d.g, device=d.dev)
    nsplit = a8.ref_nsplit(b, NKV)
    x = torch.empty(b, HIDDEN, dtype=BF16, device=d.dev)
    hold = {}

    def step():
        torch.index_select(embed, 0, tokens, out=x)
        hold["h"] = st.forward(x, pos, slot, lens, nsplit=nsplit, rowmap=False, fuse=True)

    g = _capture(step)
    return {"graph": g, "out": (hold["h"], st.kc_all, st.vc_all), "keep": (st, lens, pos, slot, x, hold),
            "weights": (layers, norm), "embed": embed, "tokens": tokens, "lens_h": lens_h}


def _prepare_slow_prefill(case, seed):
    S = 704
    ns = _lengths(case["requests"], case["shortest"], case["longest"], seed)
    a8, d, st, layers, norm, embed = _slow_stack(case, seed, len(ns) + 1, S, sum(ns))
    ns, R, pos, slot = _packed(d, case, seed)
    tokens = torch.randint(0, embed.shape[0], (R,), generator=d.g, device=d.dev)
    return {"call": "slow_prefill", "st": st, "plan": _plan(a8, ns, case, d.dev), "pos": pos, "slot": slot,
            "weights": (layers, norm), "embed": embed, "tokens": tokens, "ns": ns}


def _prepare_vocoder(case, seed):
    voc, d, b, T = _module("vocoder"), _Draws(seed), case["rows"], case["frame"]
    wts = _voc_weights(d)
    dec = voc.CLDecoder(wts, b, d.dev, frame=T, fused_ru=voc.FusedRU.DEFAULT_WIDTHS)
    x = d.randn(b, T, VOC_IN, dt=F16)
    # where the rows' streams stand: every conv's activated context
    saved = [d.randn(*s.shape, dt=F16) for s in dec.states]
    hold = {}

    def frame():
        torch._foreach_copy_(dec.states, saved)  # the engine restores its rows' snapshot before a frame
        hold["wav"] = dec(x, b)

    g = _capture(frame)
    return {"graph": g, "out": (hold["wav"], dec.states), "keep": (dec, hold), "x": x, "saved": saved, "wts": wts}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    s = state
    if s["call"] == "prefill":
        s["st"].forward(s["qkv"], s["bias"], s["pos"], s["slot"], None, plan=s["plan"], q=s["q"], outs=s["outs"],
                        fuse=True)
        return s["outs"], s["st"].kc_all, s["st"].vc_all
    if s["call"] == "prefix_copy":
        for k, v, slots in zip(s["k"], s["v"], s["slots"]):
            s["a8"].prefix_copy(k, v, s["kc"], s["vc"], slots)
        return s["kc"], s["vc"]
    x = s["embed"].index_select(0, s["tokens"])
    h = s["st"].forward(x, s["pos"], s["slot"], None, plan=s["plan"], fuse=True)
    return h, s["st"].kc_all, s["st"].vc_all


# ---------------------------------------------------------------- work

def _store_bytes(rows):
    """qkv rows, one bias, positions, slots, lengths and the cos / sin rows in; one key and value out."""
    return rows * (W * 2 + 12 + 2 * HD * 2 + 2 * NKV * HD * 2) + W * 2


def _attend_work(lens):
    keys = sum(lens)
    return (keys * 2 * NKV * HD * 2 + len(lens) * NQ * HD * 2 + _store_bytes(len(lens)), 4 * NQ * HD * keys)


def _prefill_work(ns, prefix):
    rows = sum(ns)
    pairs = sum(n * prefix + n * (n + 1) // 2 for n in ns)
    return (len(ns) * prefix * 2 * NKV * HD * 2 + rows * NQ * HD * 2 + _store_bytes(rows), 4 * NQ * HD * pairs)


_LAYER = W * HIDDEN + HIDDEN * NQ * HD + 3 * INTER * HIDDEN  # weights of a slow layer's products


def work(case):
    kind, n = case["kind"], case.get("layers", 1)
    if kind in ("attend", "slow_step"):
        lens = _spread(case["slots"], case["shortest"], case["longest"])
        by, fl = _attend_work(lens)
    elif kind == "fast_ar":
        b = case["slots"]
        by = fl = 0
        for lens in [[1, 2] * b] + [[p + 1] * b for p in range(2, case["passes"] + 1)]:
            x, y = _attend_work(lens)
            by, fl = by + x, fl + y
    elif kind in ("prefill", "slow_prefill"):
        ns = _spread(case["requests"], case["shortest"], case["longest"])
        by, fl = _prefill_work(ns, case["prefix"])
    elif kind == "prefix_copy":
        return {"bytes": 2 * n * NKV * case["prefix"] * HD * 2 * (case["slots"] + case["voices"]), "flops": 0}
    else:
        return _vocoder_work(case["rows"], case["frame"])
    if kind.startswith("slow"):
        rows = case["slots"] if kind == "slow_step" else sum(_spread(case["requests"], case["shortest"], case["longest"]))
        # of the activations only the step's own input and output have to touch memory; the attention's part keeps
        # its cache bytes
        by = by - rows * (W + NQ * HD) * 2 + 2 * _LAYER
        fl += 2 * rows * _LAYER
        return {"bytes": n * by + 2 * rows * HIDDEN * 2, "flops": n * fl}
    return {"bytes": n * by, "flops": n * fl}


def _vocoder_work(b, T):
    t, c = T, VOC_CH
    weights, states = VOC_CH * VOC_IN * VOC_K, (VOC_K - 1) * VOC_IN
    flops = 2 * b * t * VOC_CH * VOC_IN * VOC_K
    for s in VOC_RATES:
        states += c
        weights += c * (c // 2) * 2 * s
        flops += 2 * b * t * s * (c // 2) * 2 * c
        t, c = t * s, c // 2
        weights += len(VOC_DILS) * c * c * (VOC_K + 1)
        states += sum((VOC_K - 1) * d * c for d in VOC_DILS)
        flops += len(VOC_DILS) * 2 * b * t * c * c * (VOC_K + 1)
    weights += c * VOC_K
    states += (VOC_K - 1) * c
    flops += 2 * b * t * c * VOC_K
    return {"bytes": 2 * (weights + 2 * b * states + b * T * VOC_IN) + 4 * b * t, "flops": flops}


def tolerance(case):
    # About four times what each path is off 64-bit arithmetic on the same inputs: attention 0.003 (prefill 0.004:
    # q and the weights in bf16), the slow stack's layers 0.006 to 0.012, the vocoder 0.0014.
    return {"attend": {"rel": 0.012, "max": 0.1}, "fast_ar": {"rel": 0.012, "max": 0.1},
            "prefill": {"rel": 0.016, "max": 0.2}, "prefix_copy": "exact",
            "slow_step": {"rel": 0.03, "max": 0.4}, "slow_prefill": {"rel": 0.025, "max": 0.3},
            "vocoder": {"rel": 0.006, "max": 0.1}}[case["kind"]]


# ---------------------------------------------------------------- 64-bit results

def _tables(S, dev):
    """The engine's RoPE tables: fp32 phases, rounded to bf16 (they are part of the definition)."""
    fr = 1.0 / (BASE ** (torch.arange(0, HD, 2).float() / HD))
    ph = torch.outer(torch.arange(S).float(), fr)
    c, s = ph.cos().to(BF16).double(), ph.sin().to(BF16).double()
    return torch.cat([c, c], -1).to(dev), torch.cat([s, s], -1).to(dev)


def _rope(x, cos, sin):
    half = HD // 2
    return x * cos[:, None] + torch.cat([-x[..., half:], x[..., :half]], -1) * sin[:, None]


def _split_qkv(qkv, bias, pos, cos, sin):
    x = (qkv.double() + bias.double()).view(-1, NQ + 2 * NKV, HD)
    c, s = cos[pos.long()], sin[pos.long()]
    return _rope(x[:, :NQ], c, s), _rope(x[:, NQ:NQ + NKV], c, s), x[:, NQ + NKV:]


def _softmax_rows(q, kc, vc, visible):
    """q [r, NQ, HD] over keys kc / vc [NKV, n, HD], visible [r, n] (or None) -> [r, NQ, HD]."""
    r, n = q.shape[0], kc.shape[1]
    g = NQ // NKV
    out = torch.empty_like(q)
    for h in range(NKV):
        s = (q[:, h * g:(h + 1) * g].reshape(r * g, HD) @ kc[h].t()) * HD ** -0.5
        if visible is not None:
            s = s.view(r, g, n).masked_fill(~visible[:, None], float("-inf")).view(r * g, n)
        out[:, h * g:(h + 1) * g] = (torch.softmax(s, -1) @ vc[h]).view(r, g, HD)
    return out


def _decode_layer(q, kc, vc, rows, lens):
    return torch.cat([_softmax_rows(q[i:i + 1], kc[r, :, :n], vc[r, :, :n], None)
                      for i, (r, n) in enumerate(zip(rows, lens))])


def _prefill_layer(q, kc, vc, ns, prefix):
    out, r0 = [], 0
    for i, n in enumerate(ns):
        key = torch.arange(prefix + n, device=q.device)
        row = prefix + torch.arange(n, device=q.device)
        out.append(_softmax_rows(q[r0:r0 + n], kc[i, :, :prefix + n], vc[i, :, :prefix + n], key[None] <= row[:, None]))
        r0 += n
    return torch.cat(out)


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _slow_layers(x, weights, attend):
    """The slow AR's layers in 64 bits; attend(i, qkv) -> the layer's attention rows."""
    layers, norm = weights
    for i, L in enumerate(layers):
        qkv = _norm(x, L["ln1"]) @ L["wqkv"].double().t()
        x = x + attend(i, qkv).reshape(x.shape[0], -1) @ L["wo"].double().t()
        gu = _norm(x, L["ln2"]) @ L["w13"].double().t()
        x = x + (torch.nn.functional.silu(gu[:, :INTER]) * gu[:, INTER:]) @ L["w2"].double().t()
    return _norm(x, norm)


def exact(case, seed):
    if case["kind"] == "prefix_copy":
        s = prepare(case, seed)
        kc, vc = s["kc"].double(), s["vc"].double()
        for k, v, slots in zip(s["k"], s["v"], s["slots"]):
            kc[:, slots.long(), :, :k.shape[2]] = k.double().unsqueeze(1)
            vc[:, slots.long(), :, :k.shape[2]] = v.double().unsqueeze(1)
        return kc, vc
    return globals()["_exact_" + case["kind"]](case, prepare(case, seed))


def _exact_attend(case, s):
    st, lens, pos, slot, qkv, bias, _ = s["keep"]
    cos, sin = _tables(case["cache"], pos.device)
    kd, vd = st.kc_all.double(), st.vc_all.double()
    outs = []
    for i in range(case["layers"]):
        q, k, v = _split_qkv(qkv[i], bias[i], pos, cos, sin)
        kd[i][slot.long(), :, pos.long()], vd[i][slot.long(), :, pos.long()] = k, v
        outs.append(_decode_layer(q, kd[i], vd[i], range(case["slots"]), s["lens_h"]))
    return outs, kd, vd


def _exact_fast_ar(case, s):
    st, passes, qkvs, bias, _ = s["keep"]
    cos, sin = _tables(16, st.kc_all.device)
    kd, vd = st.kc_all.double(), st.vc_all.double()
    outs = []
    for (pos, slot, lens, _, nr), qkv in zip(passes, qkvs):
        got = []
        for i in range(case["layers"]):
            q, k, v = _split_qkv(qkv[i], bias[i], pos, cos, sin)
            kd[i][slot.long(), :, pos.long()], vd[i][slot.long(), :, pos.long()] = k, v
            got.append(_decode_layer(q, kd[i], vd[i], slot.tolist(), lens.tolist()))
        outs.append(got)
    return outs, kd, vd


def _exact_prefill(case, s):
    st, pos, slot = s["st"], s["pos"], s["slot"]
    cos, sin = _tables(704, pos.device)
    kd, vd = st.kc_all.double(), st.vc_all.double()
    outs = []
    for i in range(case["layers"]):
        q, k, v = _split_qkv(s["qkv"][i], s["bias"][i], pos, cos, sin)
        kd[i][slot.long(), :, pos.long()], vd[i][slot.long(), :, pos.long()] = k, v
        outs.append(_prefill_layer(q, kd[i], vd[i], s["ns"], case["prefix"]))
    return outs, kd, vd


def _exact_slow_step(case, s):
    st, lens, pos, slot = s["keep"][:4]
    cos, sin = _tables(case["cache"], pos.device)
    kd, vd = st.kc_all.double(), st.vc_all.double()

    def attend(i, qkv):
        q, k, v = _split_qkv(qkv, s["weights"][0][i]["bqkv"], pos, cos, sin)
        kd[i][slot.long(), :, pos.long()], vd[i][slot.long(), :, pos.long()] = k, v
        return _decode_layer(q, kd[i], vd[i], range(case["slots"]), s["lens_h"])

    return _slow_layers(s["embed"][s["tokens"]].double(), s["weights"], attend), kd, vd


def _exact_slow_prefill(case, s):
    st, pos, slot = s["st"], s["pos"], s["slot"]
    cos, sin = _tables(704, pos.device)
    kd, vd = st.kc_all.double(), st.vc_all.double()

    def attend(i, qkv):
        q, k, v = _split_qkv(qkv, s["weights"][0][i]["bqkv"], pos, cos, sin)
        kd[i][slot.long(), :, pos.long()], vd[i][slot.long(), :, pos.long()] = k, v
        return _prefill_layer(q, kd[i], vd[i], s["ns"], case["prefix"])

    return _slow_layers(s["embed"][s["tokens"]].double(), s["weights"], attend), kd, vd


def _exact_vocoder(case, s):
    """The decoder on its modules' weights as the kernels hold them (fp16), everything else in 64 bits."""
    w, saved, states = s["wts"], iter(s["saved"]), []

    def f16(t):
        return t.to(F16).double()

    def snake(x, alpha):
        a = alpha.double()
        return x + torch.sin(a * x).square() / (a + 1e-9)

    def conv(x, wt, b, dil=1, alpha=None):
        x = snake(x, alpha) if alpha is not None else x
        ctx = (wt.shape[2] - 1) * dil
        if ctx:
            x = torch.cat([next(saved).double(), x], 1)
            states.append(x[:, -ctx:])
        n = x.shape[1] - ctx
        return sum(x[:, j * dil:j * dil + n] @ f16(wt[:, :, j]).t() for j in range(wt.shape[2])) + f16(b)

    def up(x, wt, b, stride, alpha):
        x = torch.cat([next(saved).double(), snake(x, alpha)], 1)
        states.append(x[:, -1:])
        cur, prev = x[:, 1:], x[:, :-1]
        ph = [prev @ f16(wt[:, :, p + stride]) + cur @ f16(wt[:, :, p]) + f16(b) for p in range(stride)]
        return torch.stack(ph, 2).flatten(1, 2)

    x = conv(s["x"].double(), *w["conv_in"])
    for a0, tw, tb, stride, units in w["blocks"]:
        x = up(x, tw, tb, stride, a0)
        for a1, w1, b1, dil, a2, w2, b2 in units:
            x = x + conv(conv(x, w1, b1, dil, a1), w2, b2, 1, a2)
    af, wf, bf = w["final"]
    return torch.tanh(conv(x, wf, bf, 1, af))[..., 0], states

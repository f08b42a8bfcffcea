"""Timed cases of the MoE decode and prefill path and of the two lm_heads, through the package's
public entry points, with a float64 restatement of each.

A case is a dict of plain values; its "kind" says which entry point it runs:

  layer      LruMoELayer.apply: one MoE layer over `tokens` rows. Up to GRAPH_TOKENS rows the
             step is recorded once into a HIP graph and replayed, as a serving loop runs decode;
             above, it is called eagerly, as a prefill chunk is. `slots` = `experts` keeps every
             expert resident; fewer slots with `misses` false is the static arm (experts
             without a slot are read from the full tensor in HBM); with `misses` true the full
             tensor is pinned host memory and the step caches its misses from there.
  lru        LruCache.fused of LRU_LAYERS layers of one step (manager and both aligns), one
             graph, fed the next step of a routing trace on every pass.
  head_fp8   ops.gemm_fp8_block: the fp8 target head over `rows` hidden states.
  head_w4    w4.gemm_w4a16: the int4 draft head over `rows` hidden states.

    listed()  the cases           draw(rng)  one more of the same ranges
    prepare / run / work / tolerance / exact  of one case
"""
from __future__ import annotations

import importlib.util
import pathlib
import sys

import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent
PKG_NAME = "r9700_lru_expert_cache_amd"
DEV = "cuda"
GRAPH_TOKENS = 256
LRU_LAYERS = 8
TRACE_STEPS = 32          # routing steps a trace holds before it starts over
ZIPF = 1.1                # routing skew of the benchmark's traces
CHUNK = 32                # experts made at a time
VOCAB = 151936


def _pkg():
    if PKG_NAME in sys.modules:
        return sys.modules[PKG_NAME]
    d = ROOT / "r9700-lru-expert-cache_amd"
    spec = importlib.util.spec_from_file_location(PKG_NAME, d / "__init__.py",
                                                  submodule_search_locations=[str(d)])
    mod = importlib.util.module_from_spec(spec)
    sys.modules[PKG_NAME] = mod
    spec.loader.exec_module(mod)
    return mod


# ---- the cases ----------------------------------------------------------------------------------
# the benchmark's expert shape, and shapes of other common MoE layers
MAIN = dict(experts=512, top_k=10, hidden=2560, inter=768)
OTHER = [dict(experts=128, top_k=8, hidden=2048, inter=768),
         dict(experts=64, top_k=8, hidden=2048, inter=1024),
         dict(experts=64, top_k=6, hidden=2048, inter=1408),
         dict(experts=256, top_k=8, hidden=1536, inter=512)]


def _layer(name, tokens, shape, slots=None, corr=0.0, misses=False):
    c = dict(kind="layer", tokens=tokens, **shape, slots=slots or shape["experts"], corr=corr,
             misses=misses)
    return dict(c, name=name) if name else c


def _head(name, kind, rows, vocab=VOCAB, hidden=2560):
    c = dict(kind=kind, rows=rows, vocab=vocab, hidden=hidden)
    return dict(c, name=name) if name else c


def _lru(name, tokens, experts=512, slots=257, top_k=10, corr=0.7):
    c = dict(kind="lru", tokens=tokens, experts=experts, slots=slots, top_k=top_k, corr=corr)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the cache's bookkeeping of a 4-stream step with 5 rows each: 20 tokens, a few misses
        _lru("lru_20", 20),
        # one stream, 5 rows (the token and its drafts): the smallest step of a layer
        _layer("decode_5", 5, MAIN),
        # 4 streams: the ordinary decode step, rows of a step routed alike
        _layer("decode_20", 20, MAIN, corr=0.7),
        # 16 streams: most experts are routed, an expert has one or two rows
        _layer("decode_80", 80, MAIN),
        # the same decode step where the cache is too small and experts come from host memory
        _layer("decode_20_miss", 20, OTHER[0], slots=64, corr=0.7, misses=True),
        # a short ragged prompt
        _layer("prefill_617", 617, MAIN),
        # an ordinary prefill chunk over half the experts resident, the rest read through
        _layer("prefill_4096_half", 4096, MAIN, slots=257),
        # the largest chunk
        _layer("prefill_8192", 8192, MAIN),
        # a chunk of a model with another expert shape
        _layer("prefill_2048_h2048", 2048, OTHER[0]),
        # the target head over one 4-stream verification step
        _head("head_fp8_20", "head_fp8", 20),
        # the draft head, one row for each of 4 streams
        _head("head_w4_4", "head_w4", 4),
        # the draft head at its largest batch
        _head("head_w4_64", "head_w4", 64),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    kind = rng.choice(["layer"] * 6 + ["head_fp8", "head_fp8", "head_w4", "head_w4", "lru"])
    if kind == "layer":
        shape = MAIN if rng.random() < 0.5 else rng.choice(OTHER)
        tokens = _log_int(rng, 1, 8192 if shape is MAIN else 4096)
        slots = shape["experts"] if rng.random() < 0.6 else shape["experts"] // 2 + 1
        corr = rng.choice([0.0, 0.7]) if tokens <= GRAPH_TOKENS else 0.0
        misses = (shape is not MAIN and slots < shape["experts"] and tokens <= 64 and
                  rng.random() < 0.5)
        return _layer(None, tokens, shape, slots=slots, corr=corr, misses=misses)
    if kind == "lru":
        return _lru(None, _log_int(rng, 1, 4096), slots=rng.randint(64, 512),
                    corr=rng.choice([0.0, 0.7]))
    hidden = rng.choice([1536, 2048, 2560, 3072, 4096])
    vocab = rng.choice([32000, 50304, 102400, 128256, VOCAB])
    return _head(None, kind, _log_int(rng, 1, 64), vocab, hidden)


# ---- inputs -------------------------------------------------------------------------------------
def _gen(seed, salt=0, device=DEV):
    return torch.Generator(device=device).manual_seed(seed * 16 + salt)


def _routing(case, seed, steps=1, salt=1, device=DEV):
    """Zipf routing without replacement (Gumbel top-k): ids int32 [steps, tokens, top_k], softmax
    weights of the same shape, and the experts from the most to the least routed. A row takes
    each expert's noise from its step's first row with probability corr."""
    g = _gen(seed, salt, device)
    E, M = case["experts"], case["tokens"]
    perm = torch.randperm(E, generator=g, device=device)
    logp = torch.empty(E, device=device)
    logp[perm] = -ZIPF * torch.log(torch.arange(1, E + 1, dtype=torch.float32, device=device))
    ids, tw = [], []
    for _ in range(steps):
        u = torch.rand(M, E, generator=g, device=device).clamp(1e-7, 1 - 1e-7)
        noise = -torch.log(-torch.log(u))
        if case["corr"]:
            same = torch.rand(M, E, generator=g, device=device) < case["corr"]
            noise = torch.where(same, noise[:1].expand(M, E), noise)
        top = torch.topk(logp + noise, case["top_k"], dim=1)
        ids.append(top.indices.to(torch.int32))
        tw.append(torch.softmax(0.5 * top.values, dim=1))
    return torch.stack(ids), torch.stack(tw), perm


def _quant_blocks(w):
    """[..., N, K] float32 -> e4m3 of the same shape and its 128x128 block scales."""
    n, k = w.shape[-2:]
    b = w.reshape(-1, n // 128, 128, k // 128, 128)
    s = b.abs().amax(dim=(2, 4)).clamp(min=1e-12) / 448.0
    q = (b / s[:, :, None, :, None]).clamp(-448, 448).to(torch.float8_e4m3fn)
    return q.reshape(w.shape), s.reshape(*w.shape[:-2], n // 128, k // 128)


def _expert_chunks(case, seed):
    """(first expert, {"w13": (q, s), "w2": (q, s)}) for CHUNK experts at a time, row-major."""
    E, H, I = case["experts"], case["hidden"], case["inter"]
    g = _gen(seed, 2)
    for e0 in range(0, E, CHUNK):
        m = min(CHUNK, E - e0)
        yield e0, {name: _quant_blocks(torch.randn(m, n, k, device=DEV, generator=g) * 0.02)
                   for name, (n, k) in (("w13", (2 * I, H)), ("w2", (H, I)))}


def _hidden(seed, rows, width):
    return torch.randn(rows, width, device=DEV, generator=_gen(seed, 3)).to(torch.bfloat16)


def _experts(pkg, case, seed):
    """The expert tensors as a program loads them: fragment order, on the device."""
    E, H, I = case["experts"], case["hidden"], case["inter"]
    w = dict(w13=torch.empty(E, 2 * I, H, dtype=torch.float8_e4m3fn, device=DEV),
             s13=torch.empty(E, 2 * I // 128, H // 128, device=DEV),
             w2=torch.empty(E, H, I, dtype=torch.float8_e4m3fn, device=DEV),
             s2=torch.empty(E, H // 128, I // 128, device=DEV))
    for e0, part in _expert_chunks(case, seed):
        for wn, sn in (("w13", "s13"), ("w2", "s2")):
            q, s = part[wn]
            pkg.ops.shuffle_fp8_weight(q, out=w[wn][e0:e0 + q.shape[0]])
            w[sn][e0:e0 + q.shape[0]] = s
    return pkg.ExpertWeights(**w)


def _head_rows(case, seed):
    """(first row, the float32 head weight's next rows), 4096 * 4 rows at a time."""
    g = _gen(seed, 4)
    for r0 in range(0, case["vocab"], 16384):
        r1 = min(case["vocab"], r0 + 16384)
        yield r0, torch.randn(r1 - r0, case["hidden"], device=DEV, generator=g) * 0.02


def _w4_codes(w):
    """Round-to-nearest int4 codes per (row, 128 columns): codes, bf16 scale, integer zero."""
    n, k = w.shape
    b = w.reshape(n, k // 128, 128)
    lo, hi = b.amin(2), b.amax(2)
    s = ((hi - lo) / 15).clamp(min=1e-8).to(torch.bfloat16)
    z = torch.round(-lo / s.float()).clamp(-1024, 1024)
    q = (torch.round(b / s.float()[:, :, None]) + z[:, :, None]).clamp(0, 15)
    return q.to(torch.uint8), s, z.to(torch.int32)


def _w4_pack(q, s, z):
    """Codes [N, G, 128], scale and zero [N, G] in the documented layout of PackedW4."""
    n, g, _ = q.shape
    t = q.reshape(n // 16, 16, g, 4, 4, 8).permute(0, 2, 4, 1, 3, 5)   # strip, g, c, r, i, j
    b = t[..., [0, 4, 1, 5]] | (t[..., [2, 6, 3, 7]] << 4)
    d = (s.view(torch.int16).to(torch.int32) & 0xFFFF) | (z << 16)
    return (b.reshape(n // 16, g, 64, 16).contiguous(),
            d.reshape(n // 16, 16, g).permute(0, 2, 1).contiguous())


# ---- prepare / run ------------------------------------------------------------------------------
def _capture(fn, keep):
    """fn() recorded into a HIP graph after one eager call; the tensors of `keep` (cache state
    that the eager call moved on) are put back."""
    saved = [t.clone() for t in keep]
    torch.cuda.synchronize()
    fn()
    torch.cuda.synchronize()
    for t, v in zip(keep, saved):
        t.copy_(v)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    torch.cuda.synchronize()
    return graph


def _prepare_layer(pkg, case, seed):
    E, S, M = case["experts"], case["slots"], case["tokens"]
    full = _experts(pkg, case, seed)
    steps = TRACE_STEPS if case["misses"] else 1
    ids, tw, perm = _routing(case, seed, steps)
    hot = sorted(perm[:S].tolist())
    slots = full
    if S < E:
        at = torch.tensor(hot, device=DEV)
        slots = pkg.ExpertWeights(*[t.index_select(0, at) for t in full.tensors()])
    if case["misses"]:
        host = []
        for t in full.tensors():
            h = torch.empty(t.shape, dtype=t.dtype, pin_memory=True)
            h.copy_(t)
            host.append(h)
        full = pkg.ExpertWeights(*host)
    rank = {int(e): i for i, e in enumerate(perm.tolist())}
    layer = pkg.LruMoELayer(full, hot, rank, M, case["top_k"], DEV, slots=slots,
                            max_inserts=None if case["misses"] or S == E else 0)
    st = dict(case=case, layer=layer, x=_hidden(seed, M, case["hidden"]), ids=ids, tw=tw[0],
              step=0, out=torch.empty(M, case["hidden"], dtype=torch.bfloat16, device=DEV),
              graph=None, side=torch.cuda.Stream() if case["misses"] else None)
    # the graph's own routing buffer; recorded over experts that have a slot
    st["now"] = torch.tensor(hot[:case["top_k"]], dtype=torch.int32, device=DEV).repeat(M, 1)
    if M <= GRAPH_TOKENS:
        st["graph"] = _capture(lambda: _apply(st, st["now"]), layer.cache.state())
        st["now"].copy_(ids[0])
    return st


def _apply(st, ids):
    st["layer"].apply(st["out"], st["x"], st["tw"], ids, gather=st["case"]["misses"],
                      side=st["side"])


def _run_layer(st):
    if st["case"]["misses"]:                       # the next step's routing
        st["now"].copy_(st["ids"][st["step"] % TRACE_STEPS])
        st["step"] += 1
    if st["graph"] is not None:
        st["graph"].replay()
    else:
        _apply(st, st["ids"][0])
    cache = st["layer"].cache
    return [st["out"], cache.slot_expert, cache.slot_stamp]


def _prepare_lru(pkg, case, seed):
    M, S, E = case["tokens"], case["slots"], case["experts"]
    st = dict(case=case, step=0, caches=[], trace=[])
    for layer in range(LRU_LAYERS):
        ids, _, perm = _routing(case, seed, TRACE_STEPS if M <= GRAPH_TOKENS else 4,
                                salt=5 + layer)
        rank = {int(e): i for i, e in enumerate(perm.tolist())}
        st["caches"].append(pkg.LruCache.build(E, sorted(perm[:S].tolist()), rank, DEV))
        st["trace"].append(ids)
    st["trace"] = torch.stack(st["trace"], dim=1)                  # [steps, layers, M, top_k]
    st["now"] = st["trace"][0].clone()
    one = st["caches"][0].alloc_align(M * case["top_k"])
    st["out"] = [torch.empty(LRU_LAYERS, t.numel(), dtype=torch.int32, device=DEV) for t in one]

    def fn():
        for layer, cache in enumerate(st["caches"]):
            cache.fused(st["now"][layer], out=[t[layer] for t in st["out"]])

    st["graph"] = _capture(fn, [t for c in st["caches"] for t in c.state()])
    return st


def _run_lru(st):
    st["now"].copy_(st["trace"][st["step"] % st["trace"].shape[0]])
    st["step"] += 1
    st["graph"].replay()
    return [st["out"], [c.slot_expert for c in st["caches"]],
            [c.slot_stamp for c in st["caches"]]]


def _prepare_head_fp8(pkg, case, seed):
    q = torch.empty(case["vocab"], case["hidden"], dtype=torch.float8_e4m3fn, device=DEV)
    s = torch.empty(case["vocab"] // 128, case["hidden"] // 128, device=DEV)
    for r0, w in _head_rows(case, seed):
        wq, ws = _quant_blocks(w)
        pkg.ops.shuffle_fp8_weight(wq, out=q[r0:r0 + w.shape[0]])
        s[r0 // 128:(r0 + w.shape[0]) // 128] = ws
    return dict(case=case, x=_hidden(seed, case["rows"], case["hidden"]), wq=q, ws=s)


def _prepare_head_w4(pkg, case, seed):
    n, k = case["vocab"], case["hidden"]
    wq = torch.empty(n // 16, k // 128, 64, 16, dtype=torch.uint8, device=DEV)
    sz = torch.empty(n // 16, k // 128, 16, dtype=torch.int32, device=DEV)
    for r0, w in _head_rows(case, seed):
        a, b = r0 // 16, (r0 + w.shape[0]) // 16
        wq[a:b], sz[a:b] = _w4_pack(*_w4_codes(w))
    packed = pkg.w4.PackedW4(wq=wq, sz=sz, n=n, n_pad=n, k=k)
    return dict(case=case, x=_hidden(seed, case["rows"], k), packed=packed)


def prepare(case, seed):
    return {"layer": _prepare_layer, "lru": _prepare_lru, "head_fp8": _prepare_head_fp8,
            "head_w4": _prepare_head_w4}[case["kind"]](_pkg(), case, seed)


def run(state):
    kind = state["case"]["kind"]
    if kind == "layer":
        return _run_layer(state)
    if kind == "lru":
        return _run_lru(state)
    if kind == "head_fp8":
        return _pkg().ops.gemm_fp8_block(state["x"], state["wq"], state["ws"])
    return _pkg().w4.gemm_w4a16(state["x"], state["packed"])


# ---- work / tolerance ---------------------------------------------------------------------------
def work(case):
    if case["kind"] == "lru":
        # the ids, the state and the align outputs once, per layer
        mk = case["tokens"] * case["top_k"]
        align = min(16 * mk, mk + 15 * case["experts"])
        return dict(bytes=LRU_LAYERS * (4 * mk + 8 * case["experts"] + 12 * case["slots"] +
                                        2 * align * 4 * 17 // 16), flops=0)
    if case["kind"] == "head_fp8":
        m, n, k = case["rows"], case["vocab"], case["hidden"]
        return dict(bytes=n * k + n * k // 4096 + 2 * m * k + 2 * m * n, flops=2 * m * n * k)
    if case["kind"] == "head_w4":
        m, n, k = case["rows"], case["vocab"], case["hidden"]
        return dict(bytes=n * k // 2 + n * k // 32 + 2 * m * k + 2 * m * n, flops=2 * m * n * k)
    M, H, I, mk = case["tokens"], case["hidden"], case["inter"], case["tokens"] * case["top_k"]
    ids = _routing(case, 0, device="cpu")[0]
    experts = len(torch.unique(ids))
    return dict(bytes=experts * (3 * H * I + 4 * 3 * H * I // 16384) + 4 * M * H + 8 * mk,
                flops=6 * mk * H * I)


def tolerance(case):
    if case["kind"] == "lru":
        return "exact"
    if case["kind"] == "layer":
        # the e4m3 codes between the two products flip where a rounding before them does: 1.5e-2
        # to 1.9e-2 from the 64-bit values on every shape (2e-5 between two splits of one sum
        # by the same kernel); the cache state is whole numbers and stays the same
        return {"rel": 2e-2, "max": 0.5}
    if case["kind"] == "head_fp8":
        # 3.6e-3 from the 64-bit values, of which 1.7e-3 is the logits' bf16 rounding and the
        # rest the matrix unit's own sum over 128 products
        return {"rel": 1e-2, "max": 0.1}
    return {"rel": 1e-3, "max": 0.03}     # 1e-4 from the rounded 64-bit logits: rounding ties


# ---- the same in 64 bits ------------------------------------------------------------------------
def _quant_rows(x):
    """Group-128 e4m3 codes of [rows, K] times their float32 scales, in float64."""
    b = x.float().reshape(x.shape[0], -1, 128)
    s = (b.abs().amax(2, keepdim=True) / 448.0).clamp(min=1.0 / (448.0 * 512.0))
    q = (b / s).clamp(-448, 448).to(torch.float8_e4m3fn)
    return (q.double() * s.double()).reshape(x.shape)


def _dequant(q, s):
    n, k = q.shape
    return (q.double().reshape(n // 128, 128, k // 128, 128) *
            s.double()[:, None, :, None]).reshape(n, k)


def _exact_layer(case, seed):
    I = case["inter"]
    ids, tw, _ = _routing(case, seed, TRACE_STEPS if case["misses"] else 1)
    ids, tw = ids[0], tw[0].double()
    x = _quant_rows(_hidden(seed, case["tokens"], case["hidden"]))
    out = torch.zeros(case["tokens"], case["hidden"], dtype=torch.float64, device=DEV)
    for e0, part in _expert_chunks(case, seed):
        for j in range(part["w13"][0].shape[0]):
            rows, ks = (ids == e0 + j).nonzero(as_tuple=True)
            if len(rows):
                h = x[rows] @ _dequant(*(t[j] for t in part["w13"])).T
                a = _quant_rows(torch.nn.functional.silu(h[:, :I]) * h[:, I:])
                y = a @ _dequant(*(t[j] for t in part["w2"])).T
                out.index_add_(0, rows, y * tw[rows, ks][:, None])
    return [out, None, None]


def _exact_head(case, seed):
    x = _hidden(seed, case["rows"], case["hidden"])
    fp8 = case["kind"] == "head_fp8"
    x = _quant_rows(x) if fp8 else x.double()
    out = torch.empty(case["rows"], case["vocab"], dtype=torch.float64, device=DEV)
    for r0, w in _head_rows(case, seed):
        if fp8:
            d = _dequant(*_quant_blocks(w))
        else:
            q, s, z = _w4_codes(w)
            d = ((q.double() - z.double()[:, :, None]) * s.double()[:, :, None]).reshape(w.shape)
        out[:, r0:r0 + w.shape[0]] = x @ d.T
    return out


def exact(case, seed):
    if case["kind"] == "lru":
        return None
    return _exact_layer(case, seed) if case["kind"] == "layer" else _exact_head(case, seed)

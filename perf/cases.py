"""The work this framework is used for, one dict per case.

    listed()             the cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs, weights and captured graphs of one case, on the GPU
    run(state)           one pass through the public entry points
    work(case)           bytes and operations a pass cannot do without
    tolerance(case)      how far another correct implementation may be off
    exact(case, seed)    what run() returns, in plain torch at 64 bits

Every case has a "kind", the way a program calls the framework:

    resident  batched decode with the experts in HBM: LAYERS layers, each the
              router and the routed experts with the residual added, the step
              captured in one hipGraph and replayed
    ffn       fp8_moe_forward on many tokens (prefill), called eagerly
    a16       fp8_moe_forward with bf16 activations (the numerics of the
              dequantise-then-matmul path)
    block     the MoE block: routed experts, gated shared expert, residual
    route     the router alone, as prefill calls it
    step      decode with the experts offloaded to page-locked host memory:
              slot tables, LRU, fetch of the misses, STEPS replays of the
              captured step of LAYERS layers
    prefill   a prompt through the offload hooks: the experts the prompt
              routes to are gathered from host memory and the resident ones
              borrowed from the device cache

Shapes: hidden 2048, intermediate 512, 256 experts, top-8 (the model's own),
and the other shapes of this repository's tests.  Tokens: 1 to 128 in decode,
up to 1024 in one prefill chunk, 4096 for several chunks or prompts batched
into one call.
"""
import importlib
import math
import types

import numpy as np
import torch

importlib.import_module("drama3-offloading_amd")
import decode                                                       # noqa: E402
import devcache                                                     # noqa: E402
import hipfetch                                                     # noqa: E402
import moe                                                          # noqa: E402
import offload                                                      # noqa: E402
from fp8_moe import MODE_AUTO, MODE_GEMV_A16, fp8_moe_forward       # noqa: E402
from hostpool import HostPool, RecordLayout                         # noqa: E402

DEV = "cuda:0"
LAYERS = 4          # resident: layers of one captured step
STEP_LAYERS = 2     # step: layers of the offloaded decode
STEPS = 8           # step: tokens decoded per pass
F8 = torch.float8_e4m3fn


def _case(name, kind, tokens, hidden=2048, inter=512, experts=256, top_k=8, **more):
    c = dict(kind=kind, tokens=tokens, hidden=hidden, inter=inter, experts=experts, top_k=top_k,
             zipf=False, layout="tiles", ids64=False, wbf16=False, shared=0, capacity=0,
             logits="bf16")
    c.update(more)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # single-stream decode with everything in HBM
        _case("resident decode, 1 token", "resident", 1),
        # a small serving batch
        _case("resident decode, 8 tokens", "resident", 8),
        # an ordinary batch of a ragged size
        _case("resident decode, 29 tokens", "resident", 29),
        # a full serving batch, routed by the popularity of real traffic
        _case("resident decode, 128 tokens", "resident", 128, zipf=True),
        # a few sequences through the whole MoE block, the model's own layer
        _case("MoE block, 5 tokens", "block", 5, shared=512),
        # a prompt through the whole MoE block
        _case("MoE block, 512 tokens", "block", 512, shared=512, ids64=True),
        # one ragged prefill chunk, weights as the checkpoint stores them
        _case("expert FFN, 1021 tokens", "ffn", 1021, layout="rows", ids64=True, wbf16=True),
        # several chunks batched into one call
        _case("expert FFN, 4096 tokens", "ffn", 4096, zipf=True),
        # the router of such a call
        _case("router, 4096 tokens", "route", 4096, ids64=True),
        # decode at the precision of the CPU experts
        _case("bf16 activations, 12 tokens", "a16", 12),
        # decode with the experts offloaded, about 60 % of the picks in the cache
        _case("offloaded decode, 8 steps", "step", 1, capacity=36),
        # a prompt with the experts offloaded, some of them in the decode cache
        _case("offloaded prefill, 512 tokens", "prefill", 512, capacity=48, ids64=True),
    ]


# the shapes that this repository's tests and configurations run
_SHAPES = ((2048, 512), (2048, 512), (2048, 512), (1024, 512), (4096, 384), (2560, 256),
           (1024, 1024))


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(["resident", "resident", "ffn", "ffn", "block", "block", "route", "a16",
                       "step", "prefill"])
    hidden, inter = rng.choice(_SHAPES)
    more = dict(zipf=rng.random() < 0.5, ids64=rng.random() < 0.5, wbf16=rng.random() < 0.3,
                layout=rng.choice(["tiles", "tiles", "rows"]))
    experts, top_k = rng.choice([(256, 8), (256, 8), (128, 8), (64, 6), (192, 4)])
    if kind == "resident":
        return _case(None, kind, _log_uniform(rng, 1, 160), hidden, inter, experts, top_k,
                     zipf=more["zipf"])
    if kind == "ffn":
        return _case(None, kind, _log_uniform(rng, 17, 3600), hidden, inter, experts, top_k,
                     **more)
    if kind == "block":
        return _case(None, kind, _log_uniform(rng, 1, 1024), hidden, inter, experts, top_k,
                     shared=rng.choice([512, 512, 384]), **more)
    if kind == "route":
        return _case(None, kind, _log_uniform(rng, 1, 4096), hidden, 512, experts, top_k,
                     ids64=more["ids64"], logits=rng.choice(["bf16", "bf16", "f32"]))
    if kind == "a16":
        return _case(None, kind, _log_uniform(rng, 1, 40), hidden, inter, experts, top_k,
                     **more)
    if kind == "step":
        return _case(None, kind, 1, experts=rng.choice([128, 192, 256]),
                     capacity=rng.randint(24, 64), shared=rng.choice([0, 512]))
    return _case(None, kind, _log_uniform(rng, 33, 700), experts=rng.choice([64, 128, 192]),
                 capacity=rng.randint(12, 40), ids64=more["ids64"])


# ------------------------------------------------------------------ inputs

def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed((int(seed) * 1_000_003 + salt * 7919 + 17) % (2 ** 62))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _quantise_blocks(w):
    """[n, R, C] float32 -> e4m3 codes and float32 scales of its 128x128 blocks."""
    n, R, C = w.shape
    b = w.view(n, R // 128, 128, C // 128, 128)
    scale = b.abs().amax(dim=(2, 4)) / 448.0
    q = (b / scale[:, :, None, :, None]).to(F8)
    return q.view(torch.uint8).reshape(n, R, C), scale


def _experts(case, seed, layer, chunk=64):
    """Chunks (first expert, w13 codes, s13, w2 codes, s2) of one layer: N(0, 0.02)
    weights, block-quantised as the checkpoint's are."""
    H, I = case["hidden"], case["inter"]
    g = _gen(seed, 100 + layer)
    for e in range(0, case["experts"], chunk):
        n = min(chunk, case["experts"] - e)
        q13, s13 = _quantise_blocks(_randn(g, n, 2 * I, H) * 0.02)
        q2, s2 = _quantise_blocks(_randn(g, n, H, I) * 0.02)
        yield e, q13, s13, q2, s2


def _weights(case, seed, layer):
    """(w13, s13, w2, s2) of one layer in the case's byte order."""
    H, I, E = case["hidden"], case["inter"], case["experts"]
    if case["layout"] == "tiles":
        lay = RecordLayout(H, I)
        rec = torch.empty((E, lay.record_bytes), dtype=torch.uint8, device=DEV)
        for e, q13, s13, q2, s2 in _experts(case, seed, layer):
            rec[e:e + len(q13)] = lay.pack(q13, s13, q2, s2)
        return lay.views(rec)
    parts = list(_experts(case, seed, layer))
    w13, s13, w2, s2 = (torch.cat([p[i] for p in parts]) for i in (1, 2, 3, 4))
    return w13.view(F8), s13, w2.view(F8), s2


def _code(case):
    return hipfetch.LAYOUT_TILES if case["layout"] == "tiles" else hipfetch.LAYOUT_ROWS


def _popularity(case, g, layer):
    """Router bias [E]: zero, or a Zipf(1.1) log-popularity in a random order."""
    E = case["experts"]
    if not case["zipf"]:
        return None
    p = torch.arange(1, E + 1, dtype=torch.float64, device=DEV) ** -1.1
    return (p / p.sum()).log().float()[torch.randperm(E, generator=g, device=DEV)].contiguous()


def _routing(case, seed, tokens):
    """ids [T, K] and normalised weights [T, K]: distinct uniform picks, or draws
    without replacement from a Zipf(1.1) popularity."""
    E, K = case["experts"], case["top_k"]
    g = _gen(seed, 3)
    score = _randn(g, tokens, E)
    u = torch.rand((tokens, E), generator=g, device=DEV).clamp_(1e-9, 1 - 1e-7)
    bias = _popularity(case, g, 0)
    gumbel = -torch.log(-torch.log(u))
    ids = (gumbel if bias is None else bias + gumbel).topk(K, dim=1).indices
    w = torch.softmax(score.gather(1, ids), dim=1)
    ids = ids.to(torch.int64 if case["ids64"] else torch.int32)
    return ids.contiguous(), w.to(torch.bfloat16 if case["wbf16"] else torch.float32).contiguous()


def _hidden(case, seed, salt, tokens):
    return _randn(_gen(seed, salt), tokens, case["hidden"]).to(torch.bfloat16)


def _gate(case, seed, layer):
    return (_randn(_gen(seed, 400 + layer), case["experts"], case["hidden"]) * 0.02).to(torch.bfloat16)


def _shared(case, seed, layer, down_std):
    """Shared expert (gate, up, down, sigmoid gate) in bf16."""
    g, H, Is = _gen(seed, 600 + layer), case["hidden"], case["shared"]
    bf = lambda std, *s: (_randn(g, *s) * std).to(torch.bfloat16)   # noqa: E731
    return bf(0.02, Is, H), bf(0.02, Is, H), bf(down_std, H, Is), bf(0.02, H)


def _capture(body):
    """One captured graph of body(), after a pass outside the capture."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        body()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        body()
    return g


# ------------------------------------------------------------------- kinds

def _prepare_resident(case, seed):
    lib = hipfetch.require()
    B, H, I, E, K = (case[k] for k in ("tokens", "hidden", "inter", "experts", "top_k"))
    new = lambda dt, *s: torch.empty(s, dtype=dt, device=DEV)       # noqa: E731
    layers = []
    for l in range(LAYERS):
        layers.append(dict(
            x=_hidden(case, seed, 10 + l, B), gate=_gate(case, seed, l), w=_weights(case, seed, l),
            bias=_popularity(case, _gen(seed, 500 + l), l), out=new(torch.bfloat16, B, H),
            logits=new(torch.float32, B, E), ids=new(torch.int32, B, K),
            wts=new(torch.float32, B, K)))
    ws = new(torch.uint8, lib.fp8_moe_workspace(B, K, E, H, I))

    def body():
        for y in layers:
            w13, s13, w2, s2 = y["w"]
            if B <= 16:
                lib.router_fp8_moe_forward(y["x"], y["gate"], y["bias"], K, y["logits"], y["ids"],
                                           y["wts"], w13, s13, w2, s2, y["out"], ws,
                                           residual=y["x"], layout=_code(case))
            else:
                lib.router_topk(y["x"], y["gate"], y["bias"], K, y["logits"], y["ids"], y["wts"])
                lib.fp8_moe_forward(y["x"], y["ids"], y["wts"], w13, s13, w2, s2, y["out"], ws,
                                    residual=y["x"], layout=_code(case))
    return dict(graph=_capture(body), layers=layers, ws=ws)


def _run_resident(s):
    s["graph"].replay()
    return [{k: y[k] for k in ("out", "logits", "ids", "wts")} for y in s["layers"]]


def _prepare_ffn(case, seed):
    ids, wts = _routing(case, seed, case["tokens"])
    return dict(x=_hidden(case, seed, 1, case["tokens"]), ids=ids, wts=wts,
                w=_weights(case, seed, 0), code=_code(case),
                mode=MODE_GEMV_A16 if case["kind"] == "a16" else MODE_AUTO)


def _run_ffn(s):
    return fp8_moe_forward(s["x"], s["ids"], s["wts"], *s["w"], mode=s["mode"], layout=s["code"])


def _prepare_block(case, seed):
    s = _prepare_ffn(case, seed)
    s["lib"] = hipfetch.require()
    s["shared"] = _shared(case, seed, 0, 0.02)
    s["ws"] = torch.empty(s["lib"].fp8_moe_block_workspace(
        case["tokens"], case["top_k"], case["experts"], case["hidden"], case["inter"],
        case["shared"]), dtype=torch.uint8, device=DEV)
    return s


def _run_block(s):
    out = torch.empty_like(s["x"])
    s["lib"].fp8_moe_block_forward(s["x"], s["ids"], s["wts"], *s["w"], s["shared"], out, s["ws"],
                                   residual=s["x"], layout=s["code"])
    return out


def _prepare_route(case, seed):
    return dict(x=_hidden(case, seed, 1, case["tokens"]), gate=_gate(case, seed, 0),
                K=case["top_k"], logits=case["logits"],
                ids=torch.int64 if case["ids64"] else torch.int32)


def _run_route(s):
    ids, wts, logits = moe.route(s["x"], s["gate"], s["K"], ids_dtype=s["ids"],
                                 logit_dtype=s["logits"])
    return dict(ids=ids, wts=wts, logits=logits)


def _step_inputs(case, seed):
    """Stub matrices, gates and per-step router biases of the offloaded decode:
    Zipf(1.1) popularity per layer plus Gumbel noise, so the picks are draws from it."""
    H, E, L = case["hidden"], case["experts"], STEP_LAYERS
    g = _gen(seed, 700)
    stub = (_randn(g, L, H, H) * H ** -0.5).to(torch.bfloat16)
    gate = (_randn(g, L, E, H) * 0.002).to(torch.bfloat16)
    pop = torch.stack([_popularity(dict(case, zipf=True), g, l) for l in range(L)])
    u = torch.rand((STEPS, L, E), generator=g, device=DEV).clamp_(1e-9, 1 - 1e-7)
    bias = (pop - torch.log(-torch.log(u))).float()
    return stub, gate, bias, _hidden(case, seed, 1, 1)


def _prepare_step(case, seed):
    lay = RecordLayout(case["hidden"], case["inter"])
    pools = []
    for l in range(STEP_LAYERS):
        pool = HostPool(case["experts"], lay)
        for e, q13, s13, q2, s2 in _experts(case, seed, l):
            pool.write(e, lay.pack(q13, s13, q2, s2))
        pools.append(pool)
    cfg = decode.DecodeConfig(layers=STEP_LAYERS, n_experts=case["experts"], top_k=case["top_k"],
                              hidden=case["hidden"], inter=case["inter"],
                              capacity=case["capacity"], seed=seed, schedule_steps=STEPS,
                              shared_expert=case["shared"] > 0, shared_inter=case["shared"] or 512)
    h = decode.DecodeHarness(cfg, DEV, pools)
    stub, gate, bias, x0 = _step_inputs(case, seed)
    h.w_stub.copy_(stub)
    h.gate.copy_(gate)
    h.bias_all.copy_(bias)
    h.x0.copy_(x0)
    if case["shared"]:
        for l in range(STEP_LAYERS):
            for mine, w in zip(h.shared(l), _shared(case, seed, l, 0.005)):
                mine.copy_(w)
    h.capture()
    return h


def _run_step(h):
    h.cursor = 0
    got = []
    for _ in range(STEPS):
        h.replay()
        got.append(dict(x=h.x.clone(), logits=h.logits.clone(), ids=h.ids.clone(),
                        wts=h.wts.clone()))
    return got


def _prepare_prefill(case, seed):
    E, H, I = case["experts"], case["hidden"], case["inter"]
    experts = moe.MoEExperts(E, H, I, device="cpu")
    layer = types.SimpleNamespace(mlp=types.SimpleNamespace(experts=experts))
    model = types.SimpleNamespace(backbone=types.SimpleNamespace(
        model=types.SimpleNamespace(layers=[layer])))
    offload.pin_experts(model, torch.device(DEV))
    for e, q13, s13, q2, s2 in _experts(case, seed, 0):
        n = len(q13)
        experts.w13_weight.view(torch.uint8)[e:e + n].copy_(q13)
        experts.w2_weight.view(torch.uint8)[e:e + n].copy_(q2)
        experts.w13_scale_inv[e:e + n].copy_(s13)
        experts.w2_scale_inv[e:e + n].copy_(s2)
    devcache.install_dev_cache(model, torch.device(DEV), case["capacity"])
    # a few decoded tokens have left experts in the cache
    for t in range(6):
        ids, wts = _routing(dict(case, zipf=True), seed + 1000 + t, 1)
        experts(_hidden(case, seed, 50 + t, 1), ids, wts)
    ids, wts = _routing(case, seed, case["tokens"])
    return dict(experts=experts, x=_hidden(case, seed, 1, case["tokens"]), ids=ids, wts=wts)


def _run_prefill(s):
    return s["experts"](s["x"], s["ids"], s["wts"])


_PREPARE = dict(resident=_prepare_resident, ffn=_prepare_ffn, a16=_prepare_ffn,
                block=_prepare_block, route=_prepare_route, step=_prepare_step,
                prefill=_prepare_prefill)
_RUN = dict(resident=_run_resident, ffn=_run_ffn, a16=_run_ffn, block=_run_block,
            route=_run_route, step=_run_step, prefill=_run_prefill)


def prepare(case, seed):
    return case["kind"], _PREPARE[case["kind"]](case, int(seed))


def run(state):
    return _RUN[state[0]](state[1])


# -------------------------------------------------------------------- work

def _distinct(case, tokens):
    """Experts that `tokens` tokens' picks name, on average."""
    E, K = case["experts"], case["top_k"]
    if not case["zipf"]:
        return E * (1.0 - (1.0 - K / E) ** tokens)
    p = np.arange(1, E + 1, dtype=np.float64) ** -1.1
    # a pick without replacement is a little likelier than K single draws
    return float((1.0 - np.exp(-K * tokens * p / p.sum())).sum())


def work(case):
    T, H, I, E, K = (case[k] for k in ("tokens", "hidden", "inter", "experts", "top_k"))
    kind = case["kind"]
    record = 3 * H * I + 4 * 3 * (H // 128) * (I // 128)
    route_bytes = E * H * 2 + T * H * 2 + T * E * 4 + T * K * 8
    route_flops = 2.0 * T * E * H
    ffn_bytes = _distinct(case, T) * record + T * H * 4 + T * K * 8
    ffn_flops = 2.0 * T * K * 3 * H * I
    shared_bytes = 3 * H * case["shared"] * 2
    shared_flops = 2.0 * T * 3 * H * case["shared"]
    if kind == "route":
        return {"bytes": route_bytes, "flops": route_flops}
    if kind == "resident":
        return {"bytes": LAYERS * (route_bytes + ffn_bytes),
                "flops": LAYERS * (route_flops + ffn_flops)}
    if kind == "block":
        return {"bytes": ffn_bytes + shared_bytes, "flops": ffn_flops + shared_flops}
    if kind == "step":
        n = STEPS * STEP_LAYERS
        return {"bytes": n * (2 * H * H + route_bytes + K * record + shared_bytes),
                "flops": n * (2.0 * H * H + route_flops + ffn_flops + shared_flops)}
    return {"bytes": ffn_bytes, "flops": ffn_flops}


def tolerance(case):
    """About four times what the paths show against exact(): bf16 outputs are
    1.7e-3 off in the 2-norm by their last rounding alone, and an activation
    that quantises to the neighbouring e4m3 code adds to that."""
    kind = case["kind"]
    if kind == "route":
        return {"rel": 1e-3, "max": 0.02, "differ": 1e-3}
    if kind == "step":
        return {"rel": 1.5e-2, "max": 0.3, "differ": 0.01}
    return {"rel": 6e-3, "max": 0.1, "differ": 5e-3}


# ------------------------------------------------------------------- exact

def _bf16(v):
    """A float64 tensor rounded once to bf16, as float64 (rounding to odd into
    float32 first keeps the second rounding from being a double one)."""
    f = v.to(torch.float32)
    over = f.double().abs() > v.abs()
    bits = f.view(torch.int32)
    bits = torch.where(over, bits - 1, bits)                   # toward zero
    odd = bits.view(torch.float32).double() != v
    bits = torch.where(odd, bits | 1, bits)
    return bits.view(torch.float32).to(torch.bfloat16).double()


def _quantised(v):
    """float64 [n, C] -> the values its e4m3 codes stand for (scale amax / 448
    per 128 columns, in float32; divided by a tensor, as torch multiplies by
    the rounded reciprocal of a plain number on the GPU)."""
    f = v.float().view(v.shape[0], -1, 128)
    s = f.abs().amax(dim=2, keepdim=True) / torch.full((), 448.0, device=DEV)
    q = torch.where(s == 0, torch.zeros_like(f), f / s).clamp(-448.0, 448.0).to(F8)
    return (q.double() * s.double()).view(v.shape)


def _dequantised(codes, scale):
    n, R, C = codes.shape
    w = codes.view(F8).double().view(n, R // 128, 128, C // 128, 128)
    return (w * scale.double()[:, :, None, :, None]).view(n, R, C)


def _ffn_exact(case, seed, layer, x, ids, wts, a16=False):
    """Sum over the picks of weight * expert(x), float64 [T, H], rounded to bf16."""
    T, I, K = x.shape[0], case["inter"], case["top_k"]
    y = torch.zeros((T * K, case["hidden"]), dtype=torch.float64, device=DEV)
    xd = x.double()
    xq = xd if a16 else _quantised(xd)
    flat = ids.long().reshape(-1)
    used = set(torch.unique(flat).tolist())
    for e0, q13, s13, q2, s2 in _experts(case, seed, layer):
        for i in range(len(q13)):
            if e0 + i not in used:
                continue
            pairs = (flat == e0 + i).nonzero().view(-1)
            w13 = _dequantised(q13[i:i + 1], s13[i:i + 1])[0]
            w2 = _dequantised(q2[i:i + 1], s2[i:i + 1])[0]
            h = xq[pairs // K] @ w13.t()
            a = torch.nn.functional.silu(h[:, :I]) * h[:, I:]
            y[pairs] = (_bf16(a) if a16 else _quantised(a)) @ w2.t()
    return _bf16((y.view(T, K, -1) * wts.double().unsqueeze(2)).sum(1))


def _route_exact(x, gate, bias, K, logit_dtype):
    l = x.double() @ gate.double().t()
    l = _bf16(l).float() if logit_dtype == "bf16" else l.float()
    if bias is not None:
        l = l + bias
    ids = torch.sort(l, dim=1, descending=True, stable=True).indices[:, :K]
    return l, ids, torch.softmax(l.double().gather(1, ids), dim=1)


def _shared_exact(x, shared, routed, residual):
    wg, wu, wd, wsg = (w.double() for w in shared)
    xd = x.double()
    g, u = _bf16(xd @ wg.t()), _bf16(xd @ wu.t())
    a = _bf16(_bf16(torch.nn.functional.silu(g)) * u)
    d = _bf16(a @ wd.t())
    sig = _bf16(torch.sigmoid(_bf16(xd @ wsg.view(-1, 1))))
    return _bf16(residual.double() + _bf16(routed + _bf16(sig * d)))


def exact(case, seed):
    seed, kind, K = int(seed), case["kind"], case["top_k"]
    T = case["tokens"]
    if kind == "route":
        l, ids, wts = _route_exact(_hidden(case, seed, 1, T), _gate(case, seed, 0), None, K,
                                   case["logits"])
        return dict(ids=ids, wts=wts, logits=l.double())
    if kind == "resident":
        got = []
        for l in range(LAYERS):
            x = _hidden(case, seed, 10 + l, T)
            lg, ids, wts = _route_exact(x, _gate(case, seed, l),
                                        _popularity(case, _gen(seed, 500 + l), l), K, "bf16")
            y = _ffn_exact(case, seed, l, x, ids, wts)
            got.append(dict(out=_bf16(x.double() + y), logits=lg.double(), ids=ids, wts=wts))
        return got
    if kind == "step":
        stub, gate, bias, x0 = _step_inputs(case, seed)
        got = []
        for t in range(STEPS):
            x, ls, idl, wl = x0.double(), [], [], []
            for l in range(STEP_LAYERS):
                h = _bf16(x @ stub[l].double().t())
                lg, ids, wts = _route_exact(h, gate[l], bias[t, l], K, "bf16")
                y = _ffn_exact(case, seed, l, h, ids, wts)
                if case["shared"]:
                    x = _shared_exact(h, _shared(case, seed, l, 0.005), y, h)
                else:
                    x = _bf16(h + y)
                ls.append(lg.double()), idl.append(ids), wl.append(wts)
            got.append(dict(x=x, logits=torch.stack(ls), ids=torch.stack(idl),
                            wts=torch.stack(wl)))
        return got
    ids, wts = _routing(case, seed, T)
    x = _hidden(case, seed, 1, T)
    y = _ffn_exact(case, seed, 0, x, ids, wts, a16=kind == "a16")
    if kind == "block":
        return _shared_exact(x, _shared(case, seed, 0, 0.02), y, x)
    return y

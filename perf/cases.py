"""The work this library is measured on: layers, blocks and whole calls.

Sizes are those of the two configuration presets (``granite-1b``: hidden
1024, 32 experts; ``granite-3b``: hidden 1536, 40 experts; both top-8,
intermediate 512, 8 KV heads of 64 channels, vocabulary 49155) over the batch
sizes, prompt lengths and contexts of a generation service: one user to 128
rows, contexts to 4096, prefills from one short prompt to 48 packed ones.

A decode program records its step into a HIP graph once and replays it per
token (``execution.capture_decode``). The decode cases do the same: their
graph holds the block for several layers, each with weights (and KV pages) of
its own, as the step of a model does, so no pass finds the last one's weights
in a cache that a real step would have flushed. Prefill cases are eager calls.

Kinds (``case["op"]``):

* ``step``: one whole decode step, ``Granite.forward`` in lean decode
  (embedding, layers, final norm, LM head), logits and KV cache returned;
* ``prefill``: one whole packed prefill, ``Granite.forward`` with a
  ``PackedPrefill``, last-position logits and KV cache returned;
* ``attn_decode``: QKV projection, RoPE, KV store, flash decode, o_proj;
* ``attn_prefill``: the same block for packed ragged prompts;
* ``moe_decode``, ``moe_prefill``: the routed experts (gate/up, SiLU, down),
  the weighted combine, the residual add and the next norm;
* ``router``: residual add, norm, router logits, top-k and softmax;
* ``head``: the LM head with the greedy choice and the state update.
"""
import math

import numpy as np
import torch

from litemoe_amd import synth
from litemoe_amd.cache import KVCache
from litemoe_amd.config import preset
from litemoe_amd.ep import ExpertParallel
from litemoe_amd.execution import capture_decode
from litemoe_amd.experts import HipFusedExperts, finish_add_rmsnorm, pack_expert_weights
from litemoe_amd.flash_decode import FlashDecode
from litemoe_amd.linear import linear_dense, linear_rope_kv, linear_splitk, linear_splitk_frag, pick_splits, reduce
from litemoe_amd.model import Granite
from litemoe_amd.norm import add_rmsnorm
from litemoe_amd.packed import build_packed, varlen_attention
from litemoe_amd.router import add_rmsnorm_route, add_rmsnorm_route_splitk
from litemoe_amd.step import PackedHead, greedy_head

DEVICE = "cuda:0"
BF16 = torch.bfloat16
SPLITS_O = 4          # K slices of the o_proj partials that the decode router takes


def listed():
    return [
        # One user chatting with the small model: a whole token step, bound by
        # launches and latency (8 of its layers, the full vocabulary).
        dict(name="step_1b_b1", op="step", model="granite-1b", layers=8, rows=1, low=512, high=512),
        # A few short prompts arriving together, to their first-token logits.
        dict(name="prefill_3b_3_prompts", op="prefill", model="granite-3b", layers=2, count=3, low=61, high=389),
        # The attention block of the headline decode: 64 rows in their second thousand of tokens.
        dict(name="attn_decode_3b_b64", op="attn_decode", model="granite-3b", layers=4, rows=64, low=1025, high=1279),
        # Few users with long contexts: the key range has to be split to fill the GPU.
        dict(name="attn_decode_1b_b3_long", op="attn_decode", model="granite-1b", layers=4, rows=3, low=2049,
             high=4001),
        # Long-context serving: the largest batch over ragged contexts, bound by the KV stream.
        dict(name="attn_decode_3b_b128_ragged", op="attn_decode", model="granite-3b", layers=2, rows=128, low=1024,
             high=4095),
        # The experts of the headline decode: every expert's weights are read.
        dict(name="moe_decode_3b_b64", op="moe_decode", model="granite-3b", layers=4, rows=64, skew=0.0),
        # A handful of users: some of the experts, about one row each.
        dict(name="moe_decode_1b_b5", op="moe_decode", model="granite-1b", layers=6, rows=5, skew=0.0),
        # One ordinary prompt through the operator that stands for vLLM's fused_experts.
        dict(name="moe_prefill_3b_700", op="moe_prefill", model="granite-3b", tokens=700, skew=0.0, operator=True),
        # A packed prefill of 48 prompts whose router sends half of the routes to four experts.
        dict(name="moe_prefill_3b_46990_skewed", op="moe_prefill", model="granite-3b", tokens=46990, skew=2.2,
             operator=False),
        # The same prefill's router: every token's residual, norm and selection.
        dict(name="router_3b_46990", op="router", model="granite-3b", layers=1, tokens=46990),
        # The LM head of the headline decode with the argmax and the state update.
        dict(name="head_3b_b64", op="head", model="granite-3b", rows=64),
        # The same prefill's attention block: projections, RoPE, KV store, causal attention.
        dict(name="attn_prefill_3b_48_ragged", op="attn_prefill", model="granite-3b", count=48, low=64, high=2048),
    ]


def _log_int(rng, low, high):
    return min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 1))) - 0.5)) or low)


def draw(rng):
    op = rng.choice(["step", "prefill", "attn_decode", "attn_decode", "moe_decode", "moe_decode", "moe_prefill",
                     "moe_prefill", "router", "head", "attn_prefill"])
    case = dict(op=op, model=rng.choice(["granite-1b", "granite-3b"]))
    if op in ("step", "attn_decode"):
        low = _log_int(rng, 16, 2048)
        case.update(layers=rng.randint(2, 4), rows=_log_int(rng, 1, 64 if op == "step" else 128), low=low,
                    high=min(4095, int(low * rng.uniform(1.0, 4.0))))
    elif op in ("prefill", "attn_prefill"):
        low = _log_int(rng, 16, 1024)
        count = _log_int(rng, 1, 8 if op == "prefill" else 32)
        case.update(count=count, low=low, high=min(2048, int(low * rng.uniform(1.0, 8.0))))
        if op == "prefill":
            case.update(layers=2, high=min(case["high"], max(low, 4096 // count)))
    elif op == "moe_decode":
        case.update(layers=rng.randint(2, 4), rows=_log_int(rng, 1, 256), skew=rng.choice([0.0, 2.2]))
    elif op == "moe_prefill":
        case.update(tokens=_log_int(rng, 257, 32768), skew=rng.choice([0.0, 2.2]), operator=rng.random() < 0.5)
    elif op == "router":
        tokens = _log_int(rng, 1, 32768)
        case.update(tokens=tokens, layers=4 if tokens <= 128 else 1)
    else:
        case.update(rows=_log_int(rng, 1, 128))
    return case


# ---------------------------------------------------------------- inputs --

class _Inputs:
    """Tensors from one seed, on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed)
        self.rng = np.random.RandomState(seed % (1 << 32))

    def normal(self, *shape, std=1.0, dtype=BF16):
        return torch.empty(*shape, device=DEVICE, dtype=torch.float32).normal_(0.0, std, generator=self.gen).to(dtype)

    def norm_weight(self, hidden):
        return (1.0 + self.normal(hidden, std=0.1, dtype=torch.float32)).to(BF16)

    def lengths(self, case):
        """The case's lengths, spread evenly over its range, in an order of the seed's."""
        count = case.get("rows") or case["count"]
        return self.rng.permutation(_lengths(case, count)).tolist()

    def routes(self, tokens, cfg, skew):
        """Top-k ids and renormalised weights of random logits (std 0.8, as a
        random-init router's); ``skew`` favours four experts."""
        logits = self.normal(tokens, cfg.num_local_experts, std=0.8, dtype=torch.float32)
        if skew:
            hot = self.rng.permutation(cfg.num_local_experts)[:4].tolist()
            logits[:, hot] += skew
        top, ids = logits.topk(cfg.num_experts_per_tok, dim=-1)
        return ids.to(torch.int32), top.softmax(-1)

    def expert_weights(self, cfg):
        e, h, i = cfg.num_local_experts, cfg.hidden_size, cfg.intermediate_size
        # larger than at initialisation: the experts' part of the residual
        # stream is then of the stream's own size, as in a trained model
        return self.normal(e, 2 * i, h, std=2.5 * synth.STD), self.normal(e, h, i, std=2.5 * synth.STD)

    def attention_weights(self, cfg):
        """Packed q|k|v and o projections; the query rows are larger than at
        initialisation so that the scores spread as a trained model's do."""
        h, hq, hkv = cfg.hidden_size, cfg.num_attention_heads * 64, cfg.num_key_value_heads * 64
        qkv = torch.cat([self.normal(hq, h, std=10 * synth.STD), self.normal(2 * hkv, h, std=synth.STD)])
        return qkv, self.normal(h, hq, std=synth.STD)


def _lengths(case, count):
    return np.rint(np.linspace(case["low"], case["high"], count)).astype(np.int64)


def _capacity(longest):
    return -(-longest // 256) * 256


def _cos_sin(cfg, capacity):
    """The model's RoPE table ``[capacity, 64]``: cos | sin, bf16."""
    inv = 1.0 / cfg.rope_theta ** (torch.arange(0, 64, 2).float() / 64)
    freq = torch.outer(torch.arange(capacity, device=DEVICE).float(), inv.to(DEVICE))
    return torch.cat((freq.cos(), freq.sin()), -1).to(BF16)


def _model(case, seed, capacity):
    cfg = preset(case["model"], num_hidden_layers=case["layers"])
    w = synth.granite_weights(cfg, seed, DEVICE, method="torch")
    ep = ExpertParallel(1, 0, 1 << 16, cfg.hidden_size, cfg.num_experts_per_tok, BF16, DEVICE, HipFusedExperts())
    return Granite(cfg, w, ep, capacity, pack_weights=case["op"] == "step")


def _recorded(step, reset=lambda: None):
    """``step`` as a HIP graph, and the tensors its recording returned."""
    kept = {}

    def body():
        kept["out"] = step()

    graph = capture_decode(body, reset)
    return graph, kept["out"]


def _graph_state(inputs, step, reset=lambda: None):
    graph, out = _recorded(step, reset)
    return dict(run=lambda: (graph.replay(), out)[1], inputs=inputs, graph=graph)


# ------------------------------------------------- whole calls of a model --

def _make_step(case, seed):
    inp = _Inputs(seed)
    rows, lengths = case["rows"], inp.lengths(case)
    capacity = _capacity(case["high"] + 1)
    model = _model(case, seed, capacity)
    cfg = model.cfg
    cache = KVCache(cfg, rows, capacity, DEVICE, BF16)
    for side in (cache.k, cache.v):
        side.copy_(inp.normal(*side.shape))
    tokens = torch.tensor(inp.rng.randint(0, cfg.vocab_size, (rows, 1)), device=DEVICE)
    positions = torch.tensor(lengths, device=DEVICE)[:, None] - 1
    return dict(model=model, cache=cache, tokens=tokens, positions=positions)


def _prepare_step(case, seed):
    s = _make_step(case, seed)
    model, cache, cfg = s["model"], s["cache"], s["model"].cfg
    rows = case["rows"]
    valid = torch.ones(rows, 1, dtype=torch.bool, device=DEVICE)
    model.decode_lean = True
    model.decode_flash = FlashDecode(rows, cfg.num_key_value_heads,
                                     cfg.num_attention_heads // cfg.num_key_value_heads, cache.capacity, DEVICE,
                                     case["high"])
    return _graph_state(s, lambda: dict(logits=model.forward(s["tokens"], s["positions"], valid, cache),
                                        k=cache.k, v=cache.v))


def _make_prefill(case, seed):
    inp = _Inputs(seed)
    lengths = inp.lengths(case)
    capacity = _capacity(case["high"])
    model = _model(case, seed, capacity)
    cache = KVCache(model.cfg, case["count"], capacity, DEVICE, BF16)
    packed, ends = build_packed(lengths, DEVICE)
    tokens = torch.tensor(inp.rng.randint(0, model.cfg.vocab_size, (1, sum(lengths))), device=DEVICE)
    return dict(model=model, cache=cache, tokens=tokens, packed=packed, last=ends.long() - 1, lengths=lengths)


def _prepare_prefill(case, seed):
    s = _make_prefill(case, seed)
    model, cache = s["model"], s["cache"]
    valid = torch.ones_like(s["tokens"], dtype=torch.bool)

    def run():
        logits = model.forward(s["tokens"], s["packed"].positions[None], valid, cache, slot=s["packed"],
                               last=s["last"])
        return dict(logits=logits, k=cache.k, v=cache.v)

    return dict(run=run, inputs=s)


def _exact_model(case, s):
    """The layers and the head of ``s["model"]`` in 64 bits, for a step or a prefill."""
    model, cache = s["model"], s["cache"]
    cfg, w = model.cfg, model.w
    r, eps, scale = cfg.residual_multiplier, cfg.rms_norm_eps, cfg.attention_multiplier
    hq, hkv = cfg.num_attention_heads, cfg.num_key_value_heads
    table = _cos_sin(cfg, cache.capacity)
    x = w["embedding"].double()[s["tokens"].reshape(-1)] * cfg.embedding_multiplier
    positions = (s["packed"].positions if "packed" in s else s["positions"]).reshape(-1)
    ks, vs = cache.k.double(), cache.v.double()
    for layer, lw in enumerate(w["layers"]):
        qkv = _rmsnorm64(x, lw["input_layernorm"], eps) @ lw["self_attn.qkv_proj"].double().t()
        q, k, v = _heads64(qkv, hq, hkv, table, positions)
        if "packed" in s:
            a, row, at = [], 0, 0
            for n in s["lengths"]:
                part = slice(at, at + n)
                ks[layer, row, :, :n], vs[layer, row, :, :n] = k[part].transpose(0, 1), v[part].transpose(0, 1)
                a.append(_causal64(q[part], k[part], v[part], scale))
                row, at = row + 1, at + n
            a = torch.cat(a)
        else:
            a = _decode64(q, k, v, ks[layer], vs[layer], positions, scale)
        x = x + r * (a @ lw["self_attn.o_proj"].double().t())
        z = _rmsnorm64(x, lw["post_attention_layernorm"], eps)
        top, ids = (z @ lw["block_sparse_moe.router.layer"].double().t()).topk(cfg.num_experts_per_tok, dim=-1)
        x = x + r * _experts64(z, ids, top.softmax(-1), lw["input_linear"], lw["output_linear"])
    if "last" in s:
        x = x[s["last"]]
    logits = _rmsnorm64(x, w["norm"], eps) @ w["head"].double().t() / cfg.logits_scaling
    return dict(logits=logits[:, None], k=ks, v=vs)


# --------------------------------------------------------------- attention --

def _make_attn(case, seed):
    inp, cfg = _Inputs(seed), preset(case["model"])
    lengths = inp.lengths(case)
    prefill = case["op"] == "attn_prefill"
    layers = [inp.attention_weights(cfg) for _ in range(case.get("layers", 1))]
    capacity = _capacity(case["high"])
    cache = KVCache(preset(case["model"], num_hidden_layers=len(layers)), len(lengths), capacity, DEVICE, BF16)
    if not prefill:
        for layer in range(len(layers)):
            for side in (cache.k, cache.v):
                side[layer].copy_(inp.normal(*side.shape[1:]))
    z = [inp.normal(sum(lengths) if prefill else len(lengths), cfg.hidden_size) for _ in layers]
    return dict(cfg=cfg, lengths=lengths, layers=layers, cache=cache, z=z, table=_cos_sin(cfg, capacity))


def _prepare_attn_decode(case, seed):
    s = _make_attn(case, seed)
    cfg, cache, rows = s["cfg"], s["cache"], case["rows"]
    hq, hkv, h = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.hidden_size
    used = torch.tensor(s["lengths"], device=DEVICE, dtype=torch.int32)
    positions, active = used.long() - 1, torch.ones(rows, dtype=torch.bool, device=DEVICE)
    # a ragged batch's rows are dispatched longest first, as the engine has it
    order = torch.argsort(used, descending=True, stable=True).int() if case["high"] > 1.25 * case["low"] else None
    flash = FlashDecode(rows, hkv, hq // hkv, cache.capacity, DEVICE, case["high"])
    splits = pick_splits(rows, (hq + 2 * hkv) * 64, h), pick_splits(rows, h, hq * 64, max_splits=SPLITS_O)

    def step():
        out = []
        for layer, (qkv, o) in enumerate(s["layers"]):
            part = linear_splitk(s["z"][layer], qkv, splits[0])
            a = flash.fused_qkv(part, s["table"], positions, active, cache.k[layer], cache.v[layer],
                                cfg.attention_multiplier, used, hq, row_order=order, frag_out=True)
            out.append(reduce(linear_splitk_frag(a, o, splits[1])))
        return dict(a=out, k=cache.k, v=cache.v)

    return _graph_state((s, used, positions, active, order, flash), step)


def _exact_attn_decode(case, seed):
    s = _make_attn(case, seed)
    cfg, ks, vs = s["cfg"], s["cache"].k.double(), s["cache"].v.double()
    positions = torch.tensor(s["lengths"], device=DEVICE) - 1
    out = []
    for layer, (w, o) in enumerate(s["layers"]):
        q, k, v = _heads64(s["z"][layer].double() @ w.double().t(), cfg.num_attention_heads,
                           cfg.num_key_value_heads, s["table"], positions)
        out.append(_decode64(q, k, v, ks[layer], vs[layer], positions, cfg.attention_multiplier) @ o.double().t())
    return dict(a=out, k=ks, v=vs)


def _prepare_attn_prefill(case, seed):
    s = _make_attn(case, seed)
    cfg, cache = s["cfg"], s["cache"]
    hq, hkv = cfg.num_attention_heads, cfg.num_key_value_heads
    packed, _ = build_packed(s["lengths"], DEVICE)
    rows = sum(s["lengths"])
    active = torch.ones(rows, dtype=torch.bool, device=DEVICE)
    (w, o), z = s["layers"][0], s["z"][0]

    def run():
        qkv = linear_rope_kv(z, w, hq, hkv, packed.positions, active, s["table"], cache, 0, packed.slots)
        q, k, v = qkv.view(rows, hq + 2 * hkv, 64).split([hq, hkv, hkv], 1)
        a = varlen_attention(q, k, v, packed.cu, packed.maximum, cfg.attention_multiplier)
        return dict(a=linear_dense(a.view(rows, hq * 64), o), k=cache.k, v=cache.v)

    return dict(run=run, inputs=(s, packed, active))


def _exact_attn_prefill(case, seed):
    s = _make_attn(case, seed)
    cfg, ks, vs = s["cfg"], s["cache"].k.double(), s["cache"].v.double()
    (w, o), z, w64 = s["layers"][0], s["z"][0], s["layers"][0][0].double().t()
    out, at = [], 0
    for row, n in enumerate(s["lengths"]):
        q, k, v = _heads64(z[at:at + n].double() @ w64, cfg.num_attention_heads, cfg.num_key_value_heads, s["table"],
                           torch.arange(n, device=DEVICE))
        ks[0, row, :, :n], vs[0, row, :, :n] = k.transpose(0, 1), v.transpose(0, 1)
        out.append(_causal64(q, k, v, cfg.attention_multiplier) @ o.double().t())
        at += n
    return dict(a=torch.cat(out), k=ks, v=vs)


# ----------------------------------------------------------------- experts --

def _make_moe(case, seed):
    inp, cfg = _Inputs(seed), preset(case["model"])
    rows = case.get("rows") or case["tokens"]
    layers = []
    for _ in range(case.get("layers", 1)):
        w1, w2 = inp.expert_weights(cfg)
        ids, weights = inp.routes(rows, cfg, case["skew"])
        layers.append(dict(w1=w1, w2=w2, ids=ids, weights=weights, z=inp.normal(rows, cfg.hidden_size),
                           x=inp.normal(rows, cfg.hidden_size, std=0.25), norm=inp.norm_weight(cfg.hidden_size)))
    return cfg, layers


def _prepare_moe_decode(case, seed):
    cfg, layers = _make_moe(case, seed)
    backend = HipFusedExperts()
    for s in layers:
        s["w1"], s["w2"] = pack_expert_weights(s["w1"], s["w2"])
        s["residual"] = s["x"].clone()

    def step():
        out = []
        for s in layers:
            y = backend.routes(s["z"], s["w1"], s["w2"], s["ids"], packed=True)
            out.append(finish_add_rmsnorm(y, s["ids"], s["weights"], s["residual"], cfg.residual_multiplier,
                                          s["norm"], cfg.rms_norm_eps))
        return dict(x=[s["residual"] for s in layers], z=out)

    def reset():
        for s in layers:
            s["residual"].copy_(s["x"])

    return _graph_state((layers, backend), step, reset)


def _prepare_moe_prefill(case, seed):
    cfg, (s,) = _make_moe(case, seed)
    backend = HipFusedExperts()
    r, eps = cfg.residual_multiplier, cfg.rms_norm_eps

    def run():
        if case["operator"]:
            y = backend.operation(s["z"], s["w1"], s["w2"], s["weights"], s["ids"],
                                  apply_router_weight_on_input=False, global_num_experts=cfg.num_local_experts)
            return dict(x=[s["x"]], z=[add_rmsnorm(s["x"], y, r, s["norm"], eps)])
        y = backend.routes(s["z"], s["w1"], s["w2"], s["ids"])
        return dict(x=[s["x"]], z=[finish_add_rmsnorm(y, s["ids"], s["weights"], s["x"], r, s["norm"], eps)])

    return dict(run=run, inputs=(s, backend))


def _exact_moe(case, seed):
    cfg, layers = _make_moe(case, seed)
    xs, zs = [], []
    for s in layers:
        y = _experts64(s["z"].double(), s["ids"].long(), s["weights"].double(), s["w1"], s["w2"])
        xs.append(s["x"].double() + cfg.residual_multiplier * y)
        zs.append(_rmsnorm64(xs[-1], s["norm"], cfg.rms_norm_eps))
    return dict(x=xs, z=zs)


# ------------------------------------------------------------ router, head --

def _make_router(case, seed):
    inp, cfg = _Inputs(seed), preset(case["model"])
    rows, h = case["tokens"], cfg.hidden_size
    layers = []
    for _ in range(case["layers"]):
        s = dict(x=inp.normal(rows, h), gate=inp.normal(cfg.num_local_experts, h, std=synth.STD),
                 norm=inp.norm_weight(h))
        if rows <= 128:  # decode hands over the o_proj as split-K partials
            s["a"] = inp.normal(SPLITS_O, rows, h, std=0.5, dtype=torch.float32)
        else:
            s["a"] = inp.normal(rows, h)
        layers.append(s)
    return cfg, layers


def _prepare_router(case, seed):
    cfg, layers = _make_router(case, seed)
    decode = case["tokens"] <= 128
    route = add_rmsnorm_route_splitk if decode else add_rmsnorm_route
    for s in layers:
        s["residual"] = s["x"].clone()

    def step():
        out = dict(x=[s["residual"] for s in layers], z=[], weights=[], ids=[])
        for s in layers:
            weights, ids, z = route(s["residual"], s["a"], cfg.residual_multiplier, s["norm"], cfg.rms_norm_eps,
                                    s["gate"], cfg.num_experts_per_tok)
            for name, value in (("z", z), ("weights", weights), ("ids", ids)):
                out[name].append(value)
        return out

    def reset():
        for s in layers:
            s["residual"].copy_(s["x"])

    return _graph_state(layers, step, reset) if decode else dict(run=step, inputs=layers)


def _exact_router(case, seed):
    """x and z; the selection has no value in 64 bits (bf16 logits tie)."""
    cfg, layers = _make_router(case, seed)
    xs, zs = [], []
    for s in layers:
        a = s["a"].double()
        xs.append(s["x"].double() + cfg.residual_multiplier * (a.sum(0) if a.dim() == 3 else a))
        zs.append(_rmsnorm64(xs[-1], s["norm"], cfg.rms_norm_eps))
    return dict(x=xs, z=zs, weights=None, ids=None)


def _make_head(case, seed):
    inp, cfg = _Inputs(seed), preset(case["model"])
    return cfg, inp.normal(case["rows"], cfg.hidden_size), inp.normal(cfg.vocab_size, cfg.hidden_size, std=synth.STD)


def _prepare_head(case, seed):
    cfg, z, head = _make_head(case, seed)
    rows = case["rows"]
    packed = PackedHead(head)
    ints = lambda value: torch.full((rows,), value, dtype=torch.int64, device=DEVICE)
    state = dict(next=ints(0), length=ints(1024), generated=ints(1), budget=ints(1 << 40),
                 active=torch.ones(rows, dtype=torch.bool, device=DEVICE))
    emit = torch.zeros(rows, 3, dtype=torch.int64, device=DEVICE)
    valid, eos = state["active"].clone(), torch.tensor([cfg.eos_token_id], device=DEVICE)
    logits = torch.empty(rows, cfg.vocab_size, dtype=BF16, device=DEVICE)

    def run():
        greedy_head(z, packed, cfg.logits_scaling, valid, state, emit, eos, True, logits_out=logits)
        return dict(logits=logits, token=emit[:, 0], next=state["next"])

    return dict(run=run, inputs=(z, packed, state, emit, valid, eos))


def _exact_head(case, seed):
    _, z, head = _make_head(case, seed)
    return dict(logits=z.double() @ head.double().t(), token=None, next=None)


# --------------------------------------------------- the blocks in 64 bits --

def _rmsnorm64(x, weight, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight.double()


def _heads64(qkv, hq, hkv, table, positions):
    """q, k (rotated, neox halves) and v ``[T, heads, 64]`` of the packed projection's output."""
    q, k, v = qkv.view(-1, hq + 2 * hkv, 64).split([hq, hkv, hkv], 1)
    cos, sin = table.double()[positions][:, None].chunk(2, -1)

    def rotate(t):
        a, b = t.chunk(2, -1)
        return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)

    return rotate(q), rotate(k), v


def _decode64(q, k, v, kc, vc, positions, scale):
    """One new token per row against its page; stores k and v in it. ``[B, Hq*64]``."""
    out = []
    for b, n in enumerate(positions.tolist()):
        kc[b, :, n], vc[b, :, n] = k[b], v[b]
        keys, values = kc[b, :, :n + 1], vc[b, :, :n + 1]
        heads = q[b].view(keys.shape[0], -1, 64)
        p = (heads @ keys.transpose(1, 2).contiguous() * scale).softmax(-1)
        out.append((p @ values.contiguous()).reshape(-1))
    return torch.stack(out)


def _causal64(q, k, v, scale):
    """Causal attention of one sequence, a KV head at a time. ``[n, Hq*64]``."""
    n, hq, _ = q.shape
    group = hq // k.shape[1]
    hidden = torch.ones(n, n, dtype=torch.bool, device=q.device).triu(1)
    out = torch.empty(n, hq, 64, dtype=torch.float64, device=q.device)
    for h in range(hq):
        s = (q[:, h] @ k[:, h // group].t() * scale).masked_fill(hidden, float("-inf"))
        out[:, h] = s.softmax(-1) @ v[:, h // group]
    return out.view(n, hq * 64)


def _experts64(z, ids, weights, w1, w2):
    out, tokens = torch.zeros_like(z), torch.arange(z.shape[0], device=z.device)
    topk = ids.shape[1]
    flat, scale = ids.reshape(-1), weights.reshape(-1)
    for e in range(w1.shape[0]):
        routes = (flat == e).nonzero().flatten()
        if routes.numel():
            rows = tokens[torch.div(routes, topk, rounding_mode="floor")]
            gate, up = (z[rows] @ w1[e].double().t()).chunk(2, -1)
            y = (gate * torch.sigmoid(gate) * up) @ w2[e].double().t()
            out.index_add_(0, rows, y * scale[routes, None])
    return out


# --------------------------------------------------------------- interface --

_PREPARE = dict(step=_prepare_step, prefill=_prepare_prefill, attn_decode=_prepare_attn_decode,
                attn_prefill=_prepare_attn_prefill, moe_decode=_prepare_moe_decode,
                moe_prefill=_prepare_moe_prefill, router=_prepare_router, head=_prepare_head)
_EXACT = dict(step=lambda c, seed: _exact_model(c, _make_step(c, seed)),
              prefill=lambda c, seed: _exact_model(c, _make_prefill(c, seed)), attn_decode=_exact_attn_decode,
              attn_prefill=_exact_attn_prefill, moe_decode=_exact_moe, moe_prefill=_exact_moe, router=_exact_router,
              head=_exact_head)


def prepare(case, seed):
    with torch.inference_mode():
        return _PREPARE[case["op"]](case, seed)


def run(state):
    with torch.inference_mode():
        return state["run"]()


def exact(case, seed):
    with torch.inference_mode():
        return _EXACT[case["op"]](case, seed)


def _work_attn(cfg, lengths, prefill):
    h, hq, hkv = cfg.hidden_size, cfg.num_attention_heads * 64, cfg.num_key_value_heads * 64
    rows = int(lengths.sum()) if prefill else lengths.size
    weights = h * (2 * hq + 2 * hkv)
    keys = float((lengths * (lengths + 1) // 2).sum()) if prefill else float(lengths.sum())
    read = 0 if prefill else float((lengths - 1).sum()) * 2 * hkv
    return dict(bytes=2 * (weights + 2 * rows * h + 2 * rows * hkv + read),
                flops=2.0 * rows * weights + 4.0 * hq * keys)


def _work_moe(cfg, rows):
    e, k, h, i = cfg.num_local_experts, cfg.num_experts_per_tok, cfg.hidden_size, cfg.intermediate_size
    live = e * (1.0 - (1.0 - k / e) ** rows)  # experts that get a route, in the mean
    return dict(bytes=2 * (live * 3 * h * i + 4.0 * rows * h) + 8.0 * rows * k, flops=2.0 * rows * k * 3 * h * i)


def _work_router(cfg, rows, partials):
    h, e = cfg.hidden_size, cfg.num_local_experts
    return dict(bytes=2 * (e * h + 3.0 * rows * h) + rows * h * (4.0 * SPLITS_O if partials else 2.0)
                + 8.0 * rows * cfg.num_experts_per_tok, flops=2.0 * rows * e * h)


def work(case):
    cfg, op = preset(case["model"]), case["op"]
    lengths = _lengths(case, case.get("rows") or case["count"]) if "low" in case else None
    rows = case.get("rows") or case.get("tokens") or int(lengths.sum())
    head = lambda n: dict(bytes=2.0 * (cfg.vocab_size * (cfg.hidden_size + n) + n * cfg.hidden_size),
                          flops=2.0 * n * cfg.vocab_size * cfg.hidden_size)
    if op in ("attn_decode", "attn_prefill"):
        parts = [_work_attn(cfg, lengths, op == "attn_prefill")]
    elif op in ("moe_decode", "moe_prefill"):
        parts = [_work_moe(cfg, rows)]
    elif op == "router":
        parts = [_work_router(cfg, rows, rows <= 128)]
    elif op == "head":
        parts = [head(rows)]
    else:
        parts = [_work_attn(cfg, lengths, op == "prefill"), _work_moe(cfg, rows), _work_router(cfg, rows, False)]
    layers = case.get("layers", 1)
    total = {key: layers * sum(p[key] for p in parts) for key in ("bytes", "flops")}
    if op in ("step", "prefill"):
        last = head(rows if op == "step" else case["count"])
        total = {key: total[key] + last[key] for key in total}
    return total


def tolerance(case):
    """bf16 outputs of fp32 sums. Another order of the sums moves values by
    one bf16 rounding here and there, and the roundings between the kernels
    of a block (q, k, v, act, y) pass it on: the blocks measure 0.002 to 0.004
    from their values in 64 bits, whole calls 0.005 to 0.008 (a token's last
    expert may change with a rounding of its logit). ``differ`` is for equal
    or nearly equal router and head logits."""
    if case["op"] in ("step", "prefill"):
        return dict(rel=2e-2, max=0.5, differ=0.01)
    return dict(rel=1e-2, max=0.1, differ=0.01)

"""The work that users of this framework have it do, as cases that can be timed and checked.

A case is a dict of plain values.  `prepare` makes what a caller holds before the call (weights, caches, the opened model,
a captured step), `run` makes one pass through the public entry points, `work` counts what the pass cannot do without, and
`exact` computes the same outputs in 64 bits with plain torch.

The models have the sizes of bench.py with a few of their layers (one or two of their periods) and the same share of their
vocabulary, so that layers and head weigh in a pass as they do in the whole model; a pass over the whole model is the same
launches more often.

    moe_layer        one MoE layer of a decode step, as a host program drives it operator by operator
    moe_prompt       the grouped expert products of a prompt chunk with popular and rare experts
    attention        decode attention of a batch whose sequences differ in length, over a quantized cache
    hybrid_step      a decode step of the hybrid MoE model, captured once and replayed, as a server runs it
    hybrid_prompt    a prompt of that model
    pakirax_serve    one more token of several requests at their own positions, as the session layer runs it
    pakirax_prompt   a prompt through the session's step driver, BF16 or fully 32-bit
    kemuzen_step     a captured decode step
    kemuzen_prompt   a prompt, BF16 or fully 32-bit"""
import math

import torch

import nvmai_amd as nv
from nvmai_amd import ops
from nvmai_amd.decoder import HybridConfig, HybridDecoder, HybridWeights
from nvmai_amd.kemuzen import KemuzenConfig, KemuzenDecoder, KemuzenWeights
from nvmai_amd.pakirax import PakiraxConfig, PakiraxDecoder, PakiraxWeights

D, F, E, K = 2048, 512, 256, 8              # the MoE layer: width, expert width, experts, chosen per token
HEADS, KV_HEADS, HEAD_DIM = 16, 2, 256      # the hybrid model's attention
LAYERS, HYBRID_LAYERS = 8, 4

# width, heads, (GLA dim, vdim), (latent dim, rot_dim, vdim, kv_rank, q_rank, window), ff, vocabulary's share
PAKIRAX = {"1k": (1024, 8, (128, 128), (128, 64, 128, 256, 768, 2048), 4096, 65536 * LAYERS // 24),
           "2k": (2048, 16, (128, 128), (128, 64, 128, 512, 1536, 4096), 8192, 248320 * LAYERS // 40)}
# width, window heads, kv heads, delta heads, key heads of them, state-space heads, window, ff, vocabulary's share, side dim
KEMUZEN = {"1k": (1024, 8, 2, 16, 8, 32, 2048, 2816, 65536 * LAYERS // 24, 128),
           "2k": (2048, 16, 4, 32, 16, 64, 4096, 5632, 248320 * LAYERS // 40, 256)}
HYBRID_VOCAB = 248320 * HYBRID_LAYERS // 40


def listed():
    return [
        # the smallest call: one token, one layer, the reference's per-layer host loop
        dict(name="moe_layer_1x4bit", kind="moe_layer", batch=1, bits=4, chosen=K),
        # the layer of a full decode batch (the framework's headline figure)
        dict(name="moe_layer_32x8bit", kind="moe_layer", batch=32, bits=8, chosen=K),
        # the experts of a long prompt
        dict(name="moe_prompt_4096x4bit", kind="moe_prompt", tokens=4096, bits=4),
        # long contexts of uneven length, a batch of eight
        dict(name="attention_8x128k_8bit", kind="attention", batch=8, context=131072, bits=8),
        # one user's generation with a long context: latency and launches
        dict(name="hybrid_step_1", kind="hybrid_step", batch=1, context=32768),
        # a served batch of the same model
        dict(name="hybrid_step_16", kind="hybrid_step", batch=16, context=32768),
        # a long prompt before the first token
        dict(name="hybrid_prompt_4096", kind="hybrid_prompt", tokens=4096),
        # continuous batching: sixteen requests, each at its own position, launched call by call
        dict(name="pakirax_serve_16", kind="pakirax_serve", size="2k", batch=16, context=8192),
        # a long prompt in the session's portions
        dict(name="pakirax_prompt_4096", kind="pakirax_prompt", size="2k", tokens=4096, act="bf16"),
        # a short prompt in full precision
        dict(name="pakirax_prompt_700_fp32", kind="pakirax_prompt", size="1k", tokens=700, act="fp32"),
        # one user's generation with the third model
        dict(name="kemuzen_step_1", kind="kemuzen_step", size="2k", batch=1, context=8192),
        # an ordinary prompt of odd length
        dict(name="kemuzen_prompt_1501", kind="kemuzen_prompt", size="2k", tokens=1501, act="bf16"),
    ]


def _log(rng, lo, hi):
    """A whole number, spread evenly over the logarithm of its range; odd as often as even."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["moe_layer", "moe_prompt", "attention", "hybrid_step", "hybrid_prompt", "pakirax_serve", "pakirax_prompt",
                       "kemuzen_step", "kemuzen_prompt"])
    bits, size = rng.choice([4, 8]), rng.choice(["1k", "2k"])
    if kind == "moe_layer":
        return dict(kind=kind, batch=rng.randint(1, 32), bits=bits, chosen=rng.randint(4, K))
    if kind == "moe_prompt":
        return dict(kind=kind, tokens=_log(rng, 64, 4096), bits=bits)
    if kind == "attention":
        return dict(kind=kind, batch=rng.randint(1, 8), context=_log(rng, 512, 131072), bits=bits)
    if kind == "hybrid_step":
        return dict(kind=kind, batch=rng.randint(1, 16), context=_log(rng, 512, 32768))
    if kind == "hybrid_prompt":
        return dict(kind=kind, tokens=_log(rng, 20, 4096))
    if kind in ("pakirax_serve", "kemuzen_step"):
        return dict(kind=kind, size=size, batch=rng.randint(1, 16), context=_log(rng, 64, 8192))
    if rng.random() < 0.3:
        return dict(kind=kind, size="1k", tokens=_log(rng, 20, 800), act="fp32")
    return dict(kind=kind, size=size, tokens=_log(rng, 20, 4096), act="bf16")


# ---- weights and configurations -------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=gen).to(dtype)


def _uniform(gen, shape, lo, hi, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(lo, hi, generator=gen).to(dtype)


def _ids(gen, n, vocab):
    return torch.randint(0, vocab, (n,), generator=gen, device="cuda", dtype=torch.int32)


def _pakirax_config(case):
    width, heads, (gk, gv), (dim, rot, vdim, kv_rank, q_rank, window), ff, vocab = PAKIRAX[case["size"]]
    g = {"type": "gla", "mixer": {"heads": heads, "dim": gk, "vdim": gv, "tau": 16.0}, "mlp": None}
    at = {"type": "latent_attention", "mlp": {"kind": "dense", "ff": ff},
          "mixer": {"heads": heads, "dim": dim, "rot_dim": rot, "vdim": vdim, "kv_rank": kv_rank, "q_rank": q_rank,
                    "scale": (dim + rot) ** -0.5, "mask": {"size": window}, "rot": {"base": 10000.0, "dims": rot}}}
    return {"architecture": "Pakirax", "vocab": vocab, "width": width, "residual_mult": 0.3, "norm": {"eps": 1e-6}, "layers": [g, at] * (LAYERS // 2)}


def _pakirax_tensors(cfg, seed):
    gen, out = _gen(seed), {}
    for name, s in PakiraxConfig(cfg).tensor_shapes(lambda i: 16).items():
        if len(s) == 1:
            bias = name.endswith(".b")
            out[name] = _normal(gen, s, 0.1, 2.0 if name.endswith("a2.b") else 0.0 if bias else 1.0)
        else:
            # the residual starts at the size of what a sublayer adds to it
            out[name] = _normal(gen, s, cfg["residual_mult"] if name == "embed" else s[1] ** -0.5)
    return out


def _kemuzen_config(case):
    width, heads, kv, dheads, dkeys, sheads, window, ff, vocab, side = KEMUZEN[case["size"]]
    mlp = {"kind": "dense", "ff": ff}
    at = {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "softcap": 50.0, "mask": {"size": window, "keep_first": 4}}
    left = {k: v for k, v in at.items() if k != "softcap"}
    left["mask"] = {"size": window}
    right = {"heads": sheads, "vdim": 64, "state": 128, "groups": 1, "conv": 4, "norm_groups": 1}
    four = lambda i: [{"type": "attention", "mixer": at, "mlp": mlp},
                      {"type": "delta", "mixer": {"heads": dheads, "kv_heads": dkeys, "dim": 128, "vdim": 128, "conv": 4}, "mlp": mlp},
                      {"type": "parallel", "mixer": {"left": left, "right": right, "left_scale": 0.7, "right_scale": 0.7}, "mlp": mlp},
                      {"type": "attention", "mixer": dict(at, kv_from=i), "mlp": mlp}]
    return {"architecture": "Kemuzen", "vocab": vocab, "width": width, "embedding": {"scale": 1.0}, "norm": {"eps": 1e-6}, "logit_softcap": 30.0,
            "token_side": {"dim": side}, "layers": sum((four(i) for i in range(0, LAYERS, 4)), [])}


def _kemuzen_tensors(cfg, seed):
    gen, out = _gen(seed), {}
    for name, s in KemuzenConfig(cfg).tensor_shapes().items():
        if len(s) == 1:
            one = name.endswith(("q.norm", "k.norm", "mix.norm", "right.norm", "side.norm", ".D"))
            out[name] = _normal(gen, s, 0.1, 1.0 if one else -3.0 if name.endswith("dt_bias") else 0.0)
        else:
            out[name] = _normal(gen, s, s[1] ** -0.5)
    return out


def _hybrid(case):
    return HybridConfig(layers=HYBRID_LAYERS, vocab=HYBRID_VOCAB, expert_bits=4, attn_bits=4, kv_bits=8, head_bits=16)


DENSE = {"pakirax": (_pakirax_config, _pakirax_tensors, PakiraxConfig, PakiraxWeights, PakiraxDecoder),
         "kemuzen": (_kemuzen_config, _kemuzen_tensors, KemuzenConfig, KemuzenWeights, KemuzenDecoder)}


def _open(case, seed, batch, max_context, max_chunk):
    """A dense model opened for `batch` sequences."""
    config, tensors, Config, Weights, Decoder = DENSE[case["kind"].split("_")[0]]
    raw = config(case)
    t = tensors(raw, seed)
    ctx, cfg = nv.Context(0, nv.ACT_FP32 if case.get("act") == "fp32" else nv.ACT_BF16), Config(raw)
    w = Weights(ctx, cfg, t.__getitem__, lambda n: t[n].shape)
    return Decoder(ctx, cfg, w, batch, max_context, max_chunk)


def _recurrent(dec):
    """The recurrent parts of a decoder's state, in the order of its layers."""
    if isinstance(dec, HybridDecoder):
        return [t for L in sorted(dec.gdn_states) for t in dec.gdn_states[L]]
    return [t for L in sorted(dec.states) for t in (dec.states[L] if isinstance(dec.states[L], tuple) else (dec.states[L],))]


def _states(dec):
    """What a pass leaves in them.  Of the inputs that a short filter keeps by position only the last few mean anything:
    they come back with the next pass."""
    return [t for t in _recurrent(dec) if t.dim() == 4 or isinstance(dec, HybridDecoder)]


def _cached(dec):
    """Tensors of the dense models' caches, in the order of their layers; layers may share one."""
    out, seen = [], set()
    for L in sorted(dec.caches):
        c = dec.caches[L]
        if id(c) not in seen:
            seen.add(id(c))
            out += [c.rows] if hasattr(c, "rows") else [c.k, c.v]
    return out


def _positions(case):
    """Where the requests of a served batch stand: from half of the longest to the longest."""
    n, top = case["batch"], case["context"] - 1
    return [top - (top // 2) * b // max(1, n - 1) for b in range(n)]


def _capture(step, restore):
    """`step` as one graph.  The first call, outside it, sizes the workspaces; `restore` undoes what that call did."""
    step()
    torch.cuda.synchronize()
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            step()
    torch.cuda.synchronize()
    restore()
    return graph


# ---- prepare ---------------------------------------------------------------------------------------------------
def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state["run"](state)


def _expert_pool(ctx, gen, n, bits):
    """n experts quantized into one pool, as a model file holds them."""
    off, stride = nv.expert_offsets(D, F, bits)
    pool = torch.empty((n, stride), dtype=torch.uint8, device="cuda")
    for rows, cols, wo, so, bo in ((F, D, off.gate_w, off.gate_s, off.gate_b), (F, D, off.up_w, off.up_s, off.up_b), (D, F, off.down_w, off.down_s, off.down_b)):
        p, s, b = nv.quantize_affine(ctx, _normal(gen, (n * rows, cols), 0.02), bits)
        pool[:, wo:wo + rows * cols * bits // 8] = p.view(n, -1)
        pool[:, so:so + rows * cols // 32] = s.view(torch.uint8).view(n, -1)
        pool[:, bo:bo + rows * cols // 32] = b.view(torch.uint8).view(n, -1)
    return pool, off


def _prepare_moe_layer(case, seed):
    ctx, gen, bits = nv.Context(0, nv.ACT_BF16), _gen(seed), case["bits"]
    pool, _ = _expert_pool(ctx, gen, E + 1, bits)
    router = _normal(gen, (E, D), 0.02)
    gate = nv.quantize_affine(ctx, _normal(gen, (1, D), 0.02), 8)
    layer = nv.moe_layer_desc(D, F, E, case["chosen"], bits, nv.rows_desc(16, router.view(torch.int16)), pool[:E], pool[E], nv.rows_desc(8, *gate))
    x = _normal(gen, (case["batch"], D))
    return dict(run=_run_moe_layer, ctx=ctx, op=nv.MoE(ctx, bits), pool=pool, router=router, gate=gate, layer=layer, x=x, y=torch.empty_like(x))


def _run_moe_layer(s):
    return s["op"].decode_layer(s["layer"], s["x"], s["y"], want_routes=True)


def _prepare_moe_prompt(case, seed):
    # logits = log popularity + Gumbel noise: the top 8 then sample experts without replacement by a Zipf(1.1) law
    ctx, gen, bits, T = nv.Context(0, nv.ACT_BF16), _gen(seed), case["bits"], case["tokens"]
    pool, off = _expert_pool(ctx, gen, E, bits)
    popular = 1.0 / torch.arange(1, E + 1, device="cuda", dtype=torch.float32) ** 1.1
    popular = popular[torch.randperm(E, device="cuda", generator=gen)]
    u = torch.rand((T, E), device="cuda", generator=gen).clamp_(1e-9, 1.0)
    top = torch.topk(torch.log(popular) - torch.log(-torch.log(u)), K, dim=-1)
    new = lambda rows, cols: torch.empty((rows, cols), dtype=torch.bfloat16, device="cuda")
    return dict(run=_run_moe_prompt, ctx=ctx, bits=bits, pool=pool, off=off, x=_normal(gen, (T, D)), idx=top.indices.to(torch.int32).contiguous(),
                w=torch.softmax(top.values, -1).to(torch.float16).contiguous(), grouping=nv.PrefillMoEGrouping(ctx),
                experts=nv.PrefillGroupedRoutedMoE(ctx, bits), reduce=nv.PrefillMoE(ctx), acts=new(T * K, F), partials=new(T * K, D), out=new(T, D))


def _run_moe_prompt(s):
    routes = s["grouping"].group_routes(s["idx"], s["w"], E)
    s["experts"].encode(s["pool"], s["off"], s["x"], D, F, routes, s["acts"], s["partials"])
    return s["reduce"].encode_reduce_token_major(s["partials"], s["w"], s["x"].shape[0], K, D, s["out"])


def _fill(ctx, gen, cache):
    """A KV cache full of quantized N(0, 1) rows."""
    quant = nv.KVCacheQuantizer(ctx)
    for b in range(cache.rows.shape[0]):
        for at in range(0, cache.rows.shape[1], 32768):
            n = min(32768, cache.rows.shape[1] - at)
            quant.encode(_normal(gen, (n, cache.elements)), cache.elements, cache.view(b, at), n, cache.elements)


def _prepare_attention(case, seed):
    ctx, gen, B, n = nv.Context(0, nv.ACT_BF16), _gen(seed), case["batch"], case["context"]
    k, v = (nv.KVCache(B, n, KV_HEADS * HEAD_DIM, case["bits"]) for _ in range(2))
    for c in (k, v):
        _fill(ctx, gen, c)
    lens = [p + 1 for p in _positions(case)]
    q = _normal(gen, (B, HEADS, HEAD_DIM))
    return dict(run=_run_attention, ctx=ctx, op=nv.Attention(ctx), q=q, k=k, v=v, lens=lens, most=n, out=torch.empty_like(q),
                device_lens=torch.tensor(lens, dtype=torch.int32, device="cuda"))


def _run_attention(s):
    return s["op"].encode_ragged(s["q"], s["k"], s["v"], HEAD_DIM, HEADS, KV_HEADS, s["device_lens"], s["most"], out=s["out"])


def _prepare_hybrid_step(case, seed):
    ctx, cfg, B = nv.Context(0, nv.ACT_BF16), _hybrid(case), case["batch"]
    dec = HybridDecoder(ctx, cfg, HybridWeights(ctx, cfg, seed=seed, std=0.015), batch=B, max_context=case["context"])
    gen = _gen(seed + 1)
    for L in sorted(dec.kv):
        for c in dec.kv[L]:
            _fill(ctx, gen, c)
    dec.tokens.copy_(_ids(gen, B, cfg.vocab))
    position = case["context"] - 1
    seeds = [nv.sampler_seed_for(seed, position + b) for b in range(B)]

    def restore():
        g = _gen(seed + 2)
        for t in _recurrent(dec):
            t.normal_(0.0, 1.0 if t.dim() == 3 else 0.05, generator=g)
    restore()
    return dict(run=_run_hybrid_step, dec=dec, position=position, graph=_capture(lambda: dec.step(position, seeds), restore))


def _run_hybrid_step(s):
    s["graph"].replay()
    return dict(logits=s["dec"].logits, state=_states(s["dec"]))


def _prepare_hybrid_prompt(case, seed):
    ctx, cfg, T = nv.Context(0, nv.ACT_BF16), _hybrid(case), case["tokens"]
    dec = HybridDecoder(ctx, cfg, HybridWeights(ctx, cfg, seed=seed, std=0.015), batch=1, max_context=T)
    return dict(run=_run_hybrid_prompt, dec=dec, tokens=_ids(_gen(seed + 1), T, cfg.vocab))


def _run_hybrid_prompt(s):
    s["dec"].reset(0)
    rows = s["dec"].prefill_chunked(s["tokens"], 0, 0, 4096)
    return dict(logits=s["dec"].logits_rows(rows), state=_states(s["dec"]))


def _fill_dense(dec, seed):
    """Caches and states of the size that a long sequence leaves: a GLA state sums some hundred tokens of order one (its decays
    are near 0.99), the delta rule's and the state-space form's hold unit keys and small steps."""
    gen = _gen(seed)
    for t in _cached(dec):
        t.normal_(0.0, 1.0, generator=gen)
    for t in _recurrent(dec):
        t.normal_(0.0, 8.0 if isinstance(dec, PakiraxDecoder) else 0.1, generator=gen)


def _prepare_pakirax_serve(case, seed):
    dec = _open(case, seed, case["batch"], case["context"] + 1, 2048)
    _fill_dense(dec, seed + 1)
    return dict(run=_run_serve, dec=dec, slots=list(range(case["batch"])), positions=_positions(case),
                tokens=_ids(_gen(seed + 2), case["batch"], dec.cfg.vocab).tolist())


def _run_serve(s):
    dec = s["dec"]
    logits = dec.logits_rows(dec.decode_rows(s["slots"], s["positions"], s["tokens"]))
    ops.argmax_rows(dec.ctx, logits, out=dec.next_tokens)
    return dict(logits=logits, state=_states(dec), cache=_cached(dec))


def _prepare_kemuzen_step(case, seed):
    dec = _open(case, seed, case["batch"], case["context"] + 1, 2048)
    _fill_dense(dec, seed + 1)
    dec.tokens.copy_(_ids(_gen(seed + 2), case["batch"], dec.cfg.vocab))
    dec.positions.copy_(torch.tensor(_positions(case), dtype=torch.int32))

    def step():
        dec.forward_hidden(None)
        dec.head()
        dec.greedy()
    return dict(run=_run_kemuzen_step, dec=dec, positions=_positions(case), graph=_capture(step, lambda: _fill_dense(dec, seed + 1)))


def _run_kemuzen_step(s):
    s["graph"].replay()
    return dict(logits=s["dec"].logits_f32, state=_states(s["dec"]), cache=_cached(s["dec"]))


def _prepare_dense_prompt(case, seed):
    dec = _open(case, seed, 1, case["tokens"], 2048)
    return dict(run=_run_dense_prompt, dec=dec, tokens=_ids(_gen(seed + 2), case["tokens"], dec.cfg.vocab))


_prepare_pakirax_prompt = _prepare_kemuzen_prompt = _prepare_dense_prompt


def _run_dense_prompt(s):
    dec = s["dec"]
    dec.reset(0)
    rows = dec.prefill_rows(s["tokens"], 0, 0)
    return dict(logits=dec.logits_rows(rows), state=_states(dec), cache=_cached(dec))


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def _affine(rows, cols, bits):
    return rows * cols * bits / 8 + rows * cols / 16


def work(case):
    kind, bits = case["kind"], case.get("bits", 8)
    expert = 3 * _affine(F, D, bits)
    if kind == "moe_layer":
        B, n = case["batch"], case["chosen"]
        hit = E * (1.0 - (1.0 - n / E) ** B)
        return dict(bytes=(hit + 1) * expert + 2 * E * D + _affine(1, D, 8) + 4 * B * D, flops=2.0 * B * ((n + 1) * 3 * D * F + E * D))
    if kind == "moe_prompt":
        T = case["tokens"]
        return dict(bytes=E * (1.0 - (1.0 - K / E) ** T) * expert + 4 * T * D + 6 * T * K, flops=6.0 * T * K * D * F)
    if kind == "attention":
        rows = sum(p + 1 for p in _positions(case))
        row = KV_HEADS * HEAD_DIM
        return dict(bytes=2.0 * rows * (row * bits / 8 + row / 16) + 4 * case["batch"] * HEADS * HEAD_DIM, flops=4.0 * rows * HEADS * HEAD_DIM)
    if kind.startswith("hybrid"):
        cfg = _hybrid(case)
        kh, vh, dk, dv, _ = cfg.gdn
        lin = (cfg.gdn_qkv_dim + cfg.gdn_value_dim + 2 * vh) * D + D * cfg.gdn_value_dim
        full = (2 * cfg.q_dim + 2 * cfg.kv_dim) * D + D * cfg.q_dim
        n_lin = sum(cfg.is_linear(L) for L in range(HYBRID_LAYERS))
        per_token = n_lin * (lin + 3.0 * vh * dk * dv) + (HYBRID_LAYERS - n_lin) * full + HYBRID_LAYERS * ((K + 1) * 3 * D * F + E * D)
        if kind == "hybrid_step":
            B, n = case["batch"], case["context"]
            return dict(bytes=cfg.bytes_per_token(B, n) * B,
                        flops=2.0 * B * (per_token + cfg.vocab * D) + B * (HYBRID_LAYERS - n_lin) * 4.0 * HEADS * HEAD_DIM * n)
        T = case["tokens"]
        hit = E * (1.0 - (1.0 - K / E) ** T)
        weights = HYBRID_LAYERS * ((hit + 1) * 3 * _affine(F, D, 4) + 2 * E * D) + n_lin * _affine(1, lin, 4) + (HYBRID_LAYERS - n_lin) * _affine(1, full, 4)
        return dict(bytes=weights + 2 * cfg.vocab * D + n_lin * 4 * vh * dk * dv + (HYBRID_LAYERS - n_lin) * 2 * T * 544,
                    flops=2.0 * T * per_token + 2.0 * cfg.vocab * D + (HYBRID_LAYERS - n_lin) * 2.0 * HEADS * HEAD_DIM * T * (T + 1.0))
    name = kind.split("_")[0]
    cfg = DENSE[name][2](DENSE[name][0](case))
    matrices = cfg.matrix_elements(16) if name == "pakirax" else cfg.matrix_elements()
    if kind in ("pakirax_serve", "kemuzen_step"):
        B, at = case["batch"], _positions(case)
        return dict(bytes=2 * matrices + sum(cfg.bytes_per_token(1, p + 1) - 2 * matrices for p in at), flops=2.0 * B * matrices)
    T = case["tokens"]
    act = 4 if case["act"] == "fp32" else 2
    return dict(bytes=2 * matrices + cfg.bytes_per_token(1, T, act) - 2 * matrices, flops=cfg.prefill_flops(T))


def tolerance(case):
    """About four times the distance from `exact` that was seen over several seeds: 32-bit contexts 2e-6, one operator between
    16-bit inputs and outputs 0.0018 (0.004 where the hidden rows of the experts are 16-bit too), models in BF16 0.006 to 0.009,
    the rounding of activations carried through their layers.  Chosen experts are the same."""
    kind = case["kind"]
    if case.get("act") == "fp32":
        return {"rel": 1e-5, "max": 1e-4}
    if kind in ("moe_layer", "attention"):
        return {"rel": 7e-3, "max": 0.1, "differ": 0.0}
    if kind == "moe_prompt":
        return {"rel": 1.6e-2, "max": 0.2}
    return {"rel": 3e-2, "max": 0.9}


# ---- the same in 64 bits, with plain torch -------------------------------------------------------------------------
def _f64(t):
    return t.view(torch.bfloat16).double() if t.dtype == torch.int16 else t.double()


def _dequantized(packed, scales, biases, bits):
    rows = packed.shape[0]
    q = packed.double() if bits == 8 else torch.stack([packed & 15, packed >> 4], -1).reshape(rows, -1).double()
    return (q.view(rows, -1, 64) * _f64(scales).view(rows, -1, 1) + _f64(biases).view(rows, -1, 1)).view(rows, -1)


def _expert(blob, bits):
    """gate, up and down of one expert, whose parts lie behind one another: codes, scales, biases of each."""
    out, at = [], 0
    for rows, cols in ((F, D), (F, D), (D, F)):
        n, m = rows * cols * bits // 8, rows * cols // 32
        parts = blob[at:at + n], blob[at + n:at + n + m], blob[at + n + m:at + n + 2 * m]
        out.append(_dequantized(parts[0].view(rows, -1), parts[1].view(torch.int16).view(rows, -1), parts[2].view(torch.int16).view(rows, -1), bits))
        at += n + 2 * m
    return out


def _ffn(x, blob, bits):
    gate, up, down = _expert(blob, bits)
    return (torch.nn.functional.silu(x @ gate.T) * (x @ up.T)) @ down.T


def _routed(x, pool, bits, idx, w):
    y = torch.zeros_like(x)
    for e in idx.unique().tolist():
        t, s = (idx == e).nonzero(as_tuple=True)
        y.index_add_(0, t, _ffn(x[t], pool[e], bits) * w[t, s, None])
    return y


def _moe(x, router, pool, gate, bits, chosen=K):
    """(output, routing weights) of the MoE block over rows x; the pool's last expert is the shared one."""
    top = torch.topk(x @ _f64(router).view(E, D).T, chosen, dim=-1)
    w = torch.softmax(top.values, -1)
    shared = _ffn(x, pool[E], bits) * torch.sigmoid(x @ _dequantized(*gate, 8).view(D, 1))
    return _routed(x, pool, bits, top.indices, w) + shared, w


def _kv_rows(rows, bits):
    """[n, elements] values of quantized cache rows: codes, then a scale and then a bias in fp16 per 64."""
    n, elements = rows.shape[0], KV_HEADS * HEAD_DIM
    size, groups = elements * bits // 8, elements // 64
    codes = rows[:, :size]
    codes = codes if bits == 8 else torch.stack([codes & 15, codes >> 4], -1).reshape(n, elements)
    meta = rows[:, size:].contiguous().view(torch.float16).double()
    return (codes.double().view(n, groups, 64) * meta[:, :groups, None] + meta[:, groups:, None]).view(n, elements)


def _attend(q, k, v, scale):
    """q [heads, d], k and v [n, kv heads, d]: one query over all of its keys."""
    H, G = q.shape[0], k.shape[1]
    s = torch.einsum("ghd,ngd->ghn", q.view(G, H // G, -1), k) * scale
    return torch.einsum("ghn,ngd->ghd", torch.softmax(s, -1), v).reshape(H, -1)


def _blockwise(T, block, fn):
    return torch.cat([fn(a, min(T, a + block)) for a in range(0, T, block)])


def _masked(q, k, v, scale, visible, bias=None, cap=0.0):
    """q [T, heads, d] over k, v [n, kv heads, d]; visible(rows) -> [rows, n]; bias(rows) -> [heads, rows, n]."""
    H, G = q.shape[1], k.shape[1]
    k, v = (t.repeat_interleave(H // G, 1).transpose(0, 1) for t in (k, v))

    def rows(a, b):
        s = (q[a:b].transpose(0, 1) @ k.transpose(1, 2)) * scale
        s = cap * torch.tanh(s / cap) if cap else s
        s = s if bias is None else s + bias(a, b)
        s = s.masked_fill(~visible(a, b), -math.inf)
        return (torch.softmax(s, -1) @ v).transpose(0, 1)
    return _blockwise(q.shape[0], 512, rows)


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def exact(case, seed):
    with torch.no_grad():
        return globals()["_exact_" + case["kind"]](case, seed)


def _exact_moe_layer(case, seed):
    s = prepare(case, seed)
    y, w = _moe(s["x"].double(), s["router"], s["pool"], s["gate"], case["bits"], case["chosen"])
    return y, None, w


def _exact_moe_prompt(case, seed):
    s = prepare(case, seed)
    return _routed(s["x"].double(), s["pool"], case["bits"], s["idx"], s["w"].double())


def _exact_attention(case, seed):
    s = prepare(case, seed)
    out = []
    for b, n in enumerate(s["lens"]):
        k, v = (_kv_rows(c.rows[b, :n], case["bits"]).view(n, KV_HEADS, HEAD_DIM) for c in (s["k"], s["v"]))
        out.append(_attend(s["q"][b].double(), k, v, HEAD_DIM ** -0.5))
    return torch.stack(out)


# -- the hybrid model
def _rotate(x, positions, dims, theta):
    """x [rows, heads, d]: its first `dims` entries turned in pairs half of `dims` apart."""
    i = torch.arange(dims // 2, dtype=torch.float64, device=x.device)
    a = positions.double()[:, None, None] * theta ** (-2.0 * i / dims)
    u, v = x[..., :dims // 2], x[..., dims // 2:dims]
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin(), x[..., dims:]], -1)


def _gdn(cfg, w, proj, tail, state, one):
    """proj [rows, ...]: the rows of one sequence (one) or one row of each sequence.  tail [sequences, taps - 1, C] and
    state [sequences, heads, dv, dk] are updated."""
    kh, vh, dk, dv, taps = cfg.gdn
    C, V = cfg.gdn_qkv_dim, cfg.gdn_value_dim
    raw, z, a, b = proj.split([C, V, vh, vh], -1)
    cw = _f64(w["conv_w"])
    past = torch.cat([tail[0], raw]) if one else torch.cat([tail, raw[:, None]], 1)
    T = raw.shape[0]
    x = torch.nn.functional.silu(sum((past[j:j + T] if one else past[:, j]) * cw[:, j] for j in range(taps)))
    if one:
        tail[0] = past[-(taps - 1):]
    else:
        tail.copy_(past[:, 1:])
    q, k, v = x.split([kh * dk, kh * dk, V], -1)
    heads = lambda t, s: (_rms(t.view(T, kh, dk), 1e-6) * s).repeat_interleave(vh // kh, 1)
    q, k, v = heads(q, 1.0 / dk), heads(k, dk ** -0.5), v.view(T, vh, dv)
    g = torch.exp(-torch.exp(_f64(w["a_log"])) * torch.nn.functional.softplus(a + _f64(w["dt_bias"])))
    beta = torch.sigmoid(b)

    def token(S, q, k, v, g, beta):                          # S [.., heads, dv, dk]
        S.mul_(g[..., None, None])
        u = (v - (S @ k[..., None])[..., 0]) * beta[..., None]
        S.add_(u[..., None] * k[..., None, :])
        return (S @ q[..., None])[..., 0]
    if one:
        y = torch.stack([token(state[0], q[t], k[t], v[t], g[t], beta[t]) for t in range(T)])
    else:
        y = token(state, q, k, v, g, beta)
    y = _rms(y, 1e-6) * _f64(w["gdn_norm"]) * torch.nn.functional.silu(z.view(T, vh, dv))
    return y.reshape(T, V) @ _dequantized(*w["out_proj"], cfg.attn_bits).T


def _hybrid_rows(dec, tokens, positions, one, states, attend):
    """Final-normed rows of one sequence (one) or of one token of each; attend(layer, q, k, v): attention over the new keys and what the caches hold."""
    cfg, W = dec.cfg, dec.w
    x = _dequantized(*(t[tokens.long()] for t in W.embed), cfg.embed_bits)
    norm = lambda x, w: _rms(x, cfg.rms_eps) * _f64(w)
    T = x.shape[0]
    for L, w in enumerate(W.layers):
        h = norm(x, w["in_norm"])
        if cfg.is_linear(L):
            x = x + _gdn(cfg, w, h @ _dequantized(*w["in_proj"], cfg.attn_bits).T, *states[L], one)
        else:
            p = h @ _dequantized(*w["qkv"], cfg.attn_bits).T
            qg, k, v = p.split([2 * cfg.q_dim, cfg.kv_dim, cfg.kv_dim], -1)
            q, gate = qg.view(T, HEADS, 2, HEAD_DIM).unbind(2)
            k, v = k.view(T, KV_HEADS, HEAD_DIM), v.view(T, KV_HEADS, HEAD_DIM)
            q, k = (_rotate(norm(t, w[n]), positions, cfg.rotary_dim, cfg.rope_theta) for t, n in ((q, "q_norm"), (k, "k_norm")))
            o = attend(L, q, k, v) * torch.sigmoid(gate)
            x = x + o.reshape(T, -1) @ _dequantized(*w["o_proj"], cfg.attn_bits).T
        x = x + _moe(norm(x, w["post_norm"]), w["router"], w["pool"], w["gate"], cfg.expert_bits)[0]
    return norm(x, W.final_norm)


def _hybrid_states(dec):
    return {L: [t.double() for t in s] for L, s in dec.gdn_states.items()}


def _exact_hybrid_step(case, seed):
    s = prepare(case, seed)
    dec, n = s["dec"], s["position"]

    def attend(L, q, k, v):
        out = []
        for b in range(q.shape[0]):
            old = [_kv_rows(c.rows[b, :n], 8).view(n, KV_HEADS, HEAD_DIM) for c in dec.kv[L]]
            out.append(_attend(q[b], torch.cat([old[0], k[b:b + 1]]), torch.cat([old[1], v[b:b + 1]]), HEAD_DIM ** -0.5))
        return torch.stack(out)
    states = _hybrid_states(dec)
    rows = _hybrid_rows(dec, dec.tokens, torch.full((case["batch"],), n, device="cuda"), False, states, attend)
    return dict(logits=rows @ _f64(dec.w.lm_head[0]).T, state=[t for L in sorted(states) for t in states[L]])


def _causal(T):
    at = torch.arange(T, device="cuda")
    return lambda a, b: at[None, :] <= at[a:b, None]


def _exact_hybrid_prompt(case, seed):
    s = prepare(case, seed)
    dec, T = s["dec"], case["tokens"]
    states = _hybrid_states(dec)
    rows = _hybrid_rows(dec, s["tokens"], torch.arange(T, device="cuda"), True, states,
                        lambda L, q, k, v: _masked(q, k, v, HEAD_DIM ** -0.5, _causal(T)))
    return dict(logits=rows[-1:] @ _f64(dec.w.lm_head[0]).T, state=[t for L in sorted(states) for t in states[L]])


# -- the dense models: tensors by name from the seed; a pass is the rows of one sequence from zero or one row per sequence
def _dense_inputs(case, seed):
    """(configuration, tensors in 64 bits, prepared state, tokens, positions, whether they are one sequence's)"""
    name = case["kind"].split("_")[0]
    cfg = DENSE[name][0](case)
    t = {k: v.double() for k, v in DENSE[name][1](cfg, seed).items() if k != "embed"}
    s = prepare(case, seed)
    one = case["kind"].endswith("prompt")
    tokens = (s["tokens"] if one else torch.tensor(s["tokens"]).cuda() if "tokens" in s else s["dec"].tokens).long()
    positions = torch.arange(case["tokens"], device="cuda") if one else torch.tensor(s["positions"], device="cuda")
    return cfg, t, s["dec"], tokens, positions, one


def _layer(t, p):
    return {k[len(p):]: v for k, v in t.items() if k.startswith(p)}


def _layer_norm(x, t, name, eps):
    x = x - x.mean(-1, keepdim=True)
    return _rms(x, eps) * t[name] + t[name + ".b"]


def _store(ring, rows, index, keep):
    """Rows that are still there when the last one is written: index(position) -> place."""
    n = len(rows)
    for at in range(max(0, n - keep), n):
        ring[index(at)] = rows[at]


def _window(positions, size, keep=0):
    at = torch.arange(len(positions), device="cuda")
    return lambda a, b: (at[None, :] <= at[a:b, None]) & ((at[a:b, None] - at[None, :] < size) | (at[None, :] < keep))


def _exact_gla(t, m, eps, h, S, one):
    H, dk, dv = m["heads"], m["dim"], m["vdim"]
    T = h.shape[0]
    q, k, v = ((h @ t[n].T).view(T, H, -1) for n in "qkv")
    alpha = torch.exp(torch.nn.functional.logsigmoid((h @ t["a1"].T) @ t["a2"].T + t["a2.b"]) / m["tau"]).view(T, H, dk)

    def token(S, q, k, v, alpha):
        S.mul_(alpha[..., None]).add_(k[..., None] * v[..., None, :])
        return (q[..., None, :] @ S)[..., 0, :]
    q = q * dk ** -0.5
    y = torch.stack([token(S[0], q[i], k[i], v[i], alpha[i]) for i in range(T)]) if one else token(S, q, k, v, alpha)
    return ((_rms(y, eps) * t["norm"]).reshape(T, -1) * torch.nn.functional.silu(h @ t["g"].T)) @ t["o"].T


def _exact_latent(t, m, eps, h, ring, positions, one):
    H, dim, rot, vdim, rank, T = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], h.shape[0]
    base, size, cap = m["rot"]["base"], m["mask"]["size"], ring.shape[1]
    q = ((_rms(h @ t["dq"].T, eps) * t["dq.norm"]) @ t["uq"].T).view(T, H, dim + rot)
    qn, qr = q[..., :dim], _rotate(q[..., dim:], positions, m["rot"]["dims"], base)
    ckv = h @ t["dkv"].T
    c = _rms(ckv[:, :rank], eps) * t["dkv.norm"]
    k = _rotate(ckv[:, None, rank:], positions, m["rot"]["dims"], base)[:, 0]
    uk, uv = t["uk"].view(H, dim, rank), t["uv"].view(H, vdim, rank)
    if one:
        keys = torch.cat([torch.einsum("nr,hdr->nhd", c, uk), k[:, None].expand(-1, H, -1)], -1)
        o = _masked(torch.cat([qn, qr], -1), keys, torch.einsum("nr,hvr->nhv", c, uv), m["scale"], _window(positions, size))
        _store(ring[0], torch.cat([c, k], -1), lambda p: (p % cap, slice(0, rank + rot)), cap)
    else:
        o = []
        for b, p in enumerate(positions.tolist()):
            ring[b, p % cap, :rank + rot] = torch.cat([c[b], k[b]])
            rows = ring[b, torch.arange(max(0, p - size + 1), p + 1, device="cuda") % cap]
            cc, kk = rows[:, :rank], rows[:, rank:rank + rot]
            s = (torch.einsum("hd,hdr->hr", qn[b], uk) @ cc.T + qr[b] @ kk.T) * m["scale"]
            o.append(torch.einsum("hr,hvr->hv", torch.softmax(s, -1) @ cc, uv))
        o = torch.stack(o)
    return (o * torch.sigmoid(h @ t["g"].T)[..., None]).reshape(T, -1) @ t["o"].T


def _exact_pakirax(case, seed):
    cfg, t, dec, tokens, positions, one = _dense_inputs(case, seed)
    eps, mult = cfg["norm"]["eps"], cfg["residual_mult"]
    embed = dec.w.embed.double()
    x = embed[tokens]
    states, rings = [s.double() for s in _recurrent(dec)], [c.double() for c in _cached(dec)]
    for i, layer in enumerate(cfg["layers"]):
        lt, m = _layer(t, "l%d." % i), layer["mixer"]
        h = _layer_norm(x, lt, "norm1", eps)
        mix = _layer(lt, "mix.")
        if layer["type"] == "gla":
            y = _exact_gla(mix, m, eps, h, states[i // 2], one)
        else:
            y = _exact_latent(mix, m, eps, h, rings[i // 2], positions, one)
        x = x + mult * _layer_norm(y, lt, "norm1b", eps)
        if layer["mlp"]:
            y = torch.nn.functional.gelu(_layer_norm(x, lt, "norm2", eps) @ lt["mlp.up"].T) @ lt["mlp.down"].T
            x = x + mult * _layer_norm(y, lt, "norm2b", eps)
    x = _layer_norm(x[-1:] if one else x, t, "final.norm", eps)
    return dict(logits=x @ embed.T, state=states, cache=rings)


_exact_pakirax_serve = _exact_pakirax_prompt = _exact_pakirax


def _exact_window(t, m, eps, h, cache, positions, one, new, bias=False, alibi=False):
    """Heads' outputs [T, heads * vdim].  cache: k [slots, kv heads, rows, dim], v [slots, kv heads, vdim, rows], the pinned rows, and the
    rows of this pass, left by the layer that writes it (new) for those that share it."""
    H, G, dim, vdim, T = m["heads"], m["kv_heads"], m["dim"], m["vdim"], h.shape[0]
    b = lambda n: t[n + ".b"] if bias else 0.0
    size, keep = m["mask"]["size"], m["mask"].get("keep_first", 0)
    q = _rms((h @ t["q"].T + b("q")).view(T, H, dim), eps) * t["q.norm"]
    if new:
        k = _rms((h @ t["k"].T + b("k")).view(T, G, dim), eps) * t["k.norm"]
        v = (h @ t["v"].T + b("v")).view(T, G, vdim)
        cache["rows"] = k, v
    k, v = cache["rows"]
    K_, V_, pinned = cache["k"], cache["v"], cache["pinned"]
    ring = K_.shape[2] - pinned
    place = lambda p: p if p < pinned else pinned + p % ring          # where a position is read
    cap = m.get("softcap") or 0.0
    slopes = 2.0 ** (-8.0 * torch.arange(1, H + 1, dtype=torch.float64, device="cuda") / H)
    if one:
        if new:
            K_[0, :, [place(p) for p in range(T)]], V_[0, :, :, [place(p) for p in range(T)]] = k.transpose(0, 1), v.permute(1, 2, 0)
            turned = list(range(min(T, pinned)))                      # first tokens lie in the ring too
            K_[0, :, [pinned + p for p in turned]], V_[0, :, :, [pinned + p for p in turned]] = k[turned].transpose(0, 1), v[turned].permute(1, 2, 0)
        at = torch.arange(T, device="cuda", dtype=torch.float64)
        pull = (lambda a, c: -slopes[:, None, None] * (at[a:c, None] - at[None, :])) if alibi else None
        return _masked(q, k, v, m["scale"], _window(positions, size, keep), pull, cap).reshape(T, -1)
    out = []
    for s, p in enumerate(positions.tolist()):
        if new:
            for r in {pinned + p % ring} | ({p} if p < pinned else set()):
                K_[s, :, r], V_[s, :, :, r] = k[s], v[s]
        keys = [j for j in range(min(keep, p + 1)) if p - j >= size] + list(range(max(0, p - size + 1), p + 1))
        where = torch.tensor([place(j) for j in keys], device="cuda")
        kk, vv = K_[s][:, where], V_[s][:, :, where]
        z = torch.einsum("ghd,gnd->ghn", q[s].view(G, H // G, dim), kk) * m["scale"]
        z = cap * torch.tanh(z / cap) if cap else z
        if alibi:
            z = z - slopes.view(G, H // G, 1) * (p - torch.tensor(keys, device="cuda", dtype=torch.float64))
        out.append(torch.einsum("ghn,gvn->ghv", torch.softmax(z, -1), vv).reshape(-1))
    return torch.stack(out)


def _exact_filter(raw, weight, bias, history, positions, one):
    """silu of a causal filter per channel; history [slots, rows, channels], a ring by position, is updated."""
    taps, n, T = weight.shape[1], history.shape[1], raw.shape[0]
    if one:
        past = torch.cat([raw.new_zeros(taps - 1, raw.shape[1]), raw])
        y = sum(past[j:j + T] * weight[:, j] for j in range(taps))
        _store(history[0], raw, lambda p: p % n, taps - 1)
    else:
        y = raw * weight[:, -1]
        for s, p in enumerate(positions.tolist()):
            for back in range(1, min(taps - 1, p) + 1):
                y[s] += history[s, (p - back) % n] * weight[:, taps - 1 - back]
            history[s, p % n] = raw[s]
    return torch.nn.functional.silu(y if bias is None else y + bias)


def _exact_delta(t, m, eps, h, history, S, positions, one):
    H, G, dim, vdim, T = m["heads"], m["kv_heads"], m["dim"], m["vdim"], h.shape[0]
    raw = torch.cat([h @ t[n].T for n in "qkv"], -1)
    z = _exact_filter(raw, torch.cat([t[n + ".conv"] for n in "qkv"]), None, history, positions, one)
    q, k, v = z.split([G * dim, G * dim, H * vdim], -1)
    unit = lambda x: (x.view(T, G, dim) * torch.rsqrt((x.view(T, G, dim) ** 2).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
    q, k, v = unit(q) * dim ** -0.5, unit(k), v.view(T, H, vdim)
    beta = torch.sigmoid(h @ t["b"].T)
    g = torch.exp(-torch.exp(t["A_log"]) * torch.nn.functional.softplus(h @ t["a"].T + t["dt_bias"]))

    def token(S, q, k, v, beta, g):
        S.mul_(g[..., None, None])
        u = beta[..., None] * (v - (k[..., None, :] @ S)[..., 0, :])
        S.add_(k[..., None] * u[..., None, :])
        return (q[..., None, :] @ S)[..., 0, :]
    y = torch.stack([token(S[0], q[i], k[i], v[i], beta[i], g[i]) for i in range(T)]) if one else token(S, q, k, v, beta, g)
    return ((_rms(y, eps) * t["norm"]).reshape(T, -1) * torch.nn.functional.silu(h @ t["g"].T)) @ t["o"].T


def _exact_ssd(t, m, eps, h, history, S, positions, one):
    H, P, N, G, T = m["heads"], m["vdim"], m["state"], m["groups"], h.shape[0]
    inner, gn = H * P, G * N
    z, x, B, C, dt = (h @ t["in"].T).split([inner, inner, gn, gn, H], -1)
    order = lambda v: torch.cat([v[inner + gn:], v[inner:inner + gn], v[:inner]])        # [x | B | C] -> [C | B | x]
    y = _exact_filter(torch.cat([C, B, x], -1), order(t["conv"]), order(t["conv.b"]), history, positions, one)
    C, B, x = y.split([gn, gn, inner], -1)
    C, B = (v.view(T, G, N).repeat_interleave(H // G, 1) for v in (C, B))
    x, dt = x.view(T, H, P), torch.nn.functional.softplus(dt + t["dt_bias"])
    g = torch.exp(-torch.exp(t["A_log"]) * dt)

    def token(S, C, B, x, dt, g):
        S.mul_(g[..., None, None]).add_(B[..., None] * (dt[..., None] * x)[..., None, :])
        return (C[..., None, :] @ S)[..., 0, :]
    y = torch.stack([token(S[0], C[i], B[i], x[i], dt[i], g[i]) for i in range(T)]) if one else token(S, C, B, x, dt, g)
    y = (y + t["D"][:, None] * x).reshape(T, inner) * torch.nn.functional.silu(z)
    return (_rms(y.view(T, m["norm_groups"], -1), eps).reshape(T, inner) * t["norm"]) @ t["o"].T


def _exact_kemuzen(case, seed):
    cfg, t, dec, tokens, positions, one = _dense_inputs(case, seed)
    eps, W, side = cfg["norm"]["eps"], cfg["width"], cfg["token_side"]["dim"]
    embed = dec.w.embed.double()
    e = torch.arange(W, dtype=torch.float64, device="cuda")
    angle = positions.double()[:, None] * 10000.0 ** (-(e - e % 2) / W)
    x = embed[tokens] * cfg["embedding"]["scale"] + torch.where(e % 2 == 1, angle.cos(), angle.sin())
    states, rings = [s.double() for s in _recurrent(dec)], [c.double() for c in _cached(dec)]
    caches, n_state, n_ring = {}, 0, 0
    for i, layer in enumerate(cfg["layers"]):
        lt, m, kind = _layer(t, "l%d." % i), layer["mixer"], layer["type"]
        mix = _layer(lt, "mix.")
        a = m["left"] if kind == "parallel" else m
        if kind != "delta" and a.get("kv_from") is None:
            caches[i] = dict(k=rings[n_ring], v=rings[n_ring + 1], pinned=dec.caches[i].pinned)
            n_ring += 2
        if kind == "attention":
            y = _exact_window(mix, m, eps, x, caches[m.get("kv_from", i)], positions, one, "kv_from" not in m, bias=True) @ mix["o"].T + mix["o.b"]
        elif kind == "delta":
            y = _exact_delta(mix, m, eps, x, states[n_state], states[n_state + 1], positions, one)
            n_state += 2
        else:
            lm, rm = _layer(mix, "left."), _layer(mix, "right.")
            o = _exact_window(lm, a, eps, x, caches[i], positions, one, True, alibi=True)
            o = (o.view(len(x), a["heads"], -1) * torch.sigmoid(x @ lm["g"].T)[..., None]).reshape(len(x), -1) @ lm["o"].T
            y = m["left_scale"] * o + m["right_scale"] * _exact_ssd(rm, m["right"], eps, x, states[n_state], states[n_state + 1], positions, one)
            n_state += 2
        norm = lambda v, n: _rms(v, eps) * (1.0 + lt[n])
        x = x + norm(y, "norm1")
        x = x + norm((torch.nn.functional.silu(x @ lt["mlp.gate"].T) * (x @ lt["mlp.up"].T)) @ lt["mlp.down"].T, "norm2")
        s = torch.nn.functional.gelu(x @ lt["side.gate"].T, approximate="tanh") * t["side.embed"][tokens, i * side:(i + 1) * side]
        x = x + _rms(s @ lt["side.proj"].T, eps) * lt["side.norm"]
    x = _rms(x[-1:] if one else x, eps) * (1.0 + t["final.norm"])
    logits, cap = x @ embed.T, cfg["logit_softcap"]
    return dict(logits=cap * torch.tanh(logits / cap) if one else logits, state=states[1::2], cache=rings)


_exact_kemuzen_step = _exact_kemuzen_prompt = _exact_kemuzen

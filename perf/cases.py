"""The work that programs built on this framework have it do, as cases that can be timed and checked.

listed() names twelve of them, draw() gives more of the same ranges.  prepare() makes what such a
program holds before the call (inputs, filled caches, weights, captured graphs), run() is one pass
through the public entry points, work() the bytes and operations that a pass cannot do without,
tolerance() what another correct implementation may differ by, and exact() the same result from
plain torch in 64 bits.

Kinds of cases:
  decode   one token per sequence: (append it and) attend to the compressed cache
  prefill  a chunk of query tokens, already appended, attends to the cache
  append   a whole prompt's keys and values are compressed into a fresh cache
  mlp      add + RMSNorm, gate/up projection, SwiGLU, down projection
  model    one decode step of the example decoder, captured as a graph, to its logits
"""
from __future__ import annotations

import math

import torch

from chronoquant_mlx_amd import ChronoQuantCache, chronoquant_sdpa, patch
from chronoquant_mlx_amd.models import fused, qwen
from chronoquant_mlx_amd.synth import DecodeConfig, make_kv_device

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
EPS = 1e-6
# The codec settings in use: name -> (stride_k, stride_v, bits_k, bits_v, dead_zone_v).  "standard" is
# the package's default, "ftv3" its Full-Throttle V3 preset.
CODECS = {"standard": (32, 8, 4, 4, 0.05), "ftv3": (64, 32, 4, 3, 0.05), "plain": (32, 8, 4, 4, 0.0),
          "odd": (48, 24, 4, 4, 0.05)}


def _decode(name, batch, q_heads, kv_heads, head_dim, tokens, codec, dtype, ragged=False, append=True,
            layers=1, graph=False, dense=False):
    c = dict(kind="decode", batch=batch, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
             tokens=tokens, codec=codec, dtype=dtype, ragged=ragged, append=append, layers=layers,
             graph=graph, dense=dense)
    return dict(c, name=name) if name else c


def _prefill(name, batch, q_heads, kv_heads, head_dim, tokens, chunk, codec, dtype, mask="causal",
             dense=False):
    c = dict(kind="prefill", batch=batch, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim,
             tokens=tokens, chunk=chunk, codec=codec, dtype=dtype, mask=mask, dense=dense)
    return dict(c, name=name) if name else c


def _append(name, batch, kv_heads, head_dim, tokens, codec, dtype, token_major, dense=False):
    c = dict(kind="append", batch=batch, kv_heads=kv_heads, head_dim=head_dim, tokens=tokens,
             codec=codec, dtype=dtype, token_major=token_major, dense=dense)
    return dict(c, name=name) if name else c


def _mlp(name, rows, hidden, inter, dtype):
    c = dict(kind="mlp", rows=rows, hidden=hidden, inter=inter, dtype=dtype)
    return dict(c, name=name) if name else c


def _model(name, layers, hidden, inter, vocab, tokens, codec):
    c = dict(kind="model", layers=layers, hidden=hidden, inter=inter, vocab=vocab, tokens=tokens,
             codec=codec)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest call: one layer's attention for one token of a 4K multi-head cache, called
        # eagerly, as the reference's patched models call it
        _decode("decode_mha_4k", 1, 8, 8, 128, 4096, "plain", "f16", append=False),
        # a serving loop at batch 1: every layer appends its token and attends to 16K tokens of
        # standard-mode cache, all of it in one graph
        _decode("decode_gqa_16k_graph", 1, 32, 8, 128, 16384, "standard", "f16", layers=16, graph=True),
        # batched serving in Full-Throttle V3: 8 sequences of 32K, one layer, eager
        _decode("decode_ftv3_b8_32k", 8, 32, 8, 128, 32768, "ftv3", "f16"),
        # batched serving of sequences of every length
        _decode("decode_ragged_b32", 32, 32, 8, 128, 32767, "standard", "f16", ragged=True),
        # models with wide heads (head_dim 256 is the largest the operator takes)
        _decode("decode_d256_b4_16k", 4, 16, 4, 256, 16001, "standard", "bf16"),
        # prompt processing: the last 512-token chunk of an 8K prompt, as the end-to-end run does it
        _prefill("prefill_512_of_8k", 1, 32, 8, 128, 8192, 512, "ftv3", "bf16"),
        # the same at the largest: a 2048-token chunk that ends a 32K prompt
        _prefill("prefill_2048_of_32k", 1, 32, 8, 128, 32768, 2048, "standard", "f16"),
        # prompt processing of a model with wide heads
        _prefill("prefill_d256_512_of_8k", 1, 16, 4, 256, 8192, 512, "standard", "bf16"),
        # prompt processing under an explicit boolean mask: a layer with a sliding window, two
        # prompts of an odd length
        _prefill("prefill_window_b2", 2, 32, 8, 128, 4001, 257, "standard", "f16", mask="window"),
        # encode: a 16K prompt compressed into a fresh cache, laid out as a projection leaves it
        _append("append_prompt_16k", 1, 8, 128, 16384, "ftv3", "bf16", token_major=True),
        # one token through a layer's MLP
        _mlp("mlp_token", 1, 4096, 12288, "bf16"),
        # a whole decode step of the end-to-end model (fewer layers), 8K tokens cached
        _model("model_token_8k", 4, 4096, 12288, 151936, 8192, "ftv3"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


HEADS = ((8, 8), (32, 8), (32, 8), (16, 4), (16, 2), (32, 4))


def draw(rng):
    kind = rng.choice(("decode", "decode", "decode", "prefill", "prefill", "append", "mlp", "model"))
    codec = rng.choice(("standard", "standard", "ftv3", "ftv3", "plain", "odd"))
    dtype = rng.choice(("f16", "bf16"))
    nq, nkv = rng.choice(HEADS)
    head_dim = rng.choice((128, 128, 128, 256, 64, 80))
    dense = codec == "ftv3" and rng.random() < 0.25
    if kind == "decode":
        batch = _log(rng, 1, 32)
        # at most the largest listed cache; half of that away from head_dim 128
        most = 32 * 16384 * 8 * 128 // (1 if head_dim == 128 else 8)
        tokens = min(_log(rng, 64, 32768), most // (batch * nkv * head_dim))
        graph = batch * tokens * nkv * head_dim <= 16384 * 8 * 128
        return _decode(None, batch, nq, nkv, head_dim, tokens, codec, dtype, ragged=rng.random() < 0.4,
                       append=graph or rng.random() < 0.7, layers=rng.randint(2, 8) if graph else 1,
                       graph=graph, dense=dense)
    if kind == "prefill":
        mask = rng.choice(("causal", "causal", "causal", "none", "window"))
        # scores of one call: the largest listed chunk, or, with wide or narrow heads, a mask or
        # dense rows, the 512-token one
        most = 32 * 2048 * 32768 if head_dim == 128 and mask != "window" and not dense else 16 * 512 * 8192
        batch = _log(rng, 1, 8)
        chunk = min(_log(rng, 2, 2048), int(math.sqrt(most // (batch * nq))))
        tokens = min(_log(rng, chunk, 32768), most // (batch * nq * chunk))
        return _prefill(None, batch, nq, nkv, head_dim, max(tokens, chunk), chunk, codec, dtype, mask, dense)
    if kind == "append":
        batch = _log(rng, 1, 8)
        tokens = min(_log(rng, 16, 32768), 32768 * 8 * 128 // (batch * nkv * head_dim))
        return _append(None, batch, nkv, head_dim, tokens, codec, dtype, rng.random() < 0.5, dense)
    if kind == "mlp":
        rows = 1 if rng.random() < 0.5 else _log(rng, 2, 512)
        hidden, inter = rng.choice(((4096, 12288), (2048, 6144), (1024, 3072)))
        return _mlp(None, rows, hidden, inter, dtype)
    hidden, inter = rng.choice(((4096, 12288), (2048, 6144)))
    return _model(None, rng.randint(1, 4), hidden, inter, 151936, _log(rng, 128, 16384),
                  rng.choice(("standard", "ftv3")))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g, device="cuda").to(dtype)


def _cache(case, capacity=0):
    sk, sv, bk, bv, dz = CODECS[case["codec"]]
    return ChronoQuantCache(stride_k=sk, stride_v=sv, delta_bits_k=bk, delta_bits_v=bv, dead_zone_k=0.0,
                            dead_zone_v=dz, capacity=capacity, dense_residuals=case.get("dense", False))


def _kv(case, seed, layer=0):
    """The prompt's keys and values [batch, kv_heads, tokens, head_dim]: AR(1) streams per channel, a
    hundredth of the channels 8 times as strong as the rest."""
    cfg = DecodeConfig("prompt", case["batch"], case.get("q_heads", case["kv_heads"]), case["kv_heads"],
                       case["head_dim"], case["tokens"], 1, 1, outlier_frac=0.01)
    k, v = make_kv_device(cfg, case["tokens"], case["batch"], torch.device("cuda"),
                          seed=1_000_003 * (seed % 1_000_003) + 17 * layer)
    return k.to(DTYPES[case["dtype"]]), v.to(DTYPES[case["dtype"]])


def _decode_inputs(case, seed, layer):
    """(k, v, new k, new v, q) of one layer."""
    g = _generator(7919 * seed + layer + 1)
    dt, B, D = DTYPES[case["dtype"]], case["batch"], case["head_dim"]
    k, v = _kv(case, seed, layer)
    k1, v1 = (_normal(g, B, case["kv_heads"], 1, D, dtype=dt) for _ in range(2))
    return k, v, k1, v1, _normal(g, B, case["q_heads"], 1, D, dtype=dt)


def _lengths(case, seed):
    """Tokens cached per sequence."""
    if not case["ragged"]:
        return [case["tokens"]] * case["batch"]
    g = torch.Generator()
    g.manual_seed(seed)
    return torch.randint(max(1, case["tokens"] // 32), case["tokens"] + 1, (case["batch"],), generator=g).tolist()


def _mask(case):
    """What the attention call takes for the mask; the window is a quarter of the tokens."""
    if case["mask"] != "window":
        return "causal" if case["mask"] == "causal" else None
    T, L = case["tokens"], case["chunk"]
    q = torch.arange(T - L, T, device="cuda")[:, None]
    k = torch.arange(T, device="cuda")[None, :]
    return (q >= k) & (q < k + max(1, T // 4))


def _capture(fn):
    """fn() captured as a graph after one warm-up on the capture's stream: (graph, fn's outputs)."""
    side, here = torch.cuda.Stream(), torch.cuda.current_stream()
    side.wait_stream(here)
    with torch.cuda.stream(side), torch.no_grad():
        fn()
    here.wait_stream(side)
    side.wait_stream(here)
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph, stream=side):
        out = fn()
    here.wait_stream(side)
    return graph, out


def _prepare_decode(case, seed):
    scale = case["head_dim"] ** -0.5
    lengths = _lengths(case, seed)
    lens = torch.tensor(lengths, dtype=torch.int32, device="cuda")
    layers = []
    for i in range(case["layers"]):
        k, v, k1, v1, q = _decode_inputs(case, seed, i)
        cache = _cache(case, case["tokens"] + 1)
        cache.update_and_fetch(k, v)
        if case["append"]:  # at each sequence's end, the same place in every pass
            cache.bind_device_position(lens, case["tokens"] + 1)
        elif case["ragged"]:  # nothing is appended: the cache reads these lengths
            cache.bind_device_position(lens - 1, case["tokens"] + 1, lengths=lens, update_lengths=False)
        layers.append((cache, k1, v1, q))

    def step():
        outs = []
        for cache, k1, v1, q in layers:
            if case["append"]:
                cache.update_and_fetch(k1, v1)
            outs.append(chronoquant_sdpa(q, None, None, cache, scale))
        return outs

    state = {"step": step}
    if case["graph"]:
        state["graph"], state["out"] = _capture(step)
    return state


def _model_args(case):
    heads = case["hidden"] // 128
    return qwen.ModelArgs(hidden_size=case["hidden"], num_hidden_layers=case["layers"],
                          num_attention_heads=heads, num_key_value_heads=heads // 4, head_dim=128,
                          intermediate_size=case["inter"], vocab_size=case["vocab"], max_position=16640)


def _model_cache_case(case):
    """The decode case that the model's layers make."""
    a = _model_args(case)
    return _decode(None, 1, a.num_attention_heads, a.num_key_value_heads, 128, case["tokens"],
                   case["codec"], "bf16", layers=case["layers"])


def _model_token(case, seed):
    return torch.tensor([[seed % case["vocab"]]], device="cuda")


def _prepare_model(case, seed):
    patch.apply()
    model = qwen.random_model(_model_args(case), seed=seed)
    sub = _model_cache_case(case)
    pos = torch.tensor([case["tokens"]], dtype=torch.int32, device="cuda")
    lens = torch.empty_like(pos)
    caches = []
    for i in range(case["layers"]):
        cache = _cache(sub, case["tokens"] + 1)
        cache.update_and_fetch(*_kv(sub, seed, i))
        cache.bind_device_position(pos, case["tokens"] + 1, lengths=lens, update_lengths=i == 0)
        caches.append(cache)
    token = _model_token(case, seed)
    graph, logits = _capture(lambda: model(token, caches, positions=pos.long()[:, None]))
    return {"graph": graph, "out": logits, "model": model, "caches": caches, "token": token, "pos": pos}


def _mlp_inputs(case, seed):
    g = _generator(seed)
    dt, h, n = DTYPES[case["dtype"]], case["hidden"], case["inter"]
    return {"x": _normal(g, 1, case["rows"], h, dtype=dt), "res": _normal(g, 1, case["rows"], h, dtype=dt),
            "norm": (1 + 0.1 * _normal(g, h)).to(dt), "gate_up": (0.02 * _normal(g, 2 * n, h)).to(dt),
            "down": (0.02 * _normal(g, h, n)).to(dt)}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        return dict(_prepare_decode(case, seed), kind=kind)
    if kind == "prefill":
        k, v = _kv(case, seed)
        cache = _cache(case, case["tokens"])
        cache.update_and_fetch(k, v)
        return {"kind": kind, "cache": cache, "q": _prefill_q(case, seed), "mask": _mask(case),
                "scale": case["head_dim"] ** -0.5}
    if kind == "append":
        k, v = _kv(case, seed)
        if case["token_major"]:  # [batch, tokens, heads, dims] in memory, as a projection writes it
            k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (k, v))
        return {"kind": kind, "case": case, "k": k, "v": v}
    if kind == "mlp":
        return dict(_mlp_inputs(case, seed), kind=kind)
    return dict(_prepare_model(case, seed), kind=kind)


def _prefill_q(case, seed):
    return _normal(_generator(7919 * seed + 1), case["batch"], case["q_heads"], case["chunk"],
                   case["head_dim"], dtype=DTYPES[case["dtype"]])


def run(state):
    kind = state["kind"]
    if kind in ("decode", "model"):
        if "graph" in state:
            state["graph"].replay()
            return state["out"]
        return state["step"]()
    if kind == "prefill":
        return chronoquant_sdpa(state["q"], None, None, state["cache"], state["scale"], state["mask"])
    if kind == "append":
        cache = _cache(state["case"], state["case"]["tokens"])
        cache.update_and_fetch(state["k"], state["v"])
        return [t.view(torch.int32) if t.dtype == torch.uint32 else t for t in cache.state]
    gate_up, h = fused.linear_rms_norm(state["x"], state["res"], state["norm"], EPS, state["gate_up"],
                                       want_h=True)
    return fused.linear_silu(gate_up, state["down"]), h


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _cache_bytes(case, tokens):
    """Bytes of one sequence's compressed keys and values."""
    sk, sv, bk, bv, _ = CODECS[case["codec"]]
    H, D, total = case["kv_heads"], case["head_dim"], 0
    for stride, bits in ((sk, bk), (sv, bv)):
        anchors = -(-tokens // stride)
        field = bits if case.get("dense") else 4
        row = 4 * (-(-D * field // 32)) + 2
        total += H * (anchors * 2 * D + (tokens - anchors) * row)
    return total


def _decode_work(case, lengths):
    qo = 2 * 2 * case["batch"] * case["q_heads"] * case["head_dim"]
    kv = 2 * 2 * case["batch"] * case["kv_heads"] * case["head_dim"] if case["append"] else 0
    flops = 4 * sum(lengths) * case["q_heads"] * case["head_dim"]
    return case["layers"] * (sum(_cache_bytes(case, n) for n in lengths) + qo + kv), case["layers"] * flops


def work(case):
    kind = case["kind"]
    if kind == "decode":
        if case["ragged"]:  # lengths are uniform between these two
            mean = (max(1, case["tokens"] // 32) + case["tokens"]) // 2
        else:
            mean = case["tokens"]
        b, f = _decode_work(case, [mean + case["append"]] * case["batch"])
        return {"bytes": b, "flops": f}
    if kind == "prefill":
        B, T, L, nq, D = (case[n] for n in ("batch", "tokens", "chunk", "q_heads", "head_dim"))
        if case["mask"] == "none":
            pairs = L * T
        else:
            window = max(1, T // 4) if case["mask"] == "window" else T
            pairs = sum(min(T - L + i + 1, window) for i in range(L))
        return {"bytes": B * _cache_bytes(case, T) + 2 * 2 * B * nq * L * D, "flops": 4 * B * nq * D * pairs}
    if kind == "append":
        raw = 2 * 2 * case["batch"] * case["kv_heads"] * case["tokens"] * case["head_dim"]
        return {"bytes": raw + case["batch"] * _cache_bytes(case, case["tokens"]), "flops": 0}
    if kind == "mlp":
        weights = 3 * case["hidden"] * case["inter"]
        return {"bytes": 2 * (weights + 4 * case["rows"] * case["hidden"] + case["hidden"]),
                "flops": 2 * weights * case["rows"]}
    a = _model_args(case)
    qkv = (a.num_attention_heads + 2 * a.num_key_value_heads) * 128
    per_layer = case["hidden"] * (qkv + a.num_attention_heads * 128 + 3 * case["inter"])
    weights = case["layers"] * per_layer + case["hidden"] * case["vocab"]
    b, f = _decode_work(_model_cache_case(case), [case["tokens"] + 1])
    return {"bytes": 2 * weights + 2 * case["vocab"] + b, "flops": 2 * weights + f}


# ---------------------------------------------------------------------------
# tolerances and the 64-bit results
# ---------------------------------------------------------------------------
def tolerance(case):
    kind = case["kind"]
    if kind == "append":
        return "exact"  # codes, scales and anchors are defined bit by bit
    if kind == "model":  # measured: 0.017 from the 64-bit logits
        return {"rel": 3e-2, "max": 0.2}
    if kind == "mlp" and case["dtype"] == "bf16":  # two roundings of the rows in between: measured 0.005
        return {"rel": 2e-2, "max": 0.15}
    # one rounding of the output to 8 or 11 significant bits, and of the 16-bit attention weights or
    # of the intermediate rows before it: measured 0.0017 (bf16) and 0.0004 (fp16)
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.1}
    return {"rel": 2e-3, "max": 0.03}


def _residual_codes(x, stride, bits, dead_zone):
    """The codec in plain torch for tokens x [H, T, D] of one sequence, every operation rounded to x's
    type as the format defines: (anchors [H, n, D], codes of every token, 0 for anchors, fp16 scales)."""
    def rnd(t):
        return t.to(x.dtype).double()

    half = 2 ** (bits - 1)
    anchors = x[:, ::stride].to(torch.float16)
    group = torch.arange(x.shape[1], device=x.device) // stride
    d = rnd(x.double() - rnd(anchors)[:, group])
    # smaller denominators count as zero: 0 itself for fp16
    eps = torch.tensor(1e-10).to(x.dtype).double().item()
    top = d.abs().amax(-1, keepdim=True)
    scale = rnd(top / (half - 1))
    if dead_zone > 0:
        limit = rnd(top * torch.tensor(dead_zone).to(x.dtype).double().item())
        d = torch.where(d.abs() < limit, 0.0, d)
        kept = d.abs().amax(-1, keepdim=True)
        scale = rnd(torch.where(kept < eps, top, kept) / (half - 1))
    code = rnd(d / torch.where(scale < eps, 1.0, scale)).round().clamp(-half, half - 1).nan_to_num(0.0)
    code = torch.where(scale < eps, 0.0, code)
    code[:, ::stride] = 0
    return anchors, code, scale.to(torch.float16)


def _rebuilt(x, stride, bits, dead_zone, as_f16):
    """What the cache gives back for x [H, T, D], in 64 bits: anchor + code * scale, or (as_f16) with
    the product and the sum rounded to fp16 as the reconstruction is defined."""
    anchors, code, scale = _residual_codes(x, stride, bits, dead_zone)
    group = torch.arange(x.shape[1], device=x.device) // stride
    a, c = anchors.double()[:, group], code * scale.double()
    return (a + c.to(torch.float16).double()).to(torch.float16).double() if as_f16 else a + c


def _scaled(q, scale):
    """Queries times the scale, both of the queries' type, in 64 bits."""
    return (q.double() * torch.tensor(scale).to(q.dtype).double().item()).to(q.dtype).double()


def _attention(q, k, v, mask=None):
    """[H, G, L, D] scaled queries over k and v [H, T, D], one head at a time."""
    out = torch.empty_like(q)
    for h in range(q.shape[0]):
        for g in range(q.shape[1]):
            s = q[h, g] @ k[h].T
            if mask is not None:
                s = s.masked_fill(~mask, -math.inf)
            out[h, g] = torch.softmax(s, -1) @ v[h]
    return out


def _exact_decode_layer(case, q, k, v, lengths):
    """q [B, nq, 1, D]; k, v [B, H, T, D] with each sequence's tokens first."""
    sk, sv, bk, bv, dz = CODECS[case["codec"]]
    B, nq, _, D = q.shape
    H = k.shape[1]
    qs = _scaled(q, D ** -0.5).reshape(B, H, nq // H, 1, D)
    out = []
    for b in range(B):
        kk = _rebuilt(k[b, :, :lengths[b]], sk, bk, 0.0, False)
        vv = _rebuilt(v[b, :, :lengths[b]], sv, bv, dz, False)
        s = torch.softmax(torch.einsum("hgld,htd->hglt", qs[b], kk), -1)
        out.append(torch.einsum("hglt,htd->hgld", s, vv).reshape(nq, 1, D))
    return torch.stack(out)


def _with_token(x, token, lengths):
    """x [B, H, T, D] with one more token at each sequence's end."""
    x = torch.cat([x, torch.zeros_like(token)], 2)
    for b, n in enumerate(lengths):
        x[b, :, n] = token[b, :, 0]
    return x


def _exact_decode(case, seed):
    lengths, outs = _lengths(case, seed), []
    for i in range(case["layers"]):
        k, v, k1, v1, q = _decode_inputs(case, seed, i)
        if case["append"]:
            k, v = _with_token(k, k1, lengths), _with_token(v, v1, lengths)
        outs.append(_exact_decode_layer(case, q, k, v, [n + case["append"] for n in lengths]))
        del k, v
    return outs


def _exact_prefill(case, seed):
    sk, sv, bk, bv, dz = CODECS[case["codec"]]
    k, v = _kv(case, seed)
    q = _prefill_q(case, seed)
    B, nq, L, D = q.shape
    H, T = k.shape[1], case["tokens"]
    mask = _mask(case)
    if isinstance(mask, str):
        mask = torch.arange(T - L, T, device="cuda")[:, None] >= torch.arange(T, device="cuda")[None]
    out = []
    for b in range(B):
        kk, vv = _rebuilt(k[b], sk, bk, 0.0, True), _rebuilt(v[b], sv, bv, dz, True)
        out.append(_attention(_scaled(q[b], D ** -0.5).reshape(H, nq // H, L, D), kk, vv, mask))
    return torch.stack(out).reshape(B, nq, L, D)


def _packed(code, stride, field, bits, dense):
    """Codes [H, T, D] -> the P-frames' rows of words [H, P, W] (int32)."""
    H, T, D = code.shape
    keep = torch.arange(T, device=code.device) % stride != 0
    u = code[:, keep].long() + (2 ** (bits - 1) if dense else 8)
    words = -(-D * field // 32)
    at = field * torch.arange(D, device=code.device)
    rows = torch.zeros(H, u.shape[1], words + 1, dtype=torch.long, device=code.device)
    low = (u << (at % 32))
    rows.index_add_(2, at // 32, low & 0xFFFFFFFF)
    rows.index_add_(2, at // 32 + 1, low >> 32)
    rows = rows[..., :words]
    return (rows - ((rows >> 31) << 32)).to(torch.int32)


def _exact_append(case, seed):
    sk, sv, bk, bv, dz = CODECS[case["codec"]]
    k, v = _kv(case, seed)
    got = {}
    for name, x, stride, bits, zone in (("k", k, sk, bk, 0.0), ("v", v, sv, bv, dz)):
        dense = case["dense"] and bits < 4
        parts = []
        for b in range(x.shape[0]):
            anchors, code, scale = _residual_codes(x[b], stride, bits, zone)
            keep = torch.arange(x.shape[2], device="cuda") % stride != 0
            parts.append((anchors, _packed(code, stride, bits if dense else 4, bits, dense),
                          scale[:, keep, 0]))
        got[name] = [torch.stack(t) for t in zip(*parts)]
    return [got["k"][0], got["v"][0], got["k"][1], got["k"][2], got["v"][1], got["v"][2]]


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _gated(gate_up):
    gate, up = gate_up.chunk(2, -1)
    return torch.nn.functional.silu(gate) * up


def _exact_mlp(case, seed):
    s = _mlp_inputs(case, seed)
    h = s["x"].double() + s["res"].double()
    return _gated(_rms(h, s["norm"]) @ s["gate_up"].double().T) @ s["down"].double().T, h


def _exact_model(case, seed):
    model = qwen.random_model(_model_args(case), seed=seed)
    a, sub, n = model.args, _model_cache_case(case), case["tokens"]
    nq, nkv = a.num_attention_heads, a.num_key_value_heads
    cos, sin = model.rope.cos[n].double(), model.rope.sin[n].double()

    def turned(x):
        x1, x2 = x[..., :64], x[..., 64:]
        return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], -1)

    x = model.embed_tokens.weight[_model_token(case, seed)[0, 0]].double()
    for i, layer in enumerate(model.layers):
        att, mlp = layer.self_attn, layer.mlp
        qkv = (att.qkv_proj.weight.double() @ _rms(x, layer.input_layernorm.weight)).reshape(-1, 128)
        q = turned(_rms(qkv[:nq], att.q_norm.weight)).to(torch.bfloat16)
        k1 = turned(_rms(qkv[nq:nq + nkv], att.k_norm.weight)).to(torch.bfloat16)
        v1 = qkv[nq + nkv:].to(torch.bfloat16)
        k, v = _kv(sub, seed, i)
        k, v = (_with_token(t, u[None, :, None], [n]) for t, u in ((k, k1), (v, v1)))
        o = _exact_decode_layer(sub, q[None, :, None], k, v, [n + 1])
        x = x + att.o_proj.weight.double() @ o.reshape(-1)
        gate_up = mlp.gate_up_proj.weight.double() @ _rms(x, layer.post_attention_layernorm.weight)
        x = x + mlp.down_proj.weight.double() @ _gated(gate_up)
    return (model.lm_head.weight.double() @ _rms(x, model.norm.weight)).reshape(1, 1, -1)


def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "decode":
            return _exact_decode(case, seed)
        if kind == "prefill":
            return _exact_prefill(case, seed)
        if kind == "append":
            return _exact_append(case, seed)
        return _exact_mlp(case, seed) if kind == "mlp" else _exact_model(case, seed)

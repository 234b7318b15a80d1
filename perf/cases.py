"""What users of this framework have it do, as cases that can be timed: the operators called on their own, batch-1
generation through a session, batched decode steps and prefill passes of int8 decoders.

A case is a dict of plain values; "kind" says which path it takes:

  linear     DequantMatMul as an operator: one int8 weight matrix times M activation rows
  qlinear    DynamicQuantizeLinear of M rows, then QuantizedMatMul (the int8-activation form of a linear layer)
  attention  the attention operator over a KV cache: decode (one query row per sequence) or causal prefill
  generate   LlmSession.generate_ids: the prompt through a prefill executor, then greedy tokens, batch 1
  batch      one decode step of a batched executor over caches that already hold a context
  prefill    one pass of a prefill executor over whole prompts (logits of every row, caches filled)

The models are the two decoder shapes of this repository's benchmark (TinyLlama-1.1B and Llama-3-8B, the latter also with
fewer of its identical layers), with synthetic int8 weights.
"""
import importlib
import math

import numpy as np
import torch

mynn = importlib.import_module("my-nn-engine_amd")

MODELS = {
    "tinyllama": dict(n_layers=22, hidden=2048, n_heads=32, n_kv_heads=4, head_dim=64, ffn=5632, vocab=32000, eps=1e-5, rope_theta=10000.0),
    "llama3_8b": dict(n_layers=32, hidden=4096, n_heads=32, n_kv_heads=8, head_dim=128, ffn=14336, vocab=128256, eps=1e-5,
                      rope_theta=500000.0),
}
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
CODES = {"f32": mynn.F32, "f16": mynn.F16, "bf16": mynn.BF16}
EB = {"f32": 4, "f16": 2, "bf16": 2}
# (N, K) of the models' linear layers: q|k|v, o, gate or up, gate|up, down
LINEARS = [(2560, 2048), (2048, 2048), (5632, 2048), (11264, 2048), (2048, 5632), (6144, 4096), (4096, 4096), (14336, 4096), (28672, 4096),
           (4096, 14336)]


def listed():
    return [
        # one float row against one int8 matrix: the DequantizeLinear -> MatMul subgraph of an ONNX model on its own
        dict(name="linear_f32_m1", kind="linear", dtype="f32", m=1, n=5632, k=2048),
        # a handful of rows (a small batch's down projection)
        dict(name="linear_bf16_m6", kind="linear", dtype="bf16", m=6, n=4096, k=14336),
        # a prompt of no particular length through gate|up
        dict(name="linear_f16_m300", kind="linear", dtype="f16", m=300, n=11264, k=2048),
        # int8 activations, about a hundred rows
        dict(name="qlinear_f16_m97", kind="qlinear", dtype="f16", m=97, n=4096, k=4096),
        # attention of a decode step: four sequences, 2048 cached keys
        dict(name="attention_decode_b4", kind="attention", model="tinyllama", dtype="f16", b=4, sq=1, keys=2048, kv8=False),
        # causal attention over one ragged prompt
        dict(name="attention_prefill_777", kind="attention", model="llama3_8b", dtype="bf16", b=1, sq=777, keys=777, kv8=False),
        # a chat turn: 128 prompt tokens, then a reply, batch 1
        dict(name="generate_tinyllama", kind="generate", model="tinyllama", layers=22, dtype="f16", prompt=128, chunk=128, new=64, max_seq=384,
             kv8=False, w8a8=False),
        # the same with wide layers, a prompt that does not fill its last chunk, and a long int8 cache
        dict(name="generate_8b_kv8", kind="generate", model="llama3_8b", layers=8, dtype="f16", prompt=200, chunk=128, new=32, max_seq=4096,
             kv8=True, w8a8=False),
        # a small serving batch
        dict(name="batch8_tinyllama", kind="batch", model="tinyllama", layers=22, dtype="bf16", b=8, ctx=500, kv8=False, paged=False),
        # a full serving batch of the larger model over a paged cache
        dict(name="batch32_8b_paged", kind="batch", model="llama3_8b", layers=32, dtype="f16", b=32, ctx=2048, kv8=False, paged=True),
        # whole prompts in bulk
        dict(name="prefill_tinyllama_8x1024", kind="prefill", model="tinyllama", layers=22, dtype="f16", b=8, s=1024, w8a8=False),
        # one prompt of a user, int8 activations
        dict(name="prefill_8b_w8a8_1x500", kind="prefill", model="llama3_8b", layers=8, dtype="f16", b=1, s=500, w8a8=True),
    ]


# ------------------------------------------------------------------ drawn cases
def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_linear(rng):
    if rng.random() < 0.75:
        n, k = rng.choice(LINEARS)
    else:  # matrices of other models: any number of rows, rows of whole 16-byte pieces
        n, k = _log(rng, 500, 16000), 32 * _log(rng, 16, 256)
    return n, k


def _draw_once(rng):
    kind = rng.choice(["linear", "linear", "qlinear", "attention", "attention", "generate", "batch", "batch", "prefill", "prefill"])
    dtype = rng.choice(["f16", "bf16"])
    if kind in ("linear", "qlinear"):
        n, k = _draw_linear(rng)
        m = _log(rng, 1, 4096)
        return dict(kind=kind, dtype="f32" if kind == "linear" and m == 1 and rng.random() < 0.5 else dtype, m=m, n=n, k=k)
    model = rng.choice(["tinyllama", "llama3_8b"])
    if kind == "attention":
        if rng.random() < 0.5:
            return dict(kind=kind, model=model, dtype=dtype, b=_log(rng, 1, 32), sq=1, keys=_log(rng, 128, 8192), kv8=rng.random() < 0.3)
        s = _log(rng, 16, 2048)
        return dict(kind=kind, model=model, dtype=dtype, b=_log(rng, 1, 8), sq=s, keys=s, kv8=False)
    layers = MODELS[model]["n_layers"] if model == "tinyllama" else rng.randint(4, 10)
    if kind == "generate":
        # (an int8 cache is taken for its length)
        option = rng.choice(["plain", "plain", "kv8", "w8a8"])
        return dict(kind=kind, model=model, layers=layers, dtype="f16" if option != "plain" else dtype, prompt=_log(rng, 16, 256),
                    chunk=rng.choice([64, 128, 256]), new=_log(rng, 16, 64), max_seq=4096 if option == "kv8" else rng.choice([512, 1024, 4096]),
                    kv8=option == "kv8", w8a8=option == "w8a8")
    if kind == "batch":
        return dict(kind=kind, model=model, layers=layers, dtype=dtype, b=_log(rng, 2, 64), ctx=_log(rng, 100, 3000), kv8=rng.random() < 0.3,
                    paged=rng.random() < 0.4)
    w8a8 = rng.random() < 0.3
    return dict(kind=kind, model=model, layers=layers, dtype="f16" if w8a8 else dtype, b=_log(rng, 1, 8), s=_log(rng, 16, 1024), w8a8=w8a8)


def _cost(case):
    w = work(case)
    return w["bytes"] / 8e12 + w["flops"] / 2.5e15


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw_once(rng)
        if _cost(case) <= most:
            return case


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _codes(n, k, g):
    """int8 [n, k] as a per-channel quantiser leaves normally distributed weights: the largest of a row near 127."""
    return (torch.randn((n, k), generator=g, device="cuda") * 36.0).round_().clamp_(-127, 127).to(torch.int8)


def _linear_weight(n, k, std, dtype, g):
    """codes and scales of a matrix whose values have the given spread, a little different for every channel"""
    return _codes(n, k, g), ((torch.rand((n,), generator=g, device="cuda") * 0.2 + 0.9) * (std / 36.0)).to(dtype)


def _model_config(case, max_seq):
    return dict(MODELS[case["model"]], n_layers=case["layers"], dtype=CODES[case["dtype"]], max_seq=max_seq)


def _model_weights(cfg, dtype, g):
    """A decoder that is sure of its next token, as a trained one is: every token's embedding is the output row of another
    token, and the layers add less to the residual stream than the embedding holds, so the greedy token stays far ahead of
    the others and does not hang on the last bit of a sum.  Keys, queries, values and gates have unit variance."""
    H, F, V = cfg["hidden"], cfg["ffn"], cfg["vocab"]
    QD, KD = cfg["n_heads"] * cfg["head_dim"], cfg["n_kv_heads"] * cfg["head_dim"]

    def norm():
        return (1.0 + 0.1 * torch.randn((H,), generator=g, device="cuda")).to(dtype)

    embed = _linear_weight(V, H, 1.0, dtype, g)
    head = torch.empty_like(embed[0])
    head[torch.randperm(V, generator=g, device="cuda")] = embed[0]
    w = {"embed": embed, "lm_head": (head, ((torch.rand((V,), generator=g, device="cuda") * 0.02 + 0.99) * (20.0 / H / 36.0)).to(dtype)),
         "final_norm": norm()}
    for i in range(cfg["n_layers"]):
        for name, n, k, std in (("q", QD, H, 1.0), ("k", KD, H, 1.0), ("v", KD, H, 1.0), ("o", H, QD, 0.25), ("gate", F, H, 1.0), ("up", F, H, 1.0),
                                ("down", H, F, 0.25)):
            w["layers.%d.%s" % (i, name)] = _linear_weight(n, k, std / math.sqrt(k), dtype, g)
        w["layers.%d.norm1" % i], w["layers.%d.norm2" % i] = norm(), norm()
    return w


def _caches(cfg, batch, rows, dtype, kv8, g=None, pages=None):
    """(what Decoder takes as kv, the same memory as a few tensors): one K and one V cache per layer, zeros or (g) a random
    context; pages = (number of pages, rows per page): page pools instead of [batch, heads, rows, D] caches."""
    lead = (cfg["n_layers"], 2) + ((batch, cfg["n_kv_heads"], rows) if pages is None else (pages[0], cfg["n_kv_heads"], pages[1]))
    D = cfg["head_dim"]
    if kv8:
        codes = torch.zeros(lead + (D,), dtype=torch.int8, device="cuda")
        scale = torch.zeros(lead, dtype=dtype, device="cuda")
        if g is not None:
            for layer in range(lead[0]):
                codes[layer] = (torch.randn(lead[1:] + (D,), generator=g, device="cuda") * 45.0).round_().clamp_(-127, 127).to(torch.int8)
                scale[layer] = torch.rand(lead[1:], generator=g, device="cuda") * 0.008 + 0.018
        return [(codes[i, 0], codes[i, 1], scale[i, 0], scale[i, 1]) for i in range(lead[0])], [codes, scale]
    kv = torch.zeros(lead + (D,), dtype=dtype, device="cuda")
    if g is not None:
        for layer in range(lead[0]):
            kv[layer] = torch.randn(lead[1:] + (D,), generator=g, device="cuda")
    return [(kv[i, 0], kv[i, 1]) for i in range(lead[0])], [kv]


class _DeviceMemory:
    """Device memory of the library as a tensor's source (the executor's logits buffer).  The tensor keeps this object, and
    this object the executor whose memory it is."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<i2", data=(ptr, False), version=2)


def _logits(model, dec, dtype):
    """The executor's logits buffer, [rows, vocab]: the same memory after every step."""
    ptr = mynn.lib().mynn_model_logits_device(dec.handle)
    shape = (dec.cfg.batch * dec.cfg.seq_q, dec.cfg.vocab)
    return torch.as_tensor(_DeviceMemory(model, ptr, shape), device="cuda").view(dtype)


class _Model:
    """Executors of one model and what they hold, let go in the order the library asks for."""

    def __init__(self):
        self.parts = []

    def keep(self, part):
        self.parts.append(part)
        return part

    def __del__(self):
        for part in reversed(self.parts):
            part.close()


def prepare(case, seed):
    g, dtype = _generator(seed), DTYPES[case["dtype"]]
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        x = torch.randn((m, k), generator=g, device="cuda").to(dtype)
        wq, scale = _linear_weight(n, k, 1.0 / math.sqrt(k), dtype, g)
        return dict(kind=kind, x=x, wq=wq, scale=scale)
    if kind == "qlinear":
        m, n, k = case["m"], case["n"], case["k"]
        x = torch.randn((m, k), generator=g, device="cuda").to(dtype)
        wq, scale = _linear_weight(n, k, 1.0 / math.sqrt(k), dtype, g)
        return dict(kind=kind, x=x, wq=wq, scale=scale)
    if kind == "attention":
        c = MODELS[case["model"]]
        B, Hq, Hkv, D, L = case["b"], c["n_heads"], c["n_kv_heads"], c["head_dim"], case["keys"]
        q = torch.randn((B, Hq, case["sq"], D), generator=g, device="cuda").to(dtype)
        # a decode cache has room for the tokens to come
        rows = L if case["sq"] > 1 else (L + 256) // 256 * 256
        if case["kv8"]:
            kv = [(torch.randn((B, Hkv, rows, D), generator=g, device="cuda") * 45.0).round_().clamp_(-127, 127).to(torch.int8) for _ in range(2)]
            sc = [(torch.rand((B, Hkv, rows), generator=g, device="cuda") * 0.008 + 0.018).to(dtype) for _ in range(2)]
        else:
            kv = [torch.randn((B, Hkv, rows, D), generator=g, device="cuda").to(dtype) for _ in range(2)]
            sc = [None, None]
        return dict(kind=kind, q=q, k=kv[0], v=kv[1], k_scale=sc[0], v_scale=sc[1], scale=D ** -0.5, causal=case["sq"] > 1, active=L)

    model = _Model()
    if kind == "generate":
        cfg = _model_config(case, case["max_seq"])
        weights = _model_weights(cfg, dtype, g)
        kv, caches = _caches(cfg, 1, case["max_seq"], dtype, case["kv8"])
        prompt = torch.randint(0, cfg["vocab"], (case["prompt"],), generator=g, device="cuda").cpu().numpy()
        wset = model.keep(mynn.WeightSet(cfg, weights))
        options = dict(kv=kv, quant_kv_cache=case["kv8"], quantize_activations=case["w8a8"], weight_set=wset)
        dec = model.keep(mynn.Decoder(cfg, weights, **options))
        pre = model.keep(mynn.Decoder(cfg, weights, seq_q=case["chunk"], **options))
        session = model.keep(mynn.LlmSession(dec, pre))
        return dict(kind=kind, model=model, weights=weights, session=session, prompt=prompt, new=case["new"], caches=caches)
    if kind == "batch":
        B, ctx, page = case["b"], case["ctx"], 256
        max_seq = (ctx + 256) // 256 * 256
        cfg = _model_config(case, max_seq)
        weights = _model_weights(cfg, dtype, g)
        pages = None
        if case["paged"]:
            pool = model.keep(mynn.KvPool(B * (max_seq // page), page))
            pages = model.keep(mynn.KvPages(pool, B, max_seq))
            pages.reserve(ctx + 1)
        kv, caches = _caches(cfg, B, max_seq, dtype, case["kv8"], g, (B * (max_seq // page), page) if case["paged"] else None)
        toks = torch.randint(0, cfg["vocab"], (B,), generator=g, device="cuda").cpu().numpy()
        torch.cuda.synchronize()
        dec = model.keep(mynn.Decoder(cfg, weights, batch=B, kv=kv, quant_kv_cache=case["kv8"], kv_pages=pages))
        return dict(kind=kind, model=model, weights=weights, dec=dec, toks=toks, ctx=ctx, caches=caches, logits=_logits(model, dec, dtype))
    if kind == "prefill":
        B, S = case["b"], case["s"]
        cfg = _model_config(case, (S + 63) // 64 * 64)
        weights = _model_weights(cfg, dtype, g)
        kv, caches = _caches(cfg, B, cfg["max_seq"], dtype, False)
        ids = torch.randint(0, cfg["vocab"], (B * S,), generator=g, device="cuda").cpu().numpy()
        torch.cuda.synchronize()
        dec = model.keep(mynn.Decoder(cfg, weights, seq_q=S, batch=B, kv=kv, quantize_activations=case["w8a8"]))
        return dict(kind=kind, model=model, weights=weights, dec=dec, ids=ids, positions=np.arange(S), caches=caches, logits=_logits(model, dec, dtype))
    raise ValueError(kind)


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return mynn.dequant_matmul(state["x"], state["wq"], state["scale"])
    if kind == "qlinear":
        y, s, _ = mynn.dynamic_quantize_linear(state["x"])
        out, _ = mynn.quantized_matmul(y, s, state["wq"], state["scale"], want_acc=False)
        return [y, s, out]
    if kind == "attention":
        return mynn.attention(state["q"], state["k"], state["v"], state["scale"], is_causal=state["causal"], active=state["active"],
                              k_scale=state["k_scale"], v_scale=state["v_scale"])
    if kind == "generate":
        session = state["session"]
        session.reset()
        ids = session.generate_ids(state["prompt"], state["new"])
        return dict(ids=np.asarray(ids), caches=state["caches"])
    if kind == "batch":
        ctx = state["ctx"]
        ids, _ = state["dec"].step(state["toks"], [ctx], ctx, ctx + 1)
        return dict(ids=np.asarray(ids), logits=state["logits"], caches=state["caches"])
    dec = state["dec"]
    ids, _ = dec.step(state["ids"], state["positions"], 0, len(state["positions"]))
    return dict(ids=np.asarray(ids), logits=state["logits"], caches=state["caches"])


# ------------------------------------------------------------------ what a pass cannot do without
def _layer_weights(c):
    H, F = c["hidden"], c["ffn"]
    QD, KD = c["n_heads"] * c["head_dim"], c["n_kv_heads"] * c["head_dim"]
    return H * (QD + 2 * KD) + QD * H + 3 * F * H


def work(case):
    eb, kind = EB[case["dtype"]], case["kind"]
    if kind in ("linear", "qlinear"):
        m, n, k = case["m"], case["n"], case["k"]
        nbytes = n * k + n * eb + m * k * eb + m * n * eb
        if kind == "qlinear":
            nbytes += m * k + m * eb
        return dict(bytes=nbytes, flops=2 * m * n * k)
    c = MODELS[case["model"]]
    Hq, Hkv, D, V, H = c["n_heads"], c["n_kv_heads"], c["head_dim"], c["vocab"], c["hidden"]
    kv_row = 2 * Hkv * (D + eb if case.get("kv8") else D * eb)  # one token's keys and values
    if kind == "attention":
        B, sq, L = case["b"], case["sq"], case["keys"]
        pairs = sq * (sq + 1) // 2 if sq > 1 else L
        return dict(bytes=2 * B * Hq * sq * D * eb + B * L * kv_row, flops=4 * B * Hq * D * pairs)
    n_layers = case["layers"]
    layers, head = n_layers * _layer_weights(c), V * H

    def step(rows, seqs, past):
        """one executor step: `rows` new tokens in each of `seqs` sequences behind `past` cached ones"""
        pairs = rows * past + rows * (rows + 1) // 2
        return (layers + head + seqs * n_layers * (past + 2 * rows) * kv_row + seqs * rows * (H + V * eb),
                2 * seqs * rows * (layers + head) + 4 * seqs * n_layers * Hq * D * pairs)

    if kind == "batch":
        steps = [step(1, case["b"], case["ctx"])]
    elif kind == "prefill":
        steps = [step(case["s"], case["b"], 0)]
    else:
        prompt, chunk = case["prompt"], case["chunk"]
        steps = [step(min(chunk, prompt - p), 1, p) for p in range(0, prompt, chunk)]
        steps += [step(1, 1, prompt + i) for i in range(case["new"] - 1)]
    return dict(bytes=sum(s[0] for s in steps), flops=sum(s[1] for s in steps))


def tolerance(case):
    """Sums in f32 in any order, one rounding per stored value; a model passes those roundings on from layer to layer, and
    where activations or cached rows are quantised a rounding can move a code by one."""
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    bf16 = case["dtype"] == "bf16"
    if case["kind"] in ("linear", "qlinear", "attention"):
        return {"rel": 1e-2 if bf16 else 1.5e-3}
    if case.get("w8a8"):
        return {"rel": 3e-2, "max": 0.5}
    if case.get("kv8"):
        return {"rel": 3e-2 if bf16 else 1e-2, "max": 0.5, "differ": 1e-2}
    return {"rel": 2e-2 if bf16 else 5e-3, "max": 0.5 if bf16 else 0.2}

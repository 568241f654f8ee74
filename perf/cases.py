"""What the framework is timed on: encoder forwards as programs that embed,
search and rerank texts make them, through ``edgebert_amd.Model``.

A case is a model shape and dtype, an entry point and a batch:

* ``model``: ``minilm`` (MiniLM-L6: H 384, 12 heads of 32, FFN 1536, 6 layers)
  or ``base`` (BERT-base: H 768, 12 heads of 64, FFN 3072, 12 layers), with
  ``layers`` encoder layers of it (fewer than the whole: a block of the model);
* ``dtype``: ``fp32`` or ``bf16``, the model's compute dtype;
* ``entry``: ``device`` (``encode_device``: ids, mask and vectors stay in HBM,
  as in a serving loop), ``host`` (``encode_ids``: numpy in, numpy out,
  blocking) or ``score`` (``score_device``: cross-encoder logits);
* ``B`` x ``S`` padded positions, of which a sequence has ``lo`` .. ``hi`` tokens
  (spread evenly over that range, in an order that the seed picks).
"""
import functools
import math

import numpy as np
import torch

import edgebert_amd as eb

_SHAPES = {"minilm": (384, 12, 1536, 6), "base": (768, 12, 3072, 12)}
_VOCAB, _POS, _EPS = 30522, 512, 1e-12


def _case(name, model, dtype, entry, B, S, lo, hi, layers=None):
    return {"name": name, "model": model, "layers": layers or _SHAPES[model][3], "dtype": dtype, "entry": entry,
            "B": B, "S": S, "lo": lo, "hi": hi}


def listed():
    return [
        # One search query as an interactive program sends it: host buffers in
        # and out, nothing but latency.
        _case("query_1x16", "minilm", "fp32", "host", 1, 16, 16, 16),
        # A handful of tokens on a serving loop's own buffers.
        _case("few_2x8", "minilm", "fp32", "device", 2, 8, 8, 8),
        # A server's mixed batch of sentences, padded to the longest.
        _case("short_32x128", "minilm", "fp32", "device", 32, 128, 8, 128),
        # Bulk embedding, every sequence full: the benchmark's headline shape.
        _case("bulk_256x128", "minilm", "fp32", "device", 256, 128, 128, 128),
        # Long passages of uneven length, where attention weighs most.
        _case("long_16x512", "minilm", "fp32", "device", 16, 512, 256, 512),
        # Indexing a corpus of uneven texts from host memory.
        _case("index_256x128", "minilm", "fp32", "host", 256, 128, 8, 128),
        # Reranking the hits of one query (an odd batch) with a cross-encoder.
        _case("rerank_99x250", "minilm", "fp32", "score", 99, 250, 40, 250),
        # An odd, small batch: sizes that no tile divides.
        _case("odd_37x53", "minilm", "fp32", "device", 37, 53, 5, 53),
        # The wider model (heads of 64) in fp32.
        _case("base_fp32_48x128", "base", "fp32", "device", 48, 128, 16, 128),
        # The wider model's largest job, in bf16.
        _case("base_bf16_1024x128", "base", "bf16", "device", 1024, 128, 128, 128),
        # bf16 on long passages: two layers of the model, a block of its own.
        _case("base_bf16_40x512", "base", "bf16", "device", 40, 512, 200, 512, 2),
        # bf16 on a server's mixed batch of sentences.
        _case("base_bf16_64x128", "base", "bf16", "device", 64, 128, 8, 128, 2),
    ]


def _lengths(c):
    n = c["B"]
    return [c["lo"] + ((c["hi"] - c["lo"]) * i) // max(n - 1, 1) if n > 1 else c["hi"] for i in range(n)]


def _flops(c):
    H, _, I, _ = _SHAPES[c["model"]]
    n = _lengths(c)
    per_token = 2.0 * (4 * H * H + 2 * H * I)
    return c["layers"] * (per_token * sum(n) + 4.0 * H * sum(x * x for x in n))


# A drawn case's largest work: one pass then costs no more than the bf16 (or
# the largest fp32) listed one.
_MOST = {"bf16": 2.2e13, "fp32": 8.0e11}


def draw(rng):
    while True:
        model = rng.choice(["minilm", "minilm", "minilm", "base"])
        dtype = rng.choice(["fp32", "fp32", "bf16"]) if model == "minilm" else rng.choice(["fp32", "bf16", "bf16"])
        S = int(round(math.exp(rng.uniform(math.log(4), math.log(512)))))
        B = int(round(math.exp(rng.uniform(math.log(1), math.log(1024)))))
        entry = rng.choice(["device", "device", "host", "score"])
        if dtype == "bf16" and entry == "score":   # a logit near 0 has few bits left in bf16
            entry = "device"
        hi = S
        lo = S if rng.random() < 0.3 else rng.randint(max(1, S // 10), S)
        c = _case("", model, dtype, entry, B, S, lo, hi, rng.choice([1, 2, _SHAPES[model][3]]))
        del c["name"]
        if _flops(c) <= _MOST[dtype]:
            return c


def _weights(c, g):
    """HF-named fp32 weights on the GPU: Linear weights N(0, 0.04), LayerNorm
    gains around 1 with a few large ones (trained encoders have such outlier
    features), small biases."""
    H, _, I, _ = _SHAPES[c["model"]]

    def normal(std, *shape):
        return torch.randn(*shape, device="cuda", generator=g) * std

    def gain():
        big = (torch.rand(H, device="cuda", generator=g) < 0.01).float()
        return (1.0 + normal(0.1, H)) * (1.0 + 3.0 * big)

    w = {"embeddings.word_embeddings.weight": normal(0.05, _VOCAB, H),
         "embeddings.position_embeddings.weight": normal(0.02, _POS, H),
         "embeddings.token_type_embeddings.weight": normal(0.02, 2, H),
         "embeddings.LayerNorm.weight": gain(), "embeddings.LayerNorm.bias": normal(0.05, H)}
    for i in range(c["layers"]):
        p = f"encoder.layer.{i}."
        for name, n, k in (("attention.self.query", H, H), ("attention.self.key", H, H), ("attention.self.value", H, H),
                           ("attention.output.dense", H, H), ("intermediate.dense", I, H), ("output.dense", H, I)):
            w[p + name + ".weight"] = normal(0.04, n, k)
            w[p + name + ".bias"] = normal(0.02, n)
        for name in ("attention.output.LayerNorm", "output.LayerNorm"):
            w[p + name + ".weight"] = gain()
            w[p + name + ".bias"] = normal(0.05, H)
    if c["entry"] == "score":
        w["classifier.weight"] = normal(0.05, H)
        w["classifier.bias"] = normal(0.05, 1)
    return w


def _inputs(c, seed):
    """ids and mask [B, S]: [CLS] ids [SEP], then padding."""
    r = np.random.RandomState(seed % (1 << 32))
    B, S = c["B"], c["S"]
    n = np.array(_lengths(c))[r.permutation(B)]
    ids = r.randint(1000, _VOCAB, (B, S)).astype(np.int32)
    ids[:, 0] = 101
    ids[np.arange(B), n - 1] = 102
    mask = (np.arange(S)[None, :] < n[:, None]).astype(np.int32)
    return ids * mask, mask


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


@functools.cache
def _stream():
    """The program's one stream: passes follow one another on it."""
    return torch.cuda.Stream()


def prepare(case, seed):
    H, nh, I, _ = _SHAPES[case["model"]]
    cfg = eb.BertConfig(hidden_size=H, num_attention_heads=nh, num_hidden_layers=case["layers"], intermediate_size=I,
                        vocab_size=_VOCAB, max_position_embeddings=_POS, layer_norm_eps=_EPS)
    weights = {k: v.cpu().numpy() for k, v in _weights(case, _generator(seed)).items()}
    model = eb.Model.from_weights(weights, cfg, case["dtype"])
    ids, mask = _inputs(case, seed)
    B, S = case["B"], case["S"]
    state = {"model": model, "entry": case["entry"], "B": B, "S": S}
    if case["entry"] == "host":
        state.update(ids=ids.astype(np.uint32), mask=mask.astype(np.uint32))
    else:
        shape = (B,) if case["entry"] == "score" else (B, H)
        state.update(ids=torch.from_numpy(ids).cuda(), mask=torch.from_numpy(mask).cuda(),
                     out=torch.empty(shape, device="cuda"), stream=_stream())
    torch.cuda.synchronize()
    return state


def run(state):
    m, B, S = state["model"], state["B"], state["S"]
    if state["entry"] == "host":
        return m.encode_ids(state["ids"], state["mask"])
    out, at = state["out"], state["stream"].cuda_stream
    if state["entry"] == "score":
        m.score_device(state["ids"].data_ptr(), state["mask"].data_ptr(), B, S, out.data_ptr(), stream=at)
    else:
        m.encode_device(state["ids"].data_ptr(), state["mask"].data_ptr(), B, S, out.data_ptr(), stream=at)
    return out


def work(case):
    """The weights (in the dtype the model computes in), the embedding rows the
    tokens need, ids, mask and vectors, each once; the products of the real
    tokens and of their attention."""
    H, _, I, _ = _SHAPES[case["model"]]
    tokens, S, B = sum(_lengths(case)), case["S"], case["B"]
    size = 2 if case["dtype"] == "bf16" else 4
    weights = case["layers"] * ((4 * H * H + 2 * H * I) * size + (9 * H + I) * 4)
    rows = 4 * H * (min(tokens, _VOCAB) + S)
    out = 4 * B * (1 if case["entry"] == "score" else H)
    return {"bytes": float(weights + rows + 8 * B * S + out), "flops": _flops(case)}


def tolerance(case):
    # fp32: 24-bit products and sums through up to 12 post-LayerNorm layers,
    # measured 1e-7 .. 6.3e-7 from exact().  bf16: operands, activations and
    # residual stream of 8 bits, measured 3.1e-3 .. 3.6e-3 from exact() for two
    # layers and 1.0e-2 for twelve.
    if case["dtype"] == "fp32":
        return {"rel": 3e-6, "max": 3e-5}
    return {"rel": 1.5e-2 if case["layers"] <= 2 else 3e-2, "max": 3e-1}


def exact(case, seed):
    """The reference's forward in 64 bits on the padded batch."""
    H, nh, _, _ = _SHAPES[case["model"]]
    hd = H // nh
    w = {k: v.double() for k, v in _weights(case, _generator(seed)).items()}
    ids_all, mask_all = _inputs(case, seed)
    S = case["S"]

    def norm(x, name):
        mean = x.mean(-1, keepdim=True)
        var = ((x - mean) ** 2).mean(-1, keepdim=True)
        return (x - mean) / torch.sqrt(var + _EPS) * w[name + ".weight"] + w[name + ".bias"]

    def linear(x, name):
        return x @ w[name + ".weight"].t() + w[name + ".bias"]

    def gelu(x):
        return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))

    rows = []
    step = max(1, min(128, (1 << 25) // (nh * S * S) + 1))
    for b in range(0, case["B"], step):
        ids = torch.from_numpy(ids_all[b:b + step].astype(np.int64)).cuda()
        mask = torch.from_numpy(mask_all[b:b + step]).cuda().double()
        n = ids.shape[0]
        x = norm(w["embeddings.word_embeddings.weight"][ids] + w["embeddings.position_embeddings.weight"][:S]
                 + w["embeddings.token_type_embeddings.weight"][0], "embeddings.LayerNorm")
        hide = (1.0 - mask)[:, None, None, :].bool()
        for i in range(case["layers"]):
            p = f"encoder.layer.{i}."
            q, k, v = (linear(x, p + "attention.self." + s).view(n, S, nh, hd).transpose(1, 2).contiguous()
                       for s in ("query", "key", "value"))
            s = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(hd)
            a = torch.softmax(s.masked_fill(hide, -math.inf), -1)
            a = torch.matmul(a, v).transpose(1, 2).reshape(n, S, H)
            x = norm(x + linear(a, p + "attention.output.dense"), p + "attention.output.LayerNorm")
            f = linear(gelu(linear(x, p + "intermediate.dense")), p + "output.dense")
            x = norm(x + f, p + "output.LayerNorm")
        pooled = (x * mask[:, :, None]).sum(1) / mask.sum(1, keepdim=True).clamp(min=1.0)
        if case["entry"] == "score":
            rows.append(pooled @ w["classifier.weight"] + w["classifier.bias"])
        else:
            rows.append(pooled / pooled.norm(dim=1, keepdim=True).clamp(min=1e-12))
    return torch.cat(rows).cpu().numpy() if case["entry"] == "host" else torch.cat(rows)

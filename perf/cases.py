"""What a user of the package has it do on one GPU, as cases that can be timed and checked: whole generations, the
memory layer (decode, prompt pass, fp32, training step), the quantised value gather, the attention and feed-forward
blocks of a prompt pass, the attention block's training pass, the Engram memory (prompt pass and training step) and
the conversion of a value table to a quantised one.  Sizes are the package's configurations: d_model 384, 6 heads,
ffn 1024, vocab 32000, 4 memory heads x top-32, k_dim 512, 512 .. 4096 sub-keys per half, 16 Engram lookups of 24."""
import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "sparse-memory-lm_amd"))

from smlm_hip import kernels  # noqa: E402
from smlm_hip.engram import EngramMemory, NgramHash  # noqa: E402
from smlm_hip.model import Attention, ModelConfig, StaticKVCache, SwiGLU, Transformer  # noqa: E402
from smlm_hip.pkm import ProductKeyMemory  # noqa: E402
from smlm_hip.sparse_values import LazyRowAdam, clip_row_sparse, row_store  # noqa: E402

DEV = torch.device("cuda")
D, FFN, VOCAB = 384, 1024, 32000
HEADS, KNN, K_DIM = 4, 32, 512
ENG_LOOKUPS, ENG_DIM, ENG_ROWS, ENG_PAST = 16, 24, 524287, 9


# ---------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # greedy serving of 64 sequences on the 16.8M-row memory (the headline decode), then the generated
        # continuation scored in one pass (its logits)
        {"name": "generate", "kind": "generate", "batch": 64, "prompt": 128, "new": 64, "n_keys": 4096},
        # one token through the memory layer on its captured graph: the smallest call a serving loop makes
        {"name": "memory_decode", "kind": "memory", "batch": 1, "tokens": 1, "n_keys": 4096, "dtype": "bf16",
         "table": "bf16", "graph": True},
        # the memory layer over eight 2048-token prompts (the prefill configuration)
        {"name": "memory_prompt", "kind": "memory", "batch": 8, "tokens": 2048, "n_keys": 2048, "dtype": "bf16",
         "table": "bf16", "graph": False},
        # the memory layer alone in fp32 over 2,048 tokens
        {"name": "memory_fp32", "kind": "memory", "batch": 8, "tokens": 256, "n_keys": 1024, "dtype": "fp32",
         "table": "fp32", "graph": False},
        # the value gather of the int8 16.8M-row table with skewed lookups
        {"name": "gather_int8", "kind": "gather", "tokens": 65536, "lookups": 128, "n_keys": 4096, "table": "int8",
         "spread": "zipf"},
        # one training step of the memory layer and its table: forward, backward, clipping, lazy Adam (a 4,096-token
        # micro-batch on the 1M-row table, bf16 autocast)
        {"name": "memory_train", "kind": "memory_train", "batch": 4, "tokens": 1024, "n_keys": 1024,
         "moments": "fp32"},
        # the attention block of the same prompts
        {"name": "attention_prompt", "kind": "attention", "batch": 8, "tokens": 2048, "heads": 6, "past": -1},
        # the attention block's forward and backward at the training micro-batch
        {"name": "attention_train", "kind": "attention_train", "batch": 4, "tokens": 1024, "heads": 6},
        # the feed-forward block over prompts of an odd length
        {"name": "ffn_prompt", "kind": "ffn", "batch": 7, "tokens": 2011},
        # the Engram memory (hash, row read, gate, convolution) over prompts, and a training step of it
        {"name": "engram_prompt", "kind": "engram", "batch": 8, "tokens": 2048},
        {"name": "engram_train", "kind": "engram_train", "batch": 3, "tokens": 1021, "moments": "fp32"},
        # a trained 1M-row table converted for serving
        {"name": "quantize_int8", "kind": "quantize", "rows": 1048576, "dtype": "fp32", "table": "int8"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch_tokens(rng, most_batch, lo, hi, most):
    """A batch of sequences of lo .. hi tokens, at most `most` tokens in all."""
    t = _log(rng, lo, hi)
    return min(_log(rng, 1, most_batch), max(1, most // t)), t


def draw(rng):
    kind = rng.choice(["generate", "memory_decode", "memory_prompt", "memory_fp32", "gather", "memory_train",
                       "attention", "attention_train", "ffn", "engram", "engram_train", "quantize"])
    if kind == "generate":
        return {"kind": kind, "batch": _log(rng, 1, 64), "prompt": _log(rng, 8, 128), "new": rng.randint(16, 64),
                "n_keys": rng.choice([1024, 2048, 4096])}
    if kind == "memory_decode":
        return {"kind": "memory", "batch": _log(rng, 1, 64), "tokens": 1, "n_keys": rng.choice([512, 1024, 2048, 4096]),
                "dtype": "bf16", "table": rng.choice(["bf16", "int8", "q4"]), "graph": rng.random() < 0.7}
    if kind == "memory_prompt":
        b, t = _batch_tokens(rng, 16, 16, 2048, 16384)
        return {"kind": "memory", "batch": b, "tokens": t, "n_keys": rng.choice([512, 1024, 2048]), "dtype": "bf16",
                "table": rng.choice(["bf16", "int8", "q4"]), "graph": False}
    if kind == "memory_fp32":
        b, t = _batch_tokens(rng, 8, 16, 512, 2048)
        return {"kind": "memory", "batch": b, "tokens": t, "n_keys": rng.choice([512, 1000, 1024]), "dtype": "fp32",
                "table": "fp32", "graph": False}
    if kind == "gather":
        return {"kind": kind, "tokens": _log(rng, 64, 65536), "lookups": rng.choice([64, 96, 128]),
                "n_keys": rng.choice([1024, 2048, 4096]), "table": rng.choice(["int8", "q4"]),
                "spread": rng.choice(["zipf", "uniform"])}
    if kind == "memory_train":
        b, t = _batch_tokens(rng, 8, 64, 1024, 4096)
        return {"kind": kind, "batch": b, "tokens": t, "n_keys": rng.choice([512, 1024]),
                "moments": rng.choice(["fp32", "bf16", "int8"])}
    if kind == "attention":
        b, t = _batch_tokens(rng, 16, 16, 2048, 16384)
        return {"kind": kind, "batch": b, "tokens": t, "heads": rng.choice([3, 6, 6, 12]),
                "past": rng.choice([-1, 0, rng.randint(1, 512)])}
    if kind == "attention_train":
        b, t = _batch_tokens(rng, 8, 64, 1024, 4096)
        return {"kind": kind, "batch": b, "tokens": t, "heads": rng.choice([3, 6, 6, 12])}
    if kind == "ffn":
        b, t = _batch_tokens(rng, 16, 16, 2048, 14077)
        return {"kind": kind, "batch": b, "tokens": t}
    if kind == "engram":
        b, t = _batch_tokens(rng, 16, 16, 2048, 16384)
        return {"kind": kind, "batch": b, "tokens": t}
    if kind == "engram_train":
        b, t = _batch_tokens(rng, 8, 64, 1024, 3063)
        return {"kind": kind, "batch": b, "tokens": t, "moments": rng.choice(["fp32", "bf16"])}
    return {"kind": kind, "rows": _log(rng, 65536, 1048576), "dtype": rng.choice(["fp32", "bf16"]),
            "table": rng.choice(["int8", "q4"])}


# --------------------------------------------------------------------------------------------------- the states
def _randn(*shape, std=1.0, dtype=torch.float32):
    return torch.randn(*shape, device=DEV).mul_(std).to(dtype)


def _memory_layer(c, train=False):
    with torch.device(DEV):
        m = ProductKeyMemory(D, D, n_keys=c["n_keys"], heads=HEADS, knn=KNN, k_dim=K_DIM,
                             value_grad="row_sparse" if train else "dense")
    if train:
        return m.train()
    with torch.no_grad():           # statistics of trained queries: near what the projection of normed inputs gives
        bn = m.query_norm
        bn.running_mean.normal_(0.0, 0.05)
        bn.running_var.uniform_(0.8, 1.2).mul_(2.0 * D / (D + HEADS * K_DIM))
        bn.weight.uniform_(0.8, 1.2)
        bn.bias.normal_(0.0, 0.05)
        if c["dtype"] == "bf16":
            m = m.to(torch.bfloat16)
        if c["table"] in ("int8", "q4"):
            w = m.values.weight.detach()
            m.values.infer_table = (kernels.quantize_int8 if c["table"] == "int8" else kernels.quantize_q4)(w)
    m.eval()
    m.decode_graph = bool(c["graph"])
    return m


def _zipf_rows(n, rows, s=1.1):
    """n row numbers whose rank r has a frequency of about r^-s (the inverse of the continuous law's distribution, so
    that equal seeds give equal rows), the ranks spread over the table by a random permutation."""
    u = torch.rand(n, device=DEV, dtype=torch.float64)
    ranks = (1.0 - u * (1.0 - float(rows) ** (1.0 - s))).pow(1.0 / (1.0 - s)).long().sub_(1).clamp_(0, rows - 1)
    return torch.randperm(rows, device=DEV)[ranks]


def _attention_layer(c, max_len):
    with torch.device(DEV):
        a = Attention(ModelConfig(d_model=D, n_heads=c["heads"], max_seq_len=max_len))
    with torch.no_grad():
        a.wqkv.weight.normal_(0.0, 0.06)
        a.wo.weight.normal_(0.0, 0.05)
    return a


def _engram_layer():
    with torch.device(DEV):
        m = EngramMemory(D, ENG_LOOKUPS, ENG_DIM, ENG_ROWS)
    h = NgramHash(VOCAB, rows=ENG_ROWS, canon=torch.arange(VOCAB))
    with torch.no_grad():
        for norm in (m.h_norm, m.k_norm, m.v_norm):
            norm.weight.uniform_(0.8, 1.2)
        m.w_k.weight.normal_(0.0, 0.05)
        m.w_v.weight.normal_(0.0, 0.05)
        m.conv.weight.normal_(0.0, 0.3)
        m.values.weight.mul_(math.sqrt(D))
    return m, h.to(DEV)


def _ids(c, history):
    """Compressed token ids with word-like frequencies, `history` pad ids before each sequence."""
    ids = _zipf_rows(c["batch"] * c["tokens"], VOCAB).view(c["batch"], c["tokens"])
    return torch.cat([torch.full((c["batch"], history), VOCAB, device=DEV), ids], 1)


def prepare(c, seed):
    torch.manual_seed(seed)
    kind = c["kind"]
    if kind == "generate":
        cfg = ModelConfig(vocab_size=VOCAB, d_model=D, n_layers=6, n_heads=6, ffn_hidden=FFN,
                          max_seq_len=c["prompt"] + c["new"] + 1, mem_layers=[3], mem_n_keys=c["n_keys"],
                          mem_heads=HEADS, mem_knn=KNN, mem_k_dim=K_DIM)
        with torch.device(DEV):
            model = Transformer(cfg)
        with torch.no_grad():
            for name, p in model.named_parameters():
                if p.dim() >= 2 or name.endswith("keys"):
                    p.normal_(0.0, 0.02)
        model = model.to(torch.bfloat16).eval()
        model.set_memory_inference_table("bf16")
        prompt = torch.randint(0, VOCAB, (c["batch"], c["prompt"]), device=DEV)
        s = {"c": c, "m": model, "x": prompt}
        run(s)                      # a serving program has captured its graphs before the first request
        return s
    if kind == "memory":
        m = _memory_layer(c)
        x = _randn(c["batch"], c["tokens"], D, dtype=torch.bfloat16 if c["dtype"] == "bf16" else torch.float32)
        s = {"c": c, "m": m, "x": x}
        if c["graph"]:
            run(s)
        return s
    if kind == "gather":
        rows, quantize = c["n_keys"] ** 2, kernels.quantize_int8 if c["table"] == "int8" else kernels.quantize_q4
        parts = [quantize(_randn(min(1 << 21, rows - a), D, std=0.02)) for a in range(0, rows, 1 << 21)]
        codes, scales = (torch.cat([p[i] for p in parts]) for i in range(2))
        n = c["tokens"] * c["lookups"]
        idx = _zipf_rows(n, rows) if c["spread"] == "zipf" else torch.randint(0, rows, (n,), device=DEV)
        w = torch.softmax(_randn(c["tokens"], c["lookups"] // KNN, KNN), -1)
        return {"c": c, "codes": codes, "scales": scales, "idx": idx.view(c["tokens"], -1),
                "w": w.view(c["tokens"], -1)}
    if kind == "memory_train":
        m = _memory_layer(c, train=True)
        table = m.values.weight
        row_store(table)
        opt = LazyRowAdam([table], lr=1e-3, state_dtype=c["moments"])
        x, g = _randn(c["batch"], c["tokens"], D), _randn(c["batch"], c["tokens"], D, std=1e-2, dtype=torch.bfloat16)
        return {"c": c, "m": m, "opt": opt, "x": x.requires_grad_(), "g": g}
    if kind == "attention":
        past = max(c["past"], 0)
        a = _attention_layer(c, past + c["tokens"]).to(torch.bfloat16).eval()
        cache, hd = None, D // c["heads"]
        if c["past"] >= 0:
            cache = StaticKVCache(c["batch"], c["heads"], past + c["tokens"], hd, torch.bfloat16, DEV)
            cache.k[:, :, :past] = _randn(c["batch"], c["heads"], past, hd)
            cache.v[:, :, :past] = _randn(c["batch"], c["heads"], past, hd)
        return {"c": c, "m": a, "x": _randn(c["batch"], c["tokens"], D, dtype=torch.bfloat16), "cache": cache}
    if kind == "attention_train":
        a = _attention_layer(c, c["tokens"]).train()
        x, g = _randn(c["batch"], c["tokens"], D), _randn(c["batch"], c["tokens"], D, dtype=torch.bfloat16)
        return {"c": c, "m": a, "x": x.requires_grad_(), "g": g}
    if kind == "ffn":
        with torch.device(DEV):
            f = SwiGLU(D, FFN)
        with torch.no_grad():
            f.w13.weight.normal_(0.0, 0.06)
            f.w2.weight.normal_(0.0, 0.04)
        return {"c": c, "m": f.to(torch.bfloat16).eval(), "x": _randn(c["batch"], c["tokens"], D, dtype=torch.bfloat16)}
    if kind in ("engram", "engram_train"):
        m, h = _engram_layer()
        s = {"c": c, "hash": h, "ids": _ids(c, h.history)}
        if kind == "engram":
            s.update(m=m.to(torch.bfloat16).eval(), x=_randn(c["batch"], c["tokens"], D, dtype=torch.bfloat16))
            return s
        table = m.values.weight
        row_store(table)
        s.update(m=m.train(), x=_randn(c["batch"], c["tokens"], D).requires_grad_(),
                 g=_randn(c["batch"], c["tokens"], D), opt=LazyRowAdam([table], lr=1e-3, state_dtype=c["moments"]))
        return s
    return {"c": c, "w": _randn(c["rows"], D, std=0.05, dtype=torch.float32 if c["dtype"] == "fp32" else torch.bfloat16)}


# ----------------------------------------------------------------------------------------------------- the pass
def _no_grads(s):
    s["x"].grad = None
    for p in s["m"].parameters():
        p.grad = None


def _grads(s):
    """The gradients; a bias before the batch statistics of a BatchNorm has none but rounding."""
    return {"dx": s["x"].grad, **{"d_" + n: p.grad for n, p in s["m"].named_parameters()
                                  if p.grad is not None and n != "query_proj.bias"}}


def _train_step(s, forward):
    """Forward, backward, clipping of the table's gradient and the table's optimizer step."""
    _no_grads(s)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = forward()
    y.backward(s["g"].to(y.dtype))
    table = s["m"].values.weight
    norm = clip_row_sparse([table], 1.0)
    s["opt"].step()
    out = {"y": y, "norm": norm, "table": table, **_grads(s)}
    if s["c"]["moments"] != "int8":
        out["exp_avg"] = s["opt"].state[table]["exp_avg"]
    return out


def run(s):
    c = s["c"]
    kind = c["kind"]
    if kind == "generate":
        with torch.no_grad():
            tokens = s["m"].generate(s["x"], c["new"])
            return {"tokens": tokens, "logits": s["m"](tokens)}
    if kind in ("memory", "ffn"):
        with torch.no_grad():
            return s["m"](s["x"])
    if kind == "gather":
        return kernels.bag_infer(s["idx"], s["w"], s["codes"], s["scales"])
    if kind == "memory_train":
        return _train_step(s, lambda: s["m"](s["x"]))
    if kind == "attention":
        with torch.no_grad():
            if s["cache"] is None:
                return s["m"](s["x"])
            y = s["m"](s["x"], s["cache"], c["past"])
        return {"y": y, "k": s["cache"].k, "v": s["cache"].v}
    if kind == "attention_train":
        _no_grads(s)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = s["m"](s["x"])
        y.backward(s["g"].to(y.dtype))
        return {"y": y, **_grads(s)}
    if kind == "engram":
        with torch.no_grad():
            rows = s["hash"](s["ids"])
            return {"y": s["m"](s["x"], rows), "rows": rows}
    if kind == "engram_train":
        return _train_step(s, lambda: s["m"](s["x"], s["hash"](s["ids"])))
    return (kernels.quantize_int8 if c["table"] == "int8" else kernels.quantize_q4)(s["w"])


# ------------------------------------------------------------------------------- what a pass cannot do without
def _distinct(lookups, rows):
    """Expected distinct rows of uniform lookups."""
    return rows * -math.expm1(lookups * math.log1p(-1.0 / rows))


def _row_bytes(table):
    return {"fp32": 4 * D, "bf16": 2 * D, "int8": D + 2, "q4": D // 2 + 2}[table]


def _memory_work(n, c, esize, row_bytes):
    nq, keys = HEADS * K_DIM, HEADS * K_DIM * c["n_keys"]
    weights = D * (nq + 2 * D) + keys
    flops = 2 * n * (D * nq + keys + HEADS * KNN * D + 2 * D * D)
    return flops, esize * (2 * n * D + weights) + _distinct(n * HEADS * KNN, c["n_keys"] ** 2) * row_bytes


def _adam_bytes(moments, width, rows):
    """Per flagged row: parameter, accumulator and both moments read and written (int8: with their row scales)."""
    return rows * (2 * (8 * width + {"fp32": 8 * width, "bf16": 4 * width, "int8": 2 * width + 8}[moments]) + 1)


def work(c):
    kind = c["kind"]
    if kind == "quantize":
        return {"bytes": c["rows"] * (D * (4 if c["dtype"] == "fp32" else 2) + _row_bytes(c["table"])), "flops": 0}
    if kind == "gather":
        n, rows = c["tokens"] * c["lookups"], c["n_keys"] ** 2
        if c["spread"] == "uniform":
            read = _distinct(n, rows)
        else:                       # rank r is read with frequency f r^-1.1: the distinct ranks, by steps of a fifth
            f, read, lo = 0.1 / (1.0 - rows ** -0.1), 0.0, 1
            while lo < rows:
                hi = min(rows, max(lo + 1, int(lo * 1.2)))
                read += (hi - lo) * -math.expm1(-n * f * math.sqrt(lo * hi) ** -1.1)
                lo = hi
        return {"bytes": 12 * n + read * _row_bytes(c["table"]) + 4 * D * c["tokens"], "flops": 2 * n * D}
    n = c["batch"] * c.get("tokens", 1)
    if kind == "memory":
        fl, by = _memory_work(n, c, 2 if c["dtype"] == "bf16" else 4, _row_bytes(c["table"]))
        return {"bytes": by, "flops": fl}
    if kind == "memory_train":
        fl, by = _memory_work(n, c, 4, 4 * D)
        touched = _distinct(n * HEADS * KNN, c["n_keys"] ** 2)
        return {"bytes": 2 * by + touched * 4 * D + _adam_bytes(c["moments"], D, touched) + c["n_keys"] ** 2,
                "flops": 3 * fl}
    if kind in ("attention", "attention_train"):
        t, past = c["tokens"], max(c.get("past", 0), 0)
        pairs = c["batch"] * (t * past + t * (t + 1) / 2)
        if kind == "attention":
            return {"bytes": 2 * (2 * n * D + 4 * D * D + 2 * c["batch"] * past * D + (2 * n * D if c["past"] >= 0 else 0)),
                    "flops": 8 * n * D * D + 4 * pairs * D}
        return {"bytes": 14 * n * D + 32 * D * D, "flops": 24 * n * D * D + 14 * pairs * D}
    if kind == "ffn":
        return {"bytes": 2 * (2 * n * D + 3 * D * FFN), "flops": 6 * n * D * FFN}
    if kind in ("engram", "engram_train"):
        table = ENG_LOOKUPS * ENG_ROWS
        rows = _distinct(n, ENG_ROWS) * ENG_LOOKUPS * 0.5       # repeated n-grams read the same rows
        fl = 4 * n * D * D
        if kind == "engram":
            return {"bytes": 2 * (2 * n * D + 2 * D * D + rows * ENG_DIM) + 8 * n * (1 + ENG_LOOKUPS), "flops": fl}
        return {"bytes": 4 * (4 * n * D + 4 * D * D + rows * ENG_DIM) + 8 * n * (1 + ENG_LOOKUPS)
                + _adam_bytes(c["moments"], ENG_DIM, rows) + table, "flops": 3 * fl}
    # generate: every step reads the weights, the sub-keys, the cache and its tokens' value rows
    steps, b, layers = c["new"], c["batch"], 6
    dense = VOCAB * D + layers * 4 * D * D + (layers - 1) * 3 * D * FFN + D * (HEADS * K_DIM + 2 * D)
    keys = HEADS * K_DIM * c["n_keys"]
    per_token = dense - VOCAB * D + keys + HEADS * KNN * D
    cache = layers * b * D * sum(c["prompt"] + i for i in range(steps)) * 4
    tokens = b * (c["prompt"] + 2 * steps + 1)
    return {"bytes": 2.0 * (steps + 2) * (dense + keys) + cache + 2.0 * tokens * HEADS * KNN * D
            + 2.0 * b * (steps + 1) * VOCAB,
            "flops": 2.0 * tokens * per_token + 2.0 * b * (2 * steps + 2) * VOCAB * D}


def tolerance(c):
    """About four times the error that exact() shows, where the data type is the reason.  The memory layer in fp32 is
    1e-6 off as long as no selection changes; a pair of candidates nearer to each other than the rounding of their
    scores can change places at the end of a row's top list, and one such row of 2,048 is 2e-3 of the result."""
    return {"generate": {"rel": 0.02, "max": 0.5, "differ": 0.01},
            "memory": {"rel": 0.02, "max": 0.5} if c.get("dtype") == "bf16" else {"rel": 2e-3, "max": 0.5},
            "gather": {"rel": 1e-6, "max": 1e-4},
            "memory_train": {"rel": 0.03, "max": 0.9},
            "attention": {"rel": 0.02, "max": 0.3},
            "attention_train": {"rel": 0.03, "max": 0.5},
            "ffn": {"rel": 0.015, "max": 0.2},
            "engram": {"rel": 0.015, "max": 0.3},
            "engram_train": {"rel": 0.02, "max": 0.5},
            "quantize": "exact"}[c["kind"]]


# ------------------------------------------------------------------------------------------------ in 64 bits
class _Round(torch.autograd.Function):
    """bf16 rounding with the identity as its derivative."""

    @staticmethod
    def forward(ctx, x):
        return x.to(torch.bfloat16).to(x.dtype)

    @staticmethod
    def backward(ctx, g):
        return g


def _select64(s1, s2, nk, rounded):
    """Top-KNN pairs of s1[i] + s2[j] per row (R, nk): scores (through which gradients flow) and table rows.  Equal
    scores go to the lower row; with `rounded`, the sums are bf16 numbers."""
    v1, i1 = torch.sort(s1, dim=-1, descending=True, stable=True)
    v2, i2 = torch.sort(s2, dim=-1, descending=True, stable=True)
    pairs = [(i, j) for i in range(KNN) for j in range(KNN) if (i + 1) * (j + 1) <= KNN]
    pi, pj = (torch.tensor(p, device=DEV) for p in zip(*pairs))
    rows = i1[:, pi] * nk + i2[:, pj]
    sums = v1[:, pi] + v2[:, pj]
    if rounded:
        sums = _Round.apply(sums)
    by_row = torch.argsort(rows, -1)
    top = torch.sort(sums.detach().gather(-1, by_row), dim=-1, descending=True, stable=True)[1][:, :KNN]
    at = by_row.gather(-1, top)
    return sums.gather(-1, at), rows.gather(-1, at)


def _values64(m):
    """A function from table rows to their fp64 values."""
    t = getattr(m.values, "infer_table", None)
    if t is None:
        w = m.values.weight.detach()
        return lambda r: w[r].double()
    codes, scales = t

    def read(r):
        v = codes[r]
        v = v.double() if codes.dtype == torch.int8 else torch.cat([v & 15, v >> 4], -1).double() - 8.0
        return v * scales[r].double().unsqueeze(-1)
    return read


def _linear64(mod, x, rnd=None):
    w = mod.weight.double() if rnd is None else rnd(mod.weight.double())
    y = x @ w.t()
    return y if mod.bias is None else y + mod.bias.double()


def _memory64(m, x, c):
    bf16, out = c["dtype"] == "bf16", []
    rnd = (lambda t: t.to(torch.bfloat16).double()) if bf16 else (lambda t: t)
    bn, read, nk, half = m.query_norm, _values64(m), c["n_keys"], K_DIM // 2
    scale = bn.weight.double() / torch.sqrt(bn.running_var.double() + bn.eps)
    keys = m.keys.double()
    for xb in x.reshape(-1, D).double().split(1024):
        q = rnd((rnd(_linear64(m.query_proj, xb)) - bn.running_mean.double()) * scale + bn.bias.double())
        q = q.view(-1, HEADS, 2, half)
        s = [rnd(torch.stack([q[:, h, p] @ keys[h, p].t() for h in range(HEADS)], 1)).view(-1, nk) for p in (0, 1)]
        scores, rows = _select64(s[0], s[1], nk, bf16)
        w = torch.softmax(scores, -1).view(len(xb), 1, -1)
        bag = (w @ read(rows.view(len(xb), -1))).squeeze(1)
        out.append(_linear64(m.value_proj, bag * F.silu(_linear64(m.swilu_proj, xb))))
    return torch.cat(out).view(x.shape)


def _memory_train64(s):
    m, c, x, rnd = s["m"], s["c"], s["x"].detach().double(), _Round.apply
    P = {n: p.detach().double() for n, p in m.named_parameters() if n != "values.weight"}
    for p in (x, *P.values()):
        p.requires_grad_()
    n, nk, half = c["batch"] * c["tokens"], c["n_keys"], K_DIM // 2
    xb = rnd(x.reshape(n, D))
    lin = lambda name, v: v @ rnd(P[name + ".weight"]).t() + P[name + ".bias"]  # noqa: E731
    q = rnd(lin("query_proj", xb))
    mean, var = q.mean(0), q.var(0, unbiased=False)
    q = rnd((q - mean) / torch.sqrt(var + m.query_norm.eps) * P["query_norm.weight"] + P["query_norm.bias"])
    q, keys = q.view(n, HEADS, 2, half), rnd(P["keys"])
    s1, s2 = (rnd(torch.stack([q[:, h, p] @ keys[h, p].t() for h in range(HEADS)], 1)).view(-1, nk) for p in (0, 1))
    scores, rows = _select64(s1, s2, nk, True)
    w, rows = torch.softmax(scores, -1).view(n, -1), rows.view(n, -1)
    read = _values64(m)
    bag = torch.cat([(a.unsqueeze(1) @ read(r)).squeeze(1) for a, r in zip(w.detach().split(512), rows.split(512))])
    bag.requires_grad_()
    y = lin("value_proj", bag * F.silu(lin("swilu_proj", xb))).view(x.shape)
    y.backward(s["g"].double())
    gb = bag.grad
    w.backward(torch.cat([(read(r) @ g.unsqueeze(-1)).squeeze(-1) for g, r in zip(gb.split(512), rows.split(512))]))
    gt = torch.zeros(nk * nk, D, dtype=torch.float64, device=DEV)
    for a, r, g in zip(w.detach().split(512), rows.split(512), gb.split(512)):
        gt.index_add_(0, r.reshape(-1), (a.unsqueeze(-1) * g.unsqueeze(1)).reshape(-1, D))
    del P["query_proj.bias"]
    return _clipped64({"y": y, "dx": x.grad, **{"d_" + k: p.grad for k, p in P.items()}}, gt, c)


def _clipped64(out, gt, c):
    norm = gt.norm()
    out.update(norm=norm, table=None)
    if c["moments"] != "int8":
        out["exp_avg"] = 0.1 * gt * (1.0 / (norm + 1e-6)).clamp(max=1.0)
    return out


def _attention64(a, x, c, rnd, past_k=None, past_v=None):
    """(y, k, v) of the block; rnd rounds the weights and the input where the block gets them in bf16."""
    b, t, hd, past = c["batch"], c["tokens"], D // c["heads"], 0 if past_k is None else past_k.shape[2]
    qkv = rnd(x) @ rnd(a["wqkv"]).t()
    q, k, v = qkv.view(b, t, 3, c["heads"], hd).permute(2, 0, 3, 1, 4)
    inv = 10000.0 ** (-torch.arange(0, hd, 2, device=DEV, dtype=torch.float64) / hd)
    ang = torch.outer(torch.arange(past, past + t, device=DEV, dtype=torch.float64), inv)

    def rope(u):
        p, r = u.chunk(2, -1)
        return torch.cat([p * ang.cos() - r * ang.sin(), p * ang.sin() + r * ang.cos()], -1)
    q, k = rope(q), rope(k)
    if past:
        k, v = torch.cat([past_k, k], 2), torch.cat([past_v, v], 2)
    mask = torch.ones(t, past + t, dtype=torch.bool, device=DEV).tril(past)
    ys = []
    for i in range(b):
        s = (q[i] @ k[i].transpose(1, 2)) * hd ** -0.5
        ys.append(torch.softmax(s.masked_fill(~mask, -math.inf), -1) @ v[i])
    y = torch.stack(ys).transpose(1, 2).reshape(b, t, D)
    return y @ rnd(a["wo"]).t(), k, v


def _engram64(P, e, h, c, m):
    b, t = c["batch"], c["tokens"]

    def norm(v, w):
        return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + m.h_norm.eps) * w
    agree = (norm(h, P["h_norm.weight"]) * norm(e @ P["w_k.weight"].t(), P["k_norm.weight"])).sum(-1, keepdim=True)
    gv = torch.sigmoid(agree / math.sqrt(D)) * (e @ P["w_v.weight"].t())
    u = F.pad(norm(gv, P["v_norm.weight"]), (0, 0, ENG_PAST, 0))
    conv = sum(u[:, 3 * i:3 * i + t] * P["conv.weight"][:, 0, i] for i in range(4))
    return F.silu(conv) + gv


def exact(c, seed):
    kind = c["kind"]
    if kind in ("generate", "quantize"):
        return None                 # greedy choices follow from bf16 roundings; codes are whole numbers
    if kind == "memory" and c["graph"]:
        c = dict(c, graph=False)
    s = prepare(c, seed)
    m = s.get("m")
    if kind == "memory":
        with torch.no_grad():
            return _memory64(m, s["x"], c)
    if kind == "gather":
        codes, scales, out = s["codes"], s["scales"], []
        read = _values64(type("T", (), {"values": type("V", (), {"infer_table": (codes, scales)})})())
        for i, w in zip(s["idx"].split(1024), s["w"].split(1024)):
            out.append((w.double().unsqueeze(1) @ read(i)).squeeze(1))
        return torch.cat(out)
    if kind == "memory_train":
        return _memory_train64(s)
    same = lambda t: t  # noqa: E731
    if kind == "attention":
        W = {"wqkv": m.wqkv.weight.double(), "wo": m.wo.weight.double()}
        k = s["cache"]
        if k is None:
            with torch.no_grad():
                return _attention64(W, s["x"].double(), c, same)[0]
        with torch.no_grad():
            past = c["past"]
            y, k, v = _attention64(W, s["x"].double(), c, same, k.k[:, :, :past].double(), k.v[:, :, :past].double())
            return {"y": y, "k": k, "v": v}
    if kind == "attention_train":
        W = {n: getattr(m, n).weight.detach().double().requires_grad_() for n in ("wqkv", "wo")}
        x = s["x"].detach().double().requires_grad_()
        y = _attention64(W, x, c, _Round.apply)[0]
        y.backward(s["g"].double())
        return {"y": y, "dx": x.grad, "d_wqkv.weight": W["wqkv"].grad, "d_wo.weight": W["wo"].grad}
    if kind == "ffn":
        a, b = _linear64(m.w13, s["x"].double()).chunk(2, -1)
        return _linear64(m.w2, F.silu(a) * b).detach()
    rows = s["hash"](s["ids"])
    table = m.values.weight.detach()
    e = table[rows].double().reshape(c["batch"], c["tokens"], -1)
    P = {n: p.detach().double() for n, p in m.named_parameters() if n != "values.weight"}
    if kind == "engram":
        return {"y": _engram64(P, e, s["x"].double(), c, m), "rows": None}
    x = s["x"].detach().double()
    for p in (x, e, *P.values()):
        p.requires_grad_()
    y = _engram64(P, e, x, c, m)
    y.backward(s["g"].double())
    gt = torch.zeros(table.shape, dtype=torch.float64, device=DEV)
    gt.index_add_(0, rows.reshape(-1), e.grad.reshape(-1, ENG_DIM))
    return _clipped64({"y": y, "dx": x.grad, **{"d_" + k: p.grad for k, p in P.items()}}, gt, c)

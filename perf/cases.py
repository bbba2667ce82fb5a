"""The work that users of this package have it do, as a list of cases to be timed: each fused operator through its
module's `forward`, over the sizes of the benchmark configurations (triton_amd/configs.py, triton_amd/benchmark.py)
and of ordinary use around them -- single requests and small batches, short prompts and long ones, one new token or a
chunk of them against a cache of any length, ragged sizes throughout.

A case is a dict of plain values: "op" names the operator and form, the rest its sizes and options.  All data is fp16
apart from what the operators take or give in fp32 (KeyFormer's noise, key scores).  Values are what the paths meet in
earnest: N(0,1) activations, weights scaled to keep the projections at unit variance, norm weights around one,
Gumbel(0,1) noise.
"""
import math

import torch

from triton_amd import configs, modules

# query heads, KV heads, head_dim of the attention shapes in use: the two benchmarked models, and two small generic ones
HEADS = {
    "llama": (configs.LLAMA["n_heads"], configs.LLAMA["n_kv_heads"], configs.LLAMA["head_dim"]),
    "falcon": (configs.FALCON["n_heads"], configs.FALCON["n_kv_heads"], configs.FALCON["head_dim"]),
    "mha16": (16, 16, 64),
    "gqa8": (8, 2, 128),
}
EPS = 1e-5
MAX_ROW_PAIRS = 4096 * 4096      # batch * seq^2 of the largest attention problem


def listed():
    return [
        # RMSNorm of a whole prompt's activations: the bandwidth benchmark
        dict(name="rms_prompt", op="rms", rows=4096, cols=4096),
        # causal attention over one long prompt (the headline benchmark), and over a small batch of ragged prompts
        dict(name="attn_prompt", op="attn", heads="llama", batch=1, seq=4096),
        dict(name="attn_batch_ragged", op="attn", heads="llama", batch=4, seq=777),
        # the pre-normalised attention block: projections and attention of one prompt
        dict(name="prenorm_prompt", op="prenorm", heads="llama", batch=1, seq=2048),
        # attention with per-head norms of Q and K, many query heads on one KV head
        dict(name="qknorm_prompt", op="qknorm", heads="falcon", batch=1, seq=2048),
        # attention with key scores for cache eviction: perturbed scores with fp32 noise (the benchmark) and with
        # everything in fp16 as the drivers allocate it, and column statistics of the plain probabilities
        dict(name="keyformer_prompt", op="keyformer", heads="llama", batch=1, seq=4096, noise="fp32"),
        dict(name="keyformer_half_ragged", op="keyformer", heads="llama", batch=1, seq=1501, noise="fp16"),
        dict(name="roco_prompt", op="roco", heads="llama", batch=1, seq=4096, stats="mean_std"),
        # the drivers' own problem: a few new tokens projected, appended to the cache and attended over it
        dict(name="decode_append", op="decode", variant="vanilla", heads="llama", new=16, past=1024),
        dict(name="decode_keyformer", op="decode", variant="keyformer", heads="falcon", new=16, past=1024),
        # a chunk of a prompt against a longer cache
        dict(name="decode_chunk", op="decode", variant="prenorm", heads="llama", new=100, past=4000),
        # the smallest call: a low-rank adapted linear layer on a few tokens
        dict(name="lora_few_tokens", op="lora", tokens=16, n=1024, p=512, r=64),
    ]


def _log_int(rng, lo, hi, step=1):
    """A multiple of step in [lo, hi], uniform over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + step)))
    return max(lo, min(hi, int(v) // step * step))


def _prompt(rng, most):
    """Batch and sequence length with batch * seq^2 within the largest listed attention problem."""
    seq = _log_int(rng, 20, most)
    batch = min(_log_int(rng, 1, 8), max(1, MAX_ROW_PAIRS // (seq * seq)))
    return batch, seq


def draw(rng):
    op = rng.choice(["rms", "attn", "prenorm", "qknorm", "keyformer", "roco", "decode", "decode", "linear"])
    heads = rng.choice(["llama", "llama", "falcon", "falcon", "mha16", "gqa8"])
    if op == "rms":
        cols = _log_int(rng, 64, 8192, 8)
        return dict(op="rms", rows=_log_int(rng, 1, min(16384, (1 << 25) // cols)), cols=cols)
    if op == "decode":
        return dict(op="decode", variant=rng.choice(["vanilla", "prenorm", "qknorm", "keyformer", "roco"]), heads=heads,
                    new=_log_int(rng, 1, 128), past=_log_int(rng, 64, 16384))
    if op == "linear":
        if rng.random() < 0.5:
            return dict(op="lora", tokens=_log_int(rng, 1, 1024), n=_log_int(rng, 256, 4096, 8),
                        p=_log_int(rng, 256, 4096, 8), r=_log_int(rng, 8, 128, 8))
        return dict(op="gmlp", tokens=_log_int(rng, 1, 1024), n=_log_int(rng, 256, 4096, 8), k=_log_int(rng, 256, 4096, 8))
    batch, seq = _prompt(rng, 2048 if op == "prenorm" else 4096)
    if op == "prenorm":
        batch = max(1, min(batch, 2048 // seq))
    if op in ("keyformer", "roco"):
        # one noise value per query, key and head: at most the listed 32 heads x 4096^2
        while batch > 1 and batch * HEADS[heads][0] * seq * seq > 32 * MAX_ROW_PAIRS:
            batch -= 1
        if batch * HEADS[heads][0] * seq * seq > 32 * MAX_ROW_PAIRS:
            heads = "llama"
    case = dict(op=op, heads=heads, batch=batch, seq=seq)
    if op == "keyformer":
        case["noise"] = rng.choice(["fp32", "fp16"])
    elif op == "roco":
        case["stats"] = rng.choice(["sums", "mean_std"])
    return case


# ------------------------------------------------------------------------------------------------ inputs
def _randn(g, *shape, std=1.0, mean=0.0):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std + mean).half()


def _zeros(*shape, dtype=torch.float16):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _gumbel(g, shape, dtype):
    e = torch.empty(shape, dtype=torch.float32, device="cuda").exponential_(generator=g)
    return e.log_().neg_().to(dtype)


def prepare(case, seed):
    """Tensors by the names of the module's TENSOR_PARAMS, the module, and the names of what it writes."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    op = case["op"]
    t = {}
    if op == "rms":
        rows, cols = case["rows"], case["cols"]
        t = dict(X=_randn(g, rows, cols), gamma=_randn(g, cols, std=0.02, mean=1.0), X_norm=_zeros(rows, cols))
        mod, outs = modules.get("rms", eps=EPS), ["X_norm"]
    elif op == "lora":
        m, n, p, r = case["tokens"], case["n"], case["p"], case["r"]
        t = dict(X=_randn(g, m, n), W=_randn(g, n, p, std=n ** -0.5), A=_randn(g, n, r, std=n ** -0.5),
                 B=_randn(g, r, p, std=r ** -0.5), O=_zeros(m, p))
        mod, outs = modules.get("lora", "linear"), ["O"]
    elif op == "gmlp":
        m, n, k = case["tokens"], case["n"], case["k"]
        t = dict(X=_randn(g, m, k), W1=_randn(g, k, n, std=k ** -0.5), W2=_randn(g, k, n, std=k ** -0.5), O=_zeros(m, n))
        mod, outs = modules.get("gmlp", "linear"), ["O"]
    elif op == "decode":
        # multi-head form: every head has its own keys and values, X and the weights are [.., heads * head_dim]
        h, _, d = HEADS[case["heads"]]
        m, past, n, variant = case["new"], case["past"], h * d, case["variant"]
        t = dict(X=_randn(g, m, n), WQ=_randn(g, n, n, std=n ** -0.5), WK=_randn(g, n, n, std=n ** -0.5),
                 WV=_randn(g, n, n, std=n ** -0.5), K_cache=_randn(g, h, past + m, d), V_cache=_randn(g, h, past + m, d),
                 O2=_zeros(m, n))
        outs = ["O2", "K_cache", "V_cache"]
        if variant == "keyformer":
            t["noise"], t["C_out"] = _gumbel(g, (h, m, past + m), torch.float16), _zeros(h, past + m)
            outs.append("C_out")
        elif variant == "roco":
            # fp32: sums of squares over a long cache lie below what fp16 holds
            t["C_out1"], t["C_out2"] = (_zeros(h, past + m, dtype=torch.float32) for _ in range(2))
            outs += ["C_out1", "C_out2"]
        mod = modules.get(variant, "decode", head_dim=d, scale=d ** -0.5)
    elif op == "prenorm":
        hq, hkv, d = HEADS[case["heads"]]
        b, s, hidden = case["batch"], case["seq"], hq * d
        t = dict(X=_randn(g, b, s, hidden), gamma=_randn(g, hidden, std=0.02, mean=1.0), O=_zeros(b, s, hidden),
                 WQ=_randn(g, hidden, hq * d, std=0.02), WK=_randn(g, hidden, hkv * d, std=0.02),
                 WV=_randn(g, hidden, hkv * d, std=0.02))
        mod, outs = modules.get("prenorm", head_dim=d, eps=EPS), ["O"]
    else:
        hq, hkv, d = HEADS[case["heads"]]
        b, s = case["batch"], case["seq"]
        t = dict(Q=_randn(g, b, hq, s, d), K=_randn(g, b, hkv, s, d), V=_randn(g, b, hkv, s, d), O=_zeros(b, hq, s, d))
        outs = ["O"]
        if op == "attn":
            mod = modules.get("vanilla")
        elif op == "qknorm":
            t["gamma_q"], t["gamma_k"] = _randn(g, d, std=0.02, mean=1.0), _randn(g, d, std=0.02, mean=1.0)
            mod = modules.get("qknorm", eps=EPS)
        elif op == "keyformer":
            dtype = torch.float32 if case["noise"] == "fp32" else torch.float16
            t["noise"], t["C_out"] = _gumbel(g, (b, hq, s, s), dtype), _zeros(b, hq, s, dtype=dtype)
            mod = modules.get("keyformer", tau=1.0)
            outs.append("C_out")
        else:
            t["C_out1"], t["C_out2"] = _zeros(b, hq, s, dtype=torch.float32), _zeros(b, hq, s, dtype=torch.float32)
            mod = modules.get("roco", stats=case["stats"])
            outs += ["C_out1", "C_out2"]
    return dict(module=mod, args=[t[p] for p in mod.TENSOR_PARAMS], outputs=[t[o] for o in outs])


def run(state):
    state["module"].forward(*state["args"])
    return state["outputs"]


# ------------------------------------------------------------------------------------------------ accounting
def work(case):
    """Bytes with every input read and every output written once, and the operations of the contractions (a causal
    problem counts the visible half of its scores, and of its noise)."""
    op = case["op"]
    if op == "rms":
        n = case["rows"] * case["cols"]
        return dict(bytes=2 * (2 * n + case["cols"]), flops=4 * n)
    if op == "lora":
        m, n, p, r = case["tokens"], case["n"], case["p"], case["r"]
        return dict(bytes=2 * (m * n + n * p + n * r + r * p + m * p), flops=2 * m * (n * p + n * r + r * p))
    if op == "gmlp":
        m, n, k = case["tokens"], case["n"], case["k"]
        return dict(bytes=2 * (m * k + 2 * k * n + m * n), flops=4 * m * n * k)
    if op == "decode":
        h, _, d = HEADS[case["heads"]]
        m, keys, n, variant = case["new"], case["past"] + case["new"], h * d, case["variant"]
        size = 2 * m * n + 3 * n * n + 2 * h * keys * d
        size += h * m * keys + h * keys if variant == "keyformer" else 4 * h * keys if variant == "roco" else 0
        return dict(bytes=2 * size, flops=2 * 3 * m * n * n + 4 * h * m * keys * d)
    hq, hkv, d = HEADS[case["heads"]]
    b, s = case["batch"], case["seq"]
    if op == "prenorm":
        hidden, cols = hq * d, (hq + 2 * hkv) * d
        return dict(bytes=2 * (2 * b * s * hidden + hidden * cols + hidden),
                    flops=2 * b * s * hidden * cols + 2 * b * hq * s * s * d)
    size, flops = 2 * (2 * b * hq * s * d + 2 * b * hkv * s * d), 2 * b * hq * s * s * d
    if op == "keyformer":
        size += (4 if case["noise"] == "fp32" else 2) * (b * hq * s * (s + 1) // 2 + b * hq * s)
    elif op == "roco":
        size += 4 * 2 * b * hq * s
    return dict(bytes=size, flops=flops)


def tolerance(case):
    """About four times the distance from a float64 evaluation, measured per operator on these inputs (relative 2-norm /
    largest element): fp16 inputs to the matrix products, fp16 probabilities, fp16 outputs.  RMSNorm 2.1e-4 / 4.9e-4;
    attention 3.2e-4 / 7.6e-3, with norms of Q and K 4.1e-4 / 8.2e-3, behind the projections 7.1e-4 / 1.1e-2; decode
    4.2e-4 / 2.4e-3; linear layers 3.4e-4 / 1.4e-3."""
    op = case["op"]
    if op == "rms":
        return dict(rel=8e-4, max=2e-3)
    if op in ("lora", "gmlp"):
        return dict(rel=1.4e-3, max=6e-3)
    if op == "decode":
        return dict(rel=1.7e-3, max=1e-2)
    return dict(rel=3e-3 if op == "prenorm" else 1.7e-3, max=4e-2)

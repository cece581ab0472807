"""What this library is timed on: the calls its users make, from one decoding row to a whole prompt.

    listed()            the cases, by name
    draw(rng)           one more case of the same kinds and ranges, sizes spread over their logarithm
    prepare(case, seed) the inputs, packed weights, model and KV cache a program holds before the call
    run(state)          one pass through the public entry points
    work(case)          bytes and operations that pass cannot do without
    tolerance(case)     how far another correct implementation of the same precision may be from this one

Weights are Gaussian with log-normal column scales, quantized by the library's own quantizer; activations carry one per
cent of outlier channels at twenty times the rest.  Sizes are the layers and models of bench.py and the tests (hidden
2048, 64 and 257 experts) and the layers of models a quarter and four times that size."""
import math

import torch

import mxfp4_int8_m5_amd as scmx
from mxfp4_int8_m5_amd import fused_olmoe, fused_qwen3, fused_qwen35, pack_format

S, G, F = scmx.sc_kernels, scmx.sc_decode, scmx.sc_format
BF = torch.bfloat16
SC = F.Format()                 # the published format, named rather than left to the process-wide default
FAMILY = "e2m1/B16/M1..10"      # the deployed member of the format family
FORMATS = ("sc", "mxfp4", FAMILY)   # published 2-bit block codes; a standard MXFP4 tensor read in place; the family

# The four linears of a dense block (rows, columns, epilogue: 1 = scale, 2 = + residual, 3 = SwiGLU) at three widths.
LAYERS = {
    "small": {"qkv": (1152, 896, 1), "o": (896, 896, 2), "gate_up": (9728, 896, 3), "down": (896, 4864, 2)},
    "medium": {"qkv": (4096, 2048, 1), "o": (2048, 2048, 2), "gate_up": (12288, 2048, 3), "down": (2048, 6144, 2)},
    "large": {"qkv": (6144, 4096, 1), "o": (4096, 4096, 2), "gate_up": (24576, 4096, 3), "down": (4096, 12288, 2)},
}
HEAD = (151936, 2048, 1)        # output head


def _layer(kind, rows, shape, fmt, name=None):
    n, k, epi = shape
    case = {"kind": kind, "rows": rows, "n": n, "k": k, "epi": epi, "fmt": fmt}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one token through an attention output projection: what a batch-1 decode loop calls most
        _layer("gemv", 1, LAYERS["medium"]["o"], "sc", "gemv_o_one_row"),
        # the output head for three sequences decoding side by side
        _layer("gemv", 3, HEAD, "sc", "gemv_head_three_rows"),
        # a short prompt, or forty sequences decoding together, through the longest reduction of a block
        _layer("linear", 40, LAYERS["medium"]["down"], "sc", "linear_down_40"),
        # an ordinary prompt through the widest layer, SwiGLU included
        _layer("linear", 2048, LAYERS["medium"]["gate_up"], "sc", "linear_gate_up_2048"),
        # a long ragged prompt through a larger model's attention projections, weights as a standard MXFP4 tensor
        _layer("linear", 6001, LAYERS["large"]["qkv"], "mxfp4", "linear_mxfp4_6001"),
        # a prompt through a dense model: hidden states, the last token's logits, the filled cache
        {"name": "qwen3_prefill_1500", "kind": "qwen3_prefill", "blocks": 4, "tokens": 1500, "cached": 0},
        # one token of a served conversation, the whole step as one graph
        {"name": "qwen3_decode_3000", "kind": "qwen3_decode", "blocks": 4, "cached": 3000},
        # a prompt through a mixture-of-experts model (64 experts, top-8)
        {"name": "olmoe_prefill_3000", "kind": "olmoe_prefill", "blocks": 2, "tokens": 3000, "cached": 0},
        # one token of the same model
        {"name": "olmoe_decode_300", "kind": "olmoe_decode", "blocks": 2, "cached": 300},
        # a prompt through a sparse block with 256 routed experts and a shared one, weights in the deployed format
        {"name": "qwen35_moe_2000", "kind": "qwen35_moe", "tokens": 2000, "fmt": FAMILY},
        # packing a checkpoint's layer into the published format, and into the deployed one
        {"name": "pack_sc_gate_up", "kind": "pack", "n": 12288, "k": 2048, "fmt": "sc", "dtype": "bf16"},
        {"name": "pack_family_o", "kind": "pack", "n": 2048, "k": 2048, "fmt": FAMILY, "dtype": "bf16"},
    ]


def _spread(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "linear", "linear", "linear", "qwen3_prefill", "qwen3_decode", "olmoe_prefill",
                       "olmoe_decode", "qwen35_moe", "pack", "pack"])
    shape = rng.choice([s for w in LAYERS.values() for s in w.values()])
    fmt = rng.choice(FORMATS)
    if kind == "gemv":
        shape = rng.choice([shape, shape, HEAD])
        rows = _spread(rng, 1, 8)
        return _layer("gemv", min(rows, 4) if shape[1] > 8192 else rows, shape, fmt)
    if kind == "linear":
        most = 6001 * 6144 * 4096 // (shape[0] * shape[1])
        return _layer("linear", _spread(rng, 9, min(8192, most)), shape, fmt)
    if kind == "qwen3_prefill":
        cached = rng.choice([0, 0, _spread(rng, 1, 4000)])
        return {"kind": kind, "blocks": 4, "tokens": _spread(rng, 2, 1200), "cached": cached}
    if kind == "qwen3_decode":
        return {"kind": kind, "blocks": 4, "cached": _spread(rng, 1, 12000)}
    if kind == "olmoe_prefill":
        return {"kind": kind, "blocks": 2, "tokens": _spread(rng, 2, 3000), "cached": rng.choice([0, 0, _spread(rng, 1, 1000)])}
    if kind == "olmoe_decode":
        return {"kind": kind, "blocks": 2, "cached": _spread(rng, 1, 4000)}
    if kind == "qwen35_moe":
        return {"kind": kind, "tokens": _spread(rng, 1, 2048), "fmt": rng.choice(["sc", FAMILY])}
    n, k, _ = shape
    if fmt == FAMILY:   # several hundred trial roundings per weight: fewer rows
        n = min(n, 2048 * 2048 // k)
    return {"kind": "pack", "n": max(1, round(n * rng.uniform(0.3, 1.0))), "k": k, "fmt": "sc" if fmt == "mxfp4" else fmt,
            "dtype": rng.choice(["bf16", "f32"])}


# ---- inputs --------------------------------------------------------------------------------------------------------

class _Source:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, device="cuda", generator=self.g)

    def weights(self, n, k):
        return self.normal(n, k).mul_(0.02 * torch.exp(0.4 * self.normal(k)))

    def gain(self, n):
        return (1.0 + 0.1 * self.normal(n)).to(BF)

    def activations(self, m, k):
        scale = torch.ones(k, device="cuda")
        scale[torch.randperm(k, device="cuda", generator=self.g)[:max(1, k // 100)]] = 20.0
        return (self.normal(m, k) * scale).to(BF)

    def ids(self, n, vocab):
        return torch.randint(0, vocab, (n,), device="cuda", generator=self.g)

    def packed(self, n, k):
        return F.quantize(self.weights(n, k), SC, with_q=False)[:3]


def _packed_as(src, n, k, name):
    """(codes, block codes, row scales, format) of a layer stored as `name`."""
    if name == "sc":
        return (*src.packed(n, k), SC)
    if name == "mxfp4":
        codes, bc, ws = src.packed(n, k)
        shift = torch.stack([(bc >> (2 * i)) & 3 for i in range(4)], -1).reshape(n, k // 32)
        e8m0 = (shift + (torch.log2(ws).round().to(torch.int64) + 128).to(torch.uint8)[:, None]).contiguous()
        return codes, e8m0, F.mxfp4_row_scales(e8m0), F.MXFP4
    fmt = pack_format.sc_format_of(name)
    return (*pack_format.pack_matrix(src.weights(n, k), name, fmt)[:3], fmt)


def _fill(src, cache, rows):
    """The keys and values of `rows` earlier tokens (keys come out of a norm: unit variance)."""
    for c in cache:
        c.k[:, :rows] = src.normal(c.k.shape[0], rows, c.k.shape[2]).to(BF)
        c.v[:, :rows] = src.normal(c.v.shape[0], rows, c.v.shape[2]).to(BF)
        c.offset = rows
    return cache


# Embeddings are scaled so that the residual stream carries several times what one block adds to it, as in a trained model.
EMBED = 4.0


def _qwen3(src, blocks):
    a = fused_qwen3.Qwen3Args(num_hidden_layers=blocks)
    D, Fi, d = a.hidden_size, a.intermediate_size, a.head_dim
    hq, hk = a.num_attention_heads, a.num_key_value_heads
    shapes = {"self_attn.q_proj": (hq * d, D), "self_attn.k_proj": (hk * d, D), "self_attn.v_proj": (hk * d, D),
              "self_attn.o_proj": (D, hq * d), "mlp.gate_proj": (Fi, D), "mlp.up_proj": (Fi, D), "mlp.down_proj": (D, Fi)}
    params = {"model.embed_tokens.weight": src.normal(a.vocab_size, D) * EMBED, "model.norm.weight": src.gain(D)}
    packed = {}
    for i in range(blocks):
        p = f"model.layers.{i}."
        params.update({p + "input_layernorm.weight": src.gain(D), p + "post_attention_layernorm.weight": src.gain(D),
                       p + "self_attn.q_norm.weight": src.gain(d), p + "self_attn.k_norm.weight": src.gain(d)})
        packed.update({f"layers.{i}.{n}": src.packed(*s) for n, s in shapes.items()})
    return fused_qwen3.FusedQwen3(a, params, packed)


def _olmoe(src, blocks):
    a = fused_olmoe.OlmoeArgs(num_hidden_layers=blocks)
    D, Fi, E = a.hidden_size, a.intermediate_size, a.num_experts
    params = {"model.embed_tokens.weight": src.normal(a.vocab_size, D) * EMBED, "model.norm.weight": src.gain(D),
              "lm_head.weight": src.normal(a.vocab_size, D) * 0.02}
    flat = {}

    def stack(key, n, k):   # one launch for all experts of a projection
        c, b, w = (t.cpu().numpy() for t in src.packed(E * n, k))
        for e in range(E):
            flat[f"{key}.{e}"] = (c[e * n * k // 8:(e + 1) * n * k // 8], b[e * n:(e + 1) * n], w[e * n:(e + 1) * n])

    for i in range(blocks):
        p = f"model.layers.{i}."
        params.update({p + n + ".weight": src.gain(D) for n in ("input_layernorm", "post_attention_layernorm",
                                                                 "self_attn.q_norm", "self_attn.k_norm")})
        # experts of unequal popularity
        params[p + "mlp.gate.weight"] = src.normal(E, D) * 0.03 * torch.exp(0.3 * src.normal(E, 1))
        flat.update({f"layers.{i}.{n}": src.packed(D, D) for n in fused_olmoe.ATTN})
        stack(f"layers.{i}.experts.gate_proj", Fi, D)
        stack(f"layers.{i}.experts.up_proj", Fi, D)
        stack(f"layers.{i}.experts.down_proj", D, Fi)
    return fused_olmoe.FusedOlmoe(a, params, flat)


def _qwen35(src, fmt_name):
    a = fused_qwen35.Qwen35MoeArgs()
    D, Fi, E = a.hidden_size, a.moe_intermediate_size, a.num_experts
    fmt = None if fmt_name == "sc" else pack_format.sc_format_of(fmt_name)
    flat = {}
    for name, (n, k) in {"gate_proj": (Fi, D), "up_proj": (Fi, D), "down_proj": (D, Fi)}.items():
        if fmt is None:
            c, b, w = src.packed((E + 1) * n, k)
        else:   # Gaussian weights' codes and block multipliers tiled from a few experts: packing them all takes a second
            c, b, w = pack_format.pack_matrix(src.weights(8 * n, k), fmt_name, fmt)[:3]
            few = torch.randint(0, 8, (E + 1,), device="cuda", generator=src.g)
            c, b, w = (t.reshape(8, n, -1)[few] for t in (c, b, w))
        flat[f"experts.{name}.codes"] = c.reshape(E + 1, n, -1)
        flat[f"experts.{name}.bcodes"] = b.reshape(E + 1, n, -1)
        flat[f"experts.{name}.wscale"] = w.reshape(E + 1, n)
    flat = {k: t.cpu().numpy() for k, t in flat.items()}
    gate = src.normal(E, D) * 0.03 * torch.exp(0.3 * src.normal(E, 1))
    return fused_qwen35.Qwen35Moe(a, src.gain(D), gate, src.normal(1, D) * 0.03, flat, fmt=fmt)


def prepare(case, seed):
    src, kind = _Source(seed), case["kind"]
    if kind in ("gemv", "linear"):
        m, n, k, epi = case["rows"], case["n"], case["k"], case["epi"]
        codes, bc, ws, fmt = _packed_as(src, n, k, case["fmt"])
        st = {"x": src.activations(m, k), "codes": codes, "bcodes": bc, "wscale": ws, "fmt": fmt, "n": n, "epi": epi,
              "res": src.activations(m, n) if epi == 2 else None}
    elif kind in ("qwen3_prefill", "olmoe_prefill"):
        model = (_qwen3 if kind == "qwen3_prefill" else _olmoe)(src, case["blocks"])
        cache = _fill(src, model.make_cache(max(4096, case["cached"] + case["tokens"])), case["cached"])
        st = {"model": model, "cache": cache, "cached": case["cached"], "ids": src.ids(case["tokens"], model.args.vocab_size)}
    elif kind in ("qwen3_decode", "olmoe_decode"):
        model = (_qwen3 if kind == "qwen3_decode" else _olmoe)(src, case["blocks"])
        cache = _fill(src, model.make_cache(max(4096, case["cached"] + 64)), case["cached"])
        if kind == "qwen3_decode":
            dec = fused_qwen3.DecodeQwen3(model, fuse_prologue=True, graphs="step", head="packed")
        else:
            dec = fused_olmoe.DecodeOlmoe(model, fuse_prologue=True)
        st = {"decoder": dec, "cache": cache, "cached": case["cached"], "tok": src.ids(1, model.args.vocab_size)}
    elif kind == "qwen35_moe":
        model, L = _qwen35(src, case["fmt"]), case["tokens"]
        h = torch.zeros((S.pad_rows(L), model.args.hidden_size), dtype=BF, device="cuda")
        h[:L] = src.activations(L, model.args.hidden_size)
        st = {"model": model, "h": h, "tokens": L}
    else:
        w = src.weights(case["n"], case["k"])
        st = {"w": w.to(BF) if case["dtype"] == "bf16" else w, "fmt": case["fmt"]}
    return dict(st, kind=kind)


def _rewind(st):
    """The conversation goes back to the tokens it had (a host-side counter): the call can be made again."""
    for c in st["cache"]:
        c.offset = st["cached"]
    return st["cache"]


def run(st):
    kind = st["kind"]
    if kind == "gemv":
        return G.gemv(st["x"], st["codes"], st["bcodes"], None, st["wscale"], st["n"], st["epi"], res=st["res"], pro=1,
                      fmt=st["fmt"])
    if kind == "linear":
        return S.linear_w4a8(st["x"], st["codes"], st["bcodes"], st["wscale"], st["n"], st["epi"], st["res"], st["fmt"])
    if kind in ("qwen3_prefill", "olmoe_prefill"):
        cache = _rewind(st)
        h = st["model"].hidden(st["ids"], cache)
        return {"hidden": h, "logits": st["model"].logits(h[-1:]), "k": [c.k for c in cache], "v": [c.v for c in cache]}
    if kind in ("qwen3_decode", "olmoe_decode"):
        cache = _rewind(st)
        logits = st["decoder"].step(st["tok"], cache)
        return {"logits": logits, "k": [c.k for c in cache], "v": [c.v for c in cache]}
    if kind == "qwen35_moe":
        return st["model"].prefill(st["h"], st["tokens"])
    if st["fmt"] == "sc":
        return F.quantize(st["w"], SC, with_q=False)[:3]
    return pack_format.pack_matrix(st["w"], st["fmt"])[:3]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------

def _weight_bytes(n, k, fmt="sc"):
    return n * k * (0.5 + {"sc": 1 / 128, "mxfp4": 1 / 32, FAMILY: 1 / 32}[fmt]) + 4 * n


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "linear"):
        m, n, k = case["rows"], case["n"], case["k"]
        out = 2 * m * (n // 2 if case["epi"] == 3 else n) * (2 if case["epi"] == 2 else 1)
        return {"bytes": _weight_bytes(n, k, case["fmt"]) + 2 * m * k + out, "flops": 2.0 * m * n * k}
    if kind == "pack":
        n, k = case["n"], case["k"]
        # per weight: three exponents (or 8 row bases times 10 multipliers), each a scale, a rounding, a squared difference
        trials = 3 if case["fmt"] == "sc" else 80
        return {"bytes": n * k * (2 if case["dtype"] == "bf16" else 4) + _weight_bytes(n, k, case["fmt"]),
                "flops": n * k * trials * 5.0}
    if kind == "qwen35_moe":
        t, d, f, e = case["tokens"], 2048, 512, 256
        used = 1 + e * (1 - (1 - 8 / e) ** t)   # experts that some token visits
        return {"bytes": used * (_weight_bytes(2 * f, d, case["fmt"]) + _weight_bytes(d, f, case["fmt"])) + 2 * e * d + 4 * t * d,
                "flops": 2.0 * t * (9 * 3 * f * d + e * d)}
    t, c, blocks = case.get("tokens", 1), case["cached"], case["blocks"]
    scores = t * c + t * (t + 1) / 2     # query-key pairs
    if kind.startswith("qwen3"):
        layer = [s[:2] for s in LAYERS["medium"].values()]
        w = sum(_weight_bytes(*s) for s in layer)
        macs, kv, heads = t * sum(n * k for n, k in layer), 8 * 128, 16
        head = _weight_bytes(151936, 2048) if kind == "qwen3_decode" else 2 * 151936 * 2048
        vocab = 151936
    else:
        used = 64 * (1 - (1 - 8 / 64) ** t)
        w = (_weight_bytes(6144, 2048) + _weight_bytes(2048, 2048) + 2 * 64 * 2048
             + used * (_weight_bytes(2048, 2048) + _weight_bytes(2048, 1024)))
        macs, kv, heads = t * (4 * 2048 * 2048 + 64 * 2048 + 8 * 3 * 1024 * 2048), 16 * 128, 16
        vocab = 50304
        head = 2 * vocab * 2048
    cache = 4 * kv * (c + 2 * t)       # earlier rows read, new rows written and read
    return {"bytes": blocks * (w + cache) + head + 2 * t * 2048 * 2 + 2 * vocab,
            "flops": 2.0 * (blocks * (macs + scores * heads * 128 * 2) + vocab * 2048)}


def tolerance(case):
    # Integer sums and single roundings; a packed byte is a byte.
    if case["kind"] in ("gemv", "linear", "pack"):
        return "exact"
    # Through the blocks of a model a sum taken in another order moves a few activations to the neighbouring INT8 code.
    # With the attention replaced by float32 array operations (cut into other ranges at decode) the outputs moved by
    # up to 1.9e-2 (four dense blocks of a prompt), 1.1e-2 (a dense decode step) and 7.5e-3 (two sparse blocks).
    return {"rel": {"qwen3_prefill": 7e-2, "qwen3_decode": 4e-2}.get(case["kind"], 3e-2)}

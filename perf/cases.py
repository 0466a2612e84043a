"""What a user of this package has it do, as measurable cases.

A case is a dict of plain values; `prepare` builds the module and the inputs a serving program
holds, `run` is one forward through the public module surface (PalettizedLinear, SplitQKV,
FusedPalettizedMLP, PalettizedEmbedding), `work` counts what that forward cannot do without and
`tolerance` says how far two correct implementations may lie apart.

Ranges (what `draw` covers and the listed cases stand for):
  linear     M 1 ... 4096 tokens, N 128 ... 12288 outputs (the vocabulary head at M = 1: up to
             248320), K 1024 ... 12288 inputs, every width pair that deployed weights have, LUT
             groups of 64 ... 256 rows, float16 / bfloat16 LUTs and activations, with and without
             rotation, low-rank residual and bias
  qkv        three projections of one input, M 1 ... 1024
  mlp        gate, up, SiLU * mul, down; M 1 ... 1024
  embedding  1 ... 4096 ids, tables of 1024 ... 248320 rows, rotated and plain
Weights are uniform random indices and sorted LUT rows ~ N(0, 0.02), activations ~ N(0, 1).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "rag-cache-engineering-qwen35-9b-flute_amd"))

import palettized_modules as pm  # noqa: E402

DEVICE = "cuda"
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}


def _linear(name, M, N, K, bits=4, bits2=0, group=128, lut="f16", act="f16", rank=0, bias=False,
            rotated=False):
    return {"name": name, "kind": "linear", "M": M, "N": N, "K": K, "bits": bits, "bits2": bits2,
            "group": group, "lut": lut, "act": act, "rank": rank, "bias": bias, "rotated": rotated}


def _qkv(name, M, N, NKV, K, bits=4, bits2=0, group=128, lut="f16", act="f16", rank=0, rotated=False):
    return {"name": name, "kind": "qkv", "M": M, "N": N, "NKV": NKV, "K": K, "bits": bits,
            "bits2": bits2, "group": group, "lut": lut, "act": act, "rank": rank, "bias": False,
            "rotated": rotated}


def _mlp(name, M, N, K, bits=4, bits2=0, group=128, lut="f16", act="f16", rank=0, rotated=False):
    return {"name": name, "kind": "mlp", "M": M, "N": N, "K": K, "bits": bits, "bits2": bits2,
            "group": group, "lut": lut, "act": act, "rank": rank, "bias": False, "rotated": rotated}


def _embedding(name, M, N, K, bits=4, bits2=0, group=128, lut="f16", rotated=False):
    return {"name": name, "kind": "embedding", "M": M, "N": N, "K": K, "bits": bits, "bits2": bits2,
            "group": group, "lut": lut, "act": lut, "rank": 0, "bias": False, "rotated": rotated}


def listed():
    return [
        # one token through a key or value projection: the smallest call of a decode loop
        _linear("kv_decode", 1, 1024, 4096),
        # one token through the grouped q/k/v projections of a deployed (rotated, two-stream,
        # residual) attention block
        _qkv("qkv_decode", 1, 4096, 1024, 4096, bits=4, bits2=1, act="bf16", rank=16, rotated=True),
        # one token through the gated MLP block
        _mlp("mlp_decode", 1, 12288, 4096, act="bf16"),
        # one token through a deployed down projection: the most frequent width pair, rotated input
        _linear("down_decode_rotated", 1, 4096, 12288, bits=3, bits2=3, rotated=True),
        # one token through the vocabulary head: the largest weight stream
        _linear("lm_head_decode", 1, 248320, 4096, act="bf16"),
        # eight sequences decoded together, rotated input
        _linear("batch8_rotated", 8, 12288, 4096, act="bf16", rotated=True),
        # a ragged batch of decoding sequences through a deployed two-stream down projection
        _linear("batch48_two_streams", 48, 4096, 12288, bits=4, bits2=1, rank=16, bias=True),
        # a short prompt through the up projection
        _linear("prefill256", 256, 12288, 4096, lut="bf16", act="bf16"),
        # a prompt of odd length through the whole gated MLP block
        _mlp("prefill509_mlp", 509, 12288, 4096, act="bf16"),
        # a prompt of odd length through a deployed layer: rotation, two streams, residual
        _linear("prefill1000_deployed", 1000, 12288, 4096, bits=1, bits2=4, rank=16, rotated=True),
        # a long prompt chunk through the down projection: the largest product
        _linear("prefill4096", 4096, 4096, 12288, lut="bf16", act="bf16"),
        # the embedding rows of a prompt out of the rotated (tied) vocabulary table
        _embedding("embed_prompt", 1000, 248320, 4096, rotated=True),
    ]


def _spread(rng, lo, hi):
    """A whole number of lo ... hi, uniform over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["qkv", "mlp", "mlp", "embedding"])
    bits, bits2 = rng.choice([(4, 0), (4, 0), (4, 0), (3, 0), (4, 1), (1, 4), (3, 3), (3, 3), (2, 4), (2, 3)])
    group = rng.choice([128, 128, 128, 64, 256])
    lut, act = rng.choice([("f16", "f16"), ("f16", "bf16"), ("bf16", "bf16")])
    rank = rng.choice([0, 0, 0, 8, 16])
    rotated = rng.random() < 0.4
    K = 64 * _spread(rng, 16, 192)
    one = rng.random() < 0.35                       # a single token, as most calls of a decode loop are
    most = 4096 * 4096 * 12288                      # the largest listed product
    streams = 2 if bits2 else 1
    if kind == "linear":
        head = one and rng.random() < 0.15
        N = 128 * (_spread(rng, 400, 1940) if head else _spread(rng, 1, 96))
        if head:
            K = min(K, 4096)
        M = 1 if one else _spread(rng, 2, 4096)
        M = max(1, min(M, most // (N * K * streams)))
        return _nameless(_linear("", M, N, K, bits, bits2, group, lut, act, rank, rng.random() < 0.25, rotated))
    if kind == "qkv":
        N, NKV = 128 * _spread(rng, 4, 64), 128 * _spread(rng, 1, 16)
        M = 1 if one else _spread(rng, 2, 1024)
        M = max(1, min(M, most // ((N + 2 * NKV) * K * streams)))
        return _nameless(_qkv("", M, N, NKV, K, bits, bits2, group, lut, act, rank, rotated))
    if kind == "mlp":
        K, N = min(K, 64 * 2 * _spread(rng, 8, 32)), 128 * _spread(rng, 16, 96)
        K = K // 128 * 128                          # the block's output rows
        M = 1 if one else _spread(rng, 2, 1024)
        M = max(1, min(M, most // (3 * N * K * streams)))
        return _nameless(_mlp("", M, N, K, bits, bits2, group, lut, act, rank, rotated))
    K = min(K, 4096)
    return _nameless(_embedding("", _spread(rng, 1, 4096), 128 * _spread(rng, 8, 1940), K, bits, bits2,
                                group, lut, rotated))


def _nameless(case):
    del case["name"]
    return case


def _lut(rows, bits, scale, dtype, gen):
    v = torch.randn(rows, 1 << bits, device=DEVICE, generator=gen) * scale
    return v.sort(dim=1).values.to(dtype).contiguous()


def _operands(c, N, K, gen, rank=None, bias=None):
    """The tensors of one palettized weight (any byte string is a valid idxN blob)."""
    rank = c["rank"] if rank is None else rank
    bias = c["bias"] if bias is None else bias
    lut_t, act = DTYPES[c["lut"]], DTYPES[c["act"]]
    rows = -(-N // c["group"])

    def blob(b):
        return torch.randint(0, 256, (N * K * b // 8,), dtype=torch.uint8, device=DEVICE, generator=gen)
    kw = {"indices": blob(c["bits"]), "lut": _lut(rows, c["bits"], 0.02, lut_t, gen)}
    if c["bits2"]:
        kw["indices2"], kw["lut2"] = blob(c["bits2"]), _lut(rows, c["bits2"], 0.01, lut_t, gen)
        kw["bitwidth2"] = c["bits2"]
    if rank:
        kw["resA"] = (torch.randn(N, rank, device=DEVICE, generator=gen) * 0.05).to(act)
        kw["resB"] = (torch.randn(rank, K, device=DEVICE, generator=gen) * 0.02).to(act)
    if bias:
        kw["bias"] = (torch.randn(N, device=DEVICE, generator=gen) * 0.1).to(act)
    return kw


def _module(c, N, K, gen, seed):
    kw = _operands(c, N, K, gen)
    rot = dict(rotation_seed=seed, rotation_k=K) if c["rotated"] else {}
    return pm.PalettizedLinear(bitwidth=c["bits"], group_size=c["group"], N=N, K=K, **kw, **rot).eval()


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    c, M, N, K = case, case["M"], case["N"], case["K"]
    if c["kind"] == "embedding":
        kw = _operands(c, N, K, gen)
        rot = dict(rotation_seed=seed, rotation_k=K) if c["rotated"] else {}
        m = pm.PalettizedEmbedding(bitwidth=c["bits"], group_size=c["group"], N=N, K=K, reference=False,
                                   **kw, **rot).eval()
        return {"module": m, "x": torch.randint(0, N, (M,), device=DEVICE, generator=gen)}
    if c["kind"] == "linear":
        m = _module(c, N, K, gen, seed)
    elif c["kind"] == "qkv":
        m = pm.SplitQKV(_module(c, N, K, gen, seed), _module(c, c["NKV"], K, gen, seed),
                        _module(c, c["NKV"], K, gen, seed)).eval()
    else:
        m = pm.FusedPalettizedMLP(_module(c, N, K, gen, seed), _module(c, N, K, gen, seed),
                                  _module(c, K, N, gen, seed + 1), torch.nn.SiLU()).eval()
    x = torch.randn(M, K, device=DEVICE, generator=gen).to(DTYPES[c["act"]])
    return {"module": m, "x": x}


@torch.no_grad()
def run(state):
    return state["module"](state["x"])


def work(case):
    c, M, N, K = case, case["M"], case["N"], case["K"]
    widths = [c["bits"]] + ([c["bits2"]] if c["bits2"] else [])
    streams = len(widths)
    if c["kind"] == "embedding":
        row = sum(K * b / 8 + 2 * 2 ** b for b in widths)
        return {"bytes": M * (8 + row + 2 * K), "flops": M * K * (streams + (math.log2(K) if c["rotated"] else 0))}

    def weight(n, k):
        luts = sum(-(-n // c["group"]) * 2 * 2 ** b for b in widths)
        extra = 2 * c["rank"] * (n + k) + (2 * n if c["bias"] else 0) + (4 * k if c["rotated"] else 0)
        return sum(n * k * b / 8 for b in widths) + luts + extra

    def flops(n, k):
        return 2.0 * M * (n * k * streams + c["rank"] * (n + k)) + (M * k * math.log2(k) if c["rotated"] else 0)
    if c["kind"] == "linear":
        parts, io = [(N, K)], M * (N + K)
    elif c["kind"] == "qkv":
        parts, io = [(N, K), (c["NKV"], K), (c["NKV"], K)], M * (N + 2 * c["NKV"] + K)
    else:
        parts, io = [(N, K), (N, K), (K, N)], 2 * M * K
    return {"bytes": sum(weight(n, k) for n, k in parts) + 2 * io, "flops": sum(flops(n, k) for n, k in parts)}


def tolerance(case):
    """About four times the distance of the path from the same forward in 64 bits (the float64
    products of the dequantised weights and unrounded intermediates), which is the rounding of the
    activations' type: once at the output, and once more for each intermediate a chain rounds
    (the rotated input, one output per stream, the gated product of the MLP)."""
    f16 = case["act"] == "f16"
    if case["kind"] == "embedding":
        return {"rel": 8e-4 if f16 else 8e-3}       # seen: 2.1e-4, 2.4e-3
    if case["kind"] == "mlp":
        return {"rel": 2.4e-3 if f16 else 1.6e-2}   # seen with bfloat16: 2.6e-3 ... 4.2e-3
    return {"rel": 1.6e-3 if f16 else 1e-2}         # seen: 2.0e-4 ... 4.2e-4, 1.6e-3 ... 2.9e-3

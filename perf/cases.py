"""The calls this framework is timed on: one attention layer, as a program that serves or trains a model calls it.

A case is a dict of plain values: the call ("infer": forward without gradients, output and log-sum-exp; "train":
forward and backward, output and the gradients of q, k and v), the shape, the module's options and how the inputs
are laid out in memory.  `listed` holds the cases, `draw` gives more of the same ranges, `prepare` makes what the
program has in hand before the call (inputs and module), `run` is one pass.
"""
import math

import torch

from hyperattention_amd import HyperAttention

# What a case holds when it does not say otherwise: the module's defaults at head dim 64.
DEFAULTS = {
    "call": "infer", "batch": 1, "heads": 24, "kv_heads": 24, "seq": 4096, "dim": 64, "dtype": "bf16", "causal": True,
    "projs": 8, "block": 256, "sample": 256, "min_seq": 2048, "smooth": False,
    # "bhnd": contiguous (batch, heads, seq, dim) tensors; "bnhd": the layer's projections give (batch, seq, heads,
    # dim), which the layer hands over as transposed views
    "layout": "bhnd",
    # "normal": independent N(0, 1); "clusters": queries and keys around 64 common centroids, so that the hash
    # buckets are filled unevenly, as those of trained models are
    "data": "normal",
}


def _case(name=None, **kw):
    c = dict(DEFAULTS, **kw)
    if "kv_heads" not in kw:
        c["kv_heads"] = c["heads"]
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # a short prompt: under min_seq_len the layer is exact attention, one launch; length not a multiple of a tile
        _case("short_prompt", heads=24, seq=1000),
        # the smallest hashed layer, an encoder's: every launch of the path for little work
        _case("encoder_small", heads=4, seq=4096, dtype="fp16", causal=False),
        # the shortest prompt that the causal recursion cuts in two
        _case("prompt_4k", heads=24, seq=4096),
        # an odd length and a head dim between the two that matrix tiles like best
        _case("prompt_odd_d96", heads=16, seq=20479, dim=96),
        # a long document without causal mask
        _case("encoder_32k", heads=32, seq=32768, dtype="fp16", causal=False),
        # long-context prefill at the length the method is quoted on
        _case("prefill_131k", heads=32, seq=131072, dtype="fp16"),
        # long documents in a batch, wide heads, overlapping blocks
        _case("encoder_65k_smooth", batch=2, heads=32, seq=65536, dim=128, causal=False, block=512, sample=512, smooth=True),
        # prefill of a language model's layer: query heads that share key/value heads, projections as they come
        _case("prefill_32k_grouped", heads=32, kv_heads=2, seq=32768, dim=128, layout="bnhd", data="clusters"),
        # training on short sequences: exact attention, forward and backward
        _case("train_2k", call="train", heads=24, seq=2048),
        # training without causal mask
        _case("train_16k_encoder", call="train", heads=24, seq=16384, causal=False),
        # training of a language model's layer with grouped queries and wide heads
        _case("train_16k_grouped", call="train", heads=32, kv_heads=8, seq=16384, dim=128, layout="bnhd"),
        # long-context training
        _case("train_131k", call="train", heads=24, seq=131072),
    ]


def draw(rng):
    # the most that a drawn case computes: a third of the costliest listed one
    most = max(work(c)["flops"] for c in listed()) / 3
    while True:
        call = rng.choice(("infer", "infer", "train"))
        dim = rng.choice((64, 64, 64, 128, 128, 96, 80))
        heads = rng.choice((4, 8, 12, 16, 24, 32))
        block = rng.choice((256, 256, 256, 128, 512))
        c = _case(
            call=call, batch=rng.choice((1, 1, 1, 2, 4)), heads=heads, kv_heads=heads // rng.choice((1, 1, 1, 2, 4)),
            dim=dim, dtype=rng.choice(("bf16", "bf16", "fp16")), causal=rng.random() < 0.65, block=block, sample=block,
            projs=rng.choice((8, 8, 8, 6)), min_seq=rng.choice((2048, 2048, 4096)), smooth=rng.random() < 0.2,
            layout=rng.choice(("bhnd", "bnhd")), data=rng.choice(("normal", "clusters")))
        c["seq"] = _length(math.exp(rng.uniform(math.log(512), math.log(131072))), c, rng)
        if work(c)["flops"] <= most:
            return c


def _length(near, c, rng):
    """A length close to `near` that the layer takes: any length where attention is exact, else one whose hashed
    calls have a multiple of 128 keys; an odd one now and then where the causal recursion takes it."""
    if near < c["min_seq"]:
        return max(int(near), 1)
    if not c["causal"]:
        return max(round(near / 128) * 128, c["min_seq"])
    halvings = 0
    while near / 2 ** (halvings + 1) >= c["min_seq"]:
        halvings += 1
    n = max(round(near / 2 ** halvings / 128), c["min_seq"] // 128) * 128 * 2 ** halvings
    # odd lengths: prompts end anywhere, training sequences seldom do
    return n - 1 if rng.random() < (0.3 if c["call"] == "infer" else 0.1) else n


def _dtype(c):
    return {"fp16": torch.float16, "bf16": torch.bfloat16}[c["dtype"]]


def prepare(case, seed):
    c, dev = case, torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    dtype, n, d = _dtype(c), c["seq"], c["dim"]

    def tensor(heads):
        shape = (c["batch"], heads, n, d) if c["layout"] == "bhnd" else (c["batch"], n, heads, d)
        x = torch.randn(shape, generator=g, device=dev, dtype=dtype)
        return x if c["layout"] == "bhnd" else x.transpose(1, 2)

    q, k, v = tensor(c["heads"]), tensor(c["kv_heads"]), tensor(c["kv_heads"])
    if c["data"] == "clusters":
        centroids = 4 * torch.nn.functional.normalize(torch.randn((64, d), generator=g, device=dev), dim=-1).to(dtype)
        for x in (q, k):
            of = torch.randint(0, 64, x.shape[:3], generator=g, device=dev)
            x.mul_(0.5).add_(centroids[of])
    module = HyperAttention(
        input_dim=d, lsh_num_projs=c["projs"], block_size=c["block"], sample_size=c["sample"], min_seq_len=c["min_seq"],
        smooth_block=c["smooth"], rng=torch.Generator().manual_seed(seed)).to(device=dev, dtype=dtype)
    state = {"module": module, "causal": c["causal"], "q": q, "k": k, "v": v, "dout": None}
    if c["call"] == "train":
        state["dout"] = tensor(c["heads"])
        for x in (q, k, v):
            x.requires_grad_()
    return state


def run(state):
    q, k, v = state["q"], state["k"], state["v"]
    if state["dout"] is None:
        with torch.no_grad():
            return state["module"](q, k, v, causal=state["causal"], return_lse=True)
    out = state["module"](q, k, v, causal=state["causal"])
    return (out.detach(), *torch.autograd.grad(out, (q, k, v), state["dout"]))


def _pairs(c):
    """(query, key) pairs of one head that the layer computes: exact attention up to min_seq_len keys, else blocks
    and samples; causal: leaves and, per halving, second halves against first halves."""
    def unmasked(n):
        return n * n if c["min_seq"] > n else n * (c["block"] + c["sample"])

    n, segments, pairs = c["seq"], 1, 0
    if not c["causal"]:
        return unmasked(n)
    while n > c["min_seq"]:
        n = (n + 1) // 2
        pairs += segments * unmasked(n)
        segments *= 2
    return pairs + segments * n * (n + 1) // 2


def work(case):
    c = case
    q_rows, k_rows, d = c["batch"] * c["heads"] * c["seq"], c["batch"] * c["kv_heads"] * c["seq"], c["dim"]
    pairs = c["batch"] * c["heads"] * _pairs(c)
    if c["call"] == "infer":
        # q, k, v in; the output and its log-sum-exps out.  Two products of 2 d operations a pair
        return {"bytes": 2 * d * (2 * q_rows + 2 * k_rows) + 4 * q_rows, "flops": 4 * d * pairs}
    # q, k, v and the output's gradient in; the output and three gradients out.  Two and five products a pair
    return {"bytes": 2 * d * (4 * q_rows + 4 * k_rows), "flops": 14 * d * pairs}


def tolerance(case):
    # outputs, soft-max weights and, in the backward, the scores' gradients are rounded to the inputs' type: relative
    # errors of a few units of its last place (2^-8 for bf16, 2^-11 for fp16)
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 3e-3}

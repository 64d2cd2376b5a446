"""The work that a user of this framework has it do, as timed cases.

A case names an entry point, a shape and the options of one pass; `prepare` makes what the user's program holds before the
call (tensors on the GPU), `run` makes the call.  `listed()` are fixed cases, `draw()` gives more of the same kinds and ranges.

Fields: entry (which public entry point), b, h (kv heads), r (query groups per kv head), L (positions), d (head dim),
chunk (only shapes the views, except for the chunked operator), dtype, gates (dtype of the gates), mu (mean of the gates'
logits), train (forward + backward, else forward alone), prune (skip pairs that the decay makes negligible).
"""
import torch
import torch.nn.functional as F

from universal_attention_triton_amd.affinity import AffinityScores
from universal_attention_triton_amd.frontend import decoder_attention
from universal_attention_triton_amd.universal_attention import attention, universal_attention
from universal_attention_triton_amd.universal_attention_autograd import SMVecMatMul, UniversalAttention

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}


def _case(entry, b, h, r, L, d, dtype="bf16", train=True, chunk=128, gates=None, mu=0.0, prune=False, **name):
    return dict(name, entry=entry, b=b, h=h, r=r, L=L, d=d, chunk=chunk, dtype=dtype, gates=gates or dtype, mu=mu,
                train=train, prune=prune)


def listed():
    return [
        # the smallest call: one layer on a short float32 sequence, inference (configuration 0)
        _case("universal", 1, 4, 1, 512, 64, "fp32", train=False, chunk=64, name="infer_small_fp32"),
        # batched inference at an ordinary length (configuration 1)
        _case("universal", 2, 16, 1, 2048, 64, train=False, name="infer_batch"),
        # a decoder block reading a prompt of odd length, grouped queries, gates computed in float32
        _case("decoder", 1, 8, 4, 1531, 128, gates="fp32", train=False, name="prefill_decoder"),
        # a training step on short ragged sequences through the decoder block's front end
        _case("decoder", 2, 2, 4, 200, 64, name="train_small"),
        # a training step through the (q, k, v) calling convention, head dim and length no powers of two
        _case("gen2", 2, 4, 3, 1000, 80, name="train_gen2_ragged"),
        # training in float32, for a model that is checked against another implementation
        _case("universal", 1, 8, 1, 2048, 64, "fp32", name="train_fp32"),
        # training at the lengths models are trained on: grouped queries (configuration 3), many heads (configuration 2),
        # long context with slow decay (configuration 4)
        _case("universal", 1, 8, 4, 4096, 128, name="train_gqa"),
        _case("universal", 1, 32, 1, 8192, 128, name="train_headline"),
        _case("universal", 1, 8, 1, 32768, 128, mu=2.0, name="train_long"),
        # long context with pruning
        _case("universal", 1, 16, 1, 16384, 128, prune=True, name="train_pruned"),
        # the call sequence of the per-chunk operator and its merge, forward and backward
        _case("chunked", 1, 16, 1, 4096, 128, name="train_chunked"),
        # the decay bias alone, as a mask for another attention, forward and backward
        _case("bias", 1, 8, 1, 4096, 128, name="train_bias"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["infer_fp32", "infer", "prefill", "train_short", "gen2", "train_fp32", "train", "train", "long", "pruned",
                       "chunked", "bias"])
    d = rng.choice([64, 128])
    if kind == "infer_fp32":
        return _case("universal", rng.choice([1, 2]), rng.randint(2, 8), 1, _log(rng, 128, 2048), d, "fp32", train=False, chunk=64)
    if kind == "infer":
        return _case("universal", rng.randint(1, 4), rng.choice([4, 8, 12, 16]), rng.choice([1, 1, 2, 4]), _log(rng, 256, 4096), d,
                     train=False)
    if kind == "prefill":
        return _case("decoder", 1, rng.choice([2, 4, 8]), rng.choice([2, 4, 8]), _log(rng, 64, 4096), d,
                     gates=rng.choice(["fp32", "bf16"]), train=False)
    if kind == "train_short":
        return _case("decoder", rng.randint(1, 4), rng.choice([1, 2, 4]), rng.choice([1, 2, 4]), _log(rng, 32, 512), d,
                     gates=rng.choice(["fp32", "bf16"]))
    if kind == "gen2":
        return _case("gen2", rng.randint(1, 3), rng.choice([2, 4, 8]), rng.choice([1, 2, 3, 4]), _log(rng, 200, 2500),
                     rng.choice([48, 64, 80, 96, 112, 128]), gates=rng.choice(["fp32", "bf16"]))
    if kind == "train_fp32":
        return _case("universal", 1, rng.randint(2, 8), rng.choice([1, 1, 2]), _log(rng, 256, 3000), d, "fp32")
    if kind == "train":
        r = rng.choice([1, 1, 2, 4])
        return _case("universal", rng.choice([1, 2]), rng.choice([8, 12, 16]) // (1 if r == 1 else 2), r, _log(rng, 1024, 8192), d)
    if kind == "long":
        return _case("universal", 1, rng.choice([2, 4]), 1, _log(rng, 8192, 32768), 128, mu=2.0 * rng.random())
    if kind == "pruned":
        return _case("universal", 1, rng.choice([4, 8, 16]), 1, _log(rng, 4096, 24576), d, prune=True)
    if kind == "chunked":
        chunk = rng.choice([64, 128, 256])
        if rng.random() < 0.25:
            return _case("chunked", 1, rng.randint(2, 8), 1, chunk * max(2, _log(rng, 256, 2048) // chunk), 64, "fp32", chunk=chunk)
        return _case("chunked", 1, rng.choice([4, 8, 16]), rng.choice([1, 1, 2]), chunk * max(2, _log(rng, 512, 4096) // chunk), d,
                     chunk=chunk)
    return _case("bias", 1, rng.choice([2, 4, 8, 16]), 1, 8 * _log(rng, 48, 640), d)


def prepare(case, seed):
    """Keys of unit length, values and queries N(0,1), gates = sigmoid(N(mu,1)), upstream gradients N(0,1)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, gdt = DTYPES[case["dtype"]], DTYPES[case["gates"]]
    b, h, r, L, d = (case[k] for k in ("b", "h", "r", "L", "d"))

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    def gate(*shape):
        return torch.sigmoid(normal(*shape) + case["mu"]).to(gdt)

    entry = case["entry"]
    if entry == "decoder":                      # projections as a decoder block holds them
        args = [normal(b, L, h * r, d).to(dtype), F.normalize(normal(b, L, h, d), dim=-1).to(dtype), normal(b, L, h, d).to(dtype),
                gate(b, L, 2 * h)]
        up = (b, L, h * r, d)
    elif entry == "gen2":
        args = [normal(b, h * r, L, d).to(dtype), F.normalize(normal(b, h, L, d), dim=-1).to(dtype), normal(b, h, L, d).to(dtype),
                gate(b, h, L), gate(b, h, L)]
        up = (b, h * r, L, d)
    elif entry == "bias":
        args = [F.normalize(normal(b, h, L, d), dim=-1).to(dtype), gate(b, h, L), gate(b, h, L)]
        up = (b, h, L, L)
    else:
        c = case["chunk"] if L % case["chunk"] == 0 else L
        args = [F.normalize(normal(b, h, L // c, c, d), dim=-1).to(dtype), normal(b, h, L // c, c, d).to(dtype),
                normal(b, h, r, L, d).to(dtype), gate(b, h, L // c, c), gate(b, h, L)]
        up = (b, h, r, L, d)
    if not case["train"]:
        return {"case": case, "args": args}
    return {"case": case, "args": [a.requires_grad_() for a in args], "up": normal(*up).to(dtype)}


def run(state):
    case, args = state["case"], state["args"]
    entry = case["entry"]
    if entry == "decoder":
        out = decoder_attention(*args)
    elif entry == "gen2":
        q, k, v, src, dest = args
        out = attention(q, k, v, True, None, src, dest)
    elif entry == "bias":
        out = AffinityScores.apply(*args)
    elif entry == "chunked":
        out = SMVecMatMul.apply(*UniversalAttention.apply(*args))
    else:
        out = universal_attention(*args, prune=case["prune"])
    if not case["train"]:
        return out
    return (out, *torch.autograd.grad(out, args, state["up"]))


def work(case):
    """Bytes: every input and upstream gradient read once, the output and every gradient written once.  Operations: one
    matrix product over the causal pairs is d L^2 per head: the key-key product and its two gradients once per kv head, scores
    and output and their four gradients once per query head.  Pruned passes count the band in which a weight can matter (about
    1700 positions at d = 128 with these inputs)."""
    b, h, r, L, d = (case[k] for k in ("b", "h", "r", "L", "d"))
    size, gsize = (4 if case[k] == "fp32" else 2 for k in ("dtype", "gates"))
    keys, queries, gates = b * h * L * d * size, b * h * r * L * d * size, 2 * b * h * L * gsize
    twice = 2 if case["train"] else 1
    if case["entry"] == "bias":
        return {"bytes": twice * (keys + gates + b * h * L * L * size), "flops": (3 if case["train"] else 1) * d * L * L * b * h}
    width = min(L, 2 * 1700 * (d / 128) ** 0.5) if case["prune"] else L
    return {"bytes": twice * (2 * keys + 2 * queries + gates),
            "flops": (3 + 6 * r if case["train"] else 1 + 2 * r) * d * L * width * b * h}


def tolerance(case):
    """bf16: the rounding of the inputs to the matrix products.  float32: sums of up to L terms, and in training the key
    gradient, whose factor (k_s . k_u)^(-1/3) amplifies the rounding of small products."""
    if case["dtype"] == "bf16":
        return {"rel": 1e-2, "max": 0.5}
    return {"rel": 5e-4, "max": 0.2} if case["train"] else {"rel": 2e-5, "max": 2e-3}

"""Performance cases of the fused dependent-reduction kernels.

Each case is one call that a program using this framework makes on the GPU: a row fold, the
log-softmax readout, RMSNorm / L2-normalize, CSR segment pooling, or attention.  `listed()` names
twelve of them, from a latency-bound 4 KB reduction to a 1 GB vocabulary reduction and a
550 GFLOP attention; `draw()` makes more cases of the same ranges.  Random logits, activations
and embeddings stand in for a model's.
"""
from __future__ import annotations

import math
import pathlib
import sys

import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parent.parent / "neptune-opt_amd"))

import neptune_codegen as CG  # noqa: E402

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
SIZE = {"fp32": 4, "bf16": 2, "fp16": 2}
EPS = 1e-6
# a drawn case stays below these (the largest listed cases are just above them)
MOST_BYTES = 1.0e9
MOST_FLOPS = 5.4e11


def listed() -> list[dict]:
    return [
        # a classifier head's reduction in an eager loop: launch latency is everything
        {"name": "fold_small", "kind": "fold", "fold": "logsumexp", "dtype": "fp32",
         "rows": 8, "ncols": 128, "pad": 0, "plan": "serial"},
        # the normaliser of a language model's logits over a training batch (1.05 GB)
        {"name": "fold_vocab", "kind": "fold", "fold": "logsumexp", "dtype": "bf16",
         "rows": 16384, "ncols": 32000, "pad": 0, "plan": "serial"},
        # the same over a class count that is no multiple of a vector load
        {"name": "fold_odd", "kind": "fold", "fold": "logsumexp", "dtype": "fp16",
         "rows": 8192, "ncols": 10007, "pad": 0, "plan": "serial"},
        # a few very long rows through the explicitly requested split plan
        {"name": "fold_split", "kind": "fold", "fold": "logsumexp", "dtype": "bf16",
         "rows": 64, "ncols": 262144, "pad": 0, "plan": "split"},
        # log-probabilities over a vocabulary with a few added tokens (odd width)
        {"name": "log_softmax_odd", "kind": "log_softmax", "dtype": "bf16",
         "rows": 4096, "ncols": 32003, "pad": 0},
        # RMSNorm of a batch of tokens, called as the registered operator a fused graph calls
        {"name": "rms_norm_op", "kind": "rms_norm", "dtype": "bf16",
         "rows": 8192, "ncols": 1024, "pad": 0},
        # embedding normalisation before a similarity search, odd feature width
        {"name": "l2_normalize_odd", "kind": "l2_normalize", "dtype": "fp32",
         "rows": 20000, "ncols": 2999, "pad": 0},
        # pooling of token embeddings into 65536 variable-length sequences given by lengths
        {"name": "segment_mean_lengths", "kind": "segment", "reduce": "mean", "dtype": "fp16",
         "segments": 65536, "tokens": 1310720, "channels": 128, "offsets": False},
        # the same by CSR offsets over a channel count that is no power of two
        {"name": "segment_sum_odd", "kind": "segment", "reduce": "sum", "dtype": "bf16",
         "segments": 3000, "tokens": 120000, "channels": 300, "offsets": True},
        # causal self-attention of a long prompt (prefill), projection layout [B, S, H, D]
        {"name": "attention_prefill", "kind": "attention", "dtype": "bf16", "batch": 4,
         "heads": 32, "sq": 4096, "sk": 4096, "dim": 128, "causal": True, "lse": False,
         "layout": "bshd"},
        # one generated token per sequence against the key / value cache (decode)
        {"name": "attention_decode", "kind": "attention", "dtype": "bf16", "batch": 16,
         "heads": 32, "sq": 1, "sk": 3000, "dim": 128, "causal": False, "lse": False,
         "layout": "bhsd"},
        # an encoder layer over ragged inputs, with the logsumexp for a later merge
        {"name": "attention_encoder", "kind": "attention", "dtype": "fp16", "batch": 8,
         "heads": 12, "sq": 777, "sk": 777, "dim": 64, "causal": False, "lse": True,
         "layout": "bshd"},
    ]


# ---------------------------------------------------------------- drawn cases
def _log_int(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo: int, hi: int) -> int:
    """Half the widths are the multiples of 64 that models use, half are any number."""
    w = _log_int(rng, lo, hi)
    return max(64, w // 64 * 64) if rng.random() < 0.5 and hi >= 64 else w


def _rows(rng, lo: int, hi: int, bytes_per_row: float) -> int:
    return _log_int(rng, lo, max(lo, min(hi, MOST_BYTES / bytes_per_row)))


def draw(rng) -> dict:
    kind = rng.choice(["fold", "fold", "fold", "log_softmax", "rms_norm", "l2_normalize",
                       "segment", "segment", "attention", "attention", "attention"])
    dtype = rng.choice(["bf16", "fp16", "fp32"])
    if kind == "fold":
        # widths from a head dimension to a long sequence, 1 row to a whole batch of tokens
        ncols = _width(rng, 33, 262144)
        plan = "split" if ncols >= 16384 and rng.random() < 0.3 else "serial"
        fold = rng.choice(["logsumexp", "logsumexp", "softcap_lse", "lse_scaled", "stable_l2",
                           "rmsnorm_max"] + ([] if plan == "split" else ["variance", "std"]))
        pad = rng.choice([0, 0, 0, 8, 13])
        rows = _rows(rng, 1, 256 if plan == "split" else 32768, ncols * SIZE[dtype])
        return {"kind": kind, "fold": fold, "dtype": dtype, "rows": rows, "ncols": ncols,
                "pad": pad, "plan": plan}
    if kind in ("log_softmax", "rms_norm", "l2_normalize"):
        ncols = _width(rng, 33, 131072 if kind == "log_softmax" else 16384)
        rows = _rows(rng, 1, 32768, 2 * ncols * SIZE[dtype])
        return {"kind": kind, "dtype": dtype, "rows": rows, "ncols": ncols,
                "pad": rng.choice([0, 0, 0, 8, 13])}
    if kind == "segment":
        channels = rng.choice([64, 128, 256, 512, 768, _log_int(rng, 16, 1024)])
        mean = _log_int(rng, 2, 400)
        row = channels * SIZE[dtype]
        segments = _log_int(rng, 16, max(16, min(65536, 0.35 * MOST_BYTES / (row * (mean + 1)))))
        return {"kind": kind, "reduce": rng.choice(["sum", "mean"]), "dtype": dtype,
                "segments": segments, "tokens": segments * mean, "channels": channels,
                "offsets": rng.random() < 0.5}
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    dim = rng.choice([64, 128, 128, 256])
    batch, heads = _log_int(rng, 1, 32), rng.choice([1, 4, 8, 12, 16, 32, 40])
    mode = rng.choice(["prefill", "decode", "encoder"])
    if mode == "decode":
        # one token, or the query heads that share one key head folded into the query axis
        sq, sk = rng.choice([1, 1, 2, 4, 8, 16]), _log_int(rng, 64, 32768)
        while 4.0 * batch * heads * sk * dim > MOST_BYTES:
            sk = (sk + 1) // 2
    else:
        sq = _width(rng, 33, 8192)
        sk = sq if rng.random() < 0.7 else _width(rng, 33, 8192)
        half = 0.5 if mode == "prefill" else 1.0
        while 4.0 * batch * heads * sq * sk * dim * half > MOST_FLOPS / 2:
            sq, sk = (sq + 1) // 2, (sk + 1) // 2
    return {"kind": "attention", "dtype": dtype, "batch": batch, "heads": heads, "sq": sq,
            "sk": sk, "dim": dim, "causal": mode == "prefill", "lse": rng.random() < 0.3,
            "layout": rng.choice(["bhsd", "bshd"])}


# ---------------------------------------------------------------- inputs
def _randn(gen, shape, dtype, scale=1.0):
    """scale * N(0, 1) rounded to dtype, made in pieces so that no large fp32 copy exists."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    step = 1 << 27
    for at in range(0, flat.numel(), step):
        n = min(step, flat.numel() - at)
        piece = torch.randn(n, generator=gen, device="cuda")
        flat[at:at + n] = piece.mul_(scale)
    return out


def _rows_of(case, gen, scale):
    """[rows, ncols]; with `pad`, the leading columns of a wider tensor (a slice of a fused
    projection's output)."""
    wide = _randn(gen, (case["rows"], case["ncols"] + case["pad"]), DTYPES[case["dtype"]], scale)
    return wide[:, :case["ncols"]]


def _params(case) -> dict:
    return {"softcap_lse": {"beta": 0.5}, "lse_scaled": {"T": 2.0},
            "rmsnorm_max": {"eps": EPS}}.get(case["fold"], {})


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    dtype = DTYPES[case["dtype"]]
    if kind == "fold":
        return {"case": case, "x": _rows_of(case, gen, 3.0), "params": _params(case)}
    if kind == "log_softmax":
        return {"case": case, "x": _rows_of(case, gen, 4.0)}
    if kind == "rms_norm":
        gamma = _randn(gen, (case["ncols"],), torch.float32, 0.1).add_(1.0).to(dtype)
        return {"case": case, "x": _rows_of(case, gen, 1.0), "gamma": gamma,
                "op": CG.as_state_op("rms_norm", {"eps": EPS})}
    if kind == "l2_normalize":
        return {"case": case, "x": _rows_of(case, gen, 1.0)}
    if kind == "segment":
        data = _randn(gen, (case["tokens"], case["channels"]), dtype)
        # every token falls into a uniformly chosen segment: Poisson-like lengths, some empty
        owner = torch.randint(case["segments"], (case["tokens"],), generator=gen, device="cuda")
        lengths = torch.bincount(owner, minlength=case["segments"])
        if case["offsets"]:
            zero = lengths.new_zeros(1)
            segments = torch.cat((zero, torch.cumsum(lengths, 0))).to(torch.int32)
        else:
            segments = lengths
        return {"case": case, "data": data, "segments": segments, "lengths": lengths}
    b, h, d = case["batch"], case["heads"], case["dim"]

    def operand(s):
        if case["layout"] == "bshd":
            return _randn(gen, (b, s, h, d), dtype).transpose(1, 2)
        return _randn(gen, (b, h, s, d), dtype)

    return {"case": case, "q": operand(case["sq"]), "k": operand(case["sk"]),
            "v": operand(case["sk"])}


# ---------------------------------------------------------------- one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fold":
        return CG.run(case["fold"], state["x"], plan=case["plan"], **state["params"])
    if kind == "log_softmax":
        return CG.run_log_softmax(state["x"])
    if kind == "rms_norm":
        return state["op"](state["x"], state["gamma"])
    if kind == "l2_normalize":
        return CG.run_l2_normalize(state["x"], eps=EPS)
    if kind == "segment":
        return CG.run_segment_pool(state["data"], state["segments"], reduce=case["reduce"],
                                   offsets=case["offsets"])
    return CG.run_attention(state["q"], state["k"], state["v"], causal=case["causal"],
                            return_lse=case["lse"])


# ---------------------------------------------------------------- what a pass cannot do without
def work(case) -> dict:
    kind = case["kind"]
    size = SIZE[case["dtype"]]
    if kind == "attention":
        b, h, sq, sk, d = (case[n] for n in ("batch", "heads", "sq", "sk", "dim"))
        # causal: query i sees the keys j <= i
        seen = sum(min(i + 1, sk) for i in range(sq)) if case["causal"] else sq * sk
        keys = min(sq, sk) if case["causal"] else sk
        out = b * h * sq * (d * size + (4 if case["lse"] else 0))
        return {"bytes": b * h * d * size * (sq + 2 * keys) + out, "flops": 4 * b * h * seen * d}
    if kind == "segment":
        index = (4 if case["offsets"] else 8) * (case["segments"] + 1)
        rows = case["tokens"] + case["segments"]
        return {"bytes": rows * case["channels"] * size + index,
                "flops": case["tokens"] * case["channels"]}
    n = case["rows"] * case["ncols"]
    if kind == "fold":
        return {"bytes": n * size + case["rows"] * size, "flops": 4 * n}
    gamma = case["ncols"] * size if kind == "rms_norm" else 0
    return {"bytes": 2 * n * size + gamma, "flops": 4 * n}


# 2-norm errors against 64 bits, measured at the listed sizes and over draws: 1.2e-3 to 2.3e-3 in
# bf16 and 1.6e-4 to 2.9e-4 in fp16 (the output's rounding; RMSNorm rounds twice), 5e-8 in fp32,
# where sums in another order move by up to a few 1e-7.  The limits are about four times that;
# one element may be off by about two units in the last place.
_TOLERANCE = {"bf16": {"rel": 7e-3, "max": 2e-2}, "fp16": {"rel": 1e-3, "max": 4e-3},
              "fp32": {"rel": 2e-6, "max": 2e-5}}


def tolerance(case):
    if case["kind"] == "segment":
        return "exact"   # ordered rounding to the storage type: one defined result
    return _TOLERANCE[case["dtype"]]


# ---------------------------------------------------------------- the same in 64 bits
def _exact_fold(name, x, params):
    if name == "logsumexp":
        return torch.logsumexp(x, -1)
    if name == "softcap_lse":
        return torch.logsumexp(torch.tanh(params["beta"] * x), -1)
    if name == "lse_scaled":
        return torch.logsumexp(x / params["T"], -1)
    if name == "stable_l2":
        return torch.linalg.vector_norm(x, dim=-1)
    if name == "rmsnorm_max":
        return x.amax(-1) * torch.rsqrt(x.square().mean(-1) + params["eps"])
    var = x.var(-1, unbiased=False)
    return var if name == "variance" else var.sqrt()


def _by_rows(x, fn):
    """fn over blocks of rows in float64 (bounded memory)."""
    step = max(1, (1 << 26) // x.shape[1])
    return torch.cat([fn(x[i:i + step].double()) for i in range(0, x.shape[0], step)])


def exact(case, seed):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "fold":
        return _by_rows(state["x"], lambda x: _exact_fold(case["fold"], x, state["params"]))
    if kind == "log_softmax":
        return _by_rows(state["x"], lambda x: torch.log_softmax(x, -1))
    if kind == "rms_norm":
        g = state["gamma"].double()
        return _by_rows(state["x"], lambda x: x * torch.rsqrt(x.square().mean(-1, True) + EPS) * g)
    if kind == "l2_normalize":
        return _by_rows(state["x"], lambda x: torch.nn.functional.normalize(x, dim=-1, eps=EPS))
    if kind == "segment":
        lengths = state["lengths"]
        owner = torch.repeat_interleave(torch.arange(case["segments"], device="cuda"), lengths)
        total = torch.zeros(case["segments"], case["channels"], dtype=torch.float64, device="cuda")
        total.index_add_(0, owner, state["data"].double())
        return total if case["reduce"] == "sum" else total / lengths.double().unsqueeze(1)
    q, k, v = state["q"], state["k"], state["v"]
    b, h, sq, sk = (case[n] for n in ("batch", "heads", "sq", "sk"))
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    lse = torch.empty(q.shape[:3], dtype=torch.float64, device="cuda")
    hidden = None
    if case["causal"]:
        hidden = torch.ones(sq, sk, dtype=torch.bool, device="cuda").triu_(1)
    for i in range(b):
        for j in range(h):
            s = (q[i, j].double() / math.sqrt(case["dim"])) @ k[i, j].double().t().contiguous()
            if hidden is not None:
                s.masked_fill_(hidden, -math.inf)
            lse[i, j] = torch.logsumexp(s, -1)
            out[i, j] = torch.softmax(s, -1) @ v[i, j].double()
    return (out, lse) if case["lse"] else out

"""What the performance of this package is measured on: calls that a user's program makes, through
`intent.jit` and the example programs, over the sizes that they meet in use.

Three ways of calling are here, as programs use them: `kernel.run(...)`, which binds and allocates
on every call (one-off calls and training code with fresh tensors); a prepared call that is launched again
and again on the same buffers (a layer, a decode step or an iterative solver); and the multi-kernel
programs `PagedDecode` and `AttentionBackward`.
"""
import functools
import math
import random

import numpy as np
import torch

import intent_amd as intent
from intent_amd.examples.kernels.backward.softmax import softmax_backward_f16
from intent_amd.examples.kernels.contraction.gemm import Activation, bf16_gemm, gemm, linear_f32
from intent_amd.examples.kernels.normalization.softmax import (chunked_softmax_bf16, stable_softmax,
                                                               stable_softmax_f16)
from intent_amd.examples.kernels.sparse.csr_spmv import csr_spmv
from intent_amd.examples.kernels.streaming.attention import (flash_attention_bf16_fwd, flash_attention_fwd,
                                                             flash_gqa_attention_fwd, flash_varlen_gqa_prefill)
from intent_amd.examples.programs.attention_backward import AttentionBackward
from intent_amd.examples.programs.composition import PagedDecode

DEVICE = "cuda"


def listed():
    return [
        # The smallest call: one attention or router softmax of a small batch, called once with fresh
        # tensors, so binding, allocation and the launch are most of it. 1000 columns, the tests' ragged width.
        {"name": "softmax_f32_small", "op": "softmax_f32", "rows": 64, "cols": 1000},
        # The benchmark's training step: forward, then backward on its output, f16 storage.
        {"name": "softmax_f16_step", "op": "softmax_step", "rows": 16384, "cols": 4096},
        # Probabilities over a vocabulary: rows much longer than one wavefront holds.
        {"name": "softmax_bf16_vocabulary", "op": "softmax_bf16", "rows": 2048, "cols": 32000},
        # The benchmark's large square product.
        {"name": "gemm_bf16_8192", "op": "gemm_bf16", "m": 8192, "n": 8192, "k": 8192},
        # A feed-forward layer (the example module's 4096 x 14336 weight, ReLU) in a decode step: few rows,
        # so the weight's bytes are the work.
        {"name": "gemm_f16_relu_32_rows", "op": "gemm_f16_relu", "m": 32, "n": 14336, "k": 4096},
        # A projection over a ragged number of tokens, at a model width of 768 (three of them stacked).
        {"name": "gemm_bf16_ragged", "op": "gemm_bf16", "m": 1021, "n": 2304, "k": 768},
        # A full-precision head: 1000 outputs of a 2048-wide layer, a batch of 256.
        {"name": "linear_f32_head", "op": "linear_f32", "m": 256, "n": 1000, "k": 2048},
        # The benchmark's causal attention, the largest prefill.
        {"name": "attention_f16_causal", "op": "attention", "dtype": "f16", "batch": 4, "heads": 32, "kv_heads": 32,
         "seq": 4096, "dim": 128, "causal": True},
        # A server's prefill: packed prompts of different lengths, grouped heads.
        {"name": "attention_packed_prompts", "op": "attention_packed", "sequences": 8, "longest": 2048, "heads": 32,
         "kv_heads": 8, "dim": 128},
        # The backward of a grouped-query training layer: three kernels, three gradients.
        {"name": "attention_backward", "op": "attention_backward", "batch": 2, "heads": 32, "kv_heads": 8, "seq": 2048,
         "dim": 128, "causal": True},
        # One decode step over a paged cache at the example module's sizes (about 7300 tokens a sequence).
        {"name": "decode_paged", "op": "decode_paged", "batch": 8, "heads": 32, "kv_heads": 8, "dim": 128,
         "longest": 8191, "page": 64, "splits": 16},
        # The benchmark's sparse matrix: row lengths of a Zipf law from 1 to 65536.
        {"name": "spmv_zipf", "op": "spmv", "rows": 4194304, "cap": 65536, "c": 3.920855e8},
    ]


# ------------------------------------------------------------------------------------------ drawing
def _spread(rng, low, high, multiple=1):
    """A size between low and high, even over its logarithm, a multiple of `multiple`."""
    value = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(high // multiple, max(-(-low // multiple), round(value / multiple))) * multiple


def _within(limit, size, *others):
    """`size` cut down so that its product with `others` stays below `limit`."""
    return max(1, min(size, limit // max(1, math.prod(others))))


def draw(rng):
    """One more case. Sizes take odd values as often as the path meets them: token counts, batches,
    vocabularies and sequence lengths are arbitrary; model widths are mostly multiples of 8."""
    op = rng.choice(["softmax_f32", "softmax_step", "softmax_bf16", "gemm_bf16", "gemm_bf16_small", "gemm_f16_relu",
                     "linear_f32", "attention", "attention_packed", "attention_backward", "decode_paged", "spmv"])
    width = rng.choice([1, 8, 8, 64])
    if op == "softmax_f32":
        return {"op": op, "rows": _spread(rng, 1, 4096), "cols": _spread(rng, 16, 4096)}
    if op == "softmax_step":
        cols = _spread(rng, 128, 8192, width)
        return {"op": op, "rows": _within(1 << 26, _spread(rng, 64, 16384), cols), "cols": cols}
    if op == "softmax_bf16":
        cols = _spread(rng, 8200, 131072, width)
        return {"op": op, "rows": _within(1 << 26, _spread(rng, 16, 4096), cols), "cols": cols}
    if op == "gemm_bf16":            # large products: training and prefill projections
        m, n, k = _spread(rng, 512, 8192), _spread(rng, 1024, 8192, 64), _spread(rng, 512, 8192, 64)
        return {"op": op, "m": m, "n": n, "k": k}
    if op == "gemm_bf16_small":      # small and ragged ones
        m, n, k = _spread(rng, 16, 2048), _spread(rng, 64, 3072, width), _spread(rng, 64, 3072, width)
        return {"op": "gemm_bf16", "m": _within(1 << 32, m, n, k), "n": n, "k": k}
    if op == "gemm_f16_relu":
        return {"op": op, "m": _spread(rng, 1, 128), "n": _spread(rng, 512, 16384, 8), "k": _spread(rng, 512, 8192, 8)}
    if op == "linear_f32":
        return {"op": op, "m": _spread(rng, 1, 2048), "n": _spread(rng, 16, 4096, rng.choice([1, 4, 8])),
                "k": _spread(rng, 64, 4096, width)}
    dim = rng.choice([64, 128])
    kv_heads, group = rng.choice([(1, 8), (2, 4), (4, 4), (8, 4), (4, 8), (8, 1), (16, 2), (32, 1)])
    heads = kv_heads * group
    if op == "attention":
        seq = _spread(rng, 64, 4096)
        if rng.random() < 0.2:
            dim = rng.choice([80, 96])
        return {"op": op, "dtype": rng.choice(["f16", "bf16"]), "batch": rng.choice([1, 1, 2, 4]), "heads": heads,
                "kv_heads": kv_heads, "seq": seq, "dim": dim, "causal": rng.random() < 0.75}
    if op == "attention_packed":
        return {"op": op, "sequences": _spread(rng, 1, 32), "longest": _spread(rng, 32, 2048), "heads": heads,
                "kv_heads": kv_heads, "dim": dim}
    if op == "attention_backward":
        return {"op": op, "batch": rng.choice([1, 2]), "heads": heads, "kv_heads": kv_heads,
                "seq": _spread(rng, 64, 2048), "dim": dim, "causal": rng.random() < 0.75}
    if op == "decode_paged":
        kv_heads, group = rng.choice([(8, 4), (2, 4), (8, 1), (4, 8), (8, 8), (16, 2), (2, 16)])
        return {"op": op, "batch": _spread(rng, 1, 16), "heads": kv_heads * group, "kv_heads": kv_heads, "dim": dim,
                "longest": _spread(rng, 16, 8192), "page": rng.choice([16, 32, 64]), "splits": rng.choice([1, 4, 8, 16])}
    rows = _spread(rng, 1000, 4194304)
    cap = min(rows, _spread(rng, 64, 65536))
    heaviest = max(1.0, rng.uniform(1, 5) * rows / cap)     # rows at the cap; the mean length is about 3 times the factor
    return {"op": "spmv", "rows": rows, "cap": cap, "c": float(round(cap * heaviest ** 1.5))}


# ------------------------------------------------------------------------------------------ inputs
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _normal(g, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device=DEVICE) * scale).to(DTYPES[dtype])


def _uniform(g, shape, dtype):
    return (torch.rand(shape, generator=g, device=DEVICE) * 2 - 1).to(DTYPES[dtype])


def _scale(dim):
    return float(np.float32(dim ** -0.5))


@functools.lru_cache(maxsize=None)
def _lengths(count, longest):
    """`count` sequence lengths from 1 to `longest`, the longest among them: part of the case, not of its inputs."""
    rng = random.Random(count * 8191 + longest)
    return tuple([longest] + [rng.randint(1, longest) for _ in range(count - 1)])


def _cache_lengths(case):
    """Decode: sequences of similar age, from three quarters of the longest up."""
    longest, count = case["longest"], case["batch"]
    return [longest - (longest // 4) * i // max(1, count) for i in range(count)]


@functools.lru_cache(maxsize=4)
def _row_lengths(rows, cap, c):
    ranks = np.arange(1, rows + 1, dtype=np.float64)
    return np.minimum(cap, np.maximum(1, np.floor(c * ranks ** -1.5))).astype(np.int64)


def _softmax_inputs(case, seed):
    g = _generator(seed)
    shape = (case["rows"], case["cols"])
    if case["op"] == "softmax_f32":
        return (_normal(g, shape, "f32", 4),)
    if case["op"] == "softmax_bf16":
        return (_normal(g, shape, "bf16", 3),)
    return _normal(g, shape, "f16", 3), _normal(g, shape, "f16")


def _gemm_inputs(case, seed):
    g = _generator(seed)
    m, n, k = case["m"], case["n"], case["k"]
    if case["op"] == "gemm_bf16":
        return _uniform(g, (m, k), "bf16"), _uniform(g, (k, n), "bf16")
    if case["op"] == "gemm_f16_relu":
        return _normal(g, (m, k), "f16"), _normal(g, (k, n), "f16", k ** -0.5)
    return _normal(g, (m, k), "f32"), _normal(g, (n, k), "f32", k ** -0.5)


def _attention_inputs(case, seed):
    g = _generator(seed)
    b, hq, hk, s, d = case["batch"], case["heads"], case["kv_heads"], case["seq"], case["dim"]
    dtype = case.get("dtype", "f16")
    return _normal(g, (b, hq, s, d), dtype), _normal(g, (b, hk, s, d), dtype), _normal(g, (b, hk, s, d), dtype)


def _packed_inputs(case, seed):
    g = _generator(seed)
    lengths = _lengths(case["sequences"], case["longest"])
    total, d = sum(lengths), case["dim"]
    offsets = np.concatenate([[0], np.cumsum(lengths)])
    return (_normal(g, (total, case["heads"], d), "f16"), _normal(g, (total, case["kv_heads"], d), "f16"),
            _normal(g, (total, case["kv_heads"], d), "f16"),
            torch.tensor(lengths, dtype=torch.int32, device=DEVICE),
            torch.tensor(offsets, dtype=torch.int32, device=DEVICE))


def _causal_mask(s):
    return torch.ones((s, s), dtype=torch.bool, device=DEVICE).triu(1)


def _backward_inputs(case, seed):
    """q, k, v, the forward's output and log-sum (as the forward pass left them), and the gradient."""
    q, k, v = _attention_inputs(case, seed)
    grad = _normal(_generator(seed + 1000003), q.shape, "f16")
    out = torch.empty_like(q)
    lse = torch.empty(q.shape[:3], dtype=torch.float32, device=DEVICE)
    group, scale = case["heads"] // case["kv_heads"], _scale(case["dim"])
    mask = _causal_mask(case["seq"]) if case["causal"] else None
    for b in range(case["batch"]):
        for h in range(case["heads"]):
            scores = (q[b, h].float() @ k[b, h // group].float().t().contiguous()) * scale
            if mask is not None:
                scores.masked_fill_(mask, -math.inf)
            lse[b, h] = torch.logsumexp(scores, dim=1)
            out[b, h] = (torch.exp(scores - lse[b, h][:, None]) @ v[b, h // group].float()).half()
    return q, k, v, out, grad, lse


def _decode_inputs(case, seed):
    g = _generator(seed)
    batch, hk, d, page, splits = case["batch"], case["kv_heads"], case["dim"], case["page"], case["splits"]
    lengths = _cache_lengths(case)
    counts = [-(-n // page) for n in lengths]
    page_offsets = np.concatenate([[0], np.cumsum(counts)])
    pages = int(page_offsets[-1])
    split_offsets = [0] + [int(page_offsets[b]) + (j * counts[b]) // splits
                           for b in range(batch) for j in range(1, splits + 1)]

    def table(values):
        return torch.tensor(np.asarray(values), dtype=torch.int32, device=DEVICE)

    return (_normal(g, (batch, case["heads"], d), "f16"), _normal(g, (pages, page, hk, d), "f16"),
            _normal(g, (pages, page, hk, d), "f16"), table(page_offsets),
            torch.randperm(pages, generator=g, device=DEVICE).to(torch.int32), table(lengths), table(split_offsets))


def _spmv_inputs(case, seed):
    """Rows in random order; each row's columns are distinct, sorted and spread over the whole width (one
    in each of as many equal strata as the row has entries)."""
    g = _generator(seed)
    rows = case["rows"]
    lengths = torch.from_numpy(_row_lengths(rows, case["cap"], case["c"])).to(DEVICE)
    lengths = lengths[torch.randperm(rows, generator=g, device=DEVICE)]
    offsets = torch.zeros(rows + 1, dtype=torch.int64, device=DEVICE)
    torch.cumsum(lengths, 0, out=offsets[1:])
    nnz = int(offsets[-1])
    row = torch.repeat_interleave(torch.arange(rows, device=DEVICE), lengths, output_size=nnz)
    length = lengths[row]
    place = torch.arange(nnz, device=DEVICE) - offsets[row]
    low = place * rows // length
    span = (place + 1) * rows // length - low
    columns = low + (torch.rand(nnz, generator=g, device=DEVICE, dtype=torch.float64) * span).to(torch.int64)
    return (offsets.to(torch.int32), columns.to(torch.int32), _uniform(g, nnz, "f32"), _uniform(g, rows, "f32"))


INPUTS = {"softmax_f32": _softmax_inputs, "softmax_step": _softmax_inputs, "softmax_bf16": _softmax_inputs,
          "gemm_bf16": _gemm_inputs, "gemm_f16_relu": _gemm_inputs, "linear_f32": _gemm_inputs,
          "attention": _attention_inputs, "attention_packed": _packed_inputs, "attention_backward": _backward_inputs,
          "decode_paged": _decode_inputs, "spmv": _spmv_inputs}


# ------------------------------------------------------------------------------------------ calls
_hip = functools.partial(intent.jit, backend="hip")


@functools.lru_cache(maxsize=None)
def _kernel(definition, **constexprs):
    """A program jits a definition once and keeps the kernel."""
    return _hip(definition, constexprs=constexprs) if constexprs else _hip(definition)


@functools.lru_cache(maxsize=None)
def _backward_program(group, causal):
    return AttentionBackward.from_jit(_hip, head_group=group, causal=causal)


@functools.lru_cache(maxsize=None)
def _decode_program(page, group, splits):
    return PagedDecode.from_jit(_hip, page_size=page, head_group=group, splits=splits)


def _launched(*calls):
    """A pass that launches prepared calls in order and returns what they wrote."""
    def once():
        for call in calls:
            call.launch()
        results = tuple(call.result() for call in calls)
        return results[0] if len(results) == 1 else results
    return once


def prepare(case, seed):
    op = case["op"]
    inputs = INPUTS[op](case, seed)
    if op == "softmax_f32":
        return functools.partial(_kernel(stable_softmax).run, *inputs)
    if op == "softmax_bf16":
        return functools.partial(_kernel(chunked_softmax_bf16).run, *inputs)
    if op == "softmax_step":
        forward = _kernel(stable_softmax_f16).prepare(inputs[0])
        return _launched(forward, _kernel(softmax_backward_f16).prepare(forward.result(), inputs[1]))
    if op == "gemm_bf16":
        return _launched(_kernel(bf16_gemm).prepare(*inputs))
    if op == "gemm_f16_relu":
        return _launched(_kernel(gemm, ACTIVATION=Activation.RELU).prepare(*inputs))
    if op == "linear_f32":
        return _launched(_kernel(linear_f32).prepare(*inputs))
    if op == "spmv":
        return _launched(_kernel(csr_spmv).prepare(*inputs))
    group, scale = case["heads"] // case["kv_heads"], _scale(case["dim"])
    if op == "attention":
        if case["dtype"] == "bf16":
            kernel = _kernel(flash_attention_bf16_fwd, HEAD_GROUP=group, CAUSAL=case["causal"])
        elif group > 1:
            kernel = _kernel(flash_gqa_attention_fwd, HEAD_GROUP=group, CAUSAL=case["causal"])
        else:
            kernel = _kernel(flash_attention_fwd, CAUSAL=case["causal"])
        return functools.partial(kernel.run, *inputs, scale)
    if op == "attention_packed":
        return functools.partial(_kernel(flash_varlen_gqa_prefill, HEAD_GROUP=group).run, *inputs, scale)
    if op == "attention_backward":
        return functools.partial(_backward_program(group, case["causal"]).run, *inputs, scale)
    return _launched(_decode_program(case["page"], group, case["splits"]).prepare(*inputs, scale))


def run(state):
    return state()


# ------------------------------------------------------------------------------------------ work
SIZES = {"f32": 4, "f16": 2, "bf16": 2}


def _pairs(s, causal):
    return s * (s + 1) // 2 if causal else s * s


def work(case):
    op = case["op"]
    if op in ("softmax_f32", "softmax_bf16", "softmax_step"):
        elements = case["rows"] * case["cols"]
        if op == "softmax_step":       # x read, y written; y and dy read, dx written
            return {"bytes": elements * 10, "flops": elements * 9}
        return {"bytes": elements * 2 * (4 if op == "softmax_f32" else 2), "flops": elements * 5}
    if op in ("gemm_bf16", "gemm_f16_relu", "linear_f32"):
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m * k + k * n + m * n) * (4 if op == "linear_f32" else 2), "flops": 2 * m * n * k}
    if op == "spmv":
        nnz, rows = int(_row_lengths(case["rows"], case["cap"], case["c"]).sum()), case["rows"]
        return {"bytes": 4 * (rows + 1) + 8 * nnz + 8 * rows, "flops": 2 * nnz}
    hq, hk, d = case["heads"], case["kv_heads"], case["dim"]
    if op == "attention_packed":
        lengths = _lengths(case["sequences"], case["longest"])
        return {"bytes": sum(lengths) * d * 2 * (2 * hq + 2 * hk) + 8 * len(lengths),
                "flops": 4 * hq * d * sum(_pairs(n, True) for n in lengths)}
    if op == "decode_paged":
        tokens = sum(_cache_lengths(case))
        return {"bytes": tokens * hk * d * 4 + case["batch"] * hq * d * 4 + 4 * (tokens // case["page"]),
                "flops": 4 * tokens * hq * d}
    b, s = case["batch"], case["seq"]
    if op == "attention":
        return {"bytes": b * s * d * 2 * (2 * hq + 2 * hk), "flops": 4 * b * hq * d * _pairs(s, case["causal"])}
    # Backward: q, out, grad and k, v read; three gradients written; scores once and four products from them.
    return {"bytes": b * s * d * 2 * (4 * hq + 4 * hk) + 4 * b * hq * s,
            "flops": 10 * b * hq * d * _pairs(s, case["causal"])}


# ------------------------------------------------------------------------------------------ tolerance
# About four times the largest distance from `exact` seen over the listed cases and 60 drawn ones
# (2-norms): 2.5e-7, 3.2e-4, 1.7e-3, 1.7e-3, 2.2e-4, 1.0e-6, 2.5e-4 (f16) and 2.1e-3 (bf16), 2.5e-4, 3.0e-4,
# 2.6e-4, 1.7e-7. The 16-bit figures are the rounding of the results themselves.
TOLERANCES = {"softmax_f32": 1e-6, "softmax_step": 1.2e-3, "softmax_bf16": 7e-3, "gemm_bf16": 7e-3,
              "gemm_f16_relu": 1e-3, "linear_f32": 4e-6, "attention": 1e-3, "attention_packed": 1e-3,
              "attention_backward": 1.2e-3, "decode_paged": 1e-3, "spmv": 7e-7}


def tolerance(case):
    return {"rel": 8e-3 if case.get("dtype") == "bf16" else TOLERANCES[case["op"]]}


# ------------------------------------------------------------------------------------------ exact results
def _attend(q, k, v, scale, mask):
    """One head in 64 bits: q [S, D], k and v [T, D]."""
    scores = (q.double() @ k.double().t().contiguous()) * scale
    if mask is not None:
        scores.masked_fill_(mask, -math.inf)
    return torch.softmax(scores, dim=1) @ v.double()


def _exact_attention(case, inputs, scale):
    q, k, v = inputs
    group = case["heads"] // case["kv_heads"]
    mask = _causal_mask(case["seq"]) if case["causal"] else None
    out = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    for b in range(case["batch"]):
        for h in range(case["heads"]):
            out[b, h] = _attend(q[b, h], k[b, h // group], v[b, h // group], scale, mask)
    return out


def _exact_packed(case, inputs, scale):
    q, k, v = inputs[:3]
    group = case["heads"] // case["kv_heads"]
    out = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    start = 0
    for length in _lengths(case["sequences"], case["longest"]):
        mask, rows = _causal_mask(length), slice(start, start + length)
        for h in range(case["heads"]):
            out[rows, h] = _attend(q[rows, h], k[rows, h // group], v[rows, h // group], scale, mask)
        start += length
    return out


def _exact_backward(case, inputs, scale):
    q, k, v, out, grad, lse = inputs
    group = case["heads"] // case["kv_heads"]
    mask = _causal_mask(case["seq"]) if case["causal"] else None
    dq = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    dk, dv = (torch.zeros(k.shape, dtype=torch.float64, device=DEVICE) for _ in range(2))
    for b in range(case["batch"]):
        for h in range(case["heads"]):
            qh, kh, vh = q[b, h].double(), k[b, h // group].double(), v[b, h // group].double()
            gh = grad[b, h].double()
            p = torch.exp((qh @ kh.t().contiguous()) * scale - lse[b, h].double()[:, None])
            if mask is not None:
                p.masked_fill_(mask, 0.0)
            ds = p * ((gh @ vh.t().contiguous()) - (out[b, h].double() * gh).sum(1, keepdim=True))
            dq[b, h] = (ds @ kh) * scale
            dk[b, h // group] += (ds.t().contiguous() @ qh) * scale
            dv[b, h // group] += p.t().contiguous() @ gh
    return dq, dk, dv


def _exact_decode(case, inputs, scale):
    """Each split's rows and base-2 log-sum, then the merge's natural exponentials of those, as the two
    definitions state them."""
    q, keys, values, page_offsets, page_indices, lengths, split_offsets = inputs
    hk, d, page, splits = case["kv_heads"], case["dim"], case["page"], case["splits"]
    group = case["heads"] // hk
    starts, cuts, ends = page_offsets.tolist(), split_offsets.tolist(), lengths.tolist()
    out = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    for b in range(case["batch"]):
        rows, sums = [], []
        for j in range(splits):
            first, last = cuts[b * splits + j], cuts[b * splits + j + 1]
            live = min((last - starts[b]) * page, ends[b]) - (first - starts[b]) * page
            if live <= 0:
                continue
            pages = page_indices[first:last].long()
            k = keys[pages].reshape(-1, hk, d)[:live].permute(1, 2, 0).double().contiguous()
            v = values[pages].reshape(-1, hk, d)[:live].permute(1, 0, 2).double().contiguous()
            scores = (q[b].double().reshape(hk, group, d) @ k) * scale
            rows.append((torch.softmax(scores, dim=2) @ v).reshape(case["heads"], d))
            sums.append(torch.logsumexp(scores, dim=2).reshape(case["heads"]) / math.log(2))
        weights = torch.softmax(torch.stack(sums), dim=0)
        out[b] = (weights[:, :, None] * torch.stack(rows)).sum(0)
    return out


def exact(case, seed):
    op = case["op"]
    inputs = INPUTS[op](case, seed)
    if op in ("softmax_f32", "softmax_bf16"):
        return torch.softmax(inputs[0].double(), dim=1)
    if op == "softmax_step":
        y, dy = torch.softmax(inputs[0].double(), dim=1), inputs[1].double()
        return y, y * (dy - (y * dy).sum(1, keepdim=True))
    if op == "gemm_bf16":
        return inputs[0].double() @ inputs[1].double()
    if op == "gemm_f16_relu":
        return torch.relu(inputs[0].double() @ inputs[1].double())
    if op == "linear_f32":
        return inputs[0].double() @ inputs[1].double().t().contiguous()
    if op == "spmv":
        offsets, columns, values, x = inputs
        lengths = (offsets[1:] - offsets[:-1]).long()
        row = torch.repeat_interleave(torch.arange(case["rows"], device=DEVICE), lengths)
        products = values.double() * x.double()[columns.long()]
        return torch.zeros(case["rows"], dtype=torch.float64, device=DEVICE).index_add_(0, row, products)
    scale = _scale(case["dim"])
    return {"attention": _exact_attention, "attention_packed": _exact_packed, "attention_backward": _exact_backward,
            "decode_paged": _exact_decode}[op](case, inputs, scale)

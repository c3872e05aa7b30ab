"""The work whose speed counts: what a user of this package has it do, one pass at a time.

A case is one operator at one shape.  Its kernel is chosen as the package chooses one
without measuring on the user's machine: the stored winner of a tuning run where the table
shipped with the package has one for the shape, else the first of the cost model's ranking
of the solver's configurations that builds.  The kernel is loaded once and kept, the tensors
are the caller's, and a pass is one call of the loaded kernel.
"""

from __future__ import annotations

import functools
import math

import torch

from deca_amd import operators as ops
from deca_amd import tuned
from deca_amd.kernels import attn_bench, gemm_bench, rowwise_bench
from deca_amd.Tuner import Tuner
from deca_amd.utils.helper import GPUDetector

# The GEMM and attention solvers take multiples of 64 here and want 256 workgroups of
# their smallest tile (64 x 64 of C; 32 query rows of one head).
STEP = 64
MIN_WORKGROUPS = 256
# no drawn case is larger than the largest listed one
MAX_FLOPS = 2 * 8192**3
MAX_ROW_ELEMS = 1 << 28


def _row(name, op, M, N, dtype):
    return {"name": name, "op": op, "M": M, "N": N, "dtype": dtype}


def _gemm(name, M, N, K, dtype):
    return {"name": name, "op": "GEMM", "M": M, "N": N, "K": K, "dtype": dtype}


def _attn(name, B, H, S_q, S_kv, D, causal):
    return {"name": name, "op": "flash_attn", "B": B, "H": H, "S_q": S_q, "S_kv": S_kv, "D": D,
            "causal": causal, "dtype": "float16"}


def listed():
    return [
        # the smallest useful call: a softmax over a few hundred short rows; launch bound
        _row("softmax_small", "softmax", 256, 1024, "float16"),
        # the norm of a training or prefill step over 16k tokens at hidden size 4096
        _row("rmsnorm_prefill", "rmsnorm", 16384, 4096, "bfloat16"),
        # probabilities over a 128k vocabulary for a batch of a thousand positions
        _row("softmax_vocab", "softmax", 1024, 128256, "bfloat16"),
        # an odd number of tokens, and a hidden size that only takes 8-byte accesses
        _row("rmsnorm_ragged", "rmsnorm", 3001, 5124, "float16"),
        # one small square product, as in a small model's layers
        _gemm("gemm_small", 1024, 1024, 1024, "float16"),
        # a projection layer in serving: a batch of 256 tokens against a square weight
        _gemm("gemm_serving", 256, 4096, 4096, "bfloat16"),
        # dimensions that are multiples of 64 and of little else
        _gemm("gemm_ragged", 1344, 2816, 5440, "float16"),
        # a large training product
        _gemm("gemm_large", 8192, 8192, 8192, "bfloat16"),
        # prefill of one short prompt
        _attn("attn_short_prompt", 1, 16, 512, 512, 64, True),
        # prefill / training at the usual sequence length and head size
        _attn("attn_prefill", 4, 16, 4096, 4096, 128, True),
        # a chunk of new tokens against a long context
        _attn("attn_chunk", 1, 16, 512, 8192, 128, False),
        # an encoder over many short sequences
        _attn("attn_encoder", 32, 32, 512, 512, 64, False),
    ]


def _log_int(rng, lo, hi, step=1):
    """An integer of [lo, hi], a multiple of `step`, spread evenly over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(-(-lo // step), min(hi // step, round(v / step))) * step


def draw(rng):
    op = rng.choice(("softmax", "rmsnorm", "GEMM", "GEMM", "flash_attn", "flash_attn"))
    if op in ("softmax", "rmsnorm"):
        N = _log_int(rng, 512, 131072 if op == "softmax" else 16384, 4)
        M = _log_int(rng, 256, min(65536, MAX_ROW_ELEMS // N))
        return {"op": op, "M": M, "N": N, "dtype": rng.choice(("float16", "bfloat16"))}
    while op == "GEMM":
        M, N, K = (_log_int(rng, lo, 8192, STEP) for lo in (128, 512, 256))
        if (M // STEP) * (N // STEP) >= MIN_WORKGROUPS and 2 * M * N * K <= MAX_FLOPS:
            return {"op": op, "M": M, "N": N, "K": K, "dtype": rng.choice(("float16", "bfloat16"))}
    while True:
        D = rng.choice((64, 128))
        B, H = _log_int(rng, 1, 32), rng.choice((8, 16, 32))
        S_kv = _log_int(rng, 256, 16384, STEP)
        causal = rng.random() < 0.5
        S_q = S_kv if causal or rng.random() < 0.5 else _log_int(rng, 128, S_kv, STEP)
        if B * H * (S_q // 32) >= MIN_WORKGROUPS and 4 * B * H * S_q * S_kv * D <= MAX_FLOPS // 2:
            return {"op": op, "B": B, "H": H, "S_q": S_q, "S_kv": S_kv, "D": D, "causal": causal,
                    "dtype": "float16"}


def _shape(case):
    if case["op"] == "GEMM":
        return case["M"], case["N"], case["K"]
    if case["op"] == "flash_attn":
        return tuple(case[k] for k in ("B", "H", "S_q", "S_kv", "D"))
    return case["M"], case["N"]


@functools.lru_cache(maxsize=None)
def _arch():
    return GPUDetector.create_gpu_instance(verbose=False)


def _configs(op, shape, dtype, causal, arch):
    """The configurations of a shape in the order in which they are tried."""
    stored = tuned.lookup(tuned.make_key(op, shape, dtype, arch.gcn_arch, causal))
    if stored is not None:
        return [stored]
    tuner = Tuner(op, arch=arch, top_n=16)
    extra = {"dtype": dtype, "causal": causal}
    return tuner.tune_cpt_1(tuner.tune_cpt_0(*shape, **extra), *shape, **extra)


def _operator(op, shape, dtype, causal):
    if op == "GEMM":
        return ops.GEMMTC(*shape, dtype=dtype)
    if op == "flash_attn":
        return ops.FlashAttention(*shape, dtype=dtype, causal=causal)
    return (ops.Softmax if op == "softmax" else ops.RMSNorm)(*shape, dtype)


@functools.lru_cache(maxsize=64)
def _kernel(op, shape, dtype, causal):
    """(operator, loaded kernel), which a program keeps for as long as it needs the shape."""
    operator = _operator(op, shape, dtype, causal)
    refused = None
    for cfg in _configs(op, shape, dtype, causal, _arch()):
        try:
            return operator, operator.compile(operator.build_mod(cfg))
        except RuntimeError as err:  # the build or the loader refuses it: the next one
            refused = err
    raise refused or RuntimeError(f"no configuration for {operator.describe()}")


def _inputs(case, seed):
    op, shape, dtype = case["op"], _shape(case), case["dtype"]
    if op == "GEMM":
        return gemm_bench.make_inputs(*shape, seed=seed, dtype=getattr(torch, dtype))
    if op == "flash_attn":
        return attn_bench.make_qkv(*shape, seed=seed)
    # logits spread wider than normalised activations
    return rowwise_bench.make_inputs(op, *shape, dtype, seed=seed,
                                     std=2.0 if op == "softmax" else 1.0)


def prepare(case, seed):
    operator, kernel = _kernel(case["op"], _shape(case), case["dtype"],
                               bool(case.get("causal", False)))
    inputs = _inputs(case, seed)
    out = operator.make_output(inputs)
    return {"kernel": kernel, "args": operator.kernel_args(inputs, out), "out": out}


def run(state):
    state["kernel"](*state["args"])
    return state["out"]


def work(case):
    """Inputs read once and the output written once; the products' multiply-adds, of which a
    causal mask leaves half."""
    if case["op"] == "GEMM":
        M, N, K = _shape(case)
        return {"bytes": 2 * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    if case["op"] == "flash_attn":
        B, H, S_q, S_kv, D = _shape(case)
        return {"bytes": 2 * B * H * D * 2 * (S_q + S_kv),
                "flops": attn_bench.attn_flops(B, H, S_q, S_kv, D, case["causal"])}
    M, N = _shape(case)
    # per element: softmax subtracts, exponentiates, sums, scales; the norm squares, sums,
    # scales twice
    return {"bytes": rowwise_bench.rowwise_bytes(case["op"], M, N), "flops": 4 * M * N}


def tolerance(case):
    """About four times the distance of the path from the same operator in 64 bits, measured
    over the listed cases and sixteen drawn ones: rel 2.9e-4, max 5.6e-3 in float16 (the
    output's rounding alone: 2.1e-4); rel 2.3e-3, max 7.7e-3 in bfloat16 (1.7e-3)."""
    if case["dtype"] == "bfloat16":
        return {"rel": 1e-2, "max": 3.2e-2}
    return {"rel": 1.2e-3, "max": 2.4e-2}


def exact(case, seed):
    """The operator in 64 bits, from torch alone."""
    inputs = [t.double() for t in _inputs(case, seed)]
    if case["op"] == "GEMM":
        a, b = inputs
        return a @ b
    if case["op"] == "softmax":
        return torch.softmax(inputs[0], -1)
    if case["op"] == "rmsnorm":
        x, w = inputs
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w
    q, k, v = inputs
    out = torch.empty_like(q)
    hidden = None
    if case["causal"]:
        hidden = torch.ones(q.shape[2], k.shape[2], dtype=torch.bool, device=q.device).triu_(1)
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            s = (q[b, h] @ k[b, h].t()) * (1.0 / math.sqrt(q.shape[3]))
            if hidden is not None:
                s.masked_fill_(hidden, -math.inf)
            out[b, h] = torch.softmax(s, -1) @ v[b, h]
    return out

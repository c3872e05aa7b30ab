"""GPU parity of the row-wise HIP kernels against oracle/rowwise.py.

Inputs are drawn on the CPU from a seeded generator and copied to the device;
every launch goes through the C ABI (deca_launch via LoadedKernel).

Tolerances (written out here, from the task's accuracy gates):
  softmax  max|y - ref| <= 2e-3 (fp16), <= 1e-2 (bf16), ref = fp32 softmax
  rmsnorm  |y - ref| <= tol * max(1, |ref|) with tol = 2e-3 (fp16), 1e-2 (bf16):
           the absolute form of the gate for |ref| <= 1 and its relative form
           above, because the output grid itself is coarser than the absolute
           gate there (bf16 spacing is 3.1e-2 in [4, 8)).
On top of the gates the kernels must agree with the checker, which performs
the same roundings at the same places: softmax to within one unit in the last
place of the output dtype, RMSNorm to within two (its first rounding, of x * r,
can flip on the last bit of the hardware rsqrt and is then multiplied by w and
rounded again), and in both cases on all but a small fraction of elements.
"""

import numpy as np
import pytest
import torch

from oracle import rowwise as orw
from kernel_cases import ROWWISE_CASES, ROWWISE_FULL

pytestmark = pytest.mark.gpu

GATE = {"float16": 2e-3, "bfloat16": 1e-2}
ULP = {"float16": 2.0**-10, "bfloat16": 2.0**-7}
EPS = 1e-6


def _run(op, M, N, dtype, cfg, inputs_cpu):
    from deca_amd.kernels.rowwise_hip import build_rowwise, make_rowwise

    kern = build_rowwise(make_rowwise(op, M, N, dtype, cfg, EPS))
    dev = [t.to("cuda") for t in inputs_cpu]
    y = torch.empty_like(dev[0])
    kern(*dev, y)
    torch.cuda.synchronize()
    return y.cpu()


def _inputs(op, M, N, dtype, seed=0, std=None):
    from deca_amd.kernels.rowwise_bench import make_inputs_cpu

    std = std if std is not None else (2.0 if op == "softmax" else 1.0)
    return make_inputs_cpu(op, M, N, dtype, seed=seed, std=std)


def _oracle(op, dtype, inputs_cpu):
    if op == "softmax":
        return orw.softmax_reg(orw.to_f32(inputs_cpu[0]), dtype)
    return orw.rmsnorm(orw.to_f32(inputs_cpu[0]), orw.to_f32(inputs_cpu[1]), EPS, dtype)


def _fp32_truth(op, inputs_cpu):
    x = inputs_cpu[0].double()
    if op == "softmax":
        return torch.softmax(x, -1).numpy()
    w = inputs_cpu[1].double()
    return (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w).numpy()


def _check(op, dtype, got, inputs_cpu):
    got = orw.to_f32(got)
    want = _oracle(op, dtype, inputs_cpu)
    truth = _fp32_truth(op, inputs_cpu)
    assert np.isfinite(got).all()
    # accuracy gate
    err = np.abs(got - truth)
    if op == "softmax":
        assert err.max() <= GATE[dtype], f"max abs err {err.max():.3e}"
    else:
        assert np.all(err <= GATE[dtype] * np.maximum(1.0, np.abs(truth))), \
            f"max rel-to-grid err {(err / np.maximum(1.0, np.abs(truth))).max():.3e}"
    # parity with the checker: same roundings, so at most one ulp apart, rarely
    diff = np.abs(got - want)
    ulps = 1 if op == "softmax" else 2
    assert np.all(diff <= ulps * ULP[dtype] * np.maximum(np.abs(want), 2.0**-14) * 1.001 + 1e-12), \
        f"differs from the checker by more than {ulps} ulp: {diff.max():.3e}"
    assert (got != want).mean() < 2e-2, f"{(got != want).mean():.3%} of elements differ"


@pytest.mark.parametrize("op,M,N,dtype,cfg", ROWWISE_CASES, ids=lambda v: str(v))
def test_rowwise_parity(op, M, N, dtype, cfg):
    inputs = _inputs(op, M, N, dtype, seed=M + N)
    print(f"case {op} {M}x{N} {dtype} {cfg}", flush=True)
    _check(op, dtype, _run(op, M, N, dtype, cfg, inputs), inputs)


def test_softmax_extreme_values():
    """fp16 maximum, constant rows, a dominant entry, a very negative row."""
    from deca_amd.kernels.rowwise_hip import RowConfig

    M, N = 256, 4096
    (x,) = _inputs("softmax", M, N, "float16", seed=11)
    x[0] = 3.25
    x[1] = 0.0
    x[1, 77] = 65504.0
    x[2] = -65504.0
    x[3, :] = -30000.0
    x[3, 4095] = 30000.0
    y = orw.to_f32(_run("softmax", M, N, "float16", RowConfig(128, 1, 8), (x,)))
    assert np.isfinite(y).all()
    assert np.array_equal(y[0], np.full(N, np.float32(np.float16(1.0 / N))))
    assert y[1, 77] == 1.0 and y[1].sum() == 1.0
    assert np.array_equal(y[2], y[0])
    assert y[3, 4095] == 1.0 and y[3, :4095].max() == 0.0
    _check("softmax", "float16", torch.from_numpy(y), (x,))


def test_rmsnorm_closed_forms():
    from deca_amd.kernels.rowwise_hip import RowConfig

    M, N = 256, 4096
    x, w = _inputs("rmsnorm", M, N, "float16", seed=12)
    x[0] = 1.0
    x[1] = 0.0           # all-zero row -> zeros (eps keeps rsqrt finite)
    x[2] = x[3] * 4.0    # scale invariance
    w[:] = 1.0
    y = orw.to_f32(_run("rmsnorm", M, N, "float16", RowConfig(256, 1, 8), (x, w)))
    assert np.array_equal(y[0], np.full(N, np.float32(np.float16(1.0 / np.sqrt(1.0 + EPS)))))
    assert np.array_equal(y[1], np.zeros(N, np.float32))
    assert (y[2] != y[3]).mean() < 5e-3
    _check("rmsnorm", "float16", torch.from_numpy(y), (x, w))


@pytest.mark.parametrize("op,M,N,dtype,cfg", ROWWISE_FULL, ids=lambda v: str(v))
def test_rowwise_full_size(op, M, N, dtype, cfg):
    """Benchmark shapes: size-independent properties on every row plus the
    checker on a strided sample of rows."""
    inputs = _inputs(op, M, N, dtype, seed=0)
    print(f"full-size {op} {M}x{N} {dtype} {cfg}", flush=True)
    y = _run(op, M, N, dtype, cfg, inputs)
    yf = y.float()
    assert torch.isfinite(yf).all()
    if op == "softmax":
        sums = yf.sum(-1, dtype=torch.float64)
        assert (sums - 1.0).abs().max() <= N * ULP[dtype] / 64
        # the largest input of a row gets the largest output
        xf = inputs[0].float()
        assert torch.equal(yf.gather(1, xf.argmax(-1, keepdim=True)), yf.max(-1, keepdim=True).values)
    else:
        # dividing the weight back out leaves unit mean square
        w = inputs[1].float()
        ms = (yf / w).pow(2).mean(-1, dtype=torch.float64)
        assert (ms - 1.0).abs().max() <= 2e-2
    rows = torch.arange(0, M, max(1, M // 128))
    sub = tuple(t[rows] if t.dim() == 2 else t for t in inputs)
    _check(op, dtype, y[rows], sub)


def test_same_result_on_repeated_launches():
    """Two launches on the same input give identical bits (no dependence on
    leftover LDS contents or launch order)."""
    from deca_amd.kernels.rowwise_hip import RowConfig, build_rowwise, make_rowwise

    kern = build_rowwise(make_rowwise("softmax", 256, 4096, "float16", RowConfig(256, 2, 8), EPS))
    (x,) = _inputs("softmax", 256, 4096, "float16", seed=5)
    xd = x.cuda()
    y1, y2 = torch.empty_like(xd), torch.empty_like(xd)
    kern(xd, y1)
    kern(xd, y2)
    torch.cuda.synchronize()
    assert torch.equal(y1, y2)


def test_launch_rejects_wrong_arguments():
    from deca_amd.kernels.rowwise_hip import RowConfig, build_rowwise, make_rowwise

    kern = build_rowwise(make_rowwise("softmax", 256, 4096, "float16", RowConfig(128, 1, 8), EPS))
    x = torch.zeros(256, 4096, dtype=torch.float16, device="cuda")
    with pytest.raises(ValueError):
        kern(x)  # missing output
    with pytest.raises(ValueError):
        kern(x.cpu(), x)  # host tensor


@pytest.mark.parametrize("op,M,N,dtype,cfg", [c for c in ROWWISE_CASES if c[-1].half], ids=lambda v: str(v))
def test_half_vector_rows_end_where_they_end(op, M, N, dtype, cfg):
    """Elements behind the last row stay as they are (a whole vector stored at its end would
    reach them), and NaN there does not come into the row."""
    from deca_amd.kernels.rowwise_hip import build_rowwise, make_rowwise

    print(f"case {op} {M}x{N} {dtype} {cfg} with a guard", flush=True)
    inputs = _inputs(op, M, N, dtype, seed=M + N)
    dev = []
    for t in inputs:
        padded = torch.full((t.numel() + 64,), float("nan"), dtype=t.dtype, device="cuda")
        padded[:t.numel()] = t.cuda().flatten()
        dev.append(padded[:t.numel()].view(t.shape))
    out = torch.full((M * N + 64,), 7.0, dtype=inputs[0].dtype, device="cuda")
    kern = build_rowwise(make_rowwise(op, M, N, dtype, cfg, EPS))
    kern(*dev, out[:M * N].view(M, N))
    torch.cuda.synchronize()
    assert bool((out[M * N:] == 7.0).all())
    _check(op, dtype, out[:M * N].view(M, N).cpu(), inputs)

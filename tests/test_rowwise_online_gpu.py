"""GPU parity of the softmax form that takes the chunks of a row as they arrive, against the 64-bit
result: ordinary rows, rows masked by -inf, by the type's lowest value and by large finite numbers
down to one live element, and a row of large elements; with guards behind the output.

Tolerance: half a unit of the output type (2^-11 or 2^-8 of the element; 2^-24 below fp16's normal
range), and 2^-14 for the 32-bit part: at most 256 additions in a lane's chain (2^-16), the
rounding of exponents up to 100 (2^-17.5) and an ulp for each exp2, rescale and reciprocal.
"""

import pytest
import torch

from kernel_cases import ROWWISE_ONLINE_CASES

pytestmark = pytest.mark.gpu

HALF_UNIT = {"float16": 2.0**-11, "bfloat16": 2.0**-8}
SMALLEST = {"float16": 2.0**-24, "bfloat16": 2.0**-126}


def _rows(N, dtype):
    """Six rows, one of each kind."""
    dt = getattr(torch, dtype)
    g = torch.Generator().manual_seed(N)
    x = torch.randn(6, N, generator=g) * 2.0
    lowest = torch.finfo(dt).min
    x[1][torch.rand(N, generator=g) < 0.99] = -float("inf")
    x[2, : N // 2] = lowest
    x[3] = -1e10 if dtype == "bfloat16" else lowest
    x[3, N - 1] = 1.5
    x[4] = -float("inf")
    x[4, 17] = 3.0
    x[5] = 40000.0 + 32.0 * torch.randint(0, 2, (N,), generator=g)
    return x.to(dt)


def test_form_is_the_one_meant():
    from deca_amd.kernels.rowwise_hip import make_rowwise

    for op, M, N, dtype, cfg in ROWWISE_ONLINE_CASES:
        assert ("DECA_ONLINE", 1) in make_rowwise(op, M, N, dtype, cfg).defines


@pytest.mark.parametrize("op,M,N,dtype,cfg", ROWWISE_ONLINE_CASES, ids=lambda v: str(v))
def test_online_parity(op, M, N, dtype, cfg):
    from deca_amd.kernels.rowwise_hip import build_rowwise, make_rowwise

    print(f"case online {M}x{N} {dtype} {cfg}", flush=True)
    x = _rows(N, dtype)
    kern = build_rowwise(make_rowwise(op, M, N, dtype, cfg))
    want = torch.softmax(x.double(), -1)
    for shift in (0, 1):  # (elements: tensors may start at any of them)
        src = torch.zeros((M + 1) * N, dtype=x.dtype, device="cuda")
        src[shift: shift + M * N] = x.cuda().view(-1)
        buf = torch.full(((M + 1) * N,), 7.0, dtype=x.dtype, device="cuda")
        kern(src[shift: shift + M * N].view(M, N), buf[shift: shift + M * N].view(M, N))
        torch.cuda.synchronize()
        assert bool((buf[:shift] == 7.0).all()) and bool((buf[shift + M * N:] == 7.0).all())
        got = buf[shift: shift + M * N].view(M, N).cpu().double()
        assert bool(torch.isfinite(got).all())
        err = (got - want).abs() - (HALF_UNIT[dtype] + 2.0**-14) * want - SMALLEST[dtype]
        worst = int(err.max(-1).values.argmax())
        assert err.max().item() <= 0.0, f"shift {shift} row {worst}: {err.max().item():.3e} over the bound"

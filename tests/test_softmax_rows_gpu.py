"""GPU parity of softmax rows of every kind in forms whose vectors partly lie at the ends of a row, against
the 64-bit result, by the bound of test_rowwise_online_gpu.py: the kinds there, a row that is live at its
ends alone, with large elements, and a constant one.  (The sum and the stores must form an exponent alike:
of a large element the product with log2(e), rounded by itself, is up to 2^-9 off in float16's range and
2^-4 in that of the bfloat16 elements here.)"""

import pytest
import torch

from kernel_cases import SOFTMAX_ROW_CASES, lines_spec
from test_rowwise_online_gpu import HALF_UNIT, SMALLEST, _rows

pytestmark = pytest.mark.gpu

LARGE = {"float16": 50016.0, "bfloat16": 1003520.0}


def _more_rows(N, dtype):
    ends = torch.full((N,), torch.finfo(getattr(torch, dtype)).min)
    ends[:12] = LARGE[dtype]
    ends[-4:] = LARGE[dtype]
    more = torch.stack([ends, torch.full((N,), LARGE[dtype])])
    return torch.cat([_rows(N, dtype), more.to(getattr(torch, dtype))])


@pytest.mark.parametrize("lines", [False, True])
@pytest.mark.parametrize("M,N,dtype,cfg", SOFTMAX_ROW_CASES, ids=lambda v: str(v))
def test_rows_of_every_kind(M, N, dtype, cfg, lines):
    from deca_amd.kernels.rowwise_hip import build_rowwise, make_rowwise

    spec = (lines_spec if lines else make_rowwise)("softmax", M, N, dtype, cfg)
    assert (("DECA_LINES", 1) in spec.defines) == lines
    kern = build_rowwise(spec)
    x = _more_rows(N, dtype)
    want = torch.softmax(x.double(), -1)
    for at in (0, 4, 60):  # (elements behind a line)
        print(f"case rows {M}x{N} {dtype} {cfg} lines={lines} at {at}", flush=True)
        src = torch.full((M * N + 512,), float("nan"), dtype=x.dtype, device="cuda")
        src[128 + at: 128 + at + M * N] = x.cuda().view(-1)
        buf = torch.full((M * N + 512,), 7.0, dtype=x.dtype, device="cuda")
        y = buf[128 + at: 128 + at + M * N].view(M, N)
        kern(src[128 + at: 128 + at + M * N].view(M, N), y)
        torch.cuda.synchronize()
        assert bool((buf[: 128 + at] == 7.0).all()) and bool((buf[128 + at + M * N:] == 7.0).all())
        got = y.cpu().double()
        assert bool(torch.isfinite(got).all())
        err = (got - want).abs() - (HALF_UNIT[dtype] + 2.0**-14) * want - SMALLEST[dtype]
        worst = int(err.max(-1).values.argmax())
        assert err.max().item() <= 0.0, f"row {worst}: {err.max().item():.3e} over the bound"
    kern(torch.full_like(x, -float("inf"), device="cuda"), y)  # rows without a live element, as in torch
    torch.cuda.synchronize()
    assert bool(torch.isnan(y).all())

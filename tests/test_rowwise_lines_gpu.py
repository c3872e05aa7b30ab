"""GPU parity of the row-wise forms whose chunks start with a memory line, by the gates and the checker
of test_rowwise_gpu.py, over tensors that start at every kind of address, with guards around the
output."""

import pytest
import torch

from kernel_cases import ROWWISE_LINES_CASES, lines_spec
from test_rowwise_gpu import EPS, _check, _inputs

pytestmark = pytest.mark.gpu


def _placed(t, shift, fill):
    """`t` on the device, `shift` elements behind a line and between 256 elements of `fill` or more."""
    n = t.numel()
    buf = torch.full((n + 1024,), fill, dtype=t.dtype, device="cuda")
    buf[256 + shift: 256 + shift + n] = t.reshape(-1).cuda()
    return buf, buf[256 + shift: 256 + shift + n].view(t.shape)


@pytest.mark.parametrize("op,M,N,dtype,cfg", ROWWISE_LINES_CASES, ids=lambda v: str(v))
def test_lines_parity(op, M, N, dtype, cfg):
    from deca_amd.kernels.rowwise_hip import build_rowwise

    ins = _inputs(op, M, N, dtype, seed=N)
    kern = build_rowwise(lines_spec(op, M, N, dtype, cfg, EPS))
    for at_x, at_y in ((0, 0), (4, 4), (8, 60), (56, 0), (1, 3)):
        print(f"case lines {op} {M}x{N} {dtype} {cfg} x at {at_x}, y at {at_y}", flush=True)
        dev = [_placed(t, at_x, float("nan"))[1] for t in ins]
        buf, y = _placed(torch.full_like(ins[0], float("nan")), at_y, 7.0)
        kern(*dev, y)
        torch.cuda.synchronize()
        assert bool((buf[: 256 + at_y] == 7.0).all()) and bool((buf[256 + at_y + M * N:] == 7.0).all())
        _check(op, dtype, y.cpu(), ins)

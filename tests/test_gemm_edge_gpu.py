"""GPU parity of GEMM tiles that reach over the edge of C, and of K-tiles shared by groups of
waves, by the checks of test_gemm_gpu.py, with rows behind C and the operands that nothing may
write or need."""

import pytest
import torch

from kernel_cases import GEMM_EDGE_CASES
from test_gemm_gpu import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,cfg", GEMM_EDGE_CASES, ids=lambda v: str(v))
def test_gemm_edge_parity(M, N, K, cfg):
    from deca_amd.kernels.gemm_bench import make_inputs_cpu
    from deca_amd.kernels.gemm_hip import build_gemm_tc, make_gemm_tc

    print(f"case gemm edge {M}x{N}x{K} {cfg}", flush=True)
    a, b = make_inputs_cpu(M, N, K, seed=M + N + K)
    kern = build_gemm_tc(make_gemm_tc(M, N, K, cfg))
    # NaN behind the operands would show in C; the guard behind C must stay as it is
    pad = 256
    ad = torch.full((M + pad, K), float("nan"), dtype=torch.float16, device="cuda")
    bd = torch.full((K + pad, N), float("nan"), dtype=torch.float16, device="cuda")
    c = torch.full((M + pad, N), float("nan"), dtype=torch.float16, device="cuda")
    ad[:M], bd[:K] = a.cuda(), b.cuda()
    c[M:] = 7.0
    kern(ad[:M], bd[:K], c[:M])
    torch.cuda.synchronize()
    assert bool((c[M:] == 7.0).all())
    _check(c[:M].cpu(), a, b, K)

"""GPU parity of GEMM tiles that reach over the edge of C, and of K-tiles shared by groups of
waves, by the checks of test_gemm_gpu.py, with rows behind C that nothing may write and NaN
behind the operands, which a K-tile too many would bring into C (loads of rows and columns
behind an operand reach no result: test_gemm_edge_host.py looks at their addresses)."""

import numpy as np
import pytest
import torch

from kernel_cases import GEMM_EDGE_BF16_CASES, GEMM_EDGE_CASES
from oracle import gemm as og
from test_gemm_gpu import REL_GATE, _check

pytestmark = pytest.mark.gpu


def _run(M, N, K, cfg, a, b, dtype):
    from deca_amd.kernels.gemm_hip import build_gemm_tc, make_gemm_tc

    print(f"case gemm edge {M}x{N}x{K} {dtype} {cfg}", flush=True)
    kern = build_gemm_tc(make_gemm_tc(M, N, K, cfg, dtype))
    pad = 256
    ad = torch.full((M + pad, K), float("nan"), dtype=a.dtype, device="cuda")
    bd = torch.full((K + pad, N), float("nan"), dtype=a.dtype, device="cuda")
    c = torch.full((M + pad, N), float("nan"), dtype=a.dtype, device="cuda")
    ad[:M], bd[:K] = a.cuda(), b.cuda()
    c[M:] = 7.0
    kern(ad[:M], bd[:K], c[:M])
    torch.cuda.synchronize()
    assert bool((c[M:] == 7.0).all())
    return c[:M].cpu()


@pytest.mark.parametrize("M,N,K,cfg", GEMM_EDGE_CASES, ids=lambda v: str(v))
def test_gemm_edge_parity(M, N, K, cfg):
    from deca_amd.kernels.gemm_bench import make_inputs_cpu

    a, b = make_inputs_cpu(M, N, K, seed=M + N + K)
    _check(_run(M, N, K, cfg, a, b, "float16"), a, b, K)


@pytest.mark.parametrize("M,N,K,cfg", GEMM_EDGE_BF16_CASES, ids=lambda v: str(v))
def test_gemm_edge_bf16_parity(M, N, K, cfg):
    """The gate and the one bf16 ulp of test_gemm_gpu.test_gemm_bf16_parity."""
    from deca_amd.kernels.gemm_bench import make_inputs_cpu

    a, b = make_inputs_cpu(M, N, K, seed=M + N + K, dtype=torch.bfloat16)
    got = _run(M, N, K, cfg, a, b, "bfloat16").float().numpy()
    af, bf = a.float().numpy(), b.float().numpy()
    assert np.isfinite(got).all()
    assert og.max_rel_err(got, og.gemm_f32(af, bf)) <= REL_GATE
    want = og.gemm_bf16_out(af, bf)
    assert np.all(np.abs(got - want) <= np.maximum(np.abs(want), 2.0**-14) * 2.0**-7 * 1.001 + 1e-3)
    assert (got != want).mean() < 0.05

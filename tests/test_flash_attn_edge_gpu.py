"""GPU parity of attention whose query tiles reach over the end of the sequence, by the gate of
test_flash_attn_gpu.py, with rows behind O that nothing may write and NaN behind Q, K and V."""

import numpy as np
import pytest
import torch

from kernel_cases import FA_EDGE_CASES
from oracle import attn as oa
from test_flash_attn_gpu import GATE, _f32

pytestmark = pytest.mark.gpu


def _guarded(t, fill):
    """`t` on the device at the front of a buffer with 256 more rows of `fill`."""
    n = t.numel()
    buf = torch.full((n + 256 * t.shape[-1],), fill, dtype=t.dtype, device="cuda")
    buf[:n] = t.reshape(-1).cuda()
    return buf, buf[:n].view(t.shape)


@pytest.mark.parametrize("B,H,Sq,Skv,D,causal,cfg", FA_EDGE_CASES, ids=lambda v: str(v))
def test_edge_parity(B, H, Sq, Skv, D, causal, cfg):
    from deca_amd.kernels.attn_bench import make_qkv_cpu
    from deca_amd.kernels.flash_attn_hip import build_flash_attn, make_flash_attn_fwd

    print(f"case fa edge B{B} H{H} Sq{Sq} Skv{Skv} D{D} causal={causal} {cfg}", flush=True)
    q, k, v = make_qkv_cpu(B, H, Sq, Skv, D, seed=Sq + D)
    kern = build_flash_attn(make_flash_attn_fwd(B, H, Sq, Skv, D, cfg, None, causal))
    ins = [_guarded(t, float("nan"))[1] for t in (q, k, v)]
    buf, o = _guarded(torch.full_like(q, float("nan")), 7.0)
    kern(*ins, o)
    torch.cuda.synchronize()
    assert bool((buf[o.numel():] == 7.0).all())
    got = _f32(o.cpu())
    assert np.isfinite(got).all()
    assert np.abs(got - oa.attention_f32(_f32(q), _f32(k), _f32(v), None, causal)).max() <= GATE

"""GPU parity of the attention forms whose waves split the keys of their query rows.

The same gate as the other forms (max|o - ref| <= 2e-3 against fp32 attention).  The second
test spreads the scores so that the waves' running maxima lie far apart, and lets the largest
sit in another wave's share for every query: each wave's result then has a weight of its own
when they meet.
"""

import numpy as np
import pytest
import torch

from kernel_cases import FA_SPLIT_CASES
from oracle import attn as oa
from test_flash_attn_gpu import GATE, _f32, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Sq,Skv,D,causal,cfg", FA_SPLIT_CASES, ids=lambda v: str(v))
def test_split_parity(B, H, Sq, Skv, D, causal, cfg):
    from deca_amd.kernels.attn_bench import make_qkv_cpu

    print(f"case fa split B{B} H{H} Sq{Sq} Skv{Skv} D{D} causal={causal} {cfg}", flush=True)
    q, k, v = make_qkv_cpu(B, H, Sq, Skv, D, seed=Sq + D)
    got = _run(B, H, Sq, Skv, D, causal, cfg, q, k, v)
    assert torch.isfinite(got).all()
    assert np.abs(_f32(got) - oa.attention_f32(_f32(q), _f32(k), _f32(v), None, causal)).max() <= GATE
    if causal:  # row 0 sees key 0 only, which is in one wave's share
        assert torch.equal(got[:, :, 0], v[:, :, 0])


@pytest.mark.parametrize("B,H,Sq,Skv,D,causal,cfg", FA_SPLIT_CASES, ids=lambda v: str(v))
def test_split_shares_of_unequal_weight(B, H, Sq, Skv, D, causal, cfg):
    """Scores of tile t of query i are shifted by a multiple of 3 in (t + i) % 7: from -9 to
    +9, so shares differ by factors up to e^18."""
    from deca_amd.kernels.attn_bench import make_qkv_cpu

    print(f"case fa split shifted B{B} H{H} Sq{Sq} Skv{Skv} D{D} causal={causal} {cfg}", flush=True)
    q, k, v = make_qkv_cpu(B, H, Sq, Skv, D, seed=3)
    # seven dimensions carry the shift: one-hot of i % 7 in q, its value for each tile in k
    i, t = torch.arange(Sq), torch.arange(Skv) // cfg.Bc
    q[..., :7], k[..., :7] = 0, 0
    q[:, :, i, i % 7] = D**0.5
    for r in range(7):
        k[..., r] = (((t + r) % 7) - 3).half() * 3.0
    got = _f32(_run(B, H, Sq, Skv, D, causal, cfg, q, k, v))
    assert np.isfinite(got).all()
    # outputs dominated by single keys of |v| up to 4: fp16 rounding of P and of O, 2^-11 each
    want = oa.attention_f32(_f32(q), _f32(k), _f32(v), None, causal)
    assert np.abs(got - want).max() <= 2 * 2.0**-11 * 4 + GATE

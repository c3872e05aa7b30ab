"""Host test of the rankings on shapes where a rule once put the slower of two measured
configurations first.  Times are microseconds per launch on an MI355X, launches back to back
over buffers larger than the caches, both configurations in turn in one process."""

from dataclasses import replace

import pytest

from deca_amd import Solver, tuned
from deca_amd.arch import MI355X
from deca_amd.cost_model import CostModel as cm
from deca_amd.kernels.gemm_hip import GemmConfig
from kernel_cases import GEMM_EDGE_CASES

ARCH = MI355X()

# (operator, M, N, the slower configuration, its time, a time another one of the solver's takes)
ROWWISE = [
    # two vectors a lane, the second part empty, and half a vector at the end of the row
    ("softmax", 2713, 4116, "tpr=512,rpb=1,vec=8,mode=reg,hint=1,half=1", 11.7, 10.4),
    ("softmax", 1449, 2748, "tpr=256,rpb=1,vec=8,mode=reg,hint=1,half=1", 5.4, 4.6),
    ("softmax", 6309, 564, "tpr=64,rpb=1,vec=8,mode=reg,hint=1,half=1", 5.4, 4.9),
    ("rmsnorm", 20359, 1044, "tpr=128,rpb=1,vec=8,mode=reg,hint=1,half=1", 21.3, 18.3),
    ("rmsnorm", 611, 4820, "tpr=512,rpb=1,vec=8,mode=reg,hint=1,half=1", 4.5, 4.2),
    # ... which is nearly full here
    ("rmsnorm", 17558, 1988, "tpr=128,rpb=2,vec=4,mode=reg,hint=1", 26.7, 25.5),
    # rows all resident at once: several rows a workgroup, fewer lanes than a wave or 8-byte
    # accesses have nothing of what one wave a row gains there, nor has it with long softmax rows
    ("softmax", 7338, 3000, "tpr=32,rpb=2,vec=8,mode=reg,hint=1", 18.2, 17.0),
    ("softmax", 2718, 7408, "tpr=64,rpb=2,vec=8,mode=reg,hint=1", 17.1, 15.8),
    ("softmax", 11580, 1648, "tpr=16,rpb=4,vec=8,mode=reg,hint=1", 17.0, 14.6),
    ("rmsnorm", 4300, 3328, "tpr=64,rpb=2,vec=4,mode=reg,hint=1", 13.1, 10.6),
    ("rmsnorm", 5950, 3448, "tpr=32,rpb=2,vec=8,mode=reg,hint=1", 17.7, 16.2),
    # ... nor is one wave a row too many where there are more rows than the waves a CU needs
    ("rmsnorm", 7496, 824, "tpr=64,rpb=2,vec=4,mode=reg,hint=1", 7.0, 6.2),
    ("rmsnorm", 8181, 1028, "tpr=64,rpb=1,vec=4,mode=reg,hint=1", 9.2, 8.3),
    ("softmax", 8015, 904, "tpr=64,rpb=1,vec=4,mode=reg,hint=1", 7.5, 7.1),
    # ... but what it gains there is not lost on the half vectors at the ends of its row
    ("rmsnorm", 6760, 2460, "tpr=64,rpb=2,vec=4,mode=reg,hint=1", 14.9, 13.7),
    ("rmsnorm", 7631, 1596, "tpr=64,rpb=1,vec=4,mode=reg,hint=1", 11.4, 10.8),
    ("rmsnorm", 3027, 6932, "tpr=512,rpb=1,vec=4,mode=reg,hint=1", 17.6, 15.1),
    ("rmsnorm", 3982, 4436, "tpr=256,rpb=2,vec=8,mode=reg,hint=1,half=1", 14.6, 14.0),
    ("rmsnorm", 2439, 7132, "tpr=128,rpb=1,vec=8,mode=reg,hint=1,half=1", 14.7, 12.9),
    ("rmsnorm", 3421, 3812, "tpr=128,rpb=1,vec=8,mode=reg,hint=1,half=1", 11.6, 10.1),
    # ... where two waves a row are not nearly as good
    ("rmsnorm", 1787, 7260, "tpr=64,rpb=1,vec=8,mode=reg,hint=1,half=1", 10.1, 9.0),
    ("rmsnorm", 1820, 7220, "tpr=64,rpb=1,vec=8,mode=reg,hint=1,half=1", 11.0, 10.1),
    # long softmax rows that 8-byte accesses fit three of into a CU, 16-byte ones two
    ("softmax", 572, 64932, "tpr=512,rpb=1,vec=4,mode=reg,hint=1", 38.8, 29.9),
    ("softmax", 653, 64620, "tpr=512,rpb=1,vec=4,mode=reg,hint=1", 40.3, 38.0),
]


@pytest.mark.parametrize("op,M,N,slower,slower_us,us", ROWWISE, ids=lambda v: str(v))
def test_rowwise_first_rank_is_not_the_slower_form(op, M, N, slower, slower_us, us):
    assert us < slower_us
    first = cm.rank_rowwise_configs(Solver.solve_rowwise(ARCH, op, M, N), ARCH, op, M, N)[0]
    assert str(first) != slower


# (B, H, S_q, S_kv, D, causal, the slower configuration, its time, that of the plain form)
ATTENTION = [
    # few keys, more than two rows of 32 queries per CU: the plain forms fill the SIMDs too
    (3, 16, 384, 384, 64, False, "Br=32,Bc=32,warps=4,stages=1,q_smem=0,swz=1,kvs=1", 8.2, 7.1),
    # (of which the slot loop of two waves takes 128 keys a step)
    (3, 16, 384, 384, 64, False, "Br=64,Bc=64,warps=2,stages=2,q_smem=0,swz=1,pipe=2", 8.4, 7.1),
    (3, 16, 384, 384, 64, False, "Br=64,Bc=64,warps=2,stages=2,q_smem=0,swz=1,pipe=2,spread=8", 8.4, 7.1),
    (5, 16, 384, 384, 64, False, "Br=64,Bc=32,warps=4,stages=1,q_smem=0,swz=1,kvs=1", 10.5, 9.1),
    (8, 8, 256, 256, 64, False, "Br=64,Bc=32,warps=8,stages=1,q_smem=0,swz=1,kvs=1", 6.7, 5.9),
    (6, 16, 384, 384, 64, True, "Br=64,Bc=32,warps=4,stages=1,q_smem=0,swz=1,kvs=1", 11.0, 9.6),
    (6, 8, 768, 768, 128, True, "Br=32,Bc=32,warps=4,stages=1,q_smem=0,swz=1,kvs=1", 25.6, 21.9),
    # ... and the slot loop beats the key split there that was ahead of the plain loop of its tile
    (3, 16, 704, 704, 128, True, "Br=32,Bc=32,warps=4,stages=1,q_smem=0,swz=1,kvs=1", 22.6, 20.4),
    (1, 16, 2624, 3776, 64, False, "Br=64,Bc=32,warps=8,stages=1,q_smem=0,swz=1,kvs=1", 68.2, 60.6),
    # workgroups of eight waves that split the keys take two whole rounds for 1.2 or 1.5
    (1, 8, 1216, 12096, 128, False, "Br=32,Bc=32,warps=8,stages=1,q_smem=0,swz=1,kvs=1", 132.3, 117.2),
    (2, 32, 192, 15104, 128, False, "Br=32,Bc=32,warps=8,stages=1,q_smem=0,swz=1,kvs=1", 225.1, 215.1),
    (1, 8, 2688, 2688, 64, True, "Br=32,Bc=32,warps=8,stages=1,q_smem=0,swz=1,kvs=1", 19.6, 16.8),
    # long sequences: what the card sustains, not what a wave's own instructions would allow
    (2, 16, 8192, 8192, 128, False, "Br=256,Bc=64,warps=8,stages=2,q_smem=0,swz=1,pipe=2,spread=8", 934.8, 904.9),
    (4, 16, 4096, 4096, 128, False, "Br=256,Bc=64,warps=8,stages=2,q_smem=0,swz=1,pipe=2,spread=8", 481.9, 470.6),
    (2, 32, 8192, 8192, 64, False, "Br=128,Bc=32,warps=4,stages=2,q_smem=1,swz=1,mfma=16,roll=1,trust=1", 1176, 1038),
    (3, 32, 3840, 3840, 64, False, "Br=128,Bc=32,warps=4,stages=2,q_smem=1,swz=1,mfma=16,roll=1,trust=1", 405.2, 358.6),
    # tiles that reach over the end of the sequence against those that divide it
    (31, 8, 832, 832, 128, True, "Br=64,Bc=64,warps=2,stages=2,q_smem=0,swz=1,pipe=2,mfma=16,spread=8", 108.7, 79.7),
    (5, 32, 2368, 2368, 128, True, "Br=64,Bc=32,warps=2,stages=2,q_smem=0,swz=1,mfma=16,spread=4", 323.6, 252.4),
    (9, 16, 2880, 2880, 64, False, "Br=64,Bc=64,warps=2,stages=2,q_smem=1,swz=1,mfma=16,spread=4,trust=1", 395.1, 303.0),
    (2, 16, 1344, 1344, 192, False, "Br=64,Bc=32,warps=2,stages=2,q_smem=0,swz=1,mfma=16,trust=1", 100.5, 60.7),
    (11, 8, 2752, 2752, 192, True, "Br=64,Bc=32,warps=2,stages=2,q_smem=0,swz=1,mfma=16", 447.9, 272.8),
    (9, 8, 1600, 1600, 256, False, "Br=64,Bc=32,warps=2,stages=2,q_smem=0,swz=1,mfma=16,trust=1", 369.2, 260.6),
    # ... but for short causal ones of wide heads
    (19, 32, 448, 448, 320, True, "Br=128,Bc=64,warps=4,stages=2,q_smem=0,swz=1,pipe=2,mfma=16,spread=8,edge=1",
     578.6, 224.5),
    (20, 32, 576, 576, 320, True, "Br=128,Bc=64,warps=4,stages=2,q_smem=0,swz=1,pipe=2,mfma=16,spread=8,edge=1",
     855.1, 337.1),
    (23, 16, 576, 576, 256, True, "Br=256,Bc=32,warps=8,stages=1,q_smem=1,swz=1,mfma=16,edge=1", 187.7, 156.7),
]


@pytest.mark.parametrize("B,H,S_q,S_kv,D,causal,slower,slower_us,us", ATTENTION, ids=lambda v: str(v))
def test_attention_first_rank_is_not_the_slower_form(B, H, S_q, S_kv, D, causal, slower, slower_us, us):
    assert us < slower_us
    shape = (B, H, S_q, S_kv, D)
    first = cm.rank_fa_configs(Solver.solve_flash_attn(ARCH, *shape), ARCH, shape, causal)[0]
    assert str(first) != slower


# (B, H, S_q, S_kv, D, causal): shapes on which a key-split form was measured 1.1 ... 3.7x ahead
# of the plain form ranked first
KEY_SPLIT = [
    (1, 16, 512, 512, 64, True), (1, 16, 512, 8192, 128, False), (4, 8, 320, 384, 64, False),
    (1, 8, 1216, 12096, 128, False), (2, 16, 768, 768, 64, True),
]


@pytest.mark.parametrize("B,H,S_q,S_kv,D,causal", KEY_SPLIT)
def test_attention_first_rank_is_the_key_split_where_it_is_ahead(B, H, S_q, S_kv, D, causal):
    shape = (B, H, S_q, S_kv, D)
    assert cm.rank_fa_configs(Solver.solve_flash_attn(ARCH, *shape), ARCH, shape, causal)[0].kv_split


@pytest.mark.parametrize("D,causal", [(64, False), (64, True), (128, False), (128, True)])
def test_tuning_attention_measures_the_stored_winner(D, causal):
    """The tuning driver measures the first 16 configurations."""
    shape = (4, 16, 4096, 4096, D)
    stored = tuned.lookup(tuned.make_key("flash_attn", shape, causal=causal))
    ranked = cm.rank_fa_configs(Solver.solve_flash_attn(ARCH, *shape), ARCH, shape, causal, top_n=16)
    assert stored in ranked


@pytest.mark.parametrize("S", [2048, 8192])
@pytest.mark.parametrize("D,causal", [(64, False), (64, True), (128, False), (128, True)])
def test_no_attention_time_is_below_the_sustained_rate(S, D, causal):
    """1.25 PFLOP/s is more than any form was measured at."""
    shape = (2, 32, S, S, D)
    flops = 4.0 * 2 * 32 * S * S * D * (0.5 if causal else 1.0)
    for cfg in Solver.solve_flash_attn(ARCH, *shape):
        assert flops / cm.fa_time(cfg, ARCH, shape, causal) < 1.25e9, cfg


@pytest.mark.parametrize("M,N,K,cfg", GEMM_EDGE_CASES, ids=lambda v: str(v))
def test_every_valid_edge_form_can_be_ranked(M, N, K, cfg):
    """Also a tile body without measured step times."""
    assert cm.rank_gemm_configs([cfg], ARCH, M, N, K) == [cfg]
    assert 0.0 < cm.gemm_tc_score(cfg, ARCH, M, N, K) < 1.0


def test_edge_score_counts_useful_work_only():
    # a body without step times: half of the last row of tiles is outside of C
    cfg = GemmConfig(128, 128, 32, 64, 64, 3, 2, False, edge=True)
    full, cut = (cm.gemm_tc_score(cfg, ARCH, M, 2048, 512) for M in (2048, 1984))
    assert cut < full == cm.gemm_tc_score(replace(cfg, edge=False), ARCH, 2048, 2048, 512)


@pytest.mark.parametrize("M,N,K", [(2048, 2048, 2048), (1024, 1024, 1024), (1536, 4096, 512), (5120, 576, 512)])
def test_one_tile_has_one_score(M, N, K):
    """With and without `edge`, where the tile divides C and the two are the same code, and the
    solver has it once."""
    configs = Solver.solve_gemm_tc(ARCH, M, N, K)
    assert len({replace(c, edge=False) for c in configs}) == len(configs)
    measured = [c for c in configs if not c.edge and cm.gemm_edge_score(c, ARCH, M, N, K) is not None
                and cm.gemm_measured_form(c) == replace(c, edge=True)]
    assert measured
    for c in measured:
        assert cm.gemm_tc_score(c, ARCH, M, N, K) == cm.gemm_tc_score(replace(c, edge=True), ARCH, M, N, K)


@pytest.mark.parametrize("inputs", ["normal", "uniform"])
def test_tuning_a_small_grid_measures_the_stored_winner(inputs):
    """2048^3: 36 candidates at up to three tile orders per tile set, as its table entry was
    tuned; the entry's four-stage ring is not among the edge forms."""
    shape = (2048, 2048, 2048)
    stored = tuned.lookup(tuned.make_key("GEMM", shape, inputs=inputs))
    ranked = cm.rank_gemm_configs(Solver.solve_gemm_tc(ARCH, *shape), ARCH, *shape, top_n=36, per_tile=3)
    assert stored in ranked


# a single round of 128 x 64 or 64 x 128 tiles: wave groups were measured 4 ... 11 % ahead
KGROUPS = [(640, 1792, 2048), (1344, 1088, 2944), (2304, 704, 3072), (896, 1792, 5760),
           (1664, 1024, 7168), (512, 2880, 7936), (320, 3392, 1280)]


@pytest.mark.parametrize("M,N,K", KGROUPS)
def test_gemm_wave_groups_serve_the_grids_of_one_round(M, N, K):
    first = cm.rank_gemm_configs(Solver.solve_gemm_tc(ARCH, M, N, K), ARCH, M, N, K)[0]
    assert first.kgroups == 2 and -(-M // first.BM) * -(-N // first.BN) <= ARCH.sm_nums

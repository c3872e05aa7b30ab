"""Host check of the addresses that edge tiles load from.

What a load behind an operand brings in never reaches C (its row or column is not stored), so
no result shows it: the kernel's own offset functions are evaluated by the compiler instead,
for every chunk of the last tile row and column in their last K-tile.  Here every case is put
through the compiler, and copies of the source without the clamps must not pass."""

import shutil
import subprocess

import pytest

from deca_amd.cost_model.CostModel import GEMM_STEP_TIMES
from deca_amd.kernels.build import BASE_OPTIONS, CSRC_DIR, hipcc_path
from deca_amd.kernels.gemm_hip import GemmConfig, make_gemm_tc
from kernel_cases import GEMM_EDGE_BF16_CASES, GEMM_EDGE_CASES

# a row and 8 columns in the last tiles, and the smallest number of K-tiles, of every body that
# the solver offers
BODIES = [(bm + 1, bn + 8, bk * st, GemmConfig(bm, bn, bk, wm, wn, st, 1, True, mfma=16, kgroups=kg, edge=True))
          for bm, bn, bk, wm, wn, st, kg in GEMM_STEP_TIMES]


def _compile(spec, csrc):
    cmd = [hipcc_path(), "-fsyntax-only", "--cuda-device-only", "--offload-arch=gfx950", *BASE_OPTIONS,
           *spec.options, *spec.define_flags(), f"{csrc}/{spec.template}"]
    return subprocess.run(cmd, capture_output=True, text=True)


@pytest.mark.parametrize("M,N,K,cfg", GEMM_EDGE_CASES + GEMM_EDGE_BF16_CASES + BODIES, ids=lambda v: str(v))
def test_no_load_ends_behind_an_operand(M, N, K, cfg):
    proc = _compile(make_gemm_tc(M, N, K, cfg), CSRC_DIR)
    assert proc.returncode == 0, proc.stderr[-2000:]


@pytest.mark.parametrize("clamp,message", [
    ("(EDGE_M && row > last ? last : row)", "ends behind A"),
    ("(EDGE_N && c > last ? last : c)", "ends behind its row of B"),
])
def test_a_missing_clamp_does_not_compile(tmp_path, clamp, message):
    for name in ("gemm.hip", "gemm_tile.inc"):
        shutil.copy(f"{CSRC_DIR}/{name}", tmp_path)
    inc = tmp_path / "gemm_tile.inc"
    text = inc.read_text()
    assert text.count(clamp) == 1
    inc.write_text(text.replace(clamp, clamp.split(" : ")[1].rstrip(")")))
    M, N, K, cfg = GEMM_EDGE_CASES[0]
    proc = _compile(make_gemm_tc(M, N, K, cfg), tmp_path)
    assert proc.returncode != 0 and message in proc.stderr

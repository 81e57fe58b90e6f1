"""Causal attention over several 128-token tiles a (batch, head) pair: the workgroups take a tile of
every pair before the next tile (csrc/attention.hip, pair_tile). One token past a tile, whole tiles,
four tiles; pair counts that are no multiple of eight. Same checks and bounds as the kernel tests'."""
import pytest

import test_gpu_kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,H,dk,dv", [(3, 129, 5, 32, 32), (2, 256, 4, 64, 64), (1, 385, 3, 64, 64), (1, 130, 1, 96, 64)])
def test_causal_tiles(oracle, B, S, H, dk, dv):
    test_gpu_kernels.test_attention_fwd_bwd_vs_oracle(oracle, 1, B, S, H, dk, dv)

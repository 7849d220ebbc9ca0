"""The wrapper's dynamic-H backward at any stream count (csrc/wrapper_bwd.hip):
row counts of dP at the edges of its 16-row tiles, token counts at the edges of
its 32-token stages and of the rounds of stages, channel counts at the edges of
its 16-channel waves and 128-channel workgroups, both modes and storage types,
and a partial count of coefficient sums past the one-launch limit; against the
float64 oracle, tolerances as tests/test_gpu_wrapper_fold.py."""
import pytest
import torch

from tests.test_gpu_wrapper_fold import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["decay", "zero"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,T,C", [(2, 1, 16), (3, 31, 32), (5, 33, 160), (6, 95, 144), (7, 97, 32), (8, 193, 264),
                                   (8, 32, 120), (9, 64, 128), (16, 65, 136), (17, 40, 32), (32, 1100, 8)])
def test_shapes(device, n, T, C, dtype, mode):
    _run(device, n, T, C, dtype, mode, seed=n * T + C)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_many_tiles(device, dtype):
    # one column block: half as many token tiles as CUs, of two rounds of stages
    _run(device, 5, 256 * 97, 64, dtype, "decay", seed=3)


def test_widest_rows(device):
    """n = 2 past 1.86M channels, where a tile's 2 GiB hold less than one round of
    stages: the backward runs on the kernels for other shapes."""
    _run(device, 2, 3, 1_900_032, torch.float32, "zero", seed=4)

"""The segment-map kernels of the chunked scan (several time segments per
call) against the fp64 oracle, at the edges of their 32-row blocks and channel
tiles: ragged last blocks, one-block runs, odd and partial channel widths,
entries of the state that do not fill a tile, every dtype mix."""
import pytest
import torch

from tests._helpers import check_all, oracle_all, rand_inputs, run_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 129, 33, 9), (2, 515, 47, 16), (1, 700, 130, 24), (2, 389, 64, 32),
                                   (1, 1025, 31, 33), (3, 257, 98, 64), (1, 2049, 40, 64)])
@pytest.mark.parametrize("dtype,gate_dtype", [(torch.float32, None), (torch.bfloat16, None),
                                              (torch.bfloat16, torch.float32), (torch.float16, None)])
def test_segment_maps(gpu, shape, dtype, gate_dtype):
    b, T, D, N = shape
    ins = rand_inputs(b, T, D, N, seed=T + N, dtype=dtype, gate_dtype=gate_dtype, h0_std=0.3)
    y, g = run_hip(ins, gpu)
    ry, rg = oracle_all(ins)
    check_all(y, g, ry, rg)


def test_segment_maps_hard_gates(gpu):
    """Gates of exactly 0 and 1 across segment boundaries: a reset cuts the
    map, a run of ones carries it unchanged."""
    ins = rand_inputs(1, 640, 64, 64, seed=3, dtype=torch.bfloat16, h0_std=0.5)
    f = ins["f_logit"]
    f[:, ::7] = float("inf")
    f[:, 130] = float("-inf")
    f[:, 200:520, :32] = float("inf")
    y, g = run_hip(ins, gpu)
    ry, rg = oracle_all(ins)
    check_all(y, g, ry, rg)

"""The segment-map kernels of the chunked scan (several time segments per
call) against the fp64 oracle, at the edges of their 32-row blocks and channel
tiles: ragged last blocks, one-block runs, odd and partial channel widths,
entries of the state that do not fill a tile, every dtype mix."""
import ctypes

import pytest
import torch

from naju_amd import _lib
from tests._helpers import check, check_all, oracle_all, rand_inputs, run_hip

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


def _plan(batch, T, D, N, backward):
    """(segments, rows per segment, waves per segment map) of a call."""
    rows, waves = ctypes.c_int64(), ctypes.c_int()
    n = _lib.lib().naju_scan_time_segments(batch, T, D, N, backward, ctypes.byref(rows), ctypes.byref(waves))
    return n, rows.value, waves.value


# (batch, T, D, N), dtype, gate dtype, forward plan, backward plan. D = 33, 31:
# one channel per lane, D = 34, 64: two. 336-, 528- and 752-row segments are no
# multiple of the 32-row blocks of their waves.
PLANS = [
    ((128, 1300, 33, 16), torch.float32, None, (6, 256, 2), (4, 336, 2)),
    ((128, 1300, 34, 64), torch.bfloat16, None, (6, 256, 2), (4, 336, 2)),
    ((128, 1300, 47, 24), torch.float16, None, (6, 256, 2), (4, 336, 2)),
    ((128, 1300, 64, 100), torch.bfloat16, torch.float32, (6, 256, 2), (4, 336, 2)),
    ((256, 1500, 33, 16), torch.bfloat16, torch.float32, (3, 512, 4), (2, 752, 4)),
    ((256, 1500, 34, 64), torch.float32, None, (3, 512, 4), (2, 752, 4)),
    ((256, 1500, 33, 32), torch.float16, None, (3, 512, 4), (2, 752, 4)),
    ((256, 1500, 31, 128), torch.bfloat16, None, (3, 512, 4), (2, 752, 4)),
    ((256, 1500, 34, 65), torch.float16, torch.float32, (3, 512, 4), (2, 752, 4)),
    # the backward's last segment has 2 rows: its second wave has none
    ((32, 3842, 33, 64), torch.bfloat16, None, (31, 128, 1), (16, 256, 2)),
    ((32, 3842, 34, 128), torch.float32, None, (31, 128, 1), (16, 256, 2)),
    # ... and 466 of 528 rows in runs of 160: its fourth wave has none
    ((192, 2050, 34, 16), torch.float32, None, (17, 128, 1), (4, 528, 4)),
]


@pytest.mark.parametrize("shape,dtype,gate_dtype,fwd,bwd", PLANS)
def test_segment_maps_by_plan(gpu, shape, dtype, gate_dtype, fwd, bwd):
    """Maps formed by several waves, over blocks that the running decay and
    the prefetch cross: slow gates, so that a segment's map holds all of its
    rows. Three batch rows against the oracle (every output but dD depends on
    its own batch row alone), dD against the float64 sum."""
    b, T, D, N = shape
    assert _plan(b, T, D, N, 0) == fwd and _plan(b, T, D, N, 1) == bwd
    ins = rand_inputs(b, T, D, N, seed=T + N, dtype=dtype, gate_dtype=gate_dtype, f_shift=4.0, h0_std=0.3)
    y, g = run_hip(ins, gpu)
    rows = [0, b // 2, b - 1]
    sub = {k: v if k == "D_skip" else v[rows] for k, v in ins.items()}
    ry, rg = oracle_all(sub)
    check_all(y[rows], {k: v[rows] for k, v in g.items() if k != "dD"}, ry, rg)
    dD = (ins["dy"].to(gpu).double() * ins["u"].to(gpu).double()).sum((0, 1)).cpu().numpy()
    check("dD", g["dD"], dD, (1e-5, 1e-5))

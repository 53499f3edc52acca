"""State sizes 65 .. 128 on the matrix cores (the backward in two halves of the
entries) against the fp64 oracle: second halves of one entry up to 64, odd N
(unaligned rows of B, C and the states), ragged rows and channels, h0 and every
dtype mix."""
import pytest
import torch

from naju_amd import _lib
from tests._helpers import check_all, oracle_all, rand_inputs, run_hip


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 40, 24, 65), (2, 150, 130, 71), (1, 333, 63, 96), (2, 129, 64, 100),
                                   (1, 700, 40, 127), (2, 257, 136, 128)])
@pytest.mark.parametrize("dtype,gate_dtype", [(torch.float32, None), (torch.bfloat16, None),
                                              (torch.bfloat16, torch.float32), (torch.float16, None)])
def test_wide_state(gpu, shape, dtype, gate_dtype):
    b, T, D, N = shape
    ins = rand_inputs(b, T, D, N, seed=T + N, dtype=dtype, gate_dtype=gate_dtype, h0_std=0.3)
    y, g = run_hip(ins, gpu)
    ry, rg = oracle_all(ins)
    check_all(y, g, ry, rg)


def test_wide_state_checkpoint_interval():
    """N > 64 keeps one interval, asked for as 0 or 32 rows."""
    L = _lib.lib()
    F32 = _lib.DT_F32

    def elems(rows):
        return L.naju_scan_ckpt_elems_ex(2, 300, 96, 128, F32, F32, F32, _lib.ckpt_rows_flag(rows) if rows else 0)

    assert elems(0) == elems(32) == L.naju_scan_ckpt_elems(2, 300, 96, 128, F32, F32, F32)
    assert all(elems(r) == -1 for r in (16, 64, 128))

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
    """N > 64 serves 32 rows beside its default of 16: the checkpoint of r rows
    holds batch * ceil(T / r) * D * N floats, as the header says."""
    L = _lib.lib()
    F32 = _lib.DT_F32

    def elems(rows):
        return L.naju_scan_ckpt_elems_ex(2, 300, 96, 128, F32, F32, F32, _lib.ckpt_rows_flag(rows) if rows else 0)

    assert elems(0) == L.naju_scan_ckpt_elems(2, 300, 96, 128, F32, F32, F32) == 2 * 19 * 96 * 128
    assert elems(32) == 2 * 10 * 96 * 128
    assert all(elems(r) == -1 for r in (16, 64, 128))


@pytest.mark.gpu
@pytest.mark.parametrize("shape,dtype", [((2, 300, 96, 65), torch.float32), ((1, 129, 40, 100), torch.bfloat16),
                                         ((2, 2500, 136, 128), torch.bfloat16), ((1, 31, 16, 128), torch.float16)])
def test_wide_state_interval(gpu, shape, dtype):
    """32 rows: the forward writes the header's batch * ceil(T / 32) * D * N
    floats and nothing past them, and every output is bitwise the default's."""
    from naju_amd import naju_scan_hip
    b, T, D, N = shape
    ins = rand_inputs(b, T, D, N, seed=T, dtype=dtype, h0_std=0.3)
    keys = [k for k in ("u", "f_logit", "i_logit", "B", "C", "D_skip", "h0")]
    got = []
    for rows in (None, 32):
        xs = [ins[k].to(gpu).requires_grad_(True) for k in keys]
        y = naju_scan_hip(*xs, ckpt_rows=rows)
        y.backward(ins["dy"].to(gpu))
        got.append([y] + [x.grad for x in xs])
    assert all(torch.equal(p, q) for p, q in zip(*got))

    L = _lib.lib()
    dts = (_lib.DT_F32 if dtype == torch.float32 else (_lib.DT_BF16 if dtype == torch.bfloat16 else _lib.DT_F16),) * 3
    flags = _lib.ckpt_rows_flag(32)
    n = b * ((T + 31) // 32) * D * N
    ck = torch.full((n + 4096,), 7.0, device=gpu)
    nb = L.naju_scan_workspace_bytes_ex(b, T, D, N, *dts, flags)
    ws = torch.zeros(nb, dtype=torch.uint8, device=gpu)
    xs = [ins[k].to(gpu) for k in keys]
    y = torch.empty_like(xs[0])
    _lib.check(L.naju_scan_fwd(*[x.data_ptr() for x in xs], y.data_ptr(), ck.data_ptr(), None, b, T, D, N, *dts, flags,
                               ws.data_ptr(), nb, torch.cuda.current_stream(gpu).cuda_stream))
    torch.cuda.synchronize()
    assert bool((ck[n:] == 7.0).all()) and not bool((ck[:n] == 7.0).any())

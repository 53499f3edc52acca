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


@pytest.mark.gpu
@pytest.mark.parametrize("N", [72, 128])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_wide_state_hard_gates(gpu, N, dtype):
    """Gates of exactly 0 and 1 (the exact decay products of both halves, maps
    cut by a reset or carried unchanged): dfl is exactly 0 there."""
    ins = rand_inputs(2, 400, 64, N, seed=3, dtype=dtype, h0_std=0.5)
    f = ins["f_logit"]
    f[:, ::7] = float("inf")
    f[:, 130] = float("-inf")
    f[:, 200:320, :32] = float("inf")
    f[1, 5::9, 40:] = float("-inf")
    y, g = run_hip(ins, gpu)
    ry, rg = oracle_all(ins)
    check_all(y, g, ry, rg)
    assert bool((g["dfl"][torch.isinf(f).to(gpu)] == 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("want", [["B"], ["C"], ["u"], ["f_logit", "i_logit"], ["h0"], ["D_skip"]])
def test_wide_state_partial_gradients(gpu, want):
    """Some of the gradients only: bitwise those of the whole backward."""
    ins = rand_inputs(2, 300, 136, 96, seed=9, dtype=torch.bfloat16, h0_std=0.3)
    _, full = run_hip(ins, gpu)
    _, part = run_hip(ins, gpu, grad_names=want)
    assert len(part) == len(want)
    for k, v in part.items():
        assert torch.equal(v, full[k]), k


@pytest.mark.gpu
@pytest.mark.parametrize("N,dtype", [(65, torch.float32), (128, torch.bfloat16)])
def test_wide_state_repeats_and_replays(gpu, N, dtype):
    """Eager runs repeat bitwise, and a captured forward + backward replays
    them bitwise, also after other inputs."""
    from tests.test_graph_gpu import _setup
    outs = ("y", "du", "dfl", "dil", "dB", "dC", "dD", "dh0")
    ins = rand_inputs(2, 700, 136, N, seed=N, dtype=dtype, h0_std=0.3)
    bufs, step, status = _setup(ins, gpu)
    step()
    torch.cuda.synchronize()
    ref = {k: bufs[k].clone() for k in outs}
    step()
    torch.cuda.synchronize()
    assert all(torch.equal(bufs[k], ref[k]) for k in outs)
    s = torch.cuda.Stream(gpu)
    with torch.cuda.stream(s):
        step()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            step()
    for rep in range(3):
        for k in outs:
            bufs[k].fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(bufs[k], ref[k]) for k in outs), rep
        step()  # eager work between replays
        torch.cuda.synchronize()
        keep = bufs["_inputs"]["u"].clone()
        bufs["_inputs"]["u"].mul_(2.0)
        g.replay()
        torch.cuda.synchronize()
        assert not torch.equal(bufs["y"], ref["y"])
        bufs["_inputs"]["u"].copy_(keep)
    assert status() == 0


@pytest.mark.gpu
@pytest.mark.parametrize("shape,same_plan", [((2, 300, 96, 65), True), ((2, 2048, 1024, 128), False)])
def test_wide_state_noalloc(gpu, shape, same_plan):
    """The allocation-free forward: bitwise naju_scan_fwd where its scratch
    holds the same time segments, and to float32 rounding where it does not
    (the maps of the second shape's segments take more than the scratch)."""
    b, T, D, N = shape
    L = _lib.lib()
    dts = (_lib.DT_F32,) * 3
    ins = rand_inputs(b, T, D, N, seed=T, h0_std=0.3)
    xs = [ins[k].to(gpu) for k in ("u", "f_logit", "i_logit", "B", "C", "D_skip", "h0")]
    n_ck = L.naju_scan_ckpt_elems(b, T, D, N, *dts)
    nb = L.naju_scan_workspace_bytes(b, T, D, N, *dts)
    ws = torch.zeros(nb, dtype=torch.uint8, device=gpu)
    st = torch.cuda.current_stream(gpu).cuda_stream
    got = []
    for noalloc in (False, True):
        y, ck, hT = torch.empty_like(xs[0]), torch.empty(n_ck, device=gpu), torch.empty_like(xs[6])
        p = [x.data_ptr() for x in xs] + [y.data_ptr(), ck.data_ptr(), hT.data_ptr(), b, T, D, N, *dts, 0]
        _lib.check(L.naju_scan_fwd_noalloc(*p, st) if noalloc else L.naju_scan_fwd(*p, ws.data_ptr(), nb, st))
        torch.cuda.synchronize()
        got.append((y, ck, hT))
    for v, w in zip(*got):
        if same_plan:
            assert torch.equal(v, w)
        else:
            assert (v - w).abs().max().item() <= 1e-5 * w.abs().max().item()
    if not same_plan:
        assert not torch.equal(got[0][0], got[1][0])

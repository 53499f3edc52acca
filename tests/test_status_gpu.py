"""Failed carry hand-offs reach the caller without a synchronisation.

The N = 1 kernels hand chunk carries between workgroups with bounded waits; a
wait that gives up writes NaN outputs and sets the workspace's status word.
The kernel stores that word in pinned host memory too, and the next
naju_scan_hip call (or backward) on the same stream that finds it nonzero
raises NajuScanError, clearing both so the workspace is usable again. The failures are forced from the host with the library's
NAJU_DEBUG_SPIN_LIMIT=0 test hook (every hand-off gives up at once, every
kernel still exits normally)."""
import pytest
import torch

from tests._helpers import NAMES, rand_inputs

pytestmark = pytest.mark.gpu


def _inputs(dev, grad=False):
    ins = rand_inputs(2, 4096, 256, 1, seed=23, dtype=torch.float32)
    xs = [ins[k].to(dev).requires_grad_(grad) for k in NAMES]
    return xs, ins["dy"].to(dev)


def test_failed_forward_handoff_raises_at_the_next_call(gpu, monkeypatch):
    from naju_amd import naju_scan_hip
    from naju_amd._lib import NajuScanError
    xs, _ = _inputs(gpu)
    with torch.no_grad():
        y_ok = naju_scan_hip(*xs)
        monkeypatch.setenv("NAJU_DEBUG_SPIN_LIMIT", "0")
        y_bad = naju_scan_hip(*xs)
        monkeypatch.delenv("NAJU_DEBUG_SPIN_LIMIT")
        torch.cuda.synchronize()
        assert bool(torch.isnan(y_bad[:, 128:]).all()) and bool(torch.isfinite(y_bad[:, :128]).all())
        with pytest.raises(NajuScanError, match="earlier scan call") as ei:
            naju_scan_hip(*xs)
        assert ei.value.code == 1
        # cleared: the same workspace serves correct calls again
        y2 = naju_scan_hip(*xs)
        torch.cuda.synchronize()
    torch.testing.assert_close(y2, y_ok, rtol=1e-6, atol=1e-6)


def test_failed_backward_handoff_raises_at_the_next_call(gpu, monkeypatch):
    from naju_amd import naju_scan_hip
    from naju_amd._lib import NajuScanError
    xs, dy = _inputs(gpu, grad=True)
    y = naju_scan_hip(*xs)
    monkeypatch.setenv("NAJU_DEBUG_SPIN_LIMIT", "0")
    y.backward(dy)
    monkeypatch.delenv("NAJU_DEBUG_SPIN_LIMIT")
    torch.cuda.synchronize()
    assert bool(torch.isnan(xs[0].grad).any())
    with pytest.raises(NajuScanError) as ei:
        naju_scan_hip(*xs)
    assert ei.value.code == 1
    for x in xs:
        x.grad = None
    y = naju_scan_hip(*xs)
    y.backward(dy)
    torch.cuda.synchronize()
    assert all(bool(torch.isfinite(x.grad).all()) for x in xs)


def test_healthy_calls_never_raise(gpu):
    """Many N = 1 calls in a row on one stream without synchronisation: the
    mirror of a healthy workspace stays 0."""
    from naju_amd import naju_scan_hip
    xs, dy = _inputs(gpu, grad=True)
    for _ in range(20):
        y = naju_scan_hip(*xs)
        y.backward(dy)
    torch.cuda.synchronize()
    naju_scan_hip(*xs)
    torch.cuda.synchronize()


def test_grown_workspace_keeps_its_mirror(gpu, monkeypatch):
    """A stream's workspace that is replaced by a larger one reports failures
    through the same mirror word."""
    from naju_amd import naju_scan_hip
    from naju_amd._lib import NajuScanError
    stream = torch.cuda.Stream(gpu)
    with torch.cuda.stream(stream), torch.no_grad():
        for T in (300, 40000):
            ins = rand_inputs(2, T, 256, 1, seed=T, dtype=torch.float32)
            xs = [ins[k].to(gpu) for k in NAMES]
            naju_scan_hip(*xs)
            monkeypatch.setenv("NAJU_DEBUG_SPIN_LIMIT", "0")
            naju_scan_hip(*xs)
            monkeypatch.delenv("NAJU_DEBUG_SPIN_LIMIT")
            stream.synchronize()
            with pytest.raises(NajuScanError):
                naju_scan_hip(*xs)
            assert bool(torch.isfinite(naju_scan_hip(*xs)).all())


def test_workspace_that_was_never_zeroed(gpu):
    """Every word of the workspace holds the same arbitrary value, the ticket
    counters and what lies beside them among it: every workgroup's ticket is
    out of range, so the outputs are NaN and the status is 2, in the header and
    in the mirror that the call gave. (No address is read from the workspace.)
    Clearing the status makes it usable."""
    import ctypes
    from naju_amd import _lib
    L = _lib.lib()
    B, T, D = 2, 1000, 256
    ins = rand_inputs(B, T, D, 1, seed=5, dtype=torch.float32)
    xs = [ins[k].to(gpu) for k in NAMES]
    dts = (_lib.DT_F32,) * 3
    nb = L.naju_scan_workspace_bytes(B, T, D, 1, *dts)
    st = torch.cuda.current_stream(gpu).cuda_stream
    word = torch.zeros(1, dtype=torch.int32, pin_memory=True)

    def run(ws):
        y = torch.empty_like(xs[0])
        _lib.check(L.naju_scan_fwd_mirrored(*[x.data_ptr() for x in xs], None, y.data_ptr(), None, None, B, T, D, 1,
                                            *dts, _lib.FLAG_DETERMINISTIC, ws.data_ptr(), nb, word.data_ptr(), st))
        torch.cuda.synchronize()
        return y

    good = run(torch.zeros(nb, dtype=torch.uint8, device=gpu))
    assert int(word[0]) == 0 and bool(torch.isfinite(good).all())
    ws = torch.full((nb,), 0x40, dtype=torch.uint8, device=gpu)
    assert bool(torch.isnan(run(ws)).all()) and int(word[0]) == 2
    got = ctypes.c_uint32(0)
    _lib.check(L.naju_scan_workspace_status(ws.data_ptr(), st, ctypes.byref(got)))
    assert got.value == 2
    word.zero_()
    assert torch.equal(run(ws), good) and int(word[0]) == 0

"""Which calls go through the scan's autograd function: all but those that
nothing can record. Forward-mode AD, functorch transforms and tracing reach it
under no_grad too, as they did when every call did."""
import pytest
import torch
from torch.autograd import forward_ad

from naju_amd import scan


@pytest.fixture
def routes(monkeypatch):
    seen = []
    monkeypatch.setattr(scan, "_forward", lambda u, *a: seen.append("direct") or (u, None, None))
    monkeypatch.setattr(scan.NajuScanHip, "apply", lambda u, *a: seen.append("function") or u)
    return seen


def _call(u):
    z = torch.zeros(1, 2, 1)
    return scan.naju_scan_hip(u, u, u, z, z, torch.zeros(3))


def test_direct_only_where_nothing_records(routes):
    u = torch.zeros(1, 2, 3)
    _call(u)
    with torch.no_grad():
        _call(u)
    with torch.inference_mode():
        _call(u)
    assert routes == ["function", "direct", "direct"]


def test_transforms_keep_the_function(routes):
    u = torch.zeros(1, 2, 3)
    with torch.no_grad():
        with forward_ad.dual_level():
            _call(forward_ad.make_dual(u, torch.ones_like(u)))
        torch.vmap(_call)(u[None])
        torch.jit.trace(_call, (u,), check_trace=False)
    assert routes == ["function"] * len(routes) and len(routes) >= 3


def test_sizes_are_those_of_the_library():
    L = scan._lib.lib()
    scan._SIZES.clear()
    for flags in (0, scan._lib.ckpt_rows_flag(128)):
        for _ in range(2):
            got = scan._sizes(2, 300, 96, 64, (1, 0, 1), flags)
            assert got == (L.naju_scan_ckpt_elems_ex(2, 300, 96, 64, 1, 0, 1, flags),
                           L.naju_scan_workspace_bytes_ex(2, 300, 96, 64, 1, 0, 1, flags))
    with pytest.raises(scan._lib.NajuScanError):
        scan._sizes(2, 300, 96, 4, (0, 0, 0), scan._lib.ckpt_rows_flag(64))
    for k in range(300):  # bounded
        scan._sizes(1, k + 1, 8, 1, (0, 0, 0), 0)
    assert len(scan._SIZES) <= 256


@pytest.mark.parametrize("device", [None, "cuda", torch.device("cuda"), "cuda:1", 1])
def test_workspace_status_takes_a_device_without_an_index(monkeypatch, device):
    """"cuda" names the current device, as it does everywhere in torch."""
    asked = []
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)
    monkeypatch.setattr(scan, "_stream_handle", lambda dev: asked.append(dev.index) or 0)
    assert scan.workspace_status(device) == 0 and asked == [1]

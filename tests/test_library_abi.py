"""The C ABI library builds, loads without a GPU, and exports every function
include/warp_hip.h declares; registration declines when there is no device."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared():
    src = open(os.path.join(ROOT, "include", "warp_hip.h")).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    names = set(re.findall(r"\b((?:warp_hip|waste)_\w+)\s*\(", src))
    return sorted(n for n in names if not n.endswith("_fn"))


def test_header_declares_the_abi():
    names = declared()
    for must in ("waste_register_hip", "warp_hip_open", "warp_hip_moe_decode", "warp_hip_moe_chunk",
                 "warp_hip_vq_matvec", "warp_hip_decode_weights", "warp_hip_route"):
        assert must in names


def test_library_exports_every_declared_symbol():
    import warp_amd
    L = warp_amd.lib()
    missing = [n for n in declared() if not hasattr(L, n)]
    assert not missing, missing
    from warp_amd import hip
    assert set(declared()) <= set(hip.SIGNATURES)


def test_registration_declines_without_a_device():
    import warp_amd
    from warp_amd.device import device_count
    if device_count() > 0:
        pytest.skip("a device is present")

    class Table(ctypes.Structure):
        _fields_ = [("fn", ctypes.c_void_p * 5), ("on_device", ctypes.c_int)]

    t = Table()
    t.fn[3] = 1234
    assert warp_amd.lib().waste_register_hip(ctypes.byref(t)) is None
    assert t.fn[3] == 1234 and t.on_device == 0


def test_open_refuses_without_a_device():
    import warp_amd
    from warp_amd.device import device_count
    if device_count() > 0:
        pytest.skip("a device is present")
    with pytest.raises(warp_amd.WarpHipError):
        warp_amd.Context(hidden=128, inter=64, n_experts=8, top_k=2, n_layers=1, fmt="VQ3R",
                         rec_bytes=12288, cache_bytes=12288 * 8)


def test_run_kernels_refuse_longer_runs_than_they_take():
    """A run list made for the reduced-precision kernel holds runs of four
    jobs; the exact one would leave out two of them."""
    import warp_amd
    from warp_amd.device import device_count
    if device_count() > 0:
        pytest.skip("a device is present: the calls that are not refused would launch")
    L, buf = warp_amd.lib(), (ctypes.c_char * 4096)()
    at = (ctypes.addressof(buf) + 15) & ~15
    y = (ctypes.c_void_p * 3)(at, at, at)
    L.wk_vq_runs.argtypes = [ctypes.c_int] + [ctypes.c_void_p] * 2 + [ctypes.c_int, ctypes.c_void_p] + [
        ctypes.c_int] * 2 + [ctypes.c_void_p] * 4 + [ctypes.c_int] * 4 + [ctypes.c_void_p, ctypes.c_int,
                                                                         ctypes.c_void_p]

    def call(fp16_rows, run_j):
        return L.wk_vq_runs(9, at, at, 1, at, 0, 1, at, at, at, y, 64, 32, fp16_rows, run_j, at, 256, None)
    for fp16_rows, most in ((0, 2), (8, 4)):
        assert call(fp16_rows, most) < -1000              # passed the checks: no device to launch on
        assert [call(fp16_rows, r) for r in (0, most + 1, 5)] == [-1] * 3

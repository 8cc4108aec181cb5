"""A pass per plane of the two inner axes where it is the faster way: against a pass per axis of the
same library, at plane counts between one and three per CU (the workgroups of a CU have to be
resident together) and at the size from which arithmetic decides."""

import ctypes
import math

import pytest

pytestmark = pytest.mark.gpu


def _handle(layout, dims, real, flags):
    from fftm_amd import _lib
    h = ctypes.c_void_p()
    _lib.check(_lib.lib().fftm_mi_ffts_create(layout, _lib.i64_array(list(dims)), _lib.F32 if real == "float32" else _lib.F64,
                                              flags, ctypes.byref(h)), "create")
    return h


def _passes(h):
    from fftm_amd import _lib
    n = ctypes.c_int32()
    _lib.check(_lib.lib().fftm_mi_ffts_num_passes(h, ctypes.byref(n), None), "passes")
    return n.value


# a pass per plane takes at most a tenth more than the two passes it replaces: it moves half their
# bytes and does the same arithmetic
@pytest.mark.parametrize("real,dims", [("float64", (52, 11, 44, 39)), ("float64", (42, 15, 66, 26)), ("float64", (11, 25, 60, 22)),
                                       ("float32", (273, 32, 224)), ("float32", (324, 208, 22))])
def test_planes_share_a_cu(gpu, real, dims):
    import torch
    from fftm_amd import _lib
    L = _lib.lib()
    layout = _lib.LAYOUT_3D if len(dims) == 3 else _lib.LAYOUT_4D_SLAB
    n, nc = math.prod(dims), math.prod(dims[:-1]) * (dims[-1] // 2 + 1)
    rdt, cdt = (torch.float32, torch.complex64) if real == "float32" else (torch.float64, torch.complex128)
    u, y = torch.zeros(n, dtype=rdt, device="cuda"), torch.empty(n, dtype=rdt, device="cuda")
    X, W = torch.empty(nc, dtype=cdt, device="cuda"), torch.empty(nc, dtype=cdt, device="cuda")
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    us = {}
    for flags in (0, _lib.FLAG_NO_PLANE_FUSION):
        h = _handle(layout, dims, real, flags)
        assert _passes(h) == len(dims) - (flags == 0)
        _lib.check(L.fftm_mi_ffts_set_work_area(h, W.data_ptr()), "work")
        us[flags] = float("inf")
        for _ in range(9):
            a.record()
            for _ in range(10):
                _lib.check(L.fftm_mi_ffts_forward(h, u.data_ptr(), X.data_ptr(), 0), "forward")
                _lib.check(L.fftm_mi_ffts_backward(h, X.data_ptr(), y.data_ptr(), 0), "backward")
            b.record()
            b.synchronize()
            us[flags] = min(us[flags], a.elapsed_time(b) * 1e2)
        L.fftm_mi_ffts_destroy(h)
    print(f"[tiles] {real} {dims}: per plane {us[0]:.1f} us, per axis {us[_lib.FLAG_NO_PLANE_FUSION]:.1f}", flush=True)
    assert us[0] <= 1.1 * us[_lib.FLAG_NO_PLANE_FUSION]


@pytest.mark.parametrize("dims,passes", [((64, 64, 16, 64), 3), ((50, 48, 60, 39), 4), ((42, 40, 56, 64), 4)])
def test_large_fp32_arrays_take_a_pass_per_axis(gpu, dims, passes):
    from fftm_amd import _lib
    h = _handle(_lib.LAYOUT_4D_SLAB, dims, "float32", 0)
    assert _passes(h) == passes
    _lib.lib().fftm_mi_ffts_destroy(h)

"""Volume pass (a small transform in one workgroup) at its edges: odd row counts and lengths,
axes of one point, radices 11 and 13, several stages per axis, every layout, the largest
volumes; against the oracle, against the pass-per-axis route, adjoints and the filter."""

import ctypes
import math

import numpy as np
import pytest

import oracle
from helpers import check_close, from_gpu, roundtrip_tol, to_gpu
from test_gpu_adjoint import _make

pytestmark = pytest.mark.gpu

CASES = [("3d", (2, 1, 2)), ("3d", (1, 3, 5)), ("3d", (3, 1, 7)), ("3d", (4, 4, 4)), ("3d", (7, 5, 9)),
         ("3d", (13, 11, 26)), ("3d", (16, 16, 18)), ("3d", (17 - 1, 9, 32)), ("3d", (48, 6, 16)), ("3d", (2, 2, 1100)),
         ("3d", (900, 2, 2)), ("pencil", (3, 4, 5, 6)), ("slab", (5, 1, 3, 7)), ("xzwy", (8, 6, 10, 12)),
         ("pencil", (8, 8, 8, 12)), ("slab", (1, 1, 2, 9))]


def _forward(kind, dims, x):
    if kind == "3d":
        return oracle.ffts3d_forward(x)
    if kind == "xzwy":
        return oracle.native_xzwy_forward(x, *dims)
    return oracle.ffts4d_forward(x, kind, *dims)


@pytest.mark.parametrize("real", ["float32", "float64"])
@pytest.mark.parametrize("kind,dims", CASES)
def test_volume(gpu, kind, dims, real):
    import torch
    rdt = np.float32 if real == "float32" else np.float64
    print(f"[volume] {kind} {dims} {real}", flush=True)
    f = _make(kind, dims, real)
    assert f.num_passes() == (1, 1)
    rng = np.random.default_rng(3)
    x = rng.uniform(-1, 1, f.real_shape()).astype(rdt)
    u = to_gpu(x)
    X = f.complex_array().fill_(float("nan"))
    f.forward(u, X)
    check_close(from_gpu(X), _forward(kind, dims, x.astype(np.float64)), rdt, f"volume {kind}{dims} {real}")
    keep = X.clone()
    y = f.real_array().fill_(float("nan"))
    f.backward(X, y)
    n = math.prod(dims)
    assert torch.equal(X, keep)
    assert np.sqrt(np.mean((from_gpu(y).astype(np.float64) / n - x) ** 2)) <= roundtrip_tol(rdt)
    # backward of a spectrum that no real array has, and both adjoints, against the
    # pass-per-axis kernels of the same library (rounding only)
    from fftm_amd import _lib
    L = _lib.lib()
    layout = {"3d": _lib.LAYOUT_3D, "pencil": _lib.LAYOUT_4D_PENCIL, "slab": _lib.LAYOUT_4D_SLAB,
              "xzwy": _lib.LAYOUT_4D_XZWY}[kind]
    h = ctypes.c_void_p()
    _lib.check(L.fftm_mi_ffts_create(layout, _lib.i64_array(list(dims)), _lib.F32 if real == "float32" else _lib.F64,
                                     _lib.FLAG_NO_PLANE_FUSION, ctypes.byref(h)), "create")
    ws = ctypes.c_size_t()
    _lib.check(L.fftm_mi_ffts_get_work_size(h, ctypes.byref(ws)), "work size")
    work = torch.empty(ws.value, dtype=torch.uint8, device="cuda")
    _lib.check(L.fftm_mi_ffts_set_work_area(h, work.data_ptr()), "set work")
    G = to_gpu((rng.standard_normal(f.complex_shape()) + 1j * rng.standard_normal(f.complex_shape())).astype(
        np.complex64 if real == "float32" else np.complex128))
    for mine, call, src, out in ((f.backward, L.fftm_mi_ffts_backward, G, f.real_array()),
                                 (f.r2c_adjoint, L.fftm_mi_ffts_r2c_adjoint, G, f.real_array()),
                                 (f.c2r_adjoint, L.fftm_mi_ffts_c2r_adjoint, u, f.complex_array())):
        ref = torch.empty_like(out)
        mine(src, out)
        _lib.check(call(h, src.data_ptr(), ref.data_ptr(), 1), "per-axis route")
        check_close(from_gpu(out), from_gpu(ref).astype(np.complex128 if out.is_complex() else np.float64), rdt,
                    f"volume against passes {kind}{dims}")
    L.fftm_mi_ffts_destroy(h)
    # the filter is the same three kernels as forward, operator and backward
    v, w = f.real_array(), f.real_array()
    f.filter(u, v, "gaussian", scale=1.0 / n, sigma=2.0)
    f.spectral_apply(X, X, "gaussian", scale=1.0 / n, sigma=2.0)
    f.backward(X, w)
    assert torch.equal(v, w)
    f.close()


def test_volume_sizes(gpu):
    """Above 1536 points per axis count, and without a second axis, the axes keep their passes."""
    for kind, dims, one in (("3d", (16, 16, 18), True), ("3d", (16, 18, 18), False), ("3d", (1, 1, 64), False),
                            ("pencil", (8, 8, 8, 12), True), ("pencil", (8, 8, 8, 13), False)):
        f = _make(kind, dims)
        assert (f.num_passes()[0] == 1) == one, (kind, dims)
        f.close()

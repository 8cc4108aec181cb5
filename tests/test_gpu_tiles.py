"""Planes of the two inner axes in one launch where no plane kernel exists: odd and shortest
lengths, radices 11 and 13, few and many planes, the largest planes, in place; against the
oracle, against the pass-per-axis route of the same library, both adjoints and the filter."""

import ctypes
import math

import numpy as np
import pytest

import oracle
from helpers import check_close, from_gpu, roundtrip_tol, to_gpu
from test_gpu_adjoint import _make

pytestmark = pytest.mark.gpu

CASES = [("3d", (24, 97 - 6, 5)), ("3d", (1200, 2, 2)), ("3d", (33, 13, 22)), ("3d", (24, 7, 300)), ("3d", (100, 60, 48)),
         ("3d", (28, 343, 3)), ("3d", (72, 110, 72)), ("3d", (256, 12, 2)), ("slab", (6, 5, 9, 33)), ("slab", (1, 40, 26, 14)),
         ("slab", (40, 1, 15, 24)), ("slab", (30, 50, 24, 7))]


@pytest.mark.parametrize("real", ["float32", "float64"])
@pytest.mark.parametrize("kind,dims", CASES)
def test_tiles(gpu, kind, dims, real):
    import torch
    from fftm_amd import _lib
    rdt = np.float32 if real == "float32" else np.float64
    print(f"[tiles] {kind} {dims} {real}", flush=True)
    f = _make(kind, dims, real)
    assert f.num_passes() == (len(dims) - 1, len(dims) - 1)
    rng = np.random.default_rng(4)
    x = rng.uniform(-1, 1, f.real_shape()).astype(rdt)
    u = to_gpu(x)
    X = f.complex_array().fill_(float("nan"))
    f.forward(u, X)
    x64 = x.astype(np.float64)
    ref = oracle.ffts3d_forward(x64) if kind == "3d" else oracle.ffts4d_forward(x64, kind, *dims)
    check_close(from_gpu(X), ref, rdt, f"tiles {kind}{dims} {real}")
    keep = X.clone()
    y = f.real_array().fill_(float("nan"))
    f.backward(X, y)
    n = math.prod(dims)
    assert torch.equal(X, keep)
    assert np.sqrt(np.mean((from_gpu(y).astype(np.float64) / n - x) ** 2)) <= roundtrip_tol(rdt)
    L = _lib.lib()
    layout = _lib.LAYOUT_3D if kind == "3d" else _lib.LAYOUT_4D_SLAB
    prec = _lib.F32 if real == "float32" else _lib.F64
    h, o = ctypes.c_void_p(), ctypes.c_void_p()
    _lib.check(L.fftm_mi_ffts_create(layout, _lib.i64_array(list(dims)), prec, _lib.FLAG_NO_PLANE_FUSION, ctypes.byref(h)),
               "create")
    _lib.check(L.fftm_mi_ffts_create(layout, _lib.i64_array(list(dims)), prec, _lib.FLAG_OVERWRITE_INPUT, ctypes.byref(o)),
               "create")
    ws = ctypes.c_size_t()
    _lib.check(L.fftm_mi_ffts_get_work_size(h, ctypes.byref(ws)), "work size")
    work = torch.empty(ws.value, dtype=torch.uint8, device="cuda")
    _lib.check(L.fftm_mi_ffts_set_work_area(h, work.data_ptr()), "set work")
    G = to_gpu((rng.standard_normal(f.complex_shape()) + 1j * rng.standard_normal(f.complex_shape())).astype(
        np.complex64 if real == "float32" else np.complex128))
    for mine, call, src, out in ((f.backward, L.fftm_mi_ffts_backward, G, f.real_array()),
                                 (f.r2c_adjoint, L.fftm_mi_ffts_r2c_adjoint, G, f.real_array()),
                                 (f.c2r_adjoint, L.fftm_mi_ffts_c2r_adjoint, u, f.complex_array())):
        want = torch.empty_like(out)
        mine(src, out)
        _lib.check(call(h, src.data_ptr(), want.data_ptr(), 1), "per-axis route")
        check_close(from_gpu(out), from_gpu(want).astype(np.complex128 if out.is_complex() else np.float64), rdt,
                    f"tiles against passes {kind}{dims}")
    # in place on the spectrum: the same kernels, the same bits
    _lib.check(L.fftm_mi_ffts_backward(o, keep.data_ptr(), (z := torch.empty_like(y)).data_ptr(), 1), "in place")
    assert torch.equal(z, y)
    L.fftm_mi_ffts_destroy(h)
    L.fftm_mi_ffts_destroy(o)
    v, w = f.real_array(), f.real_array()
    f.filter(u, v, "gaussian", scale=1.0 / n, sigma=2.0)
    f.spectral_apply(X, X, "gaussian", scale=1.0 / n, sigma=2.0)
    f.backward(X, w)
    check_close(from_gpu(v), from_gpu(w).astype(np.float64), rdt, f"tiles filter {kind}{dims}")
    f.close()

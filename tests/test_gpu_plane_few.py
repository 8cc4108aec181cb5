"""Plane passes of few planes and on both sides of the thread-count rule: against the
pass-per-axis route (the FP32 / FP64 parity tolerances), and bitwise against the LDS kernel."""

import ctypes
import math

import numpy as np
import pytest

from helpers import check_close, from_gpu
from test_gpu_adjoint import _make

pytestmark = pytest.mark.gpu

CASES = [("3d", (20, 16, 16)), ("3d", (5, 32, 32)), ("3d", (1024, 32, 32)), ("3d", (1040, 32, 32)), ("3d", (2, 64, 64)),
         ("3d", (63, 64, 64)), ("3d", (1024, 64, 64)), ("3d", (1040, 64, 64)), ("3d", (1, 128, 128)), ("3d", (48, 128, 128)),
         ("3d", (256, 128, 128)), ("3d", (260, 128, 128)), ("slab", (2, 5, 32, 32)), ("pencil", (32, 3, 5, 32)),
         ("xzwy", (64, 1, 3, 64))]


@pytest.mark.parametrize("real", ["float32", "float64"])
@pytest.mark.parametrize("kind,dims", CASES)
def test_few_planes(gpu, kind, dims, real):
    import torch
    from fftm_amd import _lib
    rdt = np.float32 if real == "float32" else np.float64
    print(f"[few planes] {kind} {dims} {real}", flush=True)
    f = _make(kind, dims, real)
    fused = len(dims) - 1 if not (real == "float64" and dims == (1, 128, 128)) else len(dims)
    assert f.num_passes() == (fused, fused)
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
    g = torch.Generator(device="cuda").manual_seed(math.prod(dims))
    u = torch.rand(f.real_shape(), generator=g, device="cuda", dtype=f.real) * 2 - 1
    G = torch.complex(*(torch.rand(f.complex_shape(), generator=g, device="cuda", dtype=f.real) - 0.5 for _ in range(2)))
    calls = ((f.forward, L.fftm_mi_ffts_forward, u, f.complex_array()), (f.backward, L.fftm_mi_ffts_backward, G, f.real_array()))
    default = []
    for mine, call, src, out in calls:
        want = torch.empty_like(out)
        mine(src, out.fill_(float("nan")))
        _lib.check(call(h, src.data_ptr(), want.data_ptr(), 1), "per-axis route")
        check_close(from_gpu(out), from_gpu(want).astype(np.complex128 if out.is_complex() else np.float64), rdt,
                    f"few planes {kind}{dims}")
        default.append(out.clone())
    L.fftm_mi_ffts_destroy(h)
    if fused == len(dims) - 1:
        f.set_pass_variant(False, 0, 0)
        f.set_pass_variant(True, fused - 1, 0)
        for (mine, _, src, out), want in zip(calls, default):
            mine(src, out.fill_(float("nan")))
            assert torch.equal(out, want)
    f.close()

"""Tile shapes that untuned passes start with, where arrays of one length take several: the
measured sides of each line (create a handle, read the variant; nothing is transformed)."""

import ctypes

import pytest

pytestmark = pytest.mark.gpu


def _shape(dims, real, backward, index):
    from fftm_amd import _lib
    L = _lib.lib()
    h, v = ctypes.c_void_p(), ctypes.c_int32()
    prec = _lib.F32 if real == "float32" else _lib.F64
    _lib.check(L.fftm_mi_ffts_create(_lib.LAYOUT_3D, _lib.i64_array(list(dims)), prec, _lib.FLAG_NO_PLANE_FUSION,
                                     ctypes.byref(h)), "create")
    try:
        _lib.check(L.fftm_mi_ffts_get_pass_variant(h, backward, index, ctypes.byref(v)), "variant")
    finally:
        L.fftm_mi_ffts_destroy(h)
    return v.value % 8


# split exchange where it is faster (64 MB), the plain shape in small arrays and where the
# memory-side cache is about full (128 MB), twice the rows beyond it
@pytest.mark.parametrize("dims,shape", [((2, 16, 128), 0), ((448, 128, 128), 0), ((640, 128, 128), 6), ((1024, 128, 128), 6),
                                        ((2048, 128, 128), 0), ((3584, 128, 128), 5)])
def test_fp32_r2c_rows_of_128(gpu, dims, shape):
    assert _shape(dims, "float32", 0, 0) == shape

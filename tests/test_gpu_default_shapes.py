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


# full row segments as soon as one round of tiles does not hold the array
@pytest.mark.parametrize("real", ["float32", "float64"])
@pytest.mark.parametrize("n,mb,shape", [(2048, 8, 2), (2048, 16, 2), (2048, 20, 3), (2048, 64, 3), (4096, 12, 2), (4096, 16, 2),
                                        (4096, 24, 3), (4096, 32, 3), (1024, 64, 2)])
def test_long_columns(gpu, n, mb, shape, real):
    columns = (mb << 20) // (n * (8 if real == "float32" else 16))
    assert _shape((n, columns // 8, 14), real, 0, 2) == shape

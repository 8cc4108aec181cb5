"""Tuning records and pass lists: a record names a pass by its index, so one measured on a list
of a pass per axis is not applied to a list in which passes are fused or run another kernel."""

import ctypes

import pytest

from test_gpu_tuning import _make

pytestmark = pytest.mark.gpu


def _signature():
    from fftm_amd import _lib
    buf = ctypes.create_string_buffer(64)
    _lib.check(_lib.lib().fftm_mi_hardware_signature(buf, len(buf)), "signature")
    return buf.value.decode()


# dims, type, passes each way, whether records of the plain keys are of this list
LISTS = [((12, 10, 8), "float64", 1, False),      # one volume pass
         ((32, 64, 64), "float32", 2, False),     # 32 planes
         ((100, 60, 48), "float32", 2, False),    # planes of any lengths
         ((70, 250, 330), "float32", 3, False),   # runtime-length passes
         ((64, 64, 64), "float32", 2, True),      # 64 planes
         ((128, 64, 256), "float32", 3, True)]    # a compiled pass per axis


@pytest.mark.parametrize("dims,dt,passes,plain", LISTS)
def test_records_belong_to_a_pass_list(gpu, tmp_path, dims, dt, passes, plain):
    print(f"case tuning list {dims} {dt}", flush=True)
    f = _make(dims, dt)
    assert f.num_passes() == (passes, passes)
    before = f.pass_variants()
    cache = tmp_path / "plain.cache"
    key = "FFTM_MI_TILE_3D_%dx%dx%d_%s" % (*dims, "F32" if dt == "float32" else "F64")
    lines = ["# FFTM C++ autotune cache", "FFTM_AUTOTUNE_HARDWARE_SIGNATURE=" + _signature()]
    lines += [f"{key}_{d}{i}=8" for d in ("FWD", "BWD") for i in range(3)]
    cache.write_text("\n".join(lines) + "\n")
    assert f.load_tuning(str(cache)) == (2 * passes if plain else 0)
    assert all(v == 8 for v in f.pass_variants().values()) if plain else f.pass_variants() == before
    # its own records are applied
    own = tmp_path / "own.cache"
    chosen = f.autotune(warmup=1, iterations=2, cache_path=str(own))
    g = _make(dims, dt)
    assert g.load_tuning(str(own)) >= 2 * passes
    assert g.pass_variants() == chosen
    f.close()
    g.close()

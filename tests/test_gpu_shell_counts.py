"""The shell operators' time does not grow with the number of shells: a bin's shell is found in a
constant number of steps.  128^3 bins take microseconds either way; 1024 shells add the partial
sums of 512 blocks (4 MB written and read, 2 us) and a longer table, so twice the time with 8
shells, and 2 us for the launches' own spread, bound them."""

import pytest

pytestmark = pytest.mark.gpu


def _us(fn, reps=9, calls=20):
    import torch
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for _ in range(3):
        fn()
    best = float("inf")
    for _ in range(reps):
        a.record()
        for _ in range(calls):
            fn()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / calls)
    return best


@pytest.mark.parametrize("real", ["float32", "float64"])
@pytest.mark.parametrize("dims", [(128, 128, 128), (192, 160, 144), (32, 24, 20)])
def test_time_of_many_shells(gpu, dims, real):
    import torch
    import fftm_amd
    f = fftm_amd.ffts(real)
    f.init(*dims, options=fftm_amd.ffts_init_options(profiling_key="", memory_profiling_key="", sync=False))
    f.set_stream(torch.cuda.current_stream())
    X = torch.zeros_like(f.complex_array())
    out = torch.empty_like(X)
    t = {}
    for shells in (8, 100, 1024):
        c = torch.ones(shells, device="cuda", dtype=f.real)
        t[shells] = (_us(lambda: f.spectral_multiply(X, out, shell_coeffs=c)),
                     _us(lambda: f.shell_gradient(X, X, shells)))
    print(f"[shells] {dims} {real} us (multiply, gradient) " + str(t), flush=True)
    for shells in (100, 1024):
        for few, many in zip(t[8], t[shells]):
            assert many <= 2 * few + 2
    f.close()

"""Runtime-length passes (lengths without a compiled kernel): every radix, one to five
stages, rows, columns and row-to-column plans, odd batches, against numpy in 64 bits.
Tolerances are the parity ones of ``helpers`` (FP32 2e-6 / 1e-5, FP64 1e-12)."""

import ctypes

import numpy as np
import pytest

from helpers import check_close, from_gpu, to_gpu

# compiled lengths that take the runtime kernel in some kind, direction or precision (12, 20, 24,
# 48, 56, 72, 100, 120, 144, 224, 240, 288, 400, 480, 576, 1000, 1152, 1680, 1920) and others; 1..15: single stages; 3125 = 5^5 five stages; primes 11 and 13 alone, squared and cubed;
# the largest lengths each precision takes
LENGTHS = [1, 3, 6, 7, 9, 11, 12, 13, 14, 15, 18, 20, 22, 24, 26, 39, 45, 48, 56, 72, 99, 100, 120, 125, 143, 144, 169, 175,
           224, 234, 240, 250, 288, 330, 343, 400, 420, 480, 576, 625, 720, 1000, 1001, 1080, 1152, 1331, 1680, 1920, 2016, 2197, 3125, 3993, 4004, 4095]
MAX_LENGTH = {"float32": 4096, "float64": 2048}


def _smooth(n):
    for p in (2, 3, 5, 7, 11, 13):
        while n % p == 0:
            n //= p
    return n == 1


@pytest.mark.parametrize("real", ["float32", "float64"])
def test_accepted_lengths(real):
    """13-smooth lengths up to the single-pass limit are accepted, in both line directions
    and for every kind; others are refused (host check, no GPU)."""
    from fftm_amd import _lib
    L = _lib.lib()
    for n in range(1, 4200):
        want = _smooth(n) and (n <= MAX_LENGTH[real] or n == 2100 or n == 4096)
        for d in (1, 2, 3):
            for rows in (True, False):
                desc = _lib.PlanDesc()
                desc.dir, desc.precision = d, _lib.F32 if real == "float32" else _lib.F64
                desc.rank, desc.batch = 1, 6
                desc.n[0] = desc.inembed[0] = desc.onembed[0] = n
                desc.istride = desc.ostride = 1 if rows else 6
                desc.idist = desc.odist = n if rows else 1
                assert (L.fftm_mi_plan_validate(ctypes.byref(desc), None) == 0) == want, (n, d, rows)


def _lay(a, rows):
    """(batch, n) -> memory of the plan: rows as they are, columns transposed."""
    return np.ascontiguousarray(a if rows else a.T)


@pytest.mark.gpu
@pytest.mark.parametrize("real", ["float32", "float64"])
@pytest.mark.parametrize("n", LENGTHS)
def test_lengths(gpu, n, real):
    import fftm_amd
    D = fftm_amd.direction
    if n > MAX_LENGTH[real]:
        pytest.skip("longer than this precision's single-pass limit")
    rdt, cdt = (np.float32, np.complex64) if real == "float32" else (np.float64, np.complex128)
    nh = n // 2 + 1
    rng = np.random.default_rng(n)
    # odd batch: the last real line has no partner; 37 lines: a ragged last tile
    for batch, irows, orows in ((37, True, True), (37, False, False), (37, True, False), (18, False, True), (1, True, True)):
        print(f"[any] {real} n={n} batch={batch} rows {irows}->{orows}", flush=True)
        st = lambda m, rows: ([m], 1, m) if rows else ([m], batch, 1)
        z = (rng.uniform(-1, 1, (batch, n)) + 1j * rng.uniform(-1, 1, (batch, n))).astype(cdt)
        x = rng.uniform(-1, 1, (batch, n)).astype(rdt)
        half = np.fft.rfft(x.astype(np.float64), axis=1).astype(cdt)
        half[:, 0] += 0.5j  # ignored, as numpy's irfft ignores it
        full = z.astype(np.complex128)
        cases = [(D.C2CF, z, n, n, np.fft.fft(full, axis=1), cdt), (D.C2CB, z, n, n, np.fft.ifft(full, axis=1) * n, cdt),
                 (D.R2C, x, n, nh, np.fft.rfft(x.astype(np.float64), axis=1), cdt),
                 (D.C2R, half, nh, n, np.fft.irfft(half.astype(np.complex128), n=n, axis=1) * n, rdt)]
        for d, a, mi, mo, ref, odt in cases:
            plan = fftm_amd.fft(real, d, [n], *st(mi, irows), *st(mo, orows), batch)
            src = to_gpu(_lay(a, irows))
            out = to_gpu(_lay(np.full((batch, mo), np.nan, odt), orows))
            plan.exec(src, out)
            got = from_gpu(out)
            check_close(got if orows else got.T, ref, rdt, f"{d.name} n={n} {real}")
            if d in (D.C2CF, D.C2CB) and irows == orows:
                plan.exec(src, src)  # in place
                assert np.array_equal(from_gpu(src), got)
            plan.destroy()

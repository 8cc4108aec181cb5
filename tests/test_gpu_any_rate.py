"""Runtime-length passes take about the time of their neighbours: the same values in lines of
another length move the same bytes and need at most one LDS exchange more."""

import pytest

pytestmark = pytest.mark.gpu


def _pass_us(n, kind, rows, lines, real, reps=7, calls=10):
    """One 1D pass over `lines` lines of n points, microseconds."""
    import torch
    import fftm_amd
    D = fftm_amd.direction
    d = {"c2c": D.C2CF, "r2c": D.R2C, "c2r": D.C2R}[kind]
    nh = n // 2 + 1
    mi, mo = (nh if kind == "c2r" else n), (nh if kind == "r2c" else n)
    plans = fftm_amd.fft_wrap_many(real)
    if rows:
        plans.add_plan_1D(d, "p", n, mi, 1, mi, mo, 1, mo, lines)
    else:
        plans.add_plan_1D(d, "p", n, mi, lines, 1, mo, lines, 1, lines)
    plans.activate()
    plans.set_stream("p", torch.cuda.current_stream())
    rdt = torch.float32 if real == "float32" else torch.float64
    cdt = torch.complex64 if real == "float32" else torch.complex128
    x = torch.zeros(lines * mi, dtype=rdt if kind == "r2c" else cdt, device="cuda")
    y = torch.empty(lines * mo, dtype=rdt if kind == "c2r" else cdt, device="cuda")
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    for _ in range(3):
        plans.exec_named_no_sync("p", x, y)
    best = float("inf")
    for _ in range(reps):
        a.record()
        for _ in range(calls):
            plans.exec_named_no_sync("p", x, y)
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 1e3 / calls)
    return best


# 1440 = 10 8 6 3 is four stages, as every length here at most; a stage is under a third of the
# time that the memory takes: 1.4 holds for any of them that is not short of wavefronts
@pytest.mark.parametrize("kind", ["c2c", "r2c", "c2r"])
@pytest.mark.parametrize("n", [1350, 1500, 1575, 1960, 2016])
def test_long_fp64_rows(gpu, n, kind):
    values = 1 << 22
    ref = _pass_us(1440, kind, True, values // 1440, "float64")
    got = _pass_us(n, kind, True, values // n, "float64")
    print(f"[rate] fp64 {kind} rows of {n}: {got:.1f} us, of 1440: {ref:.1f}", flush=True)
    assert got <= 1.4 * ref


# arrays of at most 2^19 values lie in the L2 caches: strided lines cost address arithmetic, no
# more than a third of such a pass
@pytest.mark.parametrize("kind", ["r2c", "c2r"])
@pytest.mark.parametrize("n,lines", [(1029, 31), (1029, 180), (1080, 171), (1125, 164)])
def test_few_real_columns(gpu, n, lines, kind):
    ref = _pass_us(n, kind, True, lines, "float32")
    got = _pass_us(n, kind, False, lines, "float32")
    print(f"[rate] fp32 {kind} {lines} columns of {n}: {got:.1f} us, rows: {ref:.1f}", flush=True)
    assert got <= 1.4 * ref


# the same bytes the other way, and one trip through LDS more
@pytest.mark.parametrize("n,lines,rows", [(14, 13240, True), (14, 22267, True), (15, 12357, True), (14, 22267, False),
                                          (15, 20782, False)])
def test_short_c2r_lines(gpu, n, lines, rows):
    ref = _pass_us(n, "r2c", rows, lines, "float32")
    got = _pass_us(n, "c2r", rows, lines, "float32")
    print(f"[rate] fp32 {lines} lines of {n}: c2r {got:.1f} us, r2c: {ref:.1f}", flush=True)
    assert got <= 1.4 * ref

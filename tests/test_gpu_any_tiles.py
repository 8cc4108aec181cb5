"""Runtime-length passes in the tiles that large arrays take (the tile grows with the number of
lines): every line of 2^21 values, both mappings of loads and stores, a ragged last tile, a
last real line without a partner, and plans of two batch dimensions.  Tolerances are the parity
ones of ``helpers``."""

import numpy as np
import pytest

from helpers import TOL_REL_L2, TOL_REL_MAX, check_close, from_gpu, to_gpu

pytestmark = pytest.mark.gpu

# one to five stages (12: compiled, but for rows of this many values); all radices resident (45, 250, 1000), radices 11 and 13 (330, 780, 1331),
# the table in memory (from 1025 points in FP64, 2049 in FP32); 5..25: C2R columns whose threads
# are no multiple of the tile's lines
LENGTHS = {"float32": [5, 12, 14, 18, 45, 100, 250, 330, 1000, 1080, 1331, 2401, 3125, 4004],
           "float64": [5, 14, 25, 45, 100, 250, 330, 780, 1000, 1080, 1331, 1500, 1960]}
DISTINCT = 89  # input lines repeat with this period: no tile or XCD chunk has it as a size


def _whole(got, ref, rdt, what):
    """All lines of got (on the GPU) against the reference of the line modulo DISTINCT."""
    import torch
    r = torch.from_numpy(np.ascontiguousarray(ref)).cuda()
    worst, num, den = 0.0, 0.0, 0.0
    for i in range(0, got.shape[0], DISTINCT):
        g = got[i:i + DISTINCT]
        d = (g.to(r.dtype) - r[: g.shape[0]]).abs()
        assert bool(torch.isfinite(d).all()), f"{what}: line {i}.. not written"
        worst = max(worst, float(d.max()))
        num += float((d * d).sum())
        den += float((r[: g.shape[0]].abs() ** 2).sum())
    l2, mx = (num / den) ** 0.5, worst / float(r.abs().max())
    print(f"[tiles] {what}: rel_l2={l2:.2e} rel_max={mx:.2e}", flush=True)
    assert l2 <= TOL_REL_L2[rdt] and mx <= TOL_REL_MAX[rdt], what


@pytest.mark.parametrize("real,n", [(r, n) for r in LENGTHS for n in LENGTHS[r]])
def test_full_tiles(gpu, real, n):
    import torch
    import fftm_amd
    D = fftm_amd.direction
    rdt, cdt = (np.float32, np.complex64) if real == "float32" else (np.float64, np.complex128)
    lines, nh = (1 << 21) // n | 1, n // 2 + 1
    rng = np.random.default_rng(n)
    z = (rng.uniform(-1, 1, (DISTINCT, n)) + 1j * rng.uniform(-1, 1, (DISTINCT, n))).astype(cdt)
    x = rng.uniform(-1, 1, (DISTINCT, n)).astype(rdt)
    half = np.fft.rfft(x.astype(np.float64), axis=1).astype(cdt)
    cases = [(D.C2CF, z, n, n, np.fft.fft(z.astype(np.complex128), axis=1), cdt),
             (D.C2CB, z, n, n, np.fft.ifft(z.astype(np.complex128), axis=1) * n, cdt),
             (D.R2C, x, n, nh, np.fft.rfft(x.astype(np.float64), axis=1), cdt),
             (D.C2R, half, nh, n, np.fft.irfft(half.astype(np.complex128), n=n, axis=1) * n, rdt)]
    which = torch.arange(lines, device="cuda") % DISTINCT
    st = lambda m, rows: ([m], 1, m) if rows else ([m], lines, 1)
    for d, a, mi, mo, ref, odt in cases:
        base = to_gpu(a)[which]
        for irows, orows in ((True, True), (False, False), (True, False), (False, True)):
            print(f"[tiles] {real} n={n} {d.name} lines={lines} rows {irows}->{orows}", flush=True)
            plan = fftm_amd.fft(real, d, [n], *st(mi, irows), *st(mo, orows), lines)
            src = base if irows else base.T.contiguous()
            out = torch.full((lines, mo) if orows else (mo, lines), float("nan"), device="cuda",
                             dtype=to_gpu(np.zeros(1, odt)).dtype)
            plan.exec(src, out)
            _whole(out if orows else out.T, ref, rdt, f"{d.name} n={n} {real} rows {irows}->{orows}")
            plan.destroy()


@pytest.mark.parametrize("real", ["float32", "float64"])
@pytest.mark.parametrize("dims,batch", [((60, 330, 22), 5), ((26, 45, 250), 7)])
def test_two_batch_dimensions(gpu, dims, batch, real):
    """The middle axis of a rank-3 plan: columns over two batch dimensions and the batch."""
    import fftm_amd
    D = fftm_amd.direction
    rdt, cdt = (np.float32, np.complex64) if real == "float32" else (np.float64, np.complex128)
    rng = np.random.default_rng(5)
    x = rng.uniform(-1, 1, (batch, *dims)).astype(rdt)
    z = (x + 1j * rng.uniform(-1, 1, x.shape)).astype(cdt)
    for d, a, ref in ((D.C2CF, z, np.fft.fftn(z.astype(np.complex128), axes=(1, 2, 3))),
                      (D.R2C, x, np.fft.rfftn(x.astype(np.float64), axes=(1, 2, 3)))):
        plan = fftm_amd.fft(real, d, list(dims), batch=batch)
        out = to_gpu(np.full(ref.shape, np.nan, cdt))
        plan.exec(to_gpu(a), out)
        check_close(from_gpu(out), ref, rdt, f"{d.name} {dims}x{batch} {real}")
        plan.destroy()

"""C2R rows: the tile copied straight into LDS where the rows are dense and aligned against
the general loads (padded pitch, unaligned base): bitwise equal, ragged last tiles included."""

import numpy as np
import pytest

import fftm_amd
from helpers import from_gpu, torch_dtypes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("real", ["float32", "float64"])
@pytest.mark.parametrize("n", [2, 16, 64, 99, 100, 128, 144, 240, 256, 330, 512, 1000, 1024, 2048])
def test_dense_rows_equal_padded_rows(gpu, n, real):
    import torch
    rdt, cdt = torch_dtypes(np.float32 if real == "float32" else np.float64)
    nh = n // 2 + 1
    rng = np.random.default_rng(n)
    for batch in (1, 2, 37, 300):
        print(f"[dense] {real} n={n} batch={batch}", flush=True)
        X = torch.from_numpy(rng.uniform(-1, 1, (batch, nh)) + 1j * rng.uniform(-1, 1, (batch, nh))).to(cdt).cuda()
        want = np.fft.irfft(from_gpu(X).astype(np.complex128), n=n, axis=1) * n
        outs = []
        for pitch, shift in ((nh, 0), (nh + 1, 0), (nh, 1)):
            store = torch.zeros(batch * pitch + shift, dtype=cdt, device="cuda")
            src = store[shift:].view(batch, pitch)
            src[:, :nh] = X
            out = torch.full((batch, n), float("nan"), dtype=rdt, device="cuda")
            plan = fftm_amd.fft(real, fftm_amd.direction.C2R, [n], [pitch], 1, pitch, [n], 1, n, batch)
            plan.exec(src.data_ptr(), out)
            plan.destroy()
            outs.append(from_gpu(out))
        assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
        eps = np.finfo(outs[0].dtype).eps
        assert np.max(np.abs(outs[0] - want)) <= 20 * eps * np.max(np.abs(want))

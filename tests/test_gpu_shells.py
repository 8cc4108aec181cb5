"""Radial shell indices against exact integer square roots: every bin of arrays whose shell
boundaries fall on integer |k|^2, one to 1024 shells, the longest axes."""

import math

import numpy as np
import pytest

from test_gpu_adjoint import _make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("real", ["float32", "float64"])
@pytest.mark.parametrize("dims", [(6, 6, 6), (32, 32, 32), (7, 45, 12), (4096, 2, 2), (2, 3, 2048), (512, 8, 512)])
@pytest.mark.parametrize("shells", [1, 3, 32, 100, 1023, 1024])
def test_shell_index(gpu, dims, shells, real):
    import torch
    if real == "float64" and max(dims) > 2048:
        pytest.skip("longer than the double-precision single-pass limit")
    f = _make("3d", dims, real)
    k2 = sum(np.minimum(i, n - i) ** 2 for i, n in zip(np.ogrid[tuple(slice(n) for n in dims)], dims))
    k2 = k2[..., : dims[2] // 2 + 1].astype(np.int64)
    kmax2 = sum((n // 2) ** 2 for n in dims)
    table = np.array([min(shells - 1, math.isqrt(shells * shells * k // kmax2)) for k in range(kmax2 + 1)])
    c = torch.arange(1, shells + 1, device="cuda", dtype=f.real)
    X = torch.ones_like(f.complex_array())
    out = torch.empty_like(X)
    f.spectral_apply(X, out, "shell", scale=1.0, coeffs=c)
    got = out.cpu().numpy()
    assert np.array_equal(got.real, (table[k2] + 1).astype(got.real.dtype))
    assert not got.imag.any()
    f.close()

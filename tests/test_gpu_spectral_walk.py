"""Shell multiply, shell gradient and analytic operators at the edges of their row walk:
rows longer than a block, single rows, more rows than one sweep covers, extents of 1 and
2, up to 1024 shells."""

import numpy as np
import pytest

import oracle
from helpers import from_gpu, to_gpu
from test_gpu_adjoint import _logical_to_spec_mem, _make

pytestmark = pytest.mark.gpu

CASES = [("3d", (2, 2, 2), 1), ("3d", (3, 2, 4096), 7), ("3d", (1, 1, 2048), 1024), ("3d", (260, 130, 66), 100),
         ("pencil", (1000, 3, 4, 6), 33), ("pencil", (2, 128, 130, 130), 64), ("slab", (5, 12, 33, 40), 1024),
         ("xzwy", (40, 7, 9, 15), 5)]


@pytest.mark.parametrize("kind,dims,S", CASES)
@pytest.mark.parametrize("real", ["float32", "float64"])
def test_row_walk_edges(gpu, kind, dims, S, real):
    print(f"[walk] {kind} {dims} S={S} {real}", flush=True)
    f = _make(kind, dims, real)
    rdt, cdt = (np.float32, np.complex64) if real == "float32" else (np.float64, np.complex128)
    g = np.random.default_rng(7)
    X = (g.standard_normal(f.complex_shape()) + 1j * g.standard_normal(f.complex_shape())).astype(cdt)
    G = (g.standard_normal(f.complex_shape()) + 1j * g.standard_normal(f.complex_shape())).astype(cdt)
    coeffs = g.uniform(0.5, 1.5, S).astype(rdt)
    shell = _logical_to_spec_mem(kind, oracle.shell_index_logical(dims, S))
    out = f.complex_array()
    f.spectral_multiply(to_gpu(X), out, shell_coeffs=to_gpu(coeffs))
    assert np.array_equal(from_gpu(out), (X * coeffs[shell]).astype(cdt))
    Z = to_gpu(X)
    f.spectral_multiply(Z, Z, shell_coeffs=to_gpu(coeffs))  # in place
    assert np.array_equal(from_gpu(Z), (X * coeffs[shell]).astype(cdt))
    f.spectral_apply(to_gpu(X), out, "shell", coeffs=to_gpu(coeffs))
    assert np.array_equal(from_gpu(out), (X * coeffs[shell]).astype(cdt))
    # derivative along every axis: i k z, the product exact up to one rounding
    for axis in range(len(dims)):
        f.spectral_apply(to_gpu(X), out, "derivative", axis=axis)
        n = dims[axis]
        m = n // 2 + 1 if axis == len(dims) - 1 else n
        k = np.arange(m)
        if axis < len(dims) - 1:
            k = np.where(k <= n // 2, k, k - n)
        shape = [-1 if a == axis else 1 for a in range(len(dims))]
        logical = tuple(list(dims[:-1]) + [dims[-1] // 2 + 1])
        km = _logical_to_spec_mem(kind, np.broadcast_to(k.reshape(shape), logical)).astype(rdt)
        got = from_gpu(out)
        assert np.array_equal(got.real, -X.imag * km) and np.array_equal(got.imag, X.real * km)
    # gradient: a sum of n FP64 terms in some order is within n eps64 sum|terms|, then one
    # rounding to the result type
    v = G.real.astype(np.float64) * X.real + G.imag.astype(np.float64) * X.imag
    ref = np.bincount(shell.reshape(-1), weights=v.reshape(-1), minlength=S)
    mag = np.bincount(shell.reshape(-1), weights=np.abs(v).reshape(-1), minlength=S)
    got = from_gpu(f.shell_gradient(to_gpu(G), to_gpu(X), S)).astype(np.float64)
    bound = 2.0 * v.size * np.finfo(np.float64).eps * mag + np.finfo(rdt).eps * np.abs(ref)
    assert np.all(np.abs(got - ref) <= bound)

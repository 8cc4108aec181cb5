"""Workloads whose speed and results matter to a user of this library, as measurable cases.

Every case goes through the public Python entry points (``fftm_amd.ffts``,
``fftm_amd.fft_wrap_many``, ``fftm_amd.autograd.spectral_filter``) the way a program
that owns its arrays calls them: plans and work areas exist, the calls are asynchronous
on the caller's stream, nothing is tuned beforehand.

``listed()`` are the fixed cases, ``draw(rng)`` gives another one of the same ranges,
``prepare`` / ``run`` execute one, ``work`` is its minimal data movement and arithmetic
and ``exact`` the result in 64-bit arithmetic from torch / numpy alone.
"""

import math

import numpy as np
import torch

import fftm_amd
from fftm_amd.autograd import spectral_filter

# Transform lengths need prime factors up to 13.
_PRIMES = (2, 3, 5, 7, 11, 13)


def listed():
    return [
        # The smallest calls (the size of the reference's smoke test): launches and
        # latency are everything.
        {"name": "small_12x10x8_f64", "kind": "pair", "layout": "3d", "dims": "12x10x8", "dtype": "float64",
         "storage": "fp32"},
        # The ordinary double-precision round trip of a simulation code, 128^3.
        {"name": "cube_128_f64", "kind": "pair", "layout": "3d", "dims": "128x128x128", "dtype": "float64",
         "storage": "fp32"},
        # The headline throughput workload, 512^3 single precision.
        {"name": "cube_512_f32", "kind": "pair", "layout": "3d", "dims": "512x512x512", "dtype": "float32",
         "storage": "fp32"},
        # A measured volume: lengths are what the instrument gave, one of them odd.
        {"name": "ragged_175x250x330_f32", "kind": "pair", "layout": "3d", "dims": "175x250x330",
         "dtype": "float32", "storage": "fp32"},
        # Spectra kept in 16 bits between the passes, the reduced-traffic option.
        {"name": "cube_256_fp16_stored", "kind": "pair", "layout": "3d", "dims": "256x256x256",
         "dtype": "float32", "storage": "fp16"},
        # Space-time field in the pencil layout, 64^4.
        {"name": "pencil_64_f32", "kind": "pair", "layout": "4d_pencil", "dims": "64x64x64x64",
         "dtype": "float32", "storage": "fp32"},
        # Space-time field in the slab layout, unequal extents, double precision.
        {"name": "slab_36x30x40x24_f64", "kind": "pair", "layout": "4d_slab", "dims": "36x30x40x24",
         "dtype": "float64", "storage": "fp32"},
        # One image-sized 2D transform pair.
        {"name": "image_1080x1920_f32", "kind": "pair", "layout": "2d", "dims": "1080x1920",
         "dtype": "float32", "storage": "fp32"},
        # Periodic Poisson solve, real field to real field in one call.
        {"name": "poisson_512_f32", "kind": "filter", "op": "poisson", "layout": "3d", "dims": "512x512x512",
         "dtype": "float32"},
        # Gradient of a double-precision field by spectral derivatives (forward, three
        # derivatives, three backward transforms), as in a pseudo-spectral solver's step.
        {"name": "gradient_192x160x144_f64", "kind": "gradient", "layout": "3d", "dims": "192x160x144",
         "dtype": "float64"},
        # Training step of a radial spectral filter: loss, gradients with respect to the
        # field and to 32 shell coefficients.
        {"name": "loss_256_f32", "kind": "loss", "layout": "3d", "dims": "256x256x256", "dtype": "float32",
         "nshells": 32},
        # A batch of 1D complex signals through named plans, forward and inverse.
        {"name": "signals_1000x4096_f32", "kind": "signals", "dims": "1000x4096", "order": "rows",
         "dtype": "float32"},
    ]


# ---------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------
def _smooth(n):
    for p in _PRIMES:
        while n % p == 0:
            n //= p
    return n == 1


def _length(rng, lo, hi, style):
    """A transform length in [lo, hi], spread over the logarithm: a power of two, an even
    length of small factors, or any supported length (odd ones among them)."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    if style == "pow2":
        n = 1 << int(round(math.log2(v)))
        return max(lo, min(hi, n))
    n = max(lo, min(hi, int(round(v))))
    if style == "even":
        ok = [m for m in range(lo, hi + 1) if m % 2 == 0 and m // 2 and _smooth(m) and m % 11 and m % 13]
    else:
        ok = [m for m in range(lo, hi + 1) if _smooth(m)]
    return min(ok, key=lambda m: (abs(m - n), m))


def _lengths(rng, count, lo, hi, limit, styles=("pow2", "even", "any")):
    style = rng.choice(styles)
    while True:
        dims = [_length(rng, lo, hi, style) for _ in range(count)]
        if math.prod(dims) <= limit:
            return "x".join(str(n) for n in dims)


def draw(rng):
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        case = _draw(rng)
        if case not in known:
            return case


def _draw(rng):
    family = rng.choice(["small", "volume", "volume", "fp16", "field4d", "image", "filter", "gradient", "loss",
                         "signals"])
    dtype = rng.choice(["float32", "float64"])
    if family == "small":
        return {"kind": "pair", "layout": "3d", "dims": _lengths(rng, 3, 4, 32, 1 << 15), "dtype": dtype,
                "storage": "fp32"}
    if family == "volume":
        return {"kind": "pair", "layout": "3d", "dims": _lengths(rng, 3, 24, 512, 1 << 23), "dtype": dtype,
                "storage": "fp32"}
    if family == "fp16":
        return {"kind": "pair", "layout": "3d", "dims": _lengths(rng, 3, 128, 1024, 1 << 25, ("pow2",)),
                "dtype": "float32", "storage": "fp16"}
    if family == "field4d":
        return {"kind": "pair", "layout": rng.choice(["4d_pencil", "4d_slab", "4d_xzwy"]),
                "dims": _lengths(rng, 4, 6, 72, 1 << 22), "dtype": dtype, "storage": "fp32"}
    if family == "image":
        return {"kind": "pair", "layout": "2d", "dims": _lengths(rng, 2, 64, 2048, 1 << 22), "dtype": dtype,
                "storage": "fp32"}
    if family == "filter":
        layout = rng.choice(["3d", "3d", "4d_pencil", "4d_slab"])
        dims = _lengths(rng, 3, 24, 384, 1 << 23) if layout == "3d" else _lengths(rng, 4, 6, 64, 1 << 22)
        return {"kind": "filter", "op": rng.choice(["poisson", "gaussian"]), "layout": layout, "dims": dims,
                "dtype": dtype}
    if family == "gradient":
        return {"kind": "gradient", "layout": "3d", "dims": _lengths(rng, 3, 24, 256, 1 << 22), "dtype": dtype}
    if family == "loss":
        return {"kind": "loss", "layout": "3d", "dims": _lengths(rng, 3, 24, 256, 1 << 23), "dtype": "float32",
                "nshells": rng.choice([8, 16, 32, 64, 100])}
    n = _length(rng, 16, 2100, rng.choice(["pow2", "even", "any"]))
    batch = max(1, int(math.exp(rng.uniform(math.log(1 << 10), math.log(1 << 22))) / n))
    return {"kind": "signals", "dims": f"{n}x{batch}", "order": rng.choice(["rows", "columns"]), "dtype": dtype}


# ---------------------------------------------------------------------------
# running a case
# ---------------------------------------------------------------------------
def _dims(case):
    return [int(n) for n in case["dims"].split("x")]


def _types(case):
    return {"float32": (torch.float32, torch.complex64), "float64": (torch.float64, torch.complex128)}[case["dtype"]]


def _uniform(shape, real, seed, stream=0):
    g = torch.Generator(device="cuda").manual_seed(seed * 8 + stream)
    return torch.rand(shape, generator=g, device="cuda", dtype=real) * 2 - 1


def _real_shape(case):
    d = _dims(case)
    return tuple(reversed(d)) if case.get("layout") == "4d_pencil" else tuple(d)


_STRATEGY = {"4d_pencil": fftm_amd.strategy_4d_pencil_pencil, "4d_slab": fftm_amd.strategy_4d_slab_slab,
             "4d_xzwy": fftm_amd.strategy_4d_slab_native_xzwy}


def _transform(case):
    strategy = _STRATEGY[case["layout"]]() if case["layout"] in _STRATEGY else None
    f = fftm_amd.ffts(case["dtype"], strategy)
    f.init(*_dims(case), options=fftm_amd.ffts_init_options(
        profiling_key="", memory_profiling_key="", sync=False, spectrum_storage=case.get("storage", "fp32")))
    f.set_stream(torch.cuda.current_stream())
    return f


def prepare(case, seed):
    real, cplx = _types(case)
    kind = case["kind"]
    if kind == "signals":
        n, batch = _dims(case)
        plans = fftm_amd.fft_wrap_many(real)
        shape = (batch, n) if case["order"] == "rows" else (n, batch)
        stride, dist = (1, n) if case["order"] == "rows" else (batch, 1)
        for name, direction in (("forward", fftm_amd.direction.C2CF), ("inverse", fftm_amd.direction.C2CB)):
            plans.add_plan_1D(direction, name, n, n, stride, dist, n, stride, dist, batch)
        plans.activate()
        for name in ("forward", "inverse"):
            plans.set_stream(name, torch.cuda.current_stream())
        z = torch.complex(_uniform(shape, real, seed), _uniform(shape, real, seed, 1))
        return {"kind": kind, "plans": plans, "z": z, "Z": torch.empty_like(z), "y": torch.empty_like(z)}
    f = _transform(case)
    s = {"kind": kind, "f": f, "u": _uniform(_real_shape(case), real, seed), "n": math.prod(_dims(case))}
    if kind == "pair":
        s.update(X=f.complex_array(), y=f.real_array())
    elif kind == "filter":
        s.update(op=case["op"], v=f.real_array())
    elif kind == "gradient":
        s.update(X=f.complex_array(), D=f.complex_array(), g=[f.real_array() for _ in range(3)])
    elif kind == "loss":
        s["u"].requires_grad_(True)
        s["c"] = _coefficients(case, seed).requires_grad_(True)
        s["target"] = _uniform(_real_shape(case), real, seed, 2)
    return s


def _coefficients(case, seed):
    # filter values around 1, with the 1/N of the unnormalised transforms folded in
    c = _uniform((case["nshells"],), _types(case)[0], seed, 1)
    return (1 + 0.5 * c) / math.prod(_dims(case))


_SIGMA = 8.0  # width of the Gaussian low-pass, in wavenumbers


def run(s):
    if s["kind"] == "signals":
        s["plans"].exec_named_no_sync("forward", s["z"], s["Z"])
        s["plans"].exec_named_no_sync("inverse", s["Z"], s["y"])
        return [s["Z"], s["y"]]
    f = s["f"]
    if s["kind"] == "pair":
        f.forward(s["u"], s["X"])
        f.backward(s["X"], s["y"])
        return [s["X"], s["y"]]
    if s["kind"] == "filter":
        sigma = _SIGMA if s["op"] == "gaussian" else None
        f.filter(s["u"], s["v"], s["op"], scale=1.0 / s["n"], sigma=sigma)
        return s["v"]
    if s["kind"] == "gradient":
        f.forward(s["u"], s["X"])
        for axis in range(3):
            f.spectral_apply(s["X"], s["D"], "derivative", scale=1.0 / s["n"], axis=axis)
            f.backward(s["D"], s["g"][axis])
        return [s["X"]] + s["g"]
    u, c = s["u"], s["c"]
    u.grad = None
    c.grad = None
    v = spectral_filter(u, c, f)
    loss = ((v - s["target"]) ** 2).sum()
    loss.backward()
    return [loss.detach(), u.grad, c.grad]


def work(case):
    """One pass: every input read once, every output written once; 2.5 N log2 N per real
    transform, 5 N log2 N per complex one."""
    d = _dims(case)
    n = math.prod(d)
    rsz = _types(case)[0].itemsize
    if case["kind"] == "signals":
        return {"bytes": 4 * n * 2 * rsz, "flops": 2 * 5 * n * math.log2(max(d[0], 2))}
    one = 2.5 * n * math.log2(max(n, 2))
    spectrum = n // d[-1] * (d[-1] // 2 + 1) * 2 * rsz
    field = n * rsz
    if case["kind"] == "pair":
        return {"bytes": 2 * (field + spectrum), "flops": 2 * one}
    if case["kind"] == "filter":
        return {"bytes": 2 * field, "flops": 2 * one}
    if case["kind"] == "gradient":
        return {"bytes": 4 * field + spectrum, "flops": 4 * one}
    return {"bytes": 3 * field, "flops": 5 * one}


# ---------------------------------------------------------------------------
# results in 64-bit arithmetic
# ---------------------------------------------------------------------------
# Double-precision transforms are compared against extended precision where that is
# affordable on the host (an FP64 reference would be no better than the result).
_HOST_LIMIT = 1 << 23


def _rfftn(u, wide):
    if wide:
        return np.fft.rfftn(u)
    return torch.fft.rfftn(u)


def _irfftn(S, n_last, wide):
    """Normalised inverse over the logical axes; the imaginary parts of the last axis's DC
    and Nyquist bins are ignored, as numpy's irfft does."""
    lead = tuple(range(S.ndim - 1))
    if wide:
        return np.fft.irfft(np.fft.ifftn(S, axes=lead), n=n_last, axis=-1)
    T = torch.fft.ifftn(S, dim=lead)
    T[..., 0] = T[..., 0].real.to(T.dtype)
    if n_last % 2 == 0:
        T[..., -1] = T[..., -1].real.to(T.dtype)
    return torch.fft.irfft(T, n=n_last, dim=-1)


def _axis_k(dims, axis, wide):
    """Integer wavenumbers along one axis, broadcastable over the half spectrum."""
    n = dims[axis]
    m = n // 2 + 1 if axis == len(dims) - 1 else n
    k = np.arange(m, dtype=np.int64)
    if axis < len(dims) - 1:
        k = np.where(k <= n // 2, k, k - n)
    k = k.reshape([-1 if a == axis else 1 for a in range(len(dims))])
    return k if wide else torch.from_numpy(k).cuda()


def _k2(dims, wide):
    return sum(_axis_k(dims, a, wide) ** 2 for a in range(len(dims)))


def _out(t, dtype):
    """A host extended-precision or device array as a 64-bit tensor."""
    if isinstance(t, np.ndarray):
        t = torch.from_numpy(np.ascontiguousarray(t.astype(np.complex128 if np.iscomplexobj(t) else np.float64))).cuda()
    return t.to(dtype).contiguous()


def exact(case, seed):
    real = _types(case)[0]
    d = _dims(case)
    n = math.prod(d)
    wide = case["dtype"] == "float64" and n <= _HOST_LIMIT
    if case["kind"] == "signals":
        length, batch = d
        shape = (batch, length) if case["order"] == "rows" else (length, batch)
        z = torch.complex(_uniform(shape, real, seed), _uniform(shape, real, seed, 1)).to(torch.complex128)
        axis = 1 if case["order"] == "rows" else 0
        if wide:
            Z = np.fft.fft(z.cpu().numpy().astype(np.clongdouble), axis=axis)
        else:
            Z = torch.fft.fft(z, dim=axis)
        return [_out(Z, torch.complex128), z * length]
    u = _uniform(_real_shape(case), real, seed).to(torch.float64)
    pencil = case["layout"] == "4d_pencil"

    def logical(t):  # memory -> logical axis order
        return t.permute(*reversed(range(t.ndim))) if pencil else t

    def arr(t):
        t = logical(t).contiguous()
        return t.cpu().numpy().astype(np.longdouble) if wide else t

    def spectrum_memory(S):
        S = _out(S, torch.complex128)
        return S.permute(1, 2, 3, 0).contiguous() if case["layout"] in ("4d_pencil", "4d_xzwy") else S

    def real_memory(t):
        t = _out(t, torch.float64)
        return logical(t).contiguous()

    if case["kind"] == "pair":
        return [spectrum_memory(_rfftn(arr(u), wide)), u * n]
    S = _rfftn(arr(u), wide)
    if case["kind"] == "filter":
        k2 = _k2(d, wide)
        if case["op"] == "poisson":
            k2[(0,) * len(d)] = 1
            H = -1.0 / (k2.astype(np.longdouble) if wide else k2.to(torch.float64))
            H[(0,) * len(d)] = 0
        else:
            e = k2.astype(np.longdouble) if wide else k2.to(torch.float64)
            H = (np if wide else torch).exp(-e / (2 * _SIGMA * _SIGMA))
        return real_memory(_irfftn(S * H, d[-1], wide))
    if case["kind"] == "gradient":
        out = [spectrum_memory(S)]
        for axis in range(3):
            k = _axis_k(d, axis, wide)
            out.append(real_memory(_irfftn(S * (1j * (k.astype(np.longdouble) if wide else k.to(torch.float64))),
                                           d[-1], wide)))
        return out
    # loss = sum (v - t)^2, v = N irfftn(c[shell] rfftn(u)); the filter is self-adjoint
    c = _coefficients(case, seed).to(torch.float64)
    target = _uniform(_real_shape(case), real, seed, 2).to(torch.float64)
    ns = case["nshells"]
    k2 = _k2(d, False)
    kmax2 = sum((m // 2) ** 2 for m in d)
    shell = torch.sqrt(k2.to(torch.float64) * (ns * ns) / kmax2).to(torch.int64)
    shell = torch.where(shell * shell * kmax2 > ns * ns * k2, shell - 1, shell)
    shell = torch.where((shell + 1) ** 2 * kmax2 <= ns * ns * k2, shell + 1, shell).clamp(max=ns - 1)
    H = c[shell]
    v = n * _irfftn(S * H, d[-1], False)
    g = 2 * (v - target)
    G = torch.fft.rfftn(g)
    grad_u = n * _irfftn(G * H, d[-1], False)
    w = torch.full((d[-1] // 2 + 1,), 2.0, dtype=torch.float64, device="cuda")
    w[0] = 1
    if d[-1] % 2 == 0:
        w[-1] = 1
    terms = (G.conj() * S).real * w
    grad_c = torch.zeros(ns, dtype=torch.float64, device="cuda").index_add_(0, shell.flatten(), terms.flatten())
    return [((v - target) ** 2).sum(), grad_u, grad_c]

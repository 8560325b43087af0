"""The calls whose speed this framework is judged by, over the sizes they are used at.

Every case is one call, or one forward and inverse pair of calls, of the public Python API
(spectral.*, spectral.flow, spectral.rf) with the implementation that the solver and the benchmark
default to, stockham_r8. Kinds:

    c2c      spectral.fft_c2c: `batch` complex transforms of n points, one direction
    real     spectral.rfft of real rows and spectral.irfft of half spectra
    fft2     spectral.fft2: complex arrays of n1 x n2, one direction
    real2d   spectral.rfft2 of real fields and spectral.irfft2 of half spectra
    fno      spectral.rfft2_truncated of fields and spectral.irfft2_from_modes of weighted modes: the
             two transforms of a Fourier layer, m x m kept modes
    ns       spectral.flow.GpuSolver: `steps` time steps of `batch` vorticity fields of n x n, then
             the physical frame a program records
    radio    spectral.rf: an overlap-save FIR filter and the Hann spectrum of a recording
"""

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path.cwd() / "gpu-spectral-stack_amd" / "python"))

import spectral  # noqa: E402
from spectral import rf  # noqa: E402
from spectral.flow import Flow  # noqa: E402
from spectral.flow.gpu import GpuSolver  # noqa: E402

IMPL = "stockham_r8"
POINTS = 1 << 24  # of the benchmark's rows, and the most any case here holds


def listed():
    return [
        # A program that transforms one short block at a time (a control loop, an interactive
        # analysis): the call's latency is all there is.
        {"name": "real_small", "kind": "real", "n": 256, "batch": 16},
        # The headline: batched complex rows, 2^24 points.
        {"name": "c2c_1024", "kind": "c2c", "n": 1024, "batch": 16384, "inverse": False},
        # Long recordings, beyond one workgroup's LDS: a batch of 2^20-point inverses.
        {"name": "c2c_2e20", "kind": "c2c", "n": 1 << 20, "batch": 16, "inverse": True},
        # Batched real rows, both directions, 2^24 points.
        {"name": "real_1024", "kind": "real", "n": 1024, "batch": 16384},
        # Real fields of the simulation grids, both directions, 2^24 points.
        {"name": "real2d_128", "kind": "real2d", "n1": 128, "n2": 128, "batch": 1024,
         "columns": "auto"},
        {"name": "real2d_512", "kind": "real2d", "n1": 512, "n2": 512, "batch": 64,
         "columns": "auto"},
        # Complex images, an uneven number of them.
        {"name": "fft2_256", "kind": "fft2", "n1": 256, "n2": 256, "batch": 97, "inverse": False,
         "columns": "auto"},
        # A Fourier layer's transforms: 64 samples of 32 channels at 128^2 with 16 modes, and the
        # same layer at the finer grid with 32 modes.
        {"name": "fno_128", "kind": "fno", "batch": 64, "channels": 32, "n": 128, "m": 16},
        {"name": "fno_256", "kind": "fno", "batch": 8, "channels": 32, "n": 256, "m": 32},
        # The Navier-Stokes solver between two recorded frames: the benchmark's 256 trajectories
        # at 128^2, and a finer grid.
        {"name": "ns_128", "kind": "ns", "n": 128, "batch": 256, "steps": 40, "pruned": True},
        {"name": "ns_256", "kind": "ns", "n": 256, "batch": 48, "steps": 6, "pruned": True},
        # A recording filtered and looked at: 63 taps, frames of 1024 samples, 2^22 samples.
        {"name": "radio_63", "kind": "radio", "samples": 1 << 22, "taps": 63, "nfft": 1024},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """Sizes spread over their logarithm from a few thousand points to 2^24, odd batches among
    them; a call's length a power of two, as the API asks."""
    kind = rng.choice(["c2c", "real", "fft2", "real2d", "fno", "ns", "radio"])
    points = _log_uniform(rng, 1 << 13, POINTS)
    if kind == "c2c":
        n = 1 << rng.randint(4, min(22, points.bit_length() - 1))
        return {"kind": kind, "n": n, "batch": max(1, points // n), "inverse": rng.random() < 0.5}
    if kind == "real":
        n = 1 << rng.randint(4, 13)
        return {"kind": kind, "n": n, "batch": max(1, points // n)}
    if kind in ("fft2", "real2d"):
        n1, n2 = 1 << rng.randint(5, 10), 1 << rng.randint(5, 10)
        case = {"kind": kind, "n1": n1, "n2": n2, "batch": max(1, points // (n1 * n2)),
                "columns": "transpose" if rng.random() < 0.2 else "auto"}
        if kind == "fft2":
            case["inverse"] = rng.random() < 0.5
        return case
    if kind == "fno":
        n = 1 << rng.randint(6, 9)
        m = rng.randint(8, max(8, min(64, n // 8)))
        arrays = max(1, min(2048, points // (n * n)))
        channels = min(arrays, rng.choice([1, 20, 32, 64]))
        return {"kind": kind, "batch": max(1, arrays // channels), "channels": channels, "n": n,
                "m": m}
    if kind == "ns":
        n = rng.choice([64, 128, 256])
        pruned = rng.random() < 0.7
        batch = max(1, min(256, points // 4 // (n * n)))
        steps = rng.randint(1, 20) if pruned and n <= 128 else rng.randint(1, 4)
        return {"kind": kind, "n": n, "batch": batch, "steps": steps, "pruned": pruned}
    taps = _log_uniform(rng, 15, 1500)
    return {"kind": kind, "samples": _log_uniform(rng, 1 << 14, 1 << 22), "taps": taps,
            "nfft": 1 << rng.randint(8, 12)}


# --- inputs, from the seed alone ----------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _uniform_complex(g, *shape):
    x = torch.rand(*shape, 2, generator=g, device="cuda", dtype=torch.float32)
    return torch.view_as_complex(x.mul_(2.0).sub_(1.0))


def _normal_complex(g, *shape):
    return torch.view_as_complex(_normal(g, *shape, 2))


def _vorticity(g, batch, n):
    """Gaussian random fields with a k^-3 spectrum, of unit root mean square."""
    white = torch.fft.rfft2(_normal(g, batch, n, n))
    ky = torch.fft.fftfreq(n, 1.0 / n, device="cuda")[:, None]
    kx = torch.arange(n // 2 + 1, device="cuda")[None, :]
    k = torch.sqrt(ky * ky + kx * kx)
    shape = torch.where((k > 0) & (k <= n / 3), k.clamp(min=1.0) ** -2.0, torch.zeros_like(k))
    w = torch.fft.irfft2(white * shape, s=(n, n))
    return w / w.square().mean(dim=(-2, -1), keepdim=True).sqrt()


def _inputs(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind == "c2c":
        return [_uniform_complex(g, case["batch"], case["n"])]
    if kind == "fft2":
        return [_normal_complex(g, case["batch"], case["n1"], case["n2"])]
    if kind == "real":
        n, b = case["n"], case["batch"]
        return [_normal(g, b, n), _normal_complex(g, b, n // 2 + 1)]
    if kind == "real2d":
        n1, n2, b = case["n1"], case["n2"], case["batch"]
        return [_normal(g, b, n1, n2), _normal_complex(g, b, n1, n2 // 2 + 1)]
    if kind == "fno":
        b, c, n, m = case["batch"], case["channels"], case["n"], case["m"]
        return [_normal(g, b, c, n, n), _normal_complex(g, b, c, 2 * m, m)]
    if kind == "ns":
        nu = torch.rand(case["batch"], generator=g, device="cuda") * 4e-3 + 1e-3
        return [_vorticity(g, case["batch"], case["n"]), nu]
    # A tone in noise, and a windowed-sinc low-pass filter that leaves the seed's cutoff through.
    t = torch.arange(case["samples"], device="cuda", dtype=torch.float64)
    f, cut = torch.rand(2, generator=g, device="cuda").double().mul_(0.2).add_(0.05).tolist()
    tone = torch.polar(torch.ones_like(t), 2.0 * math.pi * torch.remainder(f * t, 1.0))
    x = tone.to(torch.complex64) + 0.1 * _normal_complex(g, case["samples"])
    k = torch.arange(case["taps"], device="cuda", dtype=torch.float64) - (case["taps"] - 1) / 2
    h = 2 * cut * torch.sinc(2 * cut * k)
    h = h * torch.hamming_window(case["taps"], periodic=False, dtype=torch.float64, device="cuda")
    return [x, h.float()]


_DRAG, _DT = 0.1, 2.5e-3


def prepare(case, seed):
    inputs = _inputs(case, seed)
    state = {"case": case, "inputs": inputs}
    if case["kind"] == "ns":
        w0, nu = inputs
        flow = Flow(viscosity=nu.cpu().numpy(), drag=_DRAG)
        solver = GpuSolver(case["n"], flow, _DT, fft_impl=IMPL, pruned=case["pruned"])
        state["solver"], state["inputs"] = solver, [solver.to_spectral(w0)]
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    x = state["inputs"]
    if kind == "c2c":
        return spectral.fft_c2c(x[0], inverse=case["inverse"], impl=IMPL)
    if kind == "real":
        return (spectral.rfft(x[0], impl=IMPL), spectral.irfft(x[1], case["n"], impl=IMPL))
    if kind == "fft2":
        return spectral.fft2(x[0], inverse=case["inverse"], impl=IMPL, columns=case["columns"])
    if kind == "real2d":
        return (spectral.rfft2(x[0], impl=IMPL, columns=case["columns"]),
                spectral.irfft2(x[1], case["n2"], impl=IMPL, columns=case["columns"]))
    if kind == "fno":
        return (spectral.rfft2_truncated(x[0], case["m"], case["m"], impl=IMPL),
                spectral.irfft2_from_modes(x[1], (case["n"], case["n"]), impl=IMPL))
    if kind == "ns":
        w_hat = state["solver"].advance(x[0], case["steps"])
        return (w_hat, state["solver"].to_physical(w_hat))
    return (rf.fir(x[0], x[1], fft_impl=IMPL),
            rf.spectrum(x[0], case["nfft"], window_name="hann", fft_impl=IMPL))


# --- what a pass cannot do without ----------------------------------------------------------------


def _complex_flops(n):
    return 5.0 * n * math.log2(max(n, 2))


def work(case):
    kind = case["kind"]
    if kind == "c2c":
        n, b = case["n"], case["batch"]
        return {"bytes": 16 * n * b, "flops": b * _complex_flops(n)}
    if kind == "fft2":
        n, b = case["n1"] * case["n2"], case["batch"]
        return {"bytes": 16 * n * b, "flops": b * _complex_flops(n)}
    if kind == "real":
        n, b = case["n"], case["batch"]
        return {"bytes": 2 * b * (4 * n + 8 * (n // 2 + 1)), "flops": b * _complex_flops(n)}
    if kind == "real2d":
        n1, n2, b = case["n1"], case["n2"], case["batch"]
        return {"bytes": 2 * b * (4 * n1 * n2 + 8 * n1 * (n2 // 2 + 1)),
                "flops": b * _complex_flops(n1 * n2)}
    if kind == "fno":
        n, m, b = case["n"], case["m"], case["batch"] * case["channels"]
        # Per direction: n real rows, then n-point columns of the kept m.
        return {"bytes": 2 * b * (4 * n * n + 16 * m * m),
                "flops": 2 * b * (n * _complex_flops(n) / 2 + m * _complex_flops(n))}
    if kind == "ns":
        n, b, steps = case["n"], case["batch"], case["steps"]
        m = n // 3 + 1
        modes = 16 * m * m if case["pruned"] else 8 * n * (n // 2 + 1)
        # The state in and out and the frame; per step two tendencies of five real transforms
        # over the dealiased modes.
        one = n * _complex_flops(n) / 2 + m * _complex_flops(n)
        return {"bytes": b * (2 * modes + 4 * n * n), "flops": b * (steps * 10 + 1) * one}
    s, nfft = case["samples"], case["nfft"]
    block = rf.default_nfft(case["taps"])
    blocks = -(-s // (block - case["taps"] + 1))
    return {"bytes": 4 * 8 * s, "flops": 2 * blocks * _complex_flops(block)
            + s / nfft * _complex_flops(nfft)}


def tolerance(case):
    """About four times what two orders of the same float32 sums differ by. Against 64 bits a
    transform is 1.5e-7 to 3e-7 off, the solver 1.6e-6 after 40 steps, and the filter 1e-6 of an
    output that its stop band made smaller than its input."""
    if case["kind"] == "ns":
        return {"rel": 1e-5}
    return {"rel": 6e-6 if case["kind"] == "radio" else 1.5e-6}


# --- the same in 64 bits ----------------------------------------------------------------


def _exact_ns(case, w0, nu):
    """The time steps over the full half spectrum, products dealiased by the 2/3 rule."""
    n, dt = case["n"], _DT
    m = n // 3 + 1
    ky = torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64)[:, None]
    kx = torch.arange(n // 2 + 1, device="cuda", dtype=torch.float64)[None, :]
    k2 = ky * ky + kx * kx
    mask = ((ky.abs() <= n / 3) & (kx <= n / 3)).double()
    over = torch.where(k2 > 0, 1.0 / k2.clamp(min=1.0), torch.zeros_like(k2))
    y = torch.arange(n, device="cuda", dtype=torch.float64) * (2.0 * math.pi / n)
    flow = Flow()
    k_f = flow.forcing_wavenumber
    force = -flow.forcing_amplitude * k_f * torch.cos(k_f * y)[:, None]
    force = torch.fft.rfft2(force.expand(n, n)) * mask

    def tendency(w):
        u = torch.fft.irfft2(1j * ky * over * w, s=(n, n))
        v = torch.fft.irfft2(-1j * kx * over * w, s=(n, n))
        wx = torch.fft.irfft2(1j * kx * w, s=(n, n))
        wy = torch.fft.irfft2(1j * ky * w, s=(n, n))
        return force - torch.fft.rfft2(u * wx + v * wy) * mask

    half = 0.5 * dt * (-nu.double()[:, None, None] * k2 - _DRAG)
    w = torch.fft.rfft2(w0.double()) * mask
    for _ in range(case["steps"]):
        f0 = tendency(w)
        f1 = tendency(((1 + half) * w + dt * f0) / (1 - half))
        w = ((1 + half) * w + 0.5 * dt * (f0 + f1)) / (1 - half)
    frame = torch.fft.irfft2(w, s=(n, n))
    if case["pruned"]:
        w = torch.cat([w[:, :m, :m], w[:, n - m:, :m]], dim=1)
    return (w, frame)


def exact(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    if kind == "c2c":
        f = torch.fft.ifft if case["inverse"] else torch.fft.fft
        return f(x[0].to(torch.complex128))
    if kind == "fft2":
        f = torch.fft.ifft2 if case["inverse"] else torch.fft.fft2
        return f(x[0].to(torch.complex128))
    if kind == "real":
        spec = x[1].to(torch.complex128)
        return (torch.fft.rfft(x[0].double()), _real_inverse(spec, case["n"]))
    if kind == "real2d":
        spec = torch.fft.ifft(x[1].to(torch.complex128), dim=-2)
        return (torch.fft.rfft2(x[0].double()), _real_inverse(spec, case["n2"]))
    if kind == "fno":
        n, m = case["n"], case["m"]
        modes = x[1].to(torch.complex128)
        full = modes.new_zeros((*modes.shape[:-2], n, n // 2 + 1))
        full[..., :m, :m] = modes[..., :m, :]
        full[..., n - m:, :m] = modes[..., m:, :]
        spec = torch.fft.rfft2(x[0].double())
        kept = torch.cat([spec[..., :m, :m], spec[..., n - m:, :m]], dim=-2)
        return (kept, _real_inverse(torch.fft.ifft(full, dim=-2), n))
    if kind == "ns":
        return _exact_ns(case, *x)
    signal, taps = x[0].to(torch.complex128), x[1].double()
    size = 1 << (signal.numel() + taps.numel()).bit_length()
    y = torch.fft.ifft(torch.fft.fft(signal, size) * torch.fft.fft(taps.to(signal.dtype), size))
    nfft = case["nfft"]
    frames = torch.nn.functional.pad(signal, (0, -signal.numel() % nfft)).view(-1, nfft)
    window = 0.5 - 0.5 * torch.cos(
        2 * math.pi / nfft * torch.arange(nfft, device="cuda", dtype=torch.float64))
    return (y[: signal.numel()], torch.fft.fft(frames * window))


def _real_inverse(spec, n):
    """irfft along the rows; the imaginary parts of the zero and n/2 frequencies, which have no
    real counterpart, are left out."""
    spec = spec.clone()
    spec[..., 0].imag.zero_()
    spec[..., n // 2].imag.zero_()
    return torch.fft.irfft(spec, n)

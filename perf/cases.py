"""Workloads whose time is watched: what a user of this library has it do,
through its public entry points, from one short transform to batches that fill
the GPU.

A case is a dict of plain values: ``path`` names the entry point, the other
keys give sizes and options.  ``prepare`` makes what a program holds before
the call (inputs, output buffers, the plan), ``run`` is one call, ``exact``
the same result from plain torch in 64 bits, ``work`` the bytes and operations
the call cannot do without (5 N log2 N per complex transform, 2.5 N log2 N per
real one).
"""
import math

import torch

import mufft_amd as M
from mufft_amd.autograd import FFTConv

DEV = "cuda:0"
# The largest drawn case: complex points of one transform batch.
MAX_POINTS = 1 << 26


def listed():
    return [
        # One transform through the drop-in call, host memory in and out (pinned, as mufft_alloc gives it):
        # an existing muFFT caller that switches over.  Latency only.
        {"name": "dropin_c2c_1024", "path": "dropin", "kind": "c2c", "N": 1024},
        # Spectra of overlapping frames of a short signal (ten seconds of audio, hop 1024): a small ragged batch.
        {"name": "frames_2048_x431", "path": "frames", "N": 2048, "hop": 1024, "howmany": 431},
        # The benchmark's batched complex transform.
        {"name": "c2c_4096_x16384", "path": "c2c", "N": 4096, "howmany": 16384, "direction": -1, "zero_pad": False},
        # The benchmark's real round trip: spectrum, then back to the signal.
        {"name": "real_65536_x512", "path": "real", "N": 65536, "howmany": 512},
        # 2D spectra of a batch of complex images.
        {"name": "2d_c2c_1024_x16", "path": "2d_c2c", "Nx": 1024, "Ny": 1024, "howmany": 16, "direction": -1},
        # Real images to spectra and back (2D filtering), large images.
        {"name": "2d_real_2048_x4", "path": "2d_real", "Nx": 2048, "Ny": 2048, "howmany": 4},
        # Long transforms, batched: two column launches each.
        {"name": "c2c_2^20_x64", "path": "c2c", "N": 1 << 20, "howmany": 64, "direction": -1, "zero_pad": False},
        # Very long transforms: three column launches; inverse.
        {"name": "c2c_2^24_x2", "path": "c2c", "N": 1 << 24, "howmany": 2, "direction": 1, "zero_pad": False},
        # Long real signals, there and back.
        {"name": "real_2^21_x64", "path": "real", "N": 1 << 21, "howmany": 64},
        # 640 fast convolutions of mixed sizes in one launch (512 mono, 256 to 65536 points; 128 stereo, 16384 points).
        {"name": "conv_batch_640", "path": "conv_batch", "mono": 512, "log_min": 8, "log_max": 16, "stereo": 128, "stereo_N": 16384},
        # A stretch of a stream through a long FIR filter (overlap-add).
        {"name": "ola_4096_x1024", "path": "ola", "N": 4096, "taps": 2048, "nblocks": 1024},
        # One differentiable convolution layer, forward and backward (gradients of signals and filter).
        {"name": "diff_conv_65536_x64", "path": "diff_conv", "N": 65536, "howmany": 64, "stereo": True},
    ]


def _log_int(rng, lo, hi):
    """An integer in [lo, hi], uniform in its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    path = rng.choice(["dropin", "frames", "c2c", "c2c", "real", "real", "2d_c2c", "2d_real", "conv_batch", "ola", "diff_conv"])
    if path == "dropin":
        return {"path": path, "kind": rng.choice(["c2c", "r2c", "c2r"]), "N": 1 << rng.randint(5, 14)}
    if path == "frames":
        N = 1 << rng.randint(6, 13)
        return {"path": path, "N": N, "hop": 2 * rng.randint(N // 8, N // 2), "howmany": _log_int(rng, 1, (1 << 24) // N)}
    if path == "c2c":
        N = 1 << rng.randint(4, 24)
        return {"path": path, "N": N, "howmany": _log_int(rng, 1, MAX_POINTS // N), "direction": rng.choice([-1, 1]),
                "zero_pad": rng.random() < 0.25}
    if path == "real":
        N = 1 << rng.randint(5, 24)
        return {"path": path, "N": N, "howmany": _log_int(rng, 1, MAX_POINTS // N)}
    if path == "2d_c2c":
        nx, ny = 1 << rng.randint(4, 13), 1 << rng.randint(4, 13)
        return {"path": path, "Nx": nx, "Ny": ny, "howmany": _log_int(rng, 1, max(1, (1 << 25) // (nx * ny))),
                "direction": rng.choice([-1, 1])}
    if path == "2d_real":
        nx, ny = 1 << rng.randint(4, 12), 1 << rng.randint(4, 12)
        return {"path": path, "Nx": nx, "Ny": ny, "howmany": _log_int(rng, 1, max(1, (1 << 25) // (nx * ny)))}
    if path == "conv_batch":
        lo = rng.randint(6, 12)
        return {"path": path, "mono": _log_int(rng, 3, 640), "log_min": lo, "log_max": rng.randint(lo, 16),
                "stereo": _log_int(rng, 1, 128), "stereo_N": 1 << rng.randint(8, 15)}
    if path == "ola":
        N = 1 << rng.randint(6, 16)
        return {"path": path, "N": N, "taps": rng.randint(1, N // 2), "nblocks": _log_int(rng, 1, (1 << 23) // N)}
    N = 1 << rng.randint(8, 16)
    return {"path": path, "N": N, "howmany": _log_int(rng, 1, (1 << 22) // N), "stereo": rng.random() < 0.5}


# ---- inputs (made from the seed alone) -----------------------------------------------------------------

def _gen(seed, device=DEV):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return g


def _uniform(g, shape, device=DEV):
    return torch.rand(shape, generator=g, device=device).mul_(2).sub_(1)


def _complex(g, shape, device=DEV):
    return torch.view_as_complex(_uniform(g, tuple(shape) + (2,), device))


def _taps(g, shape):
    """Exponentially decaying Gaussian taps, decay length half the filter's last axis / 2."""
    n = shape[-1]
    return torch.randn(shape, generator=g, device=DEV) * torch.exp(torch.arange(n, device=DEV, dtype=torch.float32) / (-n / 4))


def _inputs(case, seed):
    p = case["path"]
    if p == "dropin":
        g, n = _gen(seed, "cpu"), case["N"]
        if case["kind"] == "r2c":
            return _uniform(g, (n,), "cpu").pin_memory()
        if case["kind"] == "c2r":   # the spectrum of a real signal
            return torch.fft.rfft(_uniform(g, (n,), "cpu")).pin_memory()
        return _complex(g, (n,), "cpu").pin_memory()
    g = _gen(seed)
    if p == "frames":
        return _uniform(g, ((case["howmany"] - 1) * case["hop"] + case["N"],))
    if p == "c2c":
        return _complex(g, (case["howmany"], case["N"] // 2 if case["zero_pad"] else case["N"]))
    if p == "real":
        return _uniform(g, (case["howmany"], case["N"]))
    if p in ("2d_c2c", "2d_real"):   # pixels in [0, 1) plus noise
        shape = (case["howmany"], case["Ny"], case["Nx"])
        if p == "2d_c2c":
            shape += (2,)
        x = torch.rand(shape, generator=g, device=DEV).add_(torch.randn(shape, generator=g, device=DEV), alpha=0.1)
        return torch.view_as_complex(x) if p == "2d_c2c" else x
    if p == "conv_batch":
        sizes = (torch.randint(case["log_min"], case["log_max"] + 1, (case["mono"],), generator=_gen(case["mono"], "cpu"))).tolist()
        mono = [(1 << s, _uniform(g, (1 << s >> 1,)), _taps(g, (1 << s >> 1,))) for s in sizes]
        n = case["stereo_N"]
        return mono, _complex(g, (case["stereo"], n // 2)), _taps(g, (case["stereo"], n // 2))
    if p == "ola":
        return _uniform(g, (case["nblocks"] * (case["N"] // 2),)), torch.randn(case["taps"], generator=g, device=DEV) / math.sqrt(case["taps"])
    if p == "diff_conv":
        n, b = case["N"], case["howmany"]
        x = _complex(g, (b, n // 2)) if case["stereo"] else _uniform(g, (b, n // 2))
        h = torch.randn(n // 2, generator=g, device=DEV) * 1e-2
        dy = _complex(g, (b, n)) if case["stereo"] else _uniform(g, (b, n))
        return x, h, dy
    raise ValueError(p)


# ---- state, one pass, the same in 64 bits ---------------------------------------------------------------

MONO = M.CONV_METHOD_FLAG_MONO_MONO | M.CONV_METHOD_FLAG_ZERO_PAD_UPPER_HALF_FIRST | M.CONV_METHOD_FLAG_ZERO_PAD_UPPER_HALF_SECOND
STEREO = MONO | M.CONV_METHOD_FLAG_STEREO_MONO


def prepare(case, seed):
    p, x = case["path"], _inputs(case, seed)
    s = {"case": case, "x": x}
    if p == "dropin":
        n, kind = case["N"], case["kind"]
        s["plan"] = M.Plan1D(kind, n, M.INVERSE if kind == "c2r" else M.FORWARD)
        s["y"] = torch.empty(n // 2 + 1 if kind == "r2c" else n, dtype=torch.float32 if kind == "c2r" else torch.complex64, pin_memory=True)
    elif p == "frames":
        s["plan"] = M.Plan1D("r2c", case["N"])
        s["y"] = torch.empty((case["howmany"], case["N"] // 2 + 1), dtype=torch.complex64, device=DEV)
    elif p == "c2c":
        s["plan"] = M.Plan1D("c2c", case["N"], case["direction"], M.FLAG_ZERO_PAD_UPPER_HALF if case["zero_pad"] else 0)
        s["y"] = torch.empty((case["howmany"], case["N"]), dtype=torch.complex64, device=DEV)
    elif p == "real":
        s["r2c"], s["c2r"] = M.Plan1D("r2c", case["N"]), M.Plan1D("c2r", case["N"])
        s["X"] = torch.empty((case["howmany"], case["N"] // 2 + 1), dtype=torch.complex64, device=DEV)
        s["y"] = torch.empty_like(x)
    elif p == "2d_c2c":
        s["plan"] = M.Plan2D("c2c", case["Nx"], case["Ny"], case["direction"])
        s["y"] = torch.empty_like(x)
    elif p == "2d_real":
        s["r2c"], s["c2r"] = M.Plan2D("r2c", case["Nx"], case["Ny"]), M.Plan2D("c2r", case["Nx"], case["Ny"])
        # Spectrum rows hold Nx bins, of which Nx/2 + 1 are written.
        s["X"] = torch.zeros((case["howmany"], case["Ny"], case["Nx"]), dtype=torch.complex64, device=DEV)
        s["y"] = torch.empty_like(x)
    elif p == "conv_batch":
        mono, a, h = x
        s["mono"] = torch.empty(sum(n for n, _, _ in mono), dtype=torch.float32, device=DEV)
        s["stereo"] = torch.empty((case["stereo"], case["stereo_N"]), dtype=torch.complex64, device=DEV)
        outs = torch.split(s["mono"], [n for n, _, _ in mono])
        jobs = [(n, MONO, u, v, o) for (n, u, v), o in zip(mono, outs)]
        jobs += [(case["stereo_N"], STEREO, a[i], h[i], s["stereo"][i]) for i in range(case["stereo"])]
        torch.cuda.synchronize()   # the batch captures its graph on a stream of its own
        s["batch"] = M.ConvBatch(jobs)
    elif p == "ola":
        s["x"] = x[0]
        torch.cuda.synchronize()   # the filter is transformed on a stream of its own
        s["ola"] = M.OverlapAdd(case["N"], x[1])
        s["y"] = torch.empty_like(x[0])
    elif p == "diff_conv":
        s["op"] = FFTConv(case["N"], stereo=case["stereo"])
        s["x"], s["h"], s["dy"] = x[0].requires_grad_(True), x[1].requires_grad_(True), x[2]
    return s


def run(s):
    case = s["case"]
    p = case["path"]
    if p == "dropin":
        s["plan"].execute(s["y"], s["x"])
        return s["y"]
    if p == "diff_conv":
        y = s["op"](s["x"], s["h"])
        dx, dh = torch.autograd.grad(y, (s["x"], s["h"]), s["dy"])
        return y.detach(), dx, dh
    st = torch.cuda.current_stream()
    if p == "frames":
        s["plan"].execute_batched(s["y"], s["x"], case["howmany"], idist=case["hop"], stream=st)
        return s["y"]
    if p in ("c2c", "2d_c2c"):
        s["plan"].execute_batched(s["y"], s["x"], case["howmany"], stream=st)
        return s["y"]
    if p in ("real", "2d_real"):
        s["r2c"].execute_batched(s["X"], s["x"], case["howmany"], stream=st)
        s["c2r"].execute_batched(s["y"], s["X"], case["howmany"], stream=st)
        return s["X"], s["y"]
    if p == "conv_batch":
        s["batch"].execute(stream=st)
        return s["mono"], s["stereo"]
    if p == "ola":
        s["ola"](s["y"], s["x"], case["nblocks"], stream=st)
        return s["y"]
    raise ValueError(p)


def _wide(t):
    t = t.cpu()
    return t.to(torch.complex128) if t.is_complex() else t.to(torch.float64)


def _conv(x, h, n):
    """Rows of x convolved with the rows of h, the first n samples."""
    if x.is_complex():
        return torch.fft.ifft(torch.fft.fft(x, n=n) * torch.fft.fft(h, n=n))
    return torch.fft.irfft(torch.fft.rfft(x, n=n) * torch.fft.rfft(h, n=n), n=n)


def exact(case, seed):
    p, x = case["path"], _inputs(case, seed)
    if p == "dropin":
        x, n = _wide(x), case["N"]
        return torch.fft.fft(x) if case["kind"] == "c2c" else torch.fft.rfft(x) if case["kind"] == "r2c" else torch.fft.irfft(x, n=n) * n
    if p == "frames":
        return torch.fft.rfft(_wide(x).unfold(0, case["N"], case["hop"]))
    if p == "c2c":
        x, n = _wide(x), case["N"]
        return torch.fft.fft(x, n=n) if case["direction"] < 0 else torch.fft.ifft(x, n=n) * n
    if p == "real":
        x = _wide(x)
        return torch.fft.rfft(x), x * case["N"]
    if p == "2d_c2c":
        x = _wide(x)
        return torch.fft.fft2(x) if case["direction"] < 0 else torch.fft.ifft2(x) * (case["Nx"] * case["Ny"])
    if p == "2d_real":
        x, nx = _wide(x), case["Nx"]
        spec = torch.zeros(x.shape, dtype=torch.complex128)
        spec[..., : nx // 2 + 1] = torch.fft.rfft2(x)
        return spec, x * (nx * case["Ny"])
    if p == "conv_batch":
        mono, a, h = x
        return torch.cat([_conv(_wide(u), _wide(v), n) for n, u, v in mono]), _conv(_wide(a), _wide(h), case["stereo_N"])
    if p == "ola":
        x, h = _wide(x[0]), _wide(x[1])
        return _conv(x, h, 1 << (x.numel() + h.numel() - 1).bit_length())[: x.numel()]
    if p == "diff_conv":
        x, h, dy = (_wide(t) for t in x)
        n = case["N"]
        X, H, G = torch.fft.fft(x, n=n), torch.fft.fft(h, n=n), torch.fft.fft(dy)
        y, dx = torch.fft.ifft(X * H), torch.fft.ifft(G * H.conj())[:, : n // 2]
        dh = torch.fft.ifft((G * X.conj()).sum(0))[: n // 2].real
        return (y, dx, dh) if case["stereo"] else (y.real, dx.real, dh)
    raise ValueError(p)


def work(case):
    p = case["path"]

    def c(n):   # operations of a complex transform; a real one has half
        return 5.0 * n * math.log2(n)

    if p == "dropin":
        n = case["N"]
        half = case["kind"] != "c2c"
        return {"bytes": 4 * n + 8 * (n // 2 + 1) if half else 16 * n, "flops": c(n) / (2 if half else 1)}
    if p == "frames":
        n, b = case["N"], case["howmany"]
        return {"bytes": 4 * ((b - 1) * case["hop"] + n) + 8 * b * (n // 2 + 1), "flops": b * c(n) / 2}
    if p == "c2c":
        n, b = case["N"], case["howmany"]
        return {"bytes": b * n * (12 if case["zero_pad"] else 16), "flops": b * c(n)}
    if p == "real":
        n, b = case["N"], case["howmany"]
        return {"bytes": 2 * b * (4 * n + 8 * (n // 2 + 1)), "flops": b * c(n)}
    if p in ("2d_c2c", "2d_real"):
        nx, ny, b = case["Nx"], case["Ny"], case["howmany"]
        if p == "2d_c2c":
            return {"bytes": 16 * b * nx * ny, "flops": b * (ny * c(nx) + nx * c(ny))}
        return {"bytes": 2 * b * ny * (4 * nx + 8 * (nx // 2 + 1)), "flops": 2 * b * (ny * c(nx) / 2 + (nx // 2 + 1) * c(ny))}
    if p == "conv_batch":
        sizes = (torch.randint(case["log_min"], case["log_max"] + 1, (case["mono"],), generator=_gen(case["mono"], "cpu"))).tolist()
        n, b = case["stereo_N"], case["stereo"]
        return {"bytes": sum(8 * (1 << s) for s in sizes) + 14 * n * b, "flops": sum(1.5 * c(1 << s) for s in sizes) + 2.5 * b * c(n)}
    if p == "ola":   # the filter's spectrum is kept: one transform there and one back per block
        n, b = case["N"], case["nblocks"]
        return {"bytes": 4 * b * n, "flops": b * c(n)}
    if p == "diff_conv":
        # Read: signals, filter, output gradient; written: output, both gradients.
        n, b, e = case["N"], case["howmany"], 8 if case["stereo"] else 4
        t = c(n) if case["stereo"] else c(n) / 2
        return {"bytes": e * b * n * 3 + 4 * n, "flops": b * 4 * t + c(n)}
    raise ValueError(p)

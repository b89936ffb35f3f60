"""The calls whose speed this library is judged by: what a user's program hands to the GPU through the public plan
interface, from one short transform to batches that fill the card.

Every case names a `kind` (which plan runs) and its sizes. `listed` holds the fixed ones, `draw` makes more of the same
kinds over the ranges stated beside each generator, `prepare` builds inputs, output buffers and the plan, `run` is one
pass through the plan, `exact` the same result in 64 bits from torch or numpy.
"""
import math

import numpy as np
import torch

import crd_amd
from crd_amd import spectral, workloads
from crd_amd.many import ManyPlan

# Complex points of the largest drawn transform batch (2^27 points are 1 GiB per buffer).
MAX_POINTS = 1 << 27


def listed():
    return [
        # one short transform, as a control loop or an interactive tool issues it: launch and host latency
        {"name": "c2c_1k_single", "kind": "c2c", "n": 1024, "batch": 1, "inverse": False},
        # the usual batch of mid-size rows
        {"name": "c2c_4k_batch", "kind": "c2c", "n": 4096, "batch": 1024, "inverse": False},
        # long rows, a batch that streams from memory
        {"name": "c2c_64k_batch", "kind": "c2c", "n": 1 << 16, "batch": 2048, "inverse": False},
        # very long rows, the way back
        {"name": "c2c_1m_inverse", "kind": "c2c", "n": 1 << 20, "batch": 64, "inverse": True},
        # real signals to spectra and back (a filter without its product)
        {"name": "real_64k_roundtrip", "kind": "real", "n": 1 << 16, "batch": 2048},
        # many uneven smooth lengths in one call
        {"name": "mixed_20000", "kind": "many", "count": 20000, "lo": 64, "hi": 16384, "seed": 20000},
        # the split-precision form on the matrix cores
        {"name": "split_fp16_64k", "kind": "split", "n": 1 << 16, "batch": 1024, "precision": "split_fp16"},
        # power spectrum estimate of a long recording
        {"name": "welch_4k_long", "kind": "welch", "length": 1 << 26, "nperseg": 4096, "noverlap": 2048},
        # short-time transform of audio: 46 s stereo-length signal, frames of 1024 at 75 % overlap
        {"name": "stft_1k_audio", "kind": "stft", "length": 4000001, "nperseg": 1024, "noverlap": 768},
        # cosine transform of rows and its inverse (transform coding)
        {"name": "dct_4k_pair", "kind": "dct", "n": 4096, "batch": 4096},
        # a length with no small factors
        {"name": "prime_1009", "kind": "any", "n": 1009, "batch": 8192, "inverse": False},
        # a volume
        {"name": "volume_256", "kind": "nd", "dims": "256x256x256", "batch": 1, "inverse": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch(rng, n, lo_points=1 << 10, hi_points=MAX_POINTS):
    """A batch count, odd ones among them, for lo_points..hi_points points in all."""
    return max(1, min(_log_int(rng, max(1, lo_points // n), max(2, hi_points // n)), hi_points // n))


def draw(rng):
    kind = rng.choice(["c2c", "c2c", "real", "many", "split", "welch", "stft", "dct", "any", "nd"])
    if kind == "c2c":  # n = 2^4 .. 2^22, one transform up to 2^27 points (2^26 of the long rows)
        n = 1 << rng.randint(4, 22)
        return {"kind": kind, "n": n, "batch": _batch(rng, n, 1 << 10, MAX_POINTS >> (n > 1 << 17)),
                "inverse": rng.random() < 0.5}
    if kind == "real":  # n = 2^6 .. 2^22
        n = 1 << rng.randint(6, 22)
        return {"kind": kind, "n": n, "batch": _batch(rng, n)}
    if kind == "many":  # 200 .. 20000 transforms over 7-smooth lengths in [64, 16384]
        lo = _log_int(rng, 64, 1000)
        return {"kind": kind, "count": _log_int(rng, 200, 20000), "lo": lo, "hi": _log_int(rng, 4 * lo, 16384),
                "seed": rng.randint(1, 1 << 30)}
    if kind == "split":
        n = rng.choice([256, 1024, 1 << 16, 1 << 18, 1 << 20])
        return {"kind": kind, "n": n, "batch": _batch(rng, n, 1 << 16, 1 << 26),
                "precision": rng.choice(["split_bf16", "split_fp16"])}
    if kind in ("welch", "stft"):  # frames of 2^6 .. 2^14 samples, hops of an eighth of a frame up to a whole one
        nperseg = 1 << rng.randint(6, 14)
        noverlap = nperseg - rng.randint(nperseg // 8, nperseg)
        longest = (1 << 26) if kind == "welch" else (1 << 24)
        longest = max(longest * (nperseg - noverlap) // nperseg, 8 * nperseg)
        return {"kind": kind, "length": _log_int(rng, 4 * nperseg, longest), "nperseg": nperseg, "noverlap": noverlap}
    if kind == "dct":  # n = 2^4 .. 2^16
        n = 1 << rng.randint(4, 16)
        return {"kind": kind, "n": n, "batch": _batch(rng, n, 1 << 10, 1 << 25)}
    if kind == "any":  # every length, prime and smooth alike, 17 .. 100000
        n = _log_int(rng, 17, 100000)
        return {"kind": kind, "n": n, "batch": _batch(rng, n, 1 << 12, 1 << (24 if n <= 8192 else 22)),
                "inverse": rng.random() < 0.5}
    # images and volumes: axes of any length up to 2048 (images) or 160, powers of two up to 256
    axes = rng.choice([2, 2, 3])
    top = 2048 if axes == 2 else 160
    dims = [rng.choice([_log_int(rng, 24, top), 1 << rng.randint(5, 8)]) for _ in range(axes)]
    volume = math.prod(dims)
    return {"kind": kind, "dims": "x".join(str(d) for d in dims),
            "batch": _batch(rng, volume, 1 << 12, 1 << 22), "inverse": rng.random() < 0.5}


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _dims(case):
    return [int(d) for d in case["dims"].split("x")]


def _lengths(case):
    return workloads.mixed_batch(case["count"], 8, case["lo"], case["hi"], case["seed"])


def _frames(case):
    if case["length"] < case["nperseg"]:
        return 0
    return (case["length"] - case["noverlap"]) // (case["nperseg"] - case["noverlap"])


FS = 48000.0


def _input(case, seed):
    """The input on the GPU: complex64 or float32, from the seed alone."""
    g = _generator(seed)
    kind = case["kind"]
    if kind in ("c2c", "any"):
        return torch.randn(case["batch"], case["n"], dtype=torch.complex64, device="cuda", generator=g)
    if kind == "split":  # magnitudes over eight decades, any phase
        shape = (case["batch"], case["n"])
        mag = torch.pow(10.0, torch.rand(shape, device="cuda", generator=g) * 8.0 - 4.0)
        return torch.polar(mag, torch.rand(shape, device="cuda", generator=g) * (2.0 * math.pi))
    if kind in ("real", "dct"):
        return torch.randn(case["batch"], case["n"], device="cuda", generator=g)
    if kind == "many":
        return torch.view_as_complex(
            torch.rand(int(_lengths(case).sum()), 2, device="cuda", generator=g) * 2.0 - 1.0)
    if kind in ("welch", "stft"):  # noise over two tones and an offset
        t = torch.arange(case["length"], device="cuda", dtype=torch.float64) * (2.0 * math.pi / FS)
        tones = torch.sin(440.0 * t) + 0.5 * torch.sin(5000.0 * t) + 0.1
        return tones.float() + 0.3 * torch.randn(case["length"], device="cuda", generator=g)
    return torch.randn(case["batch"], *_dims(case), dtype=torch.complex64, device="cuda", generator=g)


def prepare(case, seed):
    x = _input(case, seed)
    kind = case["kind"]
    s = {"kind": kind, "x": x, "direction": crd_amd.INVERSE if case.get("inverse") else crd_amd.FORWARD}
    if kind in ("c2c", "split"):
        s["plan"] = crd_amd.FftPlan(case["n"], case["batch"], precision=case.get("precision", "fp32"))
        s["y"] = torch.empty_like(x)
    elif kind == "any":
        s["plan"] = crd_amd.BluesteinPlan(case["n"], case["batch"])
        s["y"] = torch.empty_like(x)
    elif kind == "real":
        s["plan"] = crd_amd.RealFftPlan(case["n"], case["batch"])
        s["y"] = torch.empty(case["batch"], case["n"] // 2 + 1, dtype=torch.complex64, device="cuda")
        s["z"] = torch.empty_like(x)
    elif kind == "many":
        s["plan"] = ManyPlan(_lengths(case))
        s["y"] = torch.empty_like(x)
    elif kind == "dct":
        s["plan"] = crd_amd.DctPlan(case["n"], case["batch"])
        s["y"] = torch.empty_like(x)
        s["z"] = torch.empty_like(x)
    elif kind in ("welch", "stft"):
        s["plan"] = spectral.SpectralPlan(case["nperseg"], case["noverlap"], "hann", detrend=kind == "welch")
        s["length"] = case["length"]
        bins = case["nperseg"] // 2 + 1
        s["y"] = (torch.empty(bins, device="cuda") if kind == "welch" else
                  torch.empty(_frames(case), bins, dtype=torch.complex64, device="cuda"))
    else:
        s["plan"] = crd_amd.NdFftPlan(_dims(case), case["batch"])
        s["y"] = torch.empty_like(x)
    return s


def run(s):
    kind, plan, x, y = s["kind"], s["plan"], s["x"], s["y"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "real":
        plan.rfft(x.data_ptr(), y.data_ptr(), stream)
        plan.irfft(y.data_ptr(), s["z"].data_ptr(), stream)
        return y, s["z"]
    if kind == "dct":
        plan.dct2(x.data_ptr(), y.data_ptr(), stream)
        plan.dct3(y.data_ptr(), s["z"].data_ptr(), stream)
        return y, s["z"]
    if kind == "welch":
        plan.welch(x.data_ptr(), s["length"], FS, y.data_ptr(), stream)
    elif kind == "stft":
        plan.stft(x.data_ptr(), s["length"], y.data_ptr(), stream)
    elif kind == "nd":  # the plan works in place: the volume is kept, its copy transformed
        y.copy_(x)
        plan.execute(y.data_ptr(), s["direction"], stream)
    else:
        plan.execute(x.data_ptr(), y.data_ptr(), s["direction"], stream)
    return y


def work(case):
    kind = case["kind"]
    if kind in ("c2c", "split", "any"):
        points = case["n"] * case["batch"]
        return {"bytes": 16 * points, "flops": 5 * points * math.log2(case["n"])}
    if kind == "real":
        reals, bins = case["n"] * case["batch"], (case["n"] // 2 + 1) * case["batch"]
        return {"bytes": 8 * reals + 16 * bins, "flops": 5 * reals * math.log2(case["n"])}
    if kind == "many":
        lengths = _lengths(case).astype(np.float64)
        return {"bytes": 16 * int(lengths.sum()), "flops": float((5 * lengths * np.log2(lengths)).sum())}
    if kind == "dct":
        points = case["n"] * case["batch"]
        return {"bytes": 16 * points, "flops": 5 * points * math.log2(case["n"])}
    if kind in ("welch", "stft"):
        frames, bins = _frames(case), case["nperseg"] // 2 + 1
        out = 4 * bins if kind == "welch" else 8 * bins * frames
        return {"bytes": 4 * case["length"] + out, "flops": 2.5 * frames * case["nperseg"] * math.log2(case["nperseg"])}
    points = case["batch"] * math.prod(_dims(case))
    return {"bytes": 16 * points, "flops": 5 * points * math.log2(math.prod(_dims(case)))}


def tolerance(case):
    # against the 64-bit result the FP32 transforms and the split forms measure 0.5e-7 .. 2.8e-7; chirp-z lengths run
    # two transforms of at least twice the length
    return {"rel": 2e-6 if case["kind"] in ("any", "nd") else 1.2e-6}


def exact(case, seed):
    x = _input(case, seed)
    kind = case["kind"]
    inverse = bool(case.get("inverse"))
    if kind in ("c2c", "split"):
        x = x.to(torch.complex128)
        return torch.fft.ifft(x, norm="forward") if inverse else torch.fft.fft(x)
    if kind == "any":  # the inverse of the any-length plan is scaled by 1/n
        v = x.cpu().numpy().astype(np.complex128)
        return torch.from_numpy(np.fft.ifft(v) if inverse else np.fft.fft(v)).cuda()
    if kind == "real":
        v = x.to(torch.float64)
        return torch.fft.rfft(v), v
    if kind == "many":
        v = x.cpu().numpy().astype(np.complex128)
        lengths = _lengths(case)
        starts = np.concatenate(([0], np.cumsum(lengths)[:-1]))
        out = np.empty_like(v)
        for n in np.unique(lengths):
            index = starts[lengths == n][:, None] + np.arange(n)[None, :]
            out[index] = np.fft.fft(v[index])
        return torch.from_numpy(out).cuda()
    if kind == "dct":
        n = case["n"]
        v = x.to(torch.float64)
        k = torch.arange(n, dtype=torch.float64, device="cuda")
        phase = torch.polar(torch.ones_like(k), -k * (math.pi / (2 * n)))
        return 2.0 * (torch.fft.fft(v, 2 * n)[:, :n] * phase).real, 2.0 * n * v
    if kind in ("welch", "stft"):
        m, hop = case["nperseg"], case["nperseg"] - case["noverlap"]
        window = torch.hann_window(m, periodic=True, dtype=torch.float64, device="cuda")
        frames = x.to(torch.float64).unfold(0, m, hop)[: _frames(case)]
        if kind == "stft":
            return torch.fft.rfft(frames * window)
        total = torch.zeros(m // 2 + 1, dtype=torch.float64, device="cuda")
        for block in frames.split(max(1, (1 << 26) // m)):
            spectrum = torch.fft.rfft((block - block.mean(1, keepdim=True)) * window)
            total += (spectrum.real ** 2 + spectrum.imag ** 2).sum(0)
        psd = total / (FS * (window ** 2).sum() * frames.shape[0])
        psd[1:-1] *= 2.0
        return psd
    x = x.to(torch.complex128)
    axes = tuple(range(1, 1 + len(_dims(case))))
    # the inverse of the N-D plan is scaled by 1 / volume
    return torch.fft.ifftn(x, dim=axes) if inverse else torch.fft.fftn(x, dim=axes)

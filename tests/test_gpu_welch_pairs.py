"""Welch over pairs of frames (two frames per complex transform) at the frame counts where it takes over from single frames
(512 up to 256 samples a frame, 1024 above, 769 at 8192 on 256 CUs), odd counts (half a pair), odd hops (frames on any 4-byte boundary) and both
window / detrend settings, against the oracle's FP64 restatement: rel-L2 <= 2e-6 log2(nperseg), the bar of the spectral
tests, also where a pair's squares would leave the range unscaled. A NaN sample reaches every bin, a zero signal gives zeros, reruns are bit-identical."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bound(n):
    return 2e-6 * np.log2(n)


def _signal(length, seed):
    rng = np.random.default_rng(seed)
    t = np.arange(length)
    return (np.sin(2 * np.pi * 0.013 * t) + 0.3 * rng.standard_normal(length) + 1.7).astype(np.float32)


def _welch(gpu, x, nperseg, noverlap, window, detrend, fs=250.0):
    from crd_amd import spectral

    plan = spectral.SpectralPlan(nperseg, noverlap, window, detrend=detrend)
    src = gpu.DeviceBuffer.from_array(x)
    psd = gpu.DeviceBuffer(4 * plan.nfreq)
    plan.welch(src, len(x), fs, psd)
    gpu.synchronize()
    return plan.frames(len(x)), psd.download((plan.nfreq,), np.float32)


@pytest.mark.parametrize("nperseg,hop,frames,window,detrend", [
    (8, 3, 511, "hann", True), (8, 3, 512, "hann", True), (16, 16, 700, "boxcar", False), (32, 5, 2001, "hann", False),
    (64, 63, 512, "hann", True), (128, 128, 40001, "hann", True), (256, 31, 513, "hann", True),
    (512, 7, 1023, "hann", True), (512, 7, 1024, "boxcar", True), (1024, 101, 1025, "hann", True),
    (2048, 2048, 1026, "hann", True), (4096, 64, 1024, "hann", True), (4096, 65, 5001, "hann", False),
    (8192, 33, 768, "hann", True), (8192, 33, 769, "hann", True), (8192, 33, 1027, "hann", True)])
def test_pairs_match_fp64(gpu, po, nperseg, hop, frames, window, detrend):
    print(f"welch nperseg={nperseg} hop={hop} frames={frames} {window} {detrend}", flush=True)
    length = frames * hop + nperseg - hop + min(hop - 1, 2)  # samples past the last frame are not read
    x = _signal(length, nperseg + frames)
    got_frames, w = _welch(gpu, x, nperseg, nperseg - hop, window, detrend)
    assert got_frames == frames
    rows = po.periodograms64(x.astype(np.float64), 250.0, nperseg, nperseg - hop, window=window, detrend=detrend)
    assert po.rel_l2(w, rows.mean(axis=0)) <= bound(nperseg)
    again = _welch(gpu, x, nperseg, nperseg - hop, window, detrend)[1]
    assert np.array_equal(w.view(np.uint32), again.view(np.uint32))


@pytest.mark.parametrize("nperseg", [64, 4096])
def test_nan_and_zeros(gpu, nperseg):
    x = np.zeros(nperseg * 1025, np.float32)
    assert not np.any(_welch(gpu, x, nperseg, nperseg // 2, "hann", True)[1])
    x[nperseg * 700 + 3] = np.nan
    assert np.all(np.isnan(_welch(gpu, x, nperseg, nperseg // 2, "hann", True)[1]))


@pytest.mark.parametrize("nperseg,window,fs", [(64, "hann", 48000.0), (512, "boxcar", 48000.0), (512, "hann", 1e-3),
                                               (4096, "hann", 1.0)])
def test_amplitudes_near_the_range(gpu, po, nperseg, window, fs):
    """Frames a quarter of a period apart: a bin of a pair is |A| + |B| = 2 |A|, whose square is out of range (3.4e38) where
    |A|^2 = 1.7e38 is not. The scaled sum over the frames is in range at all of these sampling rates but the smallest, where
    the amplitude is taken down by the scale's root."""
    frames, hop, k0 = 1024, nperseg // 4, 9
    w = np.ones(nperseg) if window == "boxcar" else 0.5 - 0.5 * np.cos(2 * np.pi * np.arange(nperseg) / nperseg)
    scale = 1.0 / (fs * np.sum(w * w))
    top = 1.3e19 if scale < 1 else 1.3e19 / np.sqrt(scale * frames * 4)
    t = np.arange((frames - 1) * hop + nperseg)
    x = (top / (0.5 * np.sum(w)) * np.cos(2 * np.pi * k0 * t / nperseg + 0.3)).astype(np.float32)
    got = _welch(gpu, x, nperseg, nperseg - hop, window, False, fs)[1]
    want = po.periodograms64(x.astype(np.float64), fs, nperseg, nperseg - hop, window=window, detrend=False).mean(axis=0)
    assert np.all(np.isfinite(got)) and np.all(want < 3.4e38)
    assert po.rel_l2(got, want) <= bound(nperseg)


@pytest.mark.parametrize("nperseg,frames", [(256, 2048), (2048, 1024), (4096, 1024), (8192, 1024)])
def test_mean_error_is_no_larger_than_of_single_frames(gpu, po, nperseg, frames):
    """The mean error over tone pairs at random frequencies, in noise. Single frames measure 7.3e-8 .. 8.2e-8 at these lengths
    (120 signals, standard deviation of a signal 3.8e-8); 24 signals' mean scatters by a fifth of that, so 6.5e-8 is the
    bar: pairs measure 3.6e-8 .. 5.0e-8, and 1.1e-7 from 4096 on where their constants' mean gain is left in."""
    from crd_amd import spectral

    hop = nperseg // 2
    length = (frames - 1) * hop + nperseg
    t = np.arange(length)
    plan = spectral.SpectralPlan(nperseg, nperseg - hop, "hann", detrend=True)
    psd = gpu.DeviceBuffer(4 * plan.nfreq)
    errors = []
    for seed in range(24):
        rng = np.random.default_rng(seed)
        f1, f2 = rng.random(2)
        x = (np.sin(np.pi * f1 * t) + 0.5 * np.sin(np.pi * f2 * t) + 0.1 + 0.3 * rng.standard_normal(length)).astype(np.float32)
        src = gpu.DeviceBuffer.from_array(x)
        plan.welch(src, length, 250.0, psd)
        gpu.synchronize()
        rows = po.periodograms64(x.astype(np.float64), 250.0, nperseg, nperseg - hop)
        errors.append(po.rel_l2(psd.download((plan.nfreq,), np.float32), rows.mean(axis=0)))
    assert np.mean(errors) <= 6.5e-8, np.mean(errors)

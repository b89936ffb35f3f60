"""Welch over pairs of frames (two frames per complex transform) at the frame counts where it takes over from single frames
(512 up to 256 samples a frame, 1024 above), odd counts (half a pair), odd hops (frames on any 4-byte boundary) and both
window / detrend settings, against the oracle's FP64 restatement: rel-L2 <= 2e-6 log2(nperseg), the bar of the spectral
tests. A NaN sample reaches every bin, a zero signal gives zeros, reruns are bit-identical."""
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
    (8192, 33, 1027, "hann", True)])
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

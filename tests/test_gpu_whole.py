"""The whole-transform kernel of n = 2^15 and 2^16 C2C (one workgroup per transform, persistent over rounds of one
transform per CU) at the batches where its dispatch changes: the smallest partial round it takes, full rounds, a partial
round behind full ones, and a rest that the four-step runs. Rows of every round against FP64 (rel-L2 <= 2e-6 log2 n), all
rows against a tuned four-step plan (both within that bound of FP64, so within twice the bound of each other)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bound(n):
    return 2e-6 * np.log2(n)


def _input(rng, batch, n, pitch):
    return rng.standard_normal((batch, 2 * pitch), dtype=np.float32).view(np.complex64)


def _run(gpu, plan, x, pitch_out, in_place, direction, guard):
    batch = x.shape[0]
    buf = np.full((batch, max(x.shape[1], pitch_out)), guard, np.complex64)
    if in_place:
        flat = buf.reshape(-1)
        flat[: x.size] = x.reshape(-1)
        dst = src = gpu.DeviceBuffer.from_array(buf)
    else:
        src = gpu.DeviceBuffer.from_array(x)
        dst = gpu.DeviceBuffer.from_array(np.full((batch, pitch_out), guard, np.complex64))
    plan.execute(src, dst, direction)
    gpu.synchronize()
    return dst.download((batch, pitch_out), np.complex64)


# 256 CUs: 2^15 takes a partial round from 128 transforms, 2^16 from 176; behind 1-3 full rounds from 96, behind 4 from 32
@pytest.mark.parametrize("n,batch,inverse,in_place,pad", [
    (1 << 15, 128, False, False, 0), (1 << 15, 257, True, True, 0), (1 << 15, 352, False, False, 24),
    (1 << 15, 1056, True, False, 0), (1 << 16, 176, False, False, 0), (1 << 16, 256, True, True, 8),
    (1 << 16, 259, False, True, 0), (1 << 16, 609, True, False, 40)])
def test_rounds_match_fp64_and_the_four_step(gpu, po, n, batch, inverse, in_place, pad):
    print(f"whole n={n} batch={batch} inverse={inverse} in_place={in_place} pad={pad}", flush=True)
    rng = np.random.default_rng(n + batch)
    pitch = n + pad
    x = _input(rng, batch, n, pitch)
    direction = gpu.INVERSE if inverse else gpu.FORWARD
    guard = np.complex64(complex(-3.25, 7.5))
    plan = gpu.FftPlan(n, batch, idist=pitch, odist=pitch)
    y = _run(gpu, plan, x, pitch, in_place, direction, guard)
    rows = sorted({0, 1, 127, batch // 2, 255, 256, 511, 512, batch - 1} & set(range(batch)))
    ref = po.fft64_of_f32(np.ascontiguousarray(x[rows, :n]), inverse=inverse)
    assert po.rel_l2(y[rows, :n], ref) <= bound(n)
    four = gpu.FftPlan(n, batch, idist=pitch, odist=pitch, tuning={"chunk": plan.info()["chunk"]})
    z = _run(gpu, four, x, pitch, False, direction, guard)
    for r in range(batch):
        assert po.rel_l2(y[r, :n], z[r, :n].astype(np.complex128)) <= 2 * bound(n), r
    if pad:  # the padding is the caller's: untouched out of place, the input's in place
        want = x[:, n:] if in_place else np.full((batch, pad), guard, np.complex64)
        assert np.array_equal(y[:, n:].view(np.uint32), np.ascontiguousarray(want).view(np.uint32))


def test_in_place_with_different_distances(gpu, po):
    """In place with odist > idist a workgroup's next input would be overwritten: the four-step still runs it."""
    n, batch = 1 << 15, 200
    rng = np.random.default_rng(3)
    x = _input(rng, batch, n, n)
    plan = gpu.FftPlan(n, batch, idist=n, odist=n + 16)
    a = _run(gpu, plan, x, n + 16, False, gpu.FORWARD, np.complex64(0))
    b = _run(gpu, plan, x, n + 16, True, gpu.FORWARD, np.complex64(0))
    for r in (0, 1, 57, batch - 1):
        assert po.rel_l2(b[r, :n], a[r, :n].astype(np.complex128)) <= 2 * bound(n), r


def test_rerun_is_bit_identical(gpu):
    n, batch = 1 << 16, 300
    x = _input(np.random.default_rng(5), batch, n, n)
    plan = gpu.FftPlan(n, batch)
    a = _run(gpu, plan, x, n, False, gpu.FORWARD, np.complex64(0))
    b = _run(gpu, plan, x, n, True, gpu.FORWARD, np.complex64(0))
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))

"""The whole-transform kernel of n = 2^15 and 2^16 C2C and n = 2^16 R2C / C2R (one workgroup per transform, persistent over rounds of one
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


# rows of h + 1 bins start at every residue of a 128-byte line; padded rows keep one residue
@pytest.mark.parametrize("batch,pad", [(128, 0), (257, 0), (259, 7), (352, 15), (1056, 1)])
def test_real_rounds_match_fp64_and_the_four_step(gpu, po, batch, pad):
    n = 1 << 16
    h = n // 2
    pitch = h + 1 + pad
    print(f"whole real batch={batch} pad={pad}", flush=True)
    rng = np.random.default_rng(batch + pad)
    x = rng.standard_normal((batch, n), dtype=np.float32)
    guard = np.complex64(complex(-3.25, 7.5))
    r2c = gpu.FftPlan(n, batch, "r2c", odist=pitch)
    c2r = gpu.FftPlan(n, batch, "c2r", idist=pitch)
    xin = gpu.DeviceBuffer.from_array(x)
    spec = gpu.DeviceBuffer.from_array(np.full((batch, pitch), guard, np.complex64))
    back = gpu.DeviceBuffer(4 * n * batch)
    r2c.execute(xin, spec, gpu.FORWARD)
    c2r.execute(spec, back, gpu.INVERSE)
    gpu.synchronize()
    X = spec.download((batch, pitch), np.complex64)
    rows = sorted({0, 1, 2, 15, 16, 127, batch // 2, 255, 256, batch - 1} & set(range(batch)))
    assert po.rel_l2(X[rows][:, : h + 1], po.rfft64(x[rows].astype(np.float64))) <= bound(n)
    assert not np.any(X[:, 0].imag) and not np.any(X[:, h].imag)
    assert np.array_equal(X[:, h + 1:].view(np.uint32), np.full((batch, pad), guard, np.complex64).view(np.uint32))
    xb = back.download((batch, n), np.float32)
    assert po.rel_l2(xb, x.astype(np.float64)) <= 2 * bound(n)
    # the inverse on a spectrum that is no transform of reals at 0 and h: the four-step's formula, all rows
    X[:, 0] += 1j
    X[:, h] -= 2j
    spec2 = gpu.DeviceBuffer.from_array(X)
    four_r = gpu.FftPlan(n, batch, "r2c", odist=pitch, tuning={"chunk": r2c.info()["chunk"]})
    four_c = gpu.FftPlan(n, batch, "c2r", idist=pitch, tuning={"chunk": c2r.info()["chunk"]})
    other = gpu.DeviceBuffer(4 * n * batch)
    c2r.execute(spec2, back, gpu.INVERSE)
    four_c.execute(spec2, other, gpu.INVERSE)
    four_r.execute(xin, spec, gpu.FORWARD)
    gpu.synchronize()
    a, b = back.download((batch, n), np.float32), other.download((batch, n), np.float32)
    Y = spec.download((batch, pitch), np.complex64)
    for r in range(batch):
        assert po.rel_l2(a[r], b[r].astype(np.float64)) <= 2 * bound(n), r
        if r not in rows:
            assert po.rel_l2(X[r, 1:h], Y[r, 1:h].astype(np.complex128)) <= 2 * bound(n), r


# padded reals on both sides (even distances), padded bins, and bases at every residue of a 128-byte line: the R2C stores are laid
# out by the residue of each row of bins, whichever of base and distance makes it
@pytest.mark.parametrize("pad_real,pad_bins,base_real,base_bins", [(2, 0, 0, 0), (6, 3, 1, 1), (30, 15, 2, 5), (2, 14, 0, 8),
                                                                   (10, 1, 3, 15), (0, 15, 7, 11), (64, 2, 16, 2)])
def test_real_rows_at_any_distance_and_base(gpu, po, pad_real, pad_bins, base_real, base_bins):
    """base_real pairs of reals and base_bins bins into their allocations; the gaps between rows keep what was there, and the
    values equal those of packed rows bit for bit."""
    n, batch = 1 << 16, 130
    h = n // 2
    ri, co = n + pad_real, h + 1 + pad_bins
    print(f"whole real pads {pad_real} {pad_bins} bases {base_real} {base_bins}", flush=True)
    rng = np.random.default_rng(pad_real + pad_bins)
    x = rng.standard_normal((batch, n), dtype=np.float32)
    packed = gpu.FftPlan(n, batch, "r2c")
    spec, back = gpu.DeviceBuffer(8 * (h + 1) * batch), gpu.DeviceBuffer(4 * n * batch)
    packed.execute(gpu.DeviceBuffer.from_array(x), spec, gpu.FORWARD)
    gpu.FftPlan(n, batch, "c2r").execute(spec, back, gpu.INVERSE)
    gpu.synchronize()
    X, xb = spec.download((batch, h + 1), np.complex64), back.download((batch, n), np.float32)
    rows = [0, 1, batch - 1]
    assert po.rel_l2(X[rows], po.rfft64(x[rows].astype(np.float64))) <= bound(n)
    reals = np.full(2 * base_real + batch * ri, -7.25, np.float32)
    bins = np.full(base_bins + batch * co, np.complex64(complex(2.5, -1.5)))
    reals[2 * base_real:].reshape(batch, ri)[:, :n] = x
    src, dst = gpu.DeviceBuffer.from_array(reals), gpu.DeviceBuffer.from_array(bins)
    r2c = gpu.FftPlan(n, batch, "r2c", idist=ri, odist=co)
    c2r = gpu.FftPlan(n, batch, "c2r", idist=co, odist=ri)
    assert r2c.info()["whole"] == c2r.info()["whole"] == batch
    r2c.execute(src.address + 8 * base_real, dst.address + 8 * base_bins, gpu.FORWARD)
    gpu.synchronize()
    want = bins.copy()
    want[base_bins:].reshape(batch, co)[:, : h + 1] = X
    assert np.array_equal(dst.download(want.shape, np.complex64).view(np.uint32), want.view(np.uint32))
    src.upload(np.full_like(reals, -7.25))
    c2r.execute(dst.address + 8 * base_bins, src.address + 8 * base_real, gpu.INVERSE)
    gpu.synchronize()
    want = np.full_like(reals, -7.25)
    want[2 * base_real:].reshape(batch, ri)[:, :n] = xb
    assert np.array_equal(src.download(want.shape, np.float32).view(np.uint32), want.view(np.uint32))


def test_rerun_of_the_real_forms_is_bit_identical(gpu):
    n, batch = 1 << 16, 300
    h = n // 2
    x = np.random.default_rng(6).standard_normal((batch, n), dtype=np.float32)
    r2c, c2r = gpu.FftPlan(n, batch, "r2c"), gpu.FftPlan(n, batch, "c2r")
    xin, spec, back = gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer(8 * (h + 1) * batch), gpu.DeviceBuffer(x.nbytes)
    out = []
    for _ in range(2):
        r2c.execute(xin, spec, gpu.FORWARD)
        c2r.execute(spec, back, gpu.INVERSE)
        gpu.synchronize()
        out.append((spec.download((batch, h + 1), np.complex64), back.download((batch, n), np.float32)))
    for a, b in zip(*out):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("n,batch,type", [(1 << 16, 512, "c2c"), (1 << 15, 300, "c2c"), (1 << 16, 512, "r2c"),
                                          (1 << 16, 300, "c2r")])
def test_tuning_reaches_the_planners_plan(gpu, n, batch, type):
    """Candidate 0 of the tuner, and the tuning of a record of the untuned plan, launch what an untuned plan launches."""
    import ctypes

    from crd_amd import _native as N
    from crd_amd import costmodel

    code = {"c2c": N.C2C, "r2c": N.R2C, "c2r": N.C2R}[type]
    direction = gpu.INVERSE if type == "c2r" else gpu.FORWARD
    src, dst = gpu.DeviceBuffer(8 * (n + 2) * batch), gpu.DeviceBuffer(8 * (n + 2) * batch)
    src.fill(0)

    def launches(tuning):
        plan = gpu.FftPlan(n, batch, type, tuning=tuning)
        assert plan.info()["check"] == N.CHECK_PASSED
        acc = plan.execute_profiled(src, dst, direction)
        return [acc.launches[i] for i in range(4)], [acc.points[i] for i in range(4)], plan.info()["whole"]

    plain = launches(None)
    assert plain[2] > 0
    rec = N.PlanRecord()
    N.check(N.lib().crdfft_time_plan(n, batch, code, None, 3, ctypes.byref(rec)))
    for t in (costmodel.candidates(n, batch, type)[0], rec.tuning):
        assert launches({f: getattr(t, f) for f, _ in N.Tuning._fields_}) == plain
    best = N.Tuning()
    N.check(N.lib().crdfft_autotune_plan(n, batch, code, 5, ctypes.byref(best), None, 0, None))
    N.check(N.lib().crdfft_time_plan(n, batch, code, ctypes.byref(best), 9, ctypes.byref(rec)))
    tuned = rec.ms
    N.check(N.lib().crdfft_time_plan(n, batch, code, None, 9, ctypes.byref(rec)))
    assert tuned <= 1.15 * rec.ms  # the two passes take 1.2-1.9x here


@pytest.mark.parametrize("n,batch,type", [(1 << 15, 256, "c2c"), (1 << 16, 256, "c2c"), (1 << 16, 256, "r2c"),
                                          (1 << 16, 256, "c2r")])
def test_both_forms_are_checked(gpu, n, batch, type):
    """A batch of whole transforms alone runs two passes where its buffers ask for it (below), so a plan whose two passes
    fail their check is demoted too."""
    import os

    from crd_amd import _native as N

    os.environ["CRDFFT_FAULT_SELF_CHECK"] = "3"
    try:
        plan = gpu.FftPlan(n, batch, type)
    finally:
        del os.environ["CRDFFT_FAULT_SELF_CHECK"]
    assert plan.info()["check"] == N.CHECK_DEMOTED and plan.info()["whole"] == 0
    assert plan.self_check() == N.OK
    plan = gpu.FftPlan(n, batch, type)
    assert plan.info()["check"] == N.CHECK_PASSED and plan.info()["whole"] == batch


def test_rows_between_the_rows_of_the_input(gpu, po):
    """Input and output rows in turn in one allocation: disjoint, but their ranges overlap, so two passes run them."""
    n, batch = 1 << 15, 256
    x = _input(np.random.default_rng(9), batch, n, 2 * n)
    buf = gpu.DeviceBuffer.from_array(x)
    plan = gpu.FftPlan(n, batch, idist=2 * n, odist=2 * n)
    acc = plan.execute_profiled(buf.address, buf.address + 8 * n, gpu.FORWARD)
    assert acc.launches[1] > 0
    y = buf.download((batch, 2 * n), np.complex64)
    assert np.array_equal(y[:, :n].view(np.uint32), x[:, :n].view(np.uint32))
    rows = [0, 1, 100, batch - 1]
    assert po.rel_l2(y[rows, n:], po.fft64_of_f32(np.ascontiguousarray(x[rows, :n]))) <= bound(n)


@pytest.mark.parametrize("n,type", [(1 << 15, "c2c"), (1 << 16, "c2c"), (1 << 16, "r2c")])
def test_table_bytes_count_the_whole_transforms_tables(gpu, n, type):
    plan = gpu.FftPlan(n, 256, type)
    two = gpu.FftPlan(n, 256, type, tuning={"chunk": plan.info()["chunk"]})
    points = plan.info()["complex_n"] + 256  # the four-step twiddle of 256 x n2 and W_256
    assert plan.info()["table_bytes"] == two.info()["table_bytes"] + 8 * points

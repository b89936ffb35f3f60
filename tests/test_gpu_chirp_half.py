"""The one-kernel chirp-z form at the lengths where the zero padding's half matters: n = m / 2 exactly (every slot of the
lower half in use), one less, and just above the previous m (almost half of the lower half empty too), for every m it is
instantiated at; odd batches, padded rows, both directions, against numpy's FP64 FFT. Bar: rel-L2 <= 4e-6 log2(m), twice the
plain transform's for the two transforms of m points."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", sorted({2, 3} | {v for m in range(3, 15) for v in
                                              ((1 << m) // 2, (1 << m) // 2 - 1, (1 << m) // 4 + 1)}))
def test_lengths_at_the_edges_of_m(gpu, po, n):
    print(f"chirp-z n={n}", flush=True)
    batch, pad = max(3, 20001 // n), 5
    rng = np.random.default_rng(n)
    x = rng.standard_normal((batch, 2 * (n + pad)), dtype=np.float32).view(np.complex64)
    plan = gpu.BluesteinPlan(n, batch, idist=n + pad, odist=n + pad, chirp_z=True)
    m = plan.conv_size()
    assert m >= 2 * n - 1 and plan.info()["e"] > 0
    guard = np.full((batch, n + pad), np.complex64(complex(9.0, -4.0)))
    src, dst = gpu.DeviceBuffer.from_array(x), gpu.DeviceBuffer.from_array(guard)
    for direction in (gpu.FORWARD, gpu.INVERSE):
        plan.execute(src, dst, direction)
        gpu.synchronize()
        y = dst.download((batch, n + pad), np.complex64)
        v = x[:, :n].astype(np.complex128)
        ref = np.fft.fft(v, axis=1) if direction == gpu.FORWARD else np.fft.ifft(v, axis=1)
        assert po.rel_l2(y[:, :n], ref) <= 4e-6 * np.log2(m)
        assert np.array_equal(y[:, n:].view(np.uint32), np.ascontiguousarray(guard[:, n:]).view(np.uint32))

"""Dots whose result the host polls for: the same bits as the dot that stays
on the device, at one workgroup, at the edges of the one-launch form (1,024
workgroups of 256 elements) and above it, repeated, unaligned tails included,
and sums that are no number."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 513, 65025, 262143, 262144, 262145, 1200001])
def test_host_dot_has_the_device_dots_bits(pkg, ctx, n, dtype):
    rng = np.random.default_rng(n)
    D = pkg.Vector(ctx, 1)
    for rep in range(3):
        x, y = rng.uniform(-1, 1, n), rng.uniform(-1, 1, n)
        X, Y = pkg.Vector(ctx, x, dtype), pkg.Vector(ctx, y, dtype)
        X.dot_dev(Y, D)
        want = D.numpy()[0]
        got = X.dot(Y)
        assert got == (want if dtype == np.float64 else float(np.float32(want)))
        assert X.nrm2() == X.nrm2()


@pytest.mark.parametrize("n", [100, 70000, 300000])
def test_host_dot_special_values(pkg, ctx, n):
    sentinel = np.array([0x7FF4DEAD5EEDBEEF], np.uint64).view(np.float64)[0]
    one = pkg.Vector(ctx, np.ones(n))
    for v in (np.inf, -np.inf, np.nan, sentinel):
        x = np.zeros(n)
        x[n // 2] = v
        got = pkg.Vector(ctx, x).dot(one)
        assert got == v if np.isinf(v) else np.isnan(got)
    assert one.dot(one) == n        # the next dot is not affected


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("n", [513, 65025, 262144])
def test_dot_that_gives_up_waiting(pkg, ctx, n, dtype):
    """A one-launch dot that does not wait for its partials hands over to the
    finisher: the same bits, and partials that came late reach no later dot."""
    rng = np.random.default_rng(n)
    vecs = [pkg.Vector(ctx, rng.uniform(-1, 1, n), dtype) for _ in range(6)]
    want = [v.dot(vecs[0]) for v in vecs]
    for rep in range(3):
        ctx.set_wait_polls(1)
        try:
            assert [v.dot(vecs[0]) for v in vecs] == want
        finally:
            ctx.set_wait_polls(0)
        assert [v.dot(vecs[0]) for v in vecs] == want

"""Level 1 at the sizes where a call changes its launch: below one vector, a
partial last vector, one workgroup against several (four trips of its loads),
at odd element offsets of either operand, and strided batches.

Updates are bit-exact (one operation per element); elements around the vectors
keep their bits. Reductions add FP64 partial sums of at most 4 * 16 (unit
stride) or 4 (strided) products per chain of T: the bound is 64 * eps *
sum |x_i y_i| + eps * |result|.
"""
import numpy as np
import pytest

from gpu_util import bitwise_equal, to_dev, to_host

pytestmark = pytest.mark.gpu
DT = {"S": np.float32, "D": np.float64}
# one trip of dot: 256 threads x 4 vectors (FP32 4096, FP64 2048 elements); of
# asum 16384 FP32, 4096 FP64 (512 threads)
SIZES = [1, 2, 3, 5, 1023, 1025, 8191, 8192, 8195, 16383, 16384, 16387, 65535,
         65537, 65541, 70001]


@pytest.mark.parametrize("p", ["S", "D"])
@pytest.mark.parametrize("ox,oy", [(0, 0), (1, 0), (0, 3), (1, 1)])
def test_updates_and_sums(hc, handle, orc, p, ox, oy):
    dt, api = DT[p], hc.api
    eps = np.finfo(dt).eps
    for n in SIZES:
        rng = np.random.default_rng(n + ox)
        x = rng.uniform(-1, 1, n + 8).astype(dt)
        y = rng.uniform(-1, 1, n + 8).astype(dt)
        dx, dy = to_dev(x), to_dev(y)
        px = dx.data_ptr() + ox * x.itemsize
        py = dy.data_ptr() + oy * y.itemsize
        xs, ys = x[ox:ox + n], y[oy:oy + n]
        exp = y.copy()
        exp[oy:oy + n] = orc.axpy(dt(-1.5), xs.copy(), ys.copy())
        assert getattr(api, f"hcblas{p}axpy")(handle, n, -1.5, px, 1, py, 1) == 0
        assert bitwise_equal(to_host(dy), exp), n
        exp[oy:oy + n] *= dt(0.3)
        assert getattr(api, f"hcblas{p}scal")(handle, n, float(dt(0.3)),
                                              py, 1) == 0
        assert bitwise_equal(to_host(dy), exp), n
        ys = exp[oy:oy + n].astype(np.float64)
        xs = xs.astype(np.float64)
        for _ in range(2):
            st, d = getattr(api, f"hcblas{p}dot")(handle, n, px, 1, py, 1, None)
            assert st == 0
            assert abs(d - np.dot(xs, ys)) <= 64 * eps * np.dot(
                abs(xs), abs(ys)) + eps * abs(d), n
            st, a = getattr(api, f"hcblas{p}asum")(handle, n, px, 1, None)
            assert st == 0
            assert abs(a - abs(xs).sum()) <= 65 * eps * a, n
        exp[oy:oy + n] = x[ox:ox + n]
        assert getattr(api, f"hcblas{p}copy")(handle, n, px, 1, py, 1) == 0
        assert bitwise_equal(to_host(dy), exp), n


@pytest.mark.parametrize("p", ["S", "D"])
@pytest.mark.parametrize("n,batch", [(1, 3), (300, 1), (341, 3), (1024, 1),
                                     (1025, 1), (1000, 70)])
def test_strided_batches(hc, handle, p, n, batch):
    dt, api = DT[p], hc.api
    rng = np.random.default_rng(n + batch)
    x = rng.uniform(-1, 1, 2 * n * batch).astype(dt)
    y = rng.uniform(-1, 1, 3 * n * batch).astype(dt)
    dx, dy = to_dev(x), to_dev(y)
    # the C API's batch stride is n elements: keep inc = 1 in x's batch
    inc = 2 if batch == 1 else 1
    xs = x[:n * batch * inc:inc]
    ys = y[:n * batch * inc:inc]
    eps = np.finfo(dt).eps
    st, d = getattr(api, f"hcblas{p}dotBatched")(handle, n, dx, inc, dy, inc,
                                                 None, batch)
    assert st == 0
    ref = np.dot(xs.astype(np.float64), ys.astype(np.float64))
    mag = np.dot(abs(xs).astype(np.float64), abs(ys).astype(np.float64))
    assert abs(d - ref) <= 64 * eps * mag + eps * abs(d)
    exp = y.copy()
    exp[:n * batch * inc:inc] = xs
    assert getattr(api, f"hcblas{p}copyBatched")(handle, n, dx, inc, dy, inc,
                                                 batch) == 0
    assert bitwise_equal(to_host(dy), exp)


@pytest.mark.parametrize("inc", [1, 2])
def test_short_float_sums_are_exact(hc, handle, inc):
    """Up to four trips of one workgroup, FP32 sums are held in FP64: of values
    that are multiples of 2^-24, whose sums FP64 holds exactly, the result is the
    exact sum rounded once (FP32 partial sums of two such values already round)."""
    api = hc.api
    trip_dot, trip_asum = (4096, 16384) if inc == 1 else (256, 256)
    for trip, name in ((trip_dot, "dot"), (trip_asum, "asum")):
        for n in (trip, trip + 1, trip + 4, 2 * trip, 3 * trip - 5, 4 * trip):
            rng = np.random.default_rng(n)
            x = rng.integers(1 << 23, 1 << 24, n * inc).astype(np.float64)
            x = (x * 2.0 ** -24).astype(np.float32)
            y = rng.choice([-1, 1], n * inc).astype(np.float32)
            dx, dy = to_dev(x), to_dev(y)
            xs, ys = x[::inc].astype(np.float64), y[::inc].astype(np.float64)
            if name == "dot":
                st, got = api.hcblasSdot(handle, n, dx, inc, dy, inc, None)
                want = np.float32(np.dot(xs, ys))
            else:
                st, got = api.hcblasSasum(handle, n, dx, inc, None)
                want = np.float32(xs.sum())
            assert st == 0
            assert np.float32(got) == want, (name, n, got, want)


@pytest.mark.parametrize("p", ["S", "D"])
@pytest.mark.parametrize("n,batch", [(1, 1000), (5, 300), (191, 9), (192, 9),
                                     (255, 70), (257, 70), (383, 5), (384, 5),
                                     (16, 70000), (250, 70000)])
@pytest.mark.parametrize("inc", [1, -2])
def test_strided_update_grids(hc, handle, p, n, batch, inc):
    """Batches of short vectors at a batch stride of their own: the flat grid, and
    the one by rows, with more vectors than it has rows. Gaps keep their bits."""
    dt = DT[p]
    step = n * abs(inc) + 3
    rng = np.random.default_rng(n + batch)
    x = rng.uniform(-1, 1, (batch, step)).astype(dt)
    y = rng.uniform(-1, 1, (batch, step)).astype(dt)
    dy = to_dev(y)
    assert getattr(hc.api, f"hcblas_{p.lower()}axpy_batched")(
        handle, n, -1.5, to_dev(x), inc, step, dy, abs(inc), step, 0, 0,
        batch) == 0
    xs = x[:, :n * abs(inc):abs(inc)]
    exp = y.copy()
    # one fused operation: the exact product and sum of these values rounds once
    wide = np.longdouble if p == "D" else np.float64
    s = xs[:, ::-1] if inc < 0 else xs
    exp[:, :n * abs(inc):abs(inc)] = (
        wide(-1.5) * s.astype(wide) + y[:, :n * abs(inc):abs(inc)].astype(wide)
    ).astype(dt)
    got = to_host(dy)
    gaps = np.ones(step, bool)
    gaps[:n * abs(inc):abs(inc)] = False
    assert bitwise_equal(got[:, gaps], y[:, gaps])
    # (a double rounding of the wide form differs by at most one ulp)
    assert np.all(abs(got - exp) <= np.finfo(dt).eps * abs(exp))

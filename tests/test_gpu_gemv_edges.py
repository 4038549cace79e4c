"""GEMV and GER at the sizes where the launch plan changes kernel or band, on
tightly packed matrices with any row count (the last vector of a column is
read from row R - VN on), at odd element offsets, and with non-finite rows
next to the edge.

Bound against the FP64 value: the sum of L products in any order is within
(L + 2) * eps * (|alpha| |A| |x| + |beta| |y|) componentwise, eps the unit of
the type; GER is one fused multiply-add per element and bit-exact.
"""
import numpy as np
import pytest

from gpu_util import bitwise_equal, to_dev, to_host

pytestmark = pytest.mark.gpu
COL, ROW = 1, 0
DT = {"s": np.float32, "d": np.float64}

# Storage rows R and columns: below one vector; the panel kernel (sixteen
# waves up to 512 columns, splits beyond); three quarters of a band step and
# its neighbours; bands of 1, 2, 4 and 10 row steps with partial last bands;
# few columns (short bands) and many.
SHAPES = [(1, 40), (3, 700), (5, 33), (190, 511), (255, 513), (383, 129),
          (385, 65), (767, 64), (769, 2050), (1021, 31), (1025, 300),
          (2047, 1030), (4097, 77), (5003, 600), (8193, 130), (20011, 9),
          (10007, 259)]


@pytest.mark.parametrize("p", ["s", "d"])
@pytest.mark.parametrize("trans", [0, 1])
def test_plan_edges(hc, handle, p, trans):
    dt = DT[p]
    eps = np.finfo(dt).eps
    for R, Cc in SHAPES:
        rng = np.random.default_rng(R + Cc)
        m = rng.uniform(-1, 1, (Cc, R)).astype(dt)  # column-major R x Cc
        A = np.concatenate([np.full(1, 99, dt), m.ravel(), np.full(9, 99, dt)])
        op = m if trans else m.T
        ly, lx = op.shape
        dA = to_dev(A)
        for incx in (1, -2):
            x = rng.uniform(-1, 1, lx).astype(dt)
            xs = np.zeros(1 + (lx - 1) * abs(incx), dt)
            xs[::abs(incx)] = x if incx > 0 else x[::-1]
            y = rng.uniform(-1, 1, ly + 1).astype(dt)
            dy = to_dev(y)
            st = getattr(hc.api, f"hcblas_{p}gemv")(
                handle, COL, trans, R, Cc, 1.5, dA, 1, R, to_dev(xs), 0, incx,
                -0.5, dy, 1, 1)
            assert st == 0
            got = to_host(dy)
            assert got[0] == y[0]
            o, x64, y64 = op.astype(np.float64), x.astype(np.float64), y[1:]
            ref = 1.5 * (o @ x64) - 0.5 * y64
            bound = (lx + 2) * eps * (1.5 * (abs(o) @ abs(x64)) +
                                      0.5 * abs(y64)) + eps * abs(ref)
            assert np.all(abs(got[1:] - ref) <= bound), (R, Cc, incx)


@pytest.mark.parametrize("p", ["s", "d"])
def test_edge_rows_do_not_leak(hc, handle, p):
    """An infinity in the rows that a moved last vector reads twice appears in
    each sum once: the column sums are infinite, not NaN, and no other row's
    sum sees it."""
    dt = DT[p]
    for R, Cc in [(5, 40), (259, 20), (1027, 24), (20011, 16)]:
        m = np.ones((Cc, R), dt)
        m[:, R - 2] = np.inf
        y = to_dev(np.zeros(Cc, dt))
        st = getattr(hc.api, f"hcblas{p.upper()}gemv")(
            handle, 1, R, Cc, 1.0, to_dev(m), R, to_dev(np.ones(R, dt)), 1,
            0.0, y, 1)
        assert st == 0
        assert np.all(to_host(y) == np.inf), (R, Cc)
        y = to_dev(np.zeros(R, dt))
        st = getattr(hc.api, f"hcblas{p.upper()}gemv")(
            handle, 0, R, Cc, 1.0, to_dev(m), R, to_dev(np.ones(Cc, dt)), 1,
            0.0, y, 1)
        assert st == 0
        exp = np.full(R, Cc, dt)
        exp[R - 2] = np.inf
        assert np.array_equal(to_host(y), exp), (R, Cc)


@pytest.mark.parametrize("p", ["s", "d"])
def test_ger_any_alignment(hc, handle, orc, p):
    dt = DT[p]
    for M, N in [(1, 17), (3, 16), (5, 33), (1023, 17), (1025, 40), (2051, 16)]:
        rng = np.random.default_rng(M + N)
        A = rng.uniform(-1, 1, M * N + 9).astype(dt)
        x, y = rng.uniform(-1, 1, M).astype(dt), rng.uniform(-1, 1, N).astype(dt)
        dA = to_dev(A)
        st = getattr(hc.api, f"hcblas_{p}ger")(
            handle, COL, M, N, 1.5, to_dev(x), 0, 1, to_dev(y), 0, 1, dA, 1, M)
        assert st == 0
        exp = A.copy()
        exp[1:1 + M * N] = orc.ger(COL, M, N, 1.5, x, 1, y, 1,
                                   A[1:1 + M * N].copy(), M)
        assert bitwise_equal(to_host(dA), exp), (M, N)


@pytest.mark.parametrize("p", ["s", "d"])
def test_ger_out(hc, handle, orc, p):
    """D = alpha x y^T + A: bit-exact as GER in place, other leading dimensions
    for A and D, A left alone; alpha == 0 copies A, also beside an infinity."""
    dt = DT[p]
    for M, N in [(1, 17), (3, 16), (5, 33), (1025, 40), (2051, 16)]:
        for order in (COL, ROW):
            rng = np.random.default_rng(M + N)
            R, Cc = (M, N) if order == COL else (N, M)
            lda, ldd = R + 3, R + 1
            A = rng.uniform(-1, 1, lda * Cc + 1).astype(dt)
            D = rng.uniform(-1, 1, ldd * Cc + 1).astype(dt)
            x = rng.uniform(-1, 1, M).astype(dt)
            y = rng.uniform(-1, 1, 2 * N).astype(dt)
            for alpha in (1.5, 0.0):
                if alpha == 0.0:
                    x[0] = np.inf
                dA, dD = to_dev(A), to_dev(D)
                st = getattr(hc.api, f"hcblas_{p}ger_out")(
                    handle, order, M, N, alpha, to_dev(x), 1, to_dev(y), -2,
                    dA[1:], lda, dD[1:], ldd)
                assert st == 0
                exp = D.copy()
                e = exp[1:].reshape(Cc, ldd)
                e[:, :R] = A[1:].reshape(Cc, lda)[:, :R]
                if alpha:
                    t = orc.ger(order, M, N, alpha, x, 1, y, -2,
                                np.ascontiguousarray(e[:, :R]).ravel(), R)
                    e[:, :R] = t.reshape(Cc, R)
                assert bitwise_equal(to_host(dD), exp), (M, N, order, alpha)
                assert bitwise_equal(to_host(dA), A)


# Storage rows R and columns of the pair kernel: 4 MB and just below; bands of
# 1, 2 and 4 row steps with partial last vectors, steps and bands; several
# bands and one; blocks of fewer columns than a trip, and one of 512.
PAIR = [(767, 1400), (769, 1401), (1023, 1021), (1027, 1030), (4096, 259),
        (4099, 300), (5003, 257), (8193, 130), (16389, 64), (30001, 77),
        (1025, 9001)]


@pytest.mark.parametrize("p", ["s", "d"])
def test_ger_backward_pair(hc, handle, p):
    dt = DT[p]
    eps = np.finfo(dt).eps
    for R, Cc in PAIR:
        rng = np.random.default_rng(R + Cc)
        m = rng.uniform(-1, 1, (Cc, R + 1)).astype(dt)  # ld = R + 1
        S = m[:, :R].T.astype(np.float64)
        dS = to_dev(np.concatenate([np.zeros(1, dt), m.ravel()]))
        a = rng.uniform(-1, 1, R).astype(dt)
        b = rng.uniform(-1, 1, Cc).astype(dt)
        for order in (COL, ROW):
            M, N = (R, Cc) if order == COL else (Cc, R)
            x, y = (a, b) if order == COL else (b, a)
            ys = np.zeros(2 * N - 1, dt)
            ys[::2] = y[::-1]
            dx, dy = to_dev(np.full(M, 7, dt)), to_dev(np.full(N, 7, dt))
            st = getattr(hc.api, f"hcblas_{p}ger_backward")(
                handle, order, M, N, 1.5, to_dev(x), 1, to_dev(ys), -2,
                dS[1:], R + 1, dx, dy)
            assert st == 0
            G = S if order == COL else S.T
            for got, op, v in ((dx, G, y), (dy, G.T, x)):
                v = v.astype(np.float64)
                bound = (len(v) + 2) * eps * 1.5 * (abs(op) @ abs(v))
                assert np.all(abs(to_host(got) - 1.5 * (op @ v)) <= bound), \
                    (R, Cc, order)


@pytest.mark.parametrize("p", ["s", "d"])
def test_pair_edge_rows_do_not_leak(hc, handle, p):
    """As test_edge_rows_do_not_leak, through the adjoint of GER."""
    dt = DT[p]
    for R, Cc in [(1027, 1100), (20011, 80)]:
        m = np.ones((Cc, R), dt)
        m[:, R - 2] = np.inf
        dx, dy = to_dev(np.zeros(R, dt)), to_dev(np.zeros(Cc, dt))
        st = getattr(hc.api, f"hcblas_{p}ger_backward")(
            handle, COL, R, Cc, 1.0, to_dev(np.ones(R, dt)), 1,
            to_dev(np.ones(Cc, dt)), 1, to_dev(m), R, dx, dy)
        assert st == 0
        assert np.all(to_host(dy) == np.inf), (R, Cc)
        exp = np.full(R, Cc, dt)
        exp[R - 2] = np.inf
        assert np.array_equal(to_host(dx), exp), (R, Cc)


@pytest.mark.parametrize("p", ["s", "d"])
@pytest.mark.parametrize("R,Cc", [(1, 1), (3, 17), (5, 16), (7, 33), (23, 46),
                                  (179, 125), (1022, 31), (1025, 15), (2051, 48)])
@pytest.mark.parametrize("src", [False, True])
def test_ger_edge_rows_and_columns(hc, handle, p, R, Cc, src):
    """Rows that are no whole vector beside columns that are no whole block, in
    place and into another matrix: each element is one fused operation, and
    the padding between columns keeps its bits."""
    dt = np.float32 if p == "s" else np.float64
    rng = np.random.default_rng(R + Cc)
    ld, ldd = R + 2, R + 3
    A = rng.uniform(-1, 1, (Cc, ld)).astype(dt)
    D = rng.uniform(-1, 1, (Cc, ldd)).astype(dt)
    x, y = rng.uniform(-1, 1, R).astype(dt), rng.uniform(-1, 1, Cc).astype(dt)
    dA, dD = to_dev(A), to_dev(D)
    dx, dy = to_dev(x), to_dev(y)
    if src:
        st = getattr(hc.api, f"hcblas_{p}ger_out")(
            handle, 1, R, Cc, 0.75, dx, 1, dy, 1, dA, ld, dD, ldd)
        out, pad = to_host(dD), D
        assert np.array_equal(to_host(dA), A)
    else:
        st = getattr(hc.api, f"hcblas_{p}ger")(
            handle, 1, R, Cc, 0.75, dx, 0, 1, dy, 0, 1, dA, 0, ld)
        out, pad = to_host(dA), A
    assert st == 0
    wide = np.longdouble
    # alpha * y rounds once, the fused multiply-add once (through an
    # extended type, at most one more unit)
    t = (dt(0.75) * y).astype(dt)
    want = (t.astype(wide)[:, None] * x.astype(wide) + A[:, :R].astype(wide)).astype(dt)
    assert st == 0
    eps = np.finfo(dt).eps
    assert np.all(abs(out[:, :R] - want) <= eps * abs(want))
    assert np.array_equal(out[:, R:], pad[:, R:])

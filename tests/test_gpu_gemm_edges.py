"""GEMM on operands of any alignment: every size modulo the 16-byte vector,
fewer rows than one vector, tightly packed odd leading dimensions and bases at
odd element offsets, in every order and transpose form.

The reference is the FP64 product of the stored values. The bound is that of
tests/gemm_bounds.py, c * sqrt(K) * u * (|alpha| |op(A)| |op(B)| + |beta| |C|)
plus one rounding of the result, with c = 4 and u the unit of the accumulation
type. Elements of C's buffer outside the M x N block keep their bits.
"""
import numpy as np
import pytest

from gpu_util import to_dev, to_host

pytestmark = pytest.mark.gpu
ROW, COL = 0, 1
DT = {"s": np.float32, "d": np.float64, "h": np.float16}


def _stored(rng, dt, rows, cols, order, skew):
    """rows x cols uniform values, tightly packed in `order` behind `skew`
    elements and followed by seven more: (buffer, leading dimension, the
    matrix in FP64)."""
    v = rng.uniform(-1, 1, (rows, cols)).astype(dt)
    flat = (v if order == ROW else v.T).ravel()
    buf = np.full(skew + flat.size + 7, 99, dt)
    buf[skew:skew + flat.size] = flat
    return buf, max(1, cols if order == ROW else rows), v.astype(np.float64)


def _check(hc, handle, p, order, ta, tb, M, N, K, skew, seed):
    rng = np.random.default_rng(seed)
    dt = DT[p]
    A, lda, Am = _stored(rng, dt, *((K, M) if ta else (M, K)), order, skew)
    B, ldb, Bm = _stored(rng, dt, *((N, K) if tb else (K, N)), order, skew)
    C, ldc, Cm = _stored(rng, dt, M, N, order, skew)
    Am, Bm = Am.T if ta else Am, Bm.T if tb else Bm
    bits = (lambda a: a.view(np.uint16)) if p == "h" else (lambda a: a)
    dC = to_dev(bits(C))
    st = getattr(hc.api, f"hcblas_{p}gemm")(
        handle, order, ta, tb, M, N, K, 0.75, to_dev(bits(A)), lda,
        to_dev(bits(B)), ldb, 0.5, dC, ldc, skew, skew, skew)
    assert st == 0
    got = to_host(dC).view(dt)
    what = (p, order, ta, tb, M, N, K, skew)
    assert np.array_equal(got[:skew], C[:skew]), what
    assert np.array_equal(got[skew + M * N:], C[skew + M * N:]), what
    g = got[skew:skew + M * N].astype(np.float64)
    g = g.reshape(M, N) if order == ROW else g.reshape(N, M).T
    ref = 0.75 * (Am @ Bm) + 0.5 * Cm
    u = np.finfo(np.float64 if p == "d" else np.float32).eps
    bound = 4 * np.sqrt(K) * u * (0.75 * (abs(Am) @ abs(Bm)) + 0.5 * abs(Cm))
    bound += 2 * np.finfo(dt).eps * abs(ref)
    if p == "h":
        bound += np.finfo(dt).smallest_subnormal
    assert np.all(abs(g - ref) <= bound), (what, (abs(g - ref) / bound).max())


@pytest.mark.parametrize("p", ["s", "d", "h"])
@pytest.mark.parametrize("order", [ROW, COL])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_every_residue_of_the_vector(hc, handle, p, order, ta, tb):
    # below one vector, every residue of it, and the edge of a 64-row tile
    for M, N in [(1, 6), (2, 1), (3, 7), (5, 65), (6, 66), (7, 67), (8, 61),
                 (9, 68), (63, 2), (66, 69), (70, 71), (129, 62)]:
        for K in (1, 37):
            for skew in (0, 1):
                _check(hc, handle, p, order, ta, tb, M, N, K, skew,
                       M * 1000 + N * 10 + K + skew)


# The larger tiles (128 x 64 FP64, 128 x 128 and 256 x 256 FP32 / FP16), with
# partial last tiles, a shifted last vector in either direction and a K tail.
@pytest.mark.parametrize("p,M,N,K", [("s", 2051, 2049, 75), ("d", 2051, 1777, 35),
                                     ("h", 2053, 2051, 139),
                                     ("s", 4111, 4097, 67), ("h", 4111, 4097, 67)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_large_tiles_at_odd_sizes(hc, handle, p, M, N, K, ta, tb):
    _check(hc, handle, p, COL, ta, tb, M, N, K, 1, M + N + K)


# Few tiles: 32x32 tiles with a short and a long K step (one of each type's
# thresholds on either side), split K on 32x32 tiles (fewer of them than CUs)
# and on 64x64 tiles, with slices that do not divide K.
@pytest.mark.parametrize("p,M,N,K", [("s", 33, 65, 1023), ("s", 129, 31, 1100),
                                     ("d", 33, 65, 511), ("d", 129, 31, 530),
                                     ("h", 33, 65, 1023), ("h", 129, 31, 1100),
                                     ("s", 35, 66, 2051), ("d", 35, 66, 2051),
                                     ("h", 35, 66, 2051), ("s", 515, 513, 2057),
                                     ("d", 515, 513, 2057), ("h", 515, 513, 2057)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_few_tiles(hc, handle, p, M, N, K, ta, tb):
    _check(hc, handle, p, COL, ta, tb, M, N, K, 1, M + N + K)


# Complex products (embedded by the tile loaders): operands of one element and
# one vector, odd sizes on both sides of a vector and a tile edge, K tails of
# every step length, split-K (twice K reaches 2048), 64x64 to the largest tiles.
COMPLEX = [(1, 1, 1), (1, 5, 3), (3, 1, 2), (7, 2, 1), (33, 31, 17),
           (65, 63, 33), (127, 130, 5), (70, 41, 1100), (520, 1100, 40),
           (2050, 2049, 9)]


@pytest.mark.parametrize("p", ["c", "z"])
@pytest.mark.parametrize("tb", [0, 1, 2])
@pytest.mark.parametrize("ta", [0, 1, 2])
def test_complex_edges(hc, handle, p, ta, tb):
    """Each part of an output is a sum of 2K real products of alpha * a (three
    roundings) and b in some order: within (2K + 6) eps of |alpha||A||B|."""
    dt, rt = (np.complex64, np.float32) if p == "c" else (np.complex128,
                                                          np.float64)
    eps = np.finfo(rt).eps
    for M, N, K in COMPLEX:
        rng = np.random.default_rng(M + N + K)

        def rand(r, c):
            v = rng.uniform(-1, 1, (r, c)) + 1j * rng.uniform(-1, 1, (r, c))
            return v.astype(dt)

        A = rand(K, M) if ta == 0 else rand(M, K)  # column-major storage
        B = rand(N, K) if tb == 0 else rand(K, N)
        C = rand(N, M + 1)
        alpha, beta = 1.25 - 0.5j, 0.75 + 0j
        dC = to_dev(C)
        st = getattr(hc.api, f"hcblas_{p}gemm")(
            handle, 1, ta, tb, M, N, K, alpha,
            to_dev(np.concatenate([np.zeros(1, dt), A.ravel()])), 1,
            A.shape[1], to_dev(np.concatenate([np.zeros(3, dt), B.ravel()])),
            3, B.shape[1], beta, dC, 0, M + 1)
        assert st == 0
        got = to_host(dC)

        def op(X, t):  # storage rows are the matrix's columns
            X = X.astype(np.complex128)
            return X.T if t == 0 else X if t == 1 else X.conj()

        a, b = op(A, ta), op(B, tb)
        ref = alpha * (a @ b) + beta * C.T[:M].astype(np.complex128)
        mag = abs(alpha) * (abs(a) @ abs(b)) + abs(beta * C.T[:M])
        assert np.array_equal(got.T[M], C.T[M])
        assert np.all(abs(got.T[:M] - ref) <= 2 * (2 * K + 6) * eps * mag), \
            (M, N, K)


# Operands shorter than one vector (K or rows), beside whole ones, on small and
# large outputs; K slices of a split product whose last one is a single element
# (the k-contiguous vector then begins in the slice before).
NARROW = [("s", 300, 517, 1), ("s", 300, 517, 3), ("s", 3, 517, 300),
          ("s", 517, 2, 300), ("s", 3, 65, 2305), ("s", 35, 66, 2305),
          ("s", 1100, 1030, 2), ("d", 300, 517, 1), ("d", 1, 517, 300),
          ("d", 517, 1, 130), ("d", 1, 65, 2241), ("d", 35, 66, 2241),
          ("h", 300, 517, 1), ("h", 300, 517, 7), ("h", 5, 517, 300),
          ("h", 517, 7, 300), ("h", 7, 65, 2305), ("h", 35, 66, 2305),
          ("h", 2100, 2050, 5), ("h", 2100, 7, 70)]


@pytest.mark.parametrize("p,M,N,K", NARROW)
@pytest.mark.parametrize("order", [ROW, COL])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_narrow_operands(hc, handle, p, M, N, K, order, ta, tb):
    for skew in (0, 1):
        _check(hc, handle, p, order, ta, tb, M, N, K, skew, M + N + K)


@pytest.mark.parametrize("p,K", [("c", 1), ("c", 1153), ("z", 1), ("z", 1121)])
@pytest.mark.parametrize("M,N", [(1, 40), (37, 1), (35, 66), (300, 130)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (2, 2)])
def test_narrow_complex(hc, handle, p, K, M, N, ta, tb):
    """The same for complex products, within test_complex_edges' bound."""
    dt, rt = (np.complex64, np.float32) if p == "c" else (np.complex128,
                                                          np.float64)
    rng = np.random.default_rng(M + N + K)

    def rand(r, c):
        return (rng.uniform(-1, 1, (r, c))
                + 1j * rng.uniform(-1, 1, (r, c))).astype(dt)

    A = rand(K, M) if ta == 0 else rand(M, K)  # column-major storage
    B = rand(N, K) if tb == 0 else rand(K, N)
    C = rand(N, M)
    dC = to_dev(C)
    alpha, beta = 1.25 - 0.5j, 0.75 + 0j
    assert getattr(hc.api, f"hcblas_{p}gemm")(
        handle, 1, ta, tb, M, N, K, alpha, to_dev(A), 0, A.shape[1], to_dev(B),
        0, B.shape[1], beta, dC, 0, M) == 0
    got = to_host(dC).T

    def op(X, t):
        X = X.astype(np.complex128)
        return X.T if t == 0 else X if t == 1 else X.conj()

    a, b = op(A, ta), op(B, tb)
    ref = alpha * (a @ b) + beta * C.T.astype(np.complex128)
    mag = abs(alpha) * (abs(a) @ abs(b)) + abs(beta * C.T)
    assert np.all(abs(got - ref) <= 2 * (2 * K + 6) * np.finfo(rt).eps * mag)

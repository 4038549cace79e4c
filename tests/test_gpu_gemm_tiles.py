"""GEMM on every macro tile at sizes that are odd on every side (tiles cut short, a
moved last vector in either direction, a K tail, bases at odd offsets), in the
transpose forms; gemm_tile_cases.py says which tile each size runs on."""
import numpy as np
import pytest

from gemm_tile_cases import CASES, FORMS
from gpu_util import to_dev, to_host
from test_gpu_gemm_edges import COL, _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,M,N,K", [c[:4] for c in CASES if c[0] in "sdh"])
@pytest.mark.parametrize("ta,tb", FORMS)
def test_real(hc, handle, p, M, N, K, ta, tb):
    _check(hc, handle, p, COL, ta, tb, M, N, K, 1, M + N + K)


@pytest.mark.parametrize("M,N,K", [c[1:4] for c in CASES if c[0] == "b"])
@pytest.mark.parametrize("ta,tb", FORMS)
def test_bf16(hc, handle, torch_cuda, M, N, K, ta, tb):
    """BF16 operands, FP32 sums and result: the FP32 bound of test_gpu_gemm_edges."""
    torch = torch_cuda
    g = torch.Generator().manual_seed(M + N + K)

    def rand(r, c):  # column-major r x c behind one element
        return torch.cat([torch.zeros(1), torch.rand(c * r, generator=g) * 2 - 1])

    ra, ca = (K, M) if ta else (M, K)
    rb, cb = (N, K) if tb else (K, N)
    A, B = rand(ra, ca).bfloat16(), rand(rb, cb).bfloat16()
    C = rand(M, N)
    dC = C.cuda()
    assert hc.api.hcblas_gemm_strided_batched(
        handle, hc.R_16BF, COL, ta, tb, M, N, K, 0.75, A.cuda(), ra, 1, 0,
        B.cuda(), rb, 1, 0, 0.5, dC, M, 1, 0, 1) == 0
    got = to_host(dC)
    assert got[0] == C[0]
    a = A[1:].double().numpy().reshape(ca, ra)
    b = B[1:].double().numpy().reshape(cb, rb)
    a, b = a if ta else a.T, b if tb else b.T
    c = C[1:].double().numpy().reshape(N, M).T
    ref = 0.75 * (a @ b) + 0.5 * c
    eps = np.finfo(np.float32).eps
    bound = 4 * np.sqrt(K) * eps * (0.75 * (abs(a) @ abs(b)) + 0.5 * abs(c))
    assert np.all(abs(got[1:].reshape(N, M).T - ref) <= bound + 2 * eps * abs(ref))


@pytest.mark.parametrize("p,M,N,K", [c[:4] for c in CASES if c[0] in "cz"])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 2), (1, 0), (2, 1)])
def test_complex(hc, handle, p, M, N, K, ta, tb):
    """Sums of 2K real products of alpha * a (three roundings) and b, in a
    tree or chain of unknown order: c * sqrt(2K) eps, c = 4, as for real ones, plus
    the six roundings of each product's operands and of the result."""
    dt, rt = (np.complex64, np.float32) if p == "c" else (np.complex128,
                                                          np.float64)
    rng = np.random.default_rng(M + N + K)

    def rand(r, c):
        return (rng.uniform(-1, 1, (r, c))
                + 1j * rng.uniform(-1, 1, (r, c))).astype(dt)

    A = rand(K, M) if ta == 0 else rand(M, K)  # column-major storage
    B = rand(N, K) if tb == 0 else rand(K, N)
    C = rand(N, M + 1)
    dC = to_dev(C)
    alpha, beta = 1.25 - 0.5j, 0.75 + 0j
    assert getattr(hc.api, f"hcblas_{p}gemm")(
        handle, COL, ta, tb, M, N, K, alpha,
        to_dev(np.concatenate([np.zeros(1, dt), A.ravel()])), 1, A.shape[1],
        to_dev(np.concatenate([np.zeros(3, dt), B.ravel()])), 3, B.shape[1], beta,
        dC, 0, M + 1) == 0
    got = to_host(dC)
    assert np.array_equal(got.T[M], C.T[M])

    def op(X, t):
        X = X.astype(np.complex128)
        return X.T if t == 0 else X if t == 1 else X.conj()

    a, b = op(A, ta), op(B, tb)
    ref = alpha * (a @ b) + beta * C.T[:M].astype(np.complex128)
    mag = abs(alpha) * (abs(a) @ abs(b)) + abs(beta * C.T[:M])
    # (each part has two products per complex one, each at most |a||b|)
    bound = 2 * (4 * np.sqrt(2 * K) + 6) * np.finfo(rt).eps * mag
    assert np.all(abs(got.T[:M] - ref) <= bound)

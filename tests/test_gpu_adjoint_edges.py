"""BF16 adjoints at the sizes where the mixed kernel can go wrong: every
operand orientation (order x trans), tightly packed odd leading dimensions,
sizes around the 128 and 256 tiles and around the FP32 (4) and BF16 (8)
vectors, K tails, and a cotangent with an infinity, a NaN and subnormals.

Bound: 4 sqrt(n) u |alpha| (|dC| |op(X)|) + 2 u |ref| for n products in FP32
(u = 2^-24), then one rounding to BF16 (2^-8 |ref|).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
U, UB = 2.0 ** -24, 2.0 ** -8


def _adjoints(A, B, W, ta, tb):
    from hcblas_amd import torch_ext
    A = A.clone().requires_grad_()
    B = B.clone().requires_grad_()
    torch_ext.gemm_batched(A, B, transA=ta, transB=tb).backward(W)
    return A.grad.double(), B.grad.double()


def _refs(A, B, W, ta, tb):
    a, b, w = A.double(), B.double(), W.double()
    if ta:
        a = a.mT.contiguous()
    if tb:
        b = b.mT.contiguous()
    dA = w @ b.mT.contiguous()
    dB = a.mT.contiguous() @ w
    return dA.mT if ta else dA, dB.mT if tb else dB


@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("batch,M,N,K", [(2, 3, 5, 7), (3, 9, 130, 33),
                                         (9, 130, 67, 129), (2, 257, 259, 262),
                                         (8, 300, 261, 34), (17, 33, 40, 270)])
def test_every_orientation(torch_cuda, ta, tb, batch, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)

    def rand(*s):
        return torch.rand(s, generator=g, device="cuda") * 2 - 1

    A = (rand(batch, K, M) if ta else rand(batch, M, K)).bfloat16()
    B = (rand(batch, N, K) if tb else rand(batch, K, N)).bfloat16()
    W = rand(batch, M, N)
    got = _adjoints(A, B, W, ta, tb)
    ref = _refs(A, B, W, ta, tb)
    mag = _refs(A.abs(), B.abs(), W.abs(), ta, tb)
    for d, r, m, n in zip(got, ref, mag, (N, M)):
        bound = (4 * n ** 0.5 * U * m + 2 * U * r.abs()) * (1 + UB)
        assert bool(((d - r).abs() <= bound + UB * r.abs()).all())


# Batches that fill the GPU: dA and dB on 128 and 128, 256 and 128, 128 and 256
# tiles (those above run on 64 x 64 ones).
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("batch,M,N,K", [(60, 130, 259, 200),
                                         (64, 509, 515, 261),
                                         (128, 261, 250, 257)])
def test_every_tile(torch_cuda, ta, tb, batch, M, N, K):
    test_every_orientation(torch_cuda, ta, tb, batch, M, N, K)


def test_special_cotangents(torch_cuda):
    M, N, K = 40, 48, 24
    g = torch.Generator(device="cuda").manual_seed(1)
    A = (torch.rand(1, M, K, generator=g, device="cuda") + 0.5).bfloat16()
    B = (torch.rand(1, K, N, generator=g, device="cuda") + 0.5).bfloat16()
    W = torch.rand(1, M, N, generator=g, device="cuda")
    W[0, 3, 5] = float("inf")
    W[0, 7, 9] = float("nan")
    W[0, 11, :] = 2.0 ** -140  # FP32 subnormals
    dA, dB = _adjoints(A, B, W, False, False)
    assert bool(torch.isinf(dA[0, 3]).all()) and bool((dA[0, 3] > 0).all())
    assert bool(torch.isnan(dA[0, 7]).all())
    assert bool(torch.isinf(dB[0, :, 5]).all())
    assert bool(torch.isnan(dB[0, :, 9]).all())
    rest = [i for i in range(M) if i not in (3, 7)]
    ref = _refs(A, B, torch.nan_to_num(W, 0.0, 0.0, 0.0), False, False)[0]
    assert bool(((dA[0, rest] - ref[0, rest]).abs() <=
                 2 * UB * ref[0, rest].abs() + 2.0 ** -130).all())


@pytest.mark.parametrize("e", [-112, -124, -128, -131])
def test_subnormal_cotangents_count(torch_cuda, e):
    """Cotangents around 2^e under operands large enough for normal gradients. The
    planes hold a value to within half of BF16's smallest subnormal, 2^-134; beside
    that only the result's rounding is allowed (2^-8, and 2^-15 for the sums)."""
    M, N, K = 40, 48, 24
    g = torch.Generator(device="cuda").manual_seed(1 - e)

    def rand(*s):
        return torch.rand(*s, generator=g, device="cuda") + 0.5

    A, B = (rand(1, M, K) * 2 ** 20).bfloat16(), (rand(1, K, N) * 2 ** 20).bfloat16()
    W = (rand(1, M, N).double() * 2.0 ** e).float()
    dA, dB = (d.double() for d in _adjoints(A, B, W, False, False))
    w, a, b = W.double(), A.double(), B.double()
    rA, rB = w @ b.mT.contiguous(), a.mT.contiguous() @ w
    lost = 2.0 ** -134
    for d, r, few in ((dA, rA, b.sum(2)[:, None, :]), (dB, rB, a.sum(1)[:, :, None])):
        bound = (2.0 ** -8 + 2.0 ** -15) * r + lost * few
        assert bool((bound < 0.5 * r).all())  # a flushed input fails
        assert bool(((d - r).abs() <= bound).all())


def test_special_cotangents_leave_other_columns(torch_cuda):
    """dB's columns without an Inf or NaN above them, beside those that have one."""
    M, N, K = 40, 48, 24
    g = torch.Generator(device="cuda").manual_seed(2)
    A = (torch.rand(1, M, K, generator=g, device="cuda") + 0.5).bfloat16()
    B = (torch.rand(1, K, N, generator=g, device="cuda") + 0.5).bfloat16()
    W = torch.rand(1, M, N, generator=g, device="cuda")
    W[0, 3, 5], W[0, 7, 9], W[0, 8, 47] = float("inf"), float("nan"), -float("inf")
    dB = _adjoints(A, B, W, False, False)[1]
    rest = [n for n in range(N) if n not in (5, 9, 47)]
    W[0, :, [5, 9, 47]] = 0
    ref = _refs(A, B, W, False, False)[1]
    assert bool(((dB - ref)[0][:, rest].abs() <= 2 * UB * ref[0][:, rest]).all())

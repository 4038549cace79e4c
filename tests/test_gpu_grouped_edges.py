"""Grouped GEMM over tables of odd sizes that all hold a vector: moved edge vectors
in every orientation, odd leading dimensions and offsets, beta != 0, both types.
Bit-identical to per-problem plain launches (which use the same MFMA blocks and do
not split K at these sizes), as first planned and as autotuned, in tables on both
sides of the size from which whole problems go to one XCD."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MEDIUM, SMALL = [9, 17, 33, 63, 65, 131], [9, 11, 15, 17, 31, 33]


def _table(torch, hc, seed, count, sizes):
    rng = np.random.default_rng(seed)
    meta, used = [], [0, 0]
    for _ in range(count):
        d, col, ta, tb = (int(v) for v in rng.integers(0, 2, 4))
        m, n, k = (int(rng.choice(sizes)) for _ in range(3))
        offs, lds = [], []
        for r, c in (((k, m) if ta else (m, k)), ((n, k) if tb else (k, n)), (m, n)):
            ld = (r if col else c) + int(rng.choice([0, 1, 3]))
            skew = int(rng.integers(0, 3))
            offs.append(used[d] + skew)
            lds.append(ld)
            used[d] += ld * (c if col else r) + skew + 5
        alpha, beta = float(rng.choice([1.0, -0.75])), float(rng.choice([0.0, 0.5]))
        meta.append((d, col, ta, tb, m, n, k, alpha, beta, offs, lds))
    g = torch.Generator(device="cuda").manual_seed(seed)
    arenas = [torch.rand(u, generator=g, device="cuda") * 2 - 1 for u in used]
    return meta, [arenas[0], arenas[1].half()]


@pytest.mark.parametrize("count,sizes,whole", [(60, MEDIUM, False),
                                               (700, MEDIUM, True),
                                               (300, SMALL, False),
                                               (1500, SMALL, True)])
def test_odd_tables(hc, handle, torch_cuda, count, sizes, whole):
    torch = torch_cuda
    meta, init = _table(torch, hc, count, count, sizes)
    arenas = [t.clone() for t in init]
    want = [t.clone() for t in init]
    problems = []
    for d, col, ta, tb, m, n, k, alpha, beta, offs, lds in meta:
        es = 4 if d == 0 else 2

        def at(t, i):
            return t[d].data_ptr() + offs[i] * es

        problems.append(hc.GemmProblem(
            hc.R_32F if d == 0 else hc.R_16F, col, ta, tb, m, n, k, 0, alpha, beta,
            at(arenas, 0), lds[0], at(arenas, 1), lds[1], at(arenas, 2), lds[2]))
        fn = hc.api.hcblas_sgemm if d == 0 else hc.api.hcblas_hgemm
        assert fn(handle, col, ta, tb, m, n, k, alpha, at(want, 0), lds[0],
                  at(want, 1), lds[1], beta, at(want, 2), lds[2], 0, 0, 0) == 0
    plan = hc.GroupedPlan(handle, problems)
    try:
        info = plan.info()
        cus = torch.cuda.get_device_properties(0).multi_processor_count
        assert (info["tiles"] * info["tile"] ** 2 > 2 * cus * 64 * 64) == whole
        for tune in (False, True):
            if tune:
                assert plan.autotune(1) == 0
            for _ in range(2):
                for t, u in zip(arenas, init):
                    t.copy_(u)
                assert plan.run() == 0
                torch.cuda.synchronize()
                for d, iv in ((0, torch.int32), (1, torch.int16)):
                    assert torch.equal(arenas[d].view(iv), want[d].view(iv)), (d, tune)
    finally:
        plan.destroy()

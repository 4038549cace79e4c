"""Split reductions (split-K GEMM, split GEMV, the one-pass GER adjoint) and the
memory of their partial sums: captured without a warm-up and replayed among
larger eager calls, on two streams without a wait in between, and without memory
for them.

Every call is deterministic, so its replays and its results on other streams
have the bits of one eager call; that one is compared with the FP64 product
within tests/gemm_bounds.py's c * sqrt(K) * u, c = 4 (plus a rounding of the
result)."""
import numpy as np
import pytest

from gpu_util import to_host

pytestmark = pytest.mark.gpu
ROW, COL = 0, 1
KINDS = ["s", "d", "h", "bf16", "c", "sn", "st", "dn", "dt", "sger", "dger"]


class Call:
    """One call whose reduction is split: its inputs on the GPU and their
    images in FP64. `scale` enlarges its partial sums."""

    def __init__(self, hc, torch, kind, seed, scale=1):
        self.hc, self.kind = hc, kind
        g = torch.Generator(device="cuda").manual_seed(seed)
        self.f = {"s": torch.float32, "d": torch.float64, "h": torch.float16,
                    "b": torch.bfloat16, "c": torch.complex64}[kind[0]]

        def rand(*n):
            t = torch.randn(*n, generator=g, device="cuda",
                            dtype=torch.complex64 if kind == "c" else torch.float64)
            return t.to(self.f)

        if kind in ("s", "d", "h", "bf16", "c"):
            self.m, self.n, self.k = 64 * scale, 48, 3001
            self.a, self.b = rand(self.m, self.k), rand(self.k, self.n)
            out = torch.float32 if kind == "bf16" else self.f
            self.out = [torch.zeros(self.m, self.n, dtype=out, device="cuda")]
        else:
            self.m, self.n = 300 if kind[1:] == "n" else 600, 5000 * scale
            self.a, self.x, self.y = rand(self.m, self.n), rand(self.m), rand(self.n)
            self.out = [torch.zeros_like(v) for v in
                        {"n": [self.x], "t": [self.y]}.get(kind[1:], [self.x, self.y])]

    def __call__(self, h):
        api, k = self.hc.api, self.kind
        if k == "bf16":
            st = api.hcblas_gemm_strided_batched(
                h, self.hc.R_16BF, ROW, 0, 0, self.m, self.n, self.k, 1.0, self.a,
                self.k, 0, 0, self.b, self.n, 0, 0, 0.0, self.out[0], self.n, 0, 0, 1)
        elif k == "c":
            st = api.hcblas_cgemm(
                h, ROW, 0, 0, self.m, self.n, self.k, 1.0, self.a, 0, self.k, self.b,
                0, self.n, 0.0, self.out[0], 0, self.n)
        elif len(k) == 1:
            st = getattr(api, f"hcblas_{k}gemm")(
                h, ROW, 0, 0, self.m, self.n, self.k, 1.0, self.a, self.k, self.b,
                self.n, 0.0, self.out[0], self.n, 0, 0, 0)
        elif k[1:] == "ger":
            st = getattr(api, f"hcblas_{k}_backward")(
                h, ROW, self.m, self.n, 1.0, self.x, 1, self.y, 1, self.a, self.n,
                *self.out)
        else:
            st = getattr(api, f"hcblas_{k[0]}gemv")(
                h, ROW, 0 if k[1] == "n" else 1, self.m, self.n, 1.0, self.a, 0,
                self.n, self.y if k[1] == "n" else self.x, 0, 1, 0.0, self.out[0],
                0, 1)
        assert st == 0

    def host(self):
        return [to_host(t).copy() for t in self.out]

    def clear(self):
        for t in self.out:
            t.fill_(7)

    def check(self, got):
        w = (lambda t: to_host(t.cdouble() if t.is_complex() else t.double()))
        a = w(self.a)
        if hasattr(self, "b"):
            pairs = [(a, w(self.b))]
        else:
            pairs = [(a, w(self.y))] if self.kind[1] == "n" else \
                [(a.T, w(self.x))] if self.kind[1] == "t" else \
                [(a, w(self.y)), (a.T, w(self.x))]
        assert len(pairs) == len(got)
        for (p, q), g in zip(pairs, got):
            ref, mag = p @ q, abs(p) @ abs(q)
            u = np.finfo(np.float64 if self.kind[0] == "d" else np.float32).eps
            bound = 4 * np.sqrt(2 * p.shape[1]) * u * mag
            if self.kind == "h":
                bound = bound + 2.0 ** -10 * abs(ref)
            assert np.all(abs(g - ref) <= bound), self.kind


def _same(a, b):
    return all(x.tobytes() == y.tobytes() for x, y in zip(a, b))


@pytest.mark.parametrize("kind", KINDS)
def test_captured_without_warm_up(hc, torch_cuda, kind):
    torch = torch_cuda
    call, other = Call(hc, torch, kind, 1), Call(hc, torch, kind, 2)
    large = Call(hc, torch, kind, 3, scale=4)
    with hc.Handle() as fresh:  # the bits of an eager call
        call(fresh)
        want = call.host()
        other(fresh)
        want_other = other.host()
    call.check(want)
    h = hc.Handle()
    small = Call(hc, torch, kind, 4)
    side = torch.cuda.Stream()
    graphs = []
    for c in (call, other):
        graphs.append(torch.cuda.CUDAGraph())
        torch.cuda.synchronize()
        with torch.cuda.graph(graphs[-1], stream=side):
            h.set_stream(side.cuda_stream)
            c(h)
        h.set_stream(0)
    for i in range(3):
        call.clear()
        other.clear()
        small(h)
        graphs[0].replay()
        large(h)  # the eager partials grow beside the replay
        graphs[1].replay()
        assert _same(call.host(), want), (kind, i)
        assert _same(other.host(), want_other), (kind, i)
        large.check(large.host())
        junk = torch.full((1 << 22,), float("nan"), device="cuda")
        del junk
    del graphs
    torch.cuda.synchronize()
    h.destroy()


@pytest.mark.parametrize("kind", KINDS)
def test_two_streams_without_a_wait(hc, torch_cuda, kind):
    torch = torch_cuda
    calls = [Call(hc, torch, kind, s) for s in (5, 6)]
    streams = [torch.cuda.Stream() for _ in calls]
    with hc.Handle() as h:
        want = []
        for c in calls:
            c(h)
            want.append(c.host())
        for c in calls:
            c.clear()
        torch.cuda.synchronize()
        for _ in range(40):
            for c, s in zip(calls, streams):
                h.set_stream(s.cuda_stream)
                c(h)
        torch.cuda.synchronize()
        h.set_stream(0)
        for c, w in zip(calls, want):
            assert _same(c.host(), w), kind


def test_without_memory_for_partials(hc, torch_cuda):
    """Captures whose partials fill what a handle keeps for captures: the calls
    after them run unsplit."""
    torch = torch_cuda
    m, n, k = 1024, 512, 8192
    a = torch.rand(m, k, device="cuda", dtype=torch.float64)
    b = torch.rand(k, n, device="cuda", dtype=torch.float64)
    c = torch.zeros(m, n, device="cuda", dtype=torch.float64)
    calls = [Call(hc, torch, kind, 9) for kind in KINDS]
    side = torch.cuda.Stream()
    h = hc.Handle()
    h.set_stream(side.cuda_stream)
    graphs = []

    def capture(f):
        g = torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=side):
            f()
        graphs.append(g)
        return g

    def big():
        assert hc.api.hcblas_dgemm(h, ROW, 0, 0, m, n, k, 1.0, a, k, b, n, 0.0, c,
                                   n, 0, 0, 0) == 0

    free = torch.cuda.mem_get_info()[0]
    for _ in range(40):  # 32 MiB each; 32 of them fill it
        capture(big)
    used = free - torch.cuda.mem_get_info()[0]
    assert used <= (1 << 30) + (256 << 20)
    ref = to_host(a) @ to_host(b)
    for i in (0, 39):
        c.fill_(7)
        graphs[i].replay()
        assert np.all(abs(to_host(c) - ref) <= 4 * np.sqrt(k) * 2.0 ** -52 * ref)
    for call in calls:
        g = capture(lambda: call(h))
        call.clear()
        g.replay()
        call.check(call.host())
    del g, graphs
    torch.cuda.synchronize()
    h.destroy()

"""Performance cases of hcblas_amd: the calls a program makes of this library,
through its public entry points, over the range of sizes they are made with.

A case is a dict of plain values with a "kind":

  vector   the level-1 updates of one step of an iterative solver (copy, axpy,
           scal, dot, asum), float32 / float64, unit or other increments;
  lsq      the gradient g = A^T (b - A x) of a least-squares problem: copy and
           GEMV in both directions over one matrix;
  ger      a rank-1 update through autograd, forward and backward;
  conv     one convolution layer of the conv-net shape lists as column-major
           SGEMMs: bias, forward, gradient of the columns, of the weights;
  gemm     one GEMM or one strided batch: S / D / H / C / Z, either storage
           order, every transpose form, any size;
  split    an S / D GEMM in one of the split-precision math modes;
  grouped  a table of independent small problems as one persistent launch;
  train    batched GEMM through autograd, forward and backward.

Inputs are uniform on [-1, 1]; a pass returns every output it computes.
"""
import functools
import math

import numpy as np
import torch

import hcblas_amd as hc
from hcblas_amd import torch_ext

api = hc.api

REAL = {"f32": torch.float32, "f64": torch.float64, "f16": torch.float16,
        "bf16": torch.bfloat16, "c64": torch.complex64,
        "c128": torch.complex128}
CODE = {"f32": hc.R_32F, "f64": hc.R_64F, "f16": hc.R_16F, "bf16": hc.R_16BF,
        "c64": hc.C_32F, "c128": hc.C_64F}
LETTER = {"f32": "S", "f64": "D", "f16": "H", "c64": "C", "c128": "Z"}
SIZE = {"f32": 4, "f64": 8, "f16": 2, "bf16": 2, "c64": 8, "c128": 16}


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------
def listed():
    return [
        # One step of a solver on a small system: five short calls, two of
        # which return a scalar to the host, so latency is all that counts.
        {"name": "vector_f32_small", "kind": "vector", "dtype": "f32",
         "n": 4099, "inc": 1},
        # The same on vectors far larger than the caches (the bandwidth
        # configuration's range).
        {"name": "vector_f64_large", "kind": "vector", "dtype": "f64",
         "n": 1 << 26, "inc": 1},
        # Least-squares gradient of a tall data matrix with as many samples
        # and features as the data happens to have.
        {"name": "lsq_f32_ragged", "kind": "lsq", "dtype": "f32", "m": 20011,
         "n": 4099, "order": hc.COL_MAJOR},
        # The rank-1 update of the differentiation configuration.
        {"name": "ger_f32_4096", "kind": "ger", "dtype": "f32", "m": 4096,
         "n": 4096},
        # A GoogLeNet layer (23 x 23 outputs, 3 x 3 x 128 columns, 192
        # filters): odd leading dimensions, few tiles, short calls.
        {"name": "conv_google_529x192x1152", "kind": "conv", "pixels": 529,
         "filters": 192, "columns": 1152},
        # The plain SGEMM configuration.
        {"name": "gemm_f32_rowmajor_1024", "kind": "gemm", "dtype": "f32",
         "order": hc.ROW_MAJOR, "ta": hc.OP_N, "tb": hc.OP_N, "m": 1024,
         "n": 1024, "k": 1024, "batch": 1},
        # A float64 product of matrices of odd sizes, packed tightly.
        {"name": "gemm_f64_ragged", "kind": "gemm", "dtype": "f64",
         "order": hc.COL_MAJOR, "ta": hc.OP_N, "tb": hc.OP_T, "m": 2051,
         "n": 1777, "k": 1533, "batch": 1},
        # The largest half-precision product of the benchmark.
        {"name": "gemm_f16_8192", "kind": "gemm", "dtype": "f16",
         "order": hc.COL_MAJOR, "ta": hc.OP_N, "tb": hc.OP_N, "m": 8192,
         "n": 8192, "k": 8192, "batch": 1},
        # A batch of small complex products (one per frequency or angle).
        {"name": "gemm_c64_batch_64x96", "kind": "gemm", "dtype": "c64",
         "order": hc.COL_MAJOR, "ta": hc.OP_N, "tb": hc.OP_C, "m": 96,
         "n": 96, "k": 96, "batch": 64},
        # The split-precision configuration, INT8 residue products.
        {"name": "split_f32_crt_8192", "kind": "split", "dtype": "f32",
         "mode": "crt", "ta": hc.OP_N, "tb": hc.OP_N, "m": 8192, "n": 8192,
         "k": 8192},
        # The grouped configuration.
        {"name": "grouped_4096", "kind": "grouped", "count": 4096, "lo": 16,
         "hi": 512, "multiple": 8},
        # The differentiation configuration: forward and backward in bf16.
        {"name": "train_bf16_256x256x1024x512", "kind": "train",
         "dtype": "bf16", "batch": 256, "m": 256, "n": 1024, "k": 512,
         "ta": False, "tb": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sized(rng, lo, hi):
    """A size on [lo, hi] (uniform in its logarithm): any whole number half
    of the time, otherwise a multiple of 8, 32 or 128."""
    v = _log(rng, lo, hi)
    step = rng.choice([1, 1, 1, 8, 32, 128])
    return max(lo, min(hi, v // step * step or v))


def draw(rng):
    kind = rng.choice(["vector", "lsq", "ger", "conv", "gemm", "gemm", "gemm",
                       "gemm", "split", "grouped", "train"])
    if kind == "vector":
        dt = rng.choice(["f32", "f64"])
        return {"kind": kind, "dtype": dt, "n": _sized(rng, 500, 1 << 26),
                "inc": rng.choice([1, 1, 1, 2])}
    if kind == "lsq":
        dt = rng.choice(["f32", "f64"])
        return {"kind": kind, "dtype": dt, "m": _sized(rng, 100, 20000),
                "n": _sized(rng, 100, 12000),
                "order": rng.choice([hc.ROW_MAJOR, hc.COL_MAJOR])}
    if kind == "ger":
        dt = rng.choice(["f32", "f64"])
        return {"kind": kind, "dtype": dt, "m": _sized(rng, 64, 4500),
                "n": _sized(rng, 64, 4500)}
    if kind == "conv":
        return {"kind": kind, "pixels": _sized(rng, 16, 3025),
                "filters": _sized(rng, 16, 512),
                "columns": _sized(rng, 64, 2400)}
    if kind == "gemm":
        dt = rng.choice(["f32", "f32", "f64", "f16", "c64", "c128"])
        batch = rng.choice([1, 1, _log(rng, 2, 256)])
        top = {"f32": 3e11, "f64": 1.5e11, "f16": 1e12, "c64": 3e11,
               "c128": 1.5e11}[dt]
        per = 8.0 if dt[0] == "c" else 2.0
        while True:
            hi = 8192 if batch == 1 else 1024
            m, n, k = (_sized(rng, 16, hi) for _ in range(3))
            if per * m * n * k * batch <= top and \
                    batch * (m * k + k * n + m * n) * SIZE[dt] <= 2e9:
                break
        return {"kind": kind, "dtype": dt,
                "order": rng.choice([hc.ROW_MAJOR, hc.COL_MAJOR]),
                "ta": rng.choice([hc.OP_N, hc.OP_T]),
                "tb": rng.choice([hc.OP_N, hc.OP_T]), "m": m, "n": n, "k": k,
                "batch": batch}
    if kind == "split":
        dt, mode = rng.choice([("f32", "crt"), ("f32", "bf16"),
                               ("f64", "crt")])
        hi = 8192 if dt == "f32" else 5000
        while True:
            m, n, k = (_sized(rng, 512, hi) for _ in range(3))
            if 2.0 * m * n * k <= (5e11 if dt == "f32" else 2e11):
                break
        return {"kind": kind, "dtype": dt, "mode": mode,
                "ta": rng.choice([hc.OP_N, hc.OP_T]),
                "tb": rng.choice([hc.OP_N, hc.OP_T]), "m": m, "n": n, "k": k}
    if kind == "grouped":
        return {"kind": kind, "count": _log(rng, 64, 4096),
                "lo": rng.choice([8, 16, 32]),
                "hi": rng.choice([128, 256, 512]),
                "multiple": rng.choice([1, 8, 8])}
    dt = rng.choice(["bf16", "bf16", "f32"])
    while True:
        m, n, k = (_sized(rng, 32, 1024) for _ in range(3))
        batch = _log(rng, 1, 256)
        if batch * (m * k + k * n + m * n) <= 1.5e8 and \
                6.0 * batch * m * n * k <= (2e11 if dt == "bf16" else 6e10):
            break
    return {"kind": kind, "dtype": dt, "batch": batch, "m": m, "n": n, "k": k,
            "ta": rng.choice([False, True]), "tb": rng.choice([False, True])}


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _handle():
    """The program's one handle, on torch's current stream."""
    h = hc.Handle()
    h.set_stream(torch.cuda.current_stream())
    return h


def _uniform(gen, shape, dt):
    if dt[0] == "c":
        part = "f32" if dt == "c64" else "f64"
        return torch.complex(_uniform(gen, shape, part),
                             _uniform(gen, shape, part))
    work = torch.float64 if dt == "f64" else torch.float32
    t = torch.rand(shape, generator=gen, device="cuda", dtype=work)
    return t.mul_(2).sub_(1).to(REAL[dt])


def _stored(c):
    """Shapes of A, B and C as they lie (outer, contiguous) in storage."""
    a = (c["m"], c["k"]) if c["ta"] == hc.OP_N else (c["k"], c["m"])
    b = (c["k"], c["n"]) if c["tb"] == hc.OP_N else (c["n"], c["k"])
    shapes = [a, b, (c["m"], c["n"])]
    if c.get("order", hc.COL_MAJOR) == hc.COL_MAJOR:
        shapes = [(s[1], s[0]) for s in shapes]
    return shapes


def _table(case, seed):
    """The problems of a grouped case: sizes log-uniform on [lo, hi] rounded
    to `multiple`, half float32 and half float16, in either storage order."""
    rng = np.random.default_rng(seed)
    count, step = case["count"], case["multiple"]

    def sizes():
        v = np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]), count))
        return np.maximum(step, np.round(v / step) * step).astype(np.int64)

    M, N, K = sizes(), sizes(), sizes()
    half, order = rng.integers(0, 2, count), rng.integers(0, 2, count)
    used = {0: [0, 0], 1: [0, 0]}  # elements of inputs and of outputs
    rows = []
    for m, n, k, d, o in zip(M.tolist(), N.tolist(), K.tolist(),
                             half.tolist(), order.tolist()):
        offs = []
        for out, size in ((0, m * k), (0, k * n), (1, m * n)):
            offs.append(used[d][out])
            used[d][out] += -(-size // 64) * 64
        rows.append((d, o, m, n, k, *offs))
    return rows, used


# The grouped table's sizes are the case's, not the seed's: a program builds
# its plan once and refills the buffers.
_TABLE_SEED = 2024


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    s = {"case": case, "h": _handle()}
    if kind == "vector":
        n, inc = case["n"], case["inc"]
        s["x"] = _uniform(gen, n * inc, case["dtype"])
        s["y"] = _uniform(gen, n * inc, case["dtype"])
        s["z"] = torch.zeros_like(s["y"])
    elif kind == "lsq":
        m, n = case["m"], case["n"]
        s["A"] = _uniform(gen, m * n, case["dtype"])
        s["x"] = _uniform(gen, n, case["dtype"])
        s["b"] = _uniform(gen, m, case["dtype"])
        s["r"] = torch.empty_like(s["b"])
        s["g"] = torch.empty_like(s["x"])
    elif kind == "ger":
        torch_ext.load()
        m, n = case["m"], case["n"]
        for name, shape in (("x", m), ("y", n), ("A", (m, n))):
            s[name] = _uniform(gen, shape, case["dtype"]).requires_grad_()
        s["W"] = _uniform(gen, (m, n), case["dtype"])
    elif kind == "conv":
        p, f, c = case["pixels"], case["filters"], case["columns"]
        s["ones"] = torch.ones(p, device="cuda")
        s["bias"] = _uniform(gen, f, "f32")
        s["cols"] = _uniform(gen, p * c, "f32")
        s["weight"] = _uniform(gen, c * f, "f32")
        s["dout"] = _uniform(gen, p * f, "f32")
        s["out"] = torch.empty_like(s["dout"])
        s["dcols"] = torch.empty_like(s["cols"])
        s["dweight"] = torch.empty_like(s["weight"])
    elif kind in ("gemm", "split"):
        batch = case.get("batch", 1)
        a, b, c = _stored(case)
        s["A"] = _uniform(gen, (batch, *a), case["dtype"])
        s["B"] = _uniform(gen, (batch, *b), case["dtype"])
        s["C"] = torch.empty((batch, *c), device="cuda",
                             dtype=REAL[case["dtype"]])
    elif kind == "grouped":
        rows, used = _table(case, _TABLE_SEED)
        inputs = [_uniform(gen, max(64, used[d][0]), dt)
                  for d, dt in ((0, "f32"), (1, "f16"))]
        outputs = [torch.zeros(max(64, used[d][1]), device="cuda",
                               dtype=REAL[dt])
                   for d, dt in ((0, "f32"), (1, "f16"))]
        problems = []
        for d, o, m, n, k, ao, bo, co in rows:
            size = 4 - 2 * d
            row = o == hc.ROW_MAJOR
            problems.append(hc.GemmProblem(
                hc.R_16F if d else hc.R_32F, o, hc.OP_N, hc.OP_N, m, n, k, 0,
                1.0, 0.0, inputs[d].data_ptr() + ao * size, k if row else m,
                inputs[d].data_ptr() + bo * size, n if row else k,
                outputs[d].data_ptr() + co * size, n if row else m))
        s["inputs"], s["outputs"] = inputs, outputs
        s["plan"] = hc.GroupedPlan(s["h"], problems)
        hc.check("hcblasGroupedPlanAutotune", s["plan"].autotune())
    else:
        torch_ext.load()
        b, m, n, k = (case[v] for v in ("batch", "m", "n", "k"))
        dt = case["dtype"]
        s["A"] = _uniform(gen, (b, k, m) if case["ta"] else (b, m, k),
                          dt).requires_grad_()
        s["B"] = _uniform(gen, (b, n, k) if case["tb"] else (b, k, n),
                          dt).requires_grad_()
        s["W"] = _uniform(gen, (b, m, n), "f32")
    return s


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------
def run(s):
    return globals()["_run_" + s["case"]["kind"]](s)


def _run_vector(s):
    case, h = s["case"], s["h"]
    n, inc, p = case["n"], case["inc"], LETTER[case["dtype"]]
    x, y, z = s["x"], s["y"], s["z"]
    hc.check("copy", getattr(api, f"hcblas{p}copy")(h, n, y, inc, z, inc))
    hc.check("axpy", getattr(api, f"hcblas{p}axpy")(h, n, 1.5, x, inc, z, inc))
    hc.check("scal", getattr(api, f"hcblas{p}scal")(h, n, -0.75, z, inc))
    st, d = getattr(api, f"hcblas{p}dot")(h, n, z, inc, x, inc, None)
    hc.check("dot", st)
    st, a = getattr(api, f"hcblas{p}asum")(h, n, z, inc, None)
    hc.check("asum", st)
    scalar = np.float32 if p == "S" else np.float64
    return {"z": z, "dot": scalar(d), "asum": scalar(a)}


def _run_lsq(s):
    case, h = s["case"], s["h"]
    m, n, o, p = case["m"], case["n"], case["order"], LETTER[case["dtype"]]
    lda = m if o == hc.COL_MAJOR else n
    gemv = getattr(api, f"hcblas_{p.lower()}gemv")
    hc.check("copy", getattr(api, f"hcblas{p}copy")(h, m, s["b"], 1, s["r"],
                                                    1))
    hc.check("gemv", gemv(h, o, hc.OP_N, m, n, -1.0, s["A"], 0, lda, s["x"],
                          0, 1, 1.0, s["r"], 0, 1))
    hc.check("gemv", gemv(h, o, hc.OP_T, m, n, 1.0, s["A"], 0, lda, s["r"], 0,
                          1, 0.0, s["g"], 0, 1))
    return {"r": s["r"], "g": s["g"]}


def _run_ger(s):
    x, y, A = s["x"], s["y"], s["A"]
    x.grad = y.grad = A.grad = None
    out = torch_ext.ger(x, y, A, 1.5)
    out.backward(s["W"])
    return {"out": out, "dx": x.grad, "dy": y.grad, "dA": A.grad}


def _run_conv(s):
    case, h = s["case"], s["h"]
    p, f, c = case["pixels"], case["filters"], case["columns"]
    N, T = hc.OP_N, hc.OP_T
    gemm = api.hcblasSgemm
    hc.check("bias", gemm(h, T, N, p, f, 1, 1.0, s["ones"], 1, s["bias"], 1,
                          0.0, s["out"], p))
    hc.check("forward", gemm(h, N, N, p, f, c, 1.0, s["cols"], p, s["weight"],
                             c, 1.0, s["out"], p))
    hc.check("columns", gemm(h, N, T, p, c, f, 1.0, s["dout"], p, s["weight"],
                             c, 0.0, s["dcols"], p))
    hc.check("weights", gemm(h, T, N, c, f, p, 1.0, s["cols"], p, s["dout"],
                             p, 0.0, s["dweight"], c))
    return {"out": s["out"], "dcols": s["dcols"], "dweight": s["dweight"]}


def _run_gemm(s):
    c, h = s["case"], s["h"]
    m, n, k = c["m"], c["n"], c["k"]
    A, B, C = s["A"], s["B"], s["C"]
    lda, ldb, ldc = A.size(2), B.size(2), C.size(2)
    p, o, ta, tb = LETTER[c["dtype"]], c["order"], c["ta"], c["tb"]
    if c["batch"] > 1:
        st = api.hcblas_gemm_strided_batched(
            h, CODE[c["dtype"]], o, ta, tb, m, n, k, 1.0, A, lda, 0,
            A.stride(0), B, ldb, 0, B.stride(0), 0.0, C, ldc, 0, C.stride(0),
            c["batch"])
    elif o == hc.COL_MAJOR:
        st = getattr(api, f"hcblas{p}gemm")(h, ta, tb, m, n, k, 1.0, A, lda,
                                            B, ldb, 0.0, C, ldc)
    elif p in "CZ":
        st = getattr(api, f"hcblas_{p.lower()}gemm")(
            h, o, ta, tb, m, n, k, 1.0, A, 0, lda, B, 0, ldb, 0.0, C, 0, ldc)
    else:
        st = getattr(api, f"hcblas_{p.lower()}gemm")(
            h, o, ta, tb, m, n, k, 1.0, A, lda, B, ldb, 0.0, C, ldc, 0, 0, 0)
    hc.check("gemm", st)
    return C


_SPLIT = {("f32", "crt"): "hcblas_sgemm_ozaki_crt",
          ("f32", "bf16"): "hcblas_sgemm_split_bf16",
          ("f64", "crt"): "hcblas_dgemm_ozaki_crt"}


def _run_split(s):
    c, h = s["case"], s["h"]
    A, B, C = s["A"], s["B"], s["C"]
    hc.check("split", getattr(api, _SPLIT[c["dtype"], c["mode"]])(
        h, hc.COL_MAJOR, c["ta"], c["tb"], c["m"], c["n"], c["k"], 1.0, A,
        A.size(2), B, B.size(2), 0.0, C, C.size(2), 0, 0, 0))
    return C


def _run_grouped(s):
    hc.check("hcblasGroupedGemm", s["plan"].run())
    return s["outputs"]


def _run_train(s):
    c, A, B = s["case"], s["A"], s["B"]
    A.grad = B.grad = None
    out = torch_ext.gemm_batched(A, B, transA=c["ta"], transB=c["tb"])
    out.backward(s["W"])
    return {"out": out, "dA": A.grad, "dB": B.grad}


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    size = SIZE[case.get("dtype", "f32")]
    if kind == "vector":
        n = case["n"]  # copy 2, axpy 3, scal 2, dot 2, asum 1 per element
        return {"bytes": 10.0 * n * size, "flops": 6.0 * n}
    if kind == "lsq":
        m, n = case["m"], case["n"]
        return {"bytes": size * (2.0 * m * n + 2 * n + 4 * m),
                "flops": 4.0 * m * n}
    if kind == "ger":  # forward reads A and writes out; backward reads W
        m, n = case["m"], case["n"]
        return {"bytes": size * (3.0 * m * n + 3 * (m + n)),
                "flops": 6.0 * m * n}
    if kind == "conv":
        p, f, c = case["pixels"], case["filters"], case["columns"]
        return {"bytes": 4.0 * (p + f + 2 * p * c + 2 * c * f + 2 * p * f),
                "flops": 6.0 * p * f * c}
    if kind in ("gemm", "split"):
        m, n, k, b = case["m"], case["n"], case["k"], case.get("batch", 1)
        per = 8.0 if case["dtype"][0] == "c" else 2.0
        return {"bytes": float(size * b * (m * k + k * n + m * n)),
                "flops": per * b * m * n * k}
    if kind == "grouped":
        rows, _ = _table(case, _TABLE_SEED)
        return {"bytes": float(sum((4 - 2 * d) * (m * k + k * n + m * n)
                                   for d, _, m, n, k, *_ in rows)),
                "flops": float(sum(2 * m * n * k
                                   for _, _, m, n, k, *_ in rows))}
    b, m, n, k = (case[v] for v in ("batch", "m", "n", "k"))
    return {"bytes": float(b * (2 * size * (m * k + k * n) + 8 * m * n)),
            "flops": 6.0 * b * m * n * k}


# --------------------------------------------------------------------------
# The same outputs in 64 bits
# --------------------------------------------------------------------------
def _wide(t):
    return t.detach().to(torch.complex128 if t.is_complex()
                         else torch.float64)


def exact(case, seed):
    s = prepare_inputs(case, seed)
    kind = case["kind"]
    if kind == "vector":
        x, y, inc = _wide(s["x"]), _wide(s["y"]), case["inc"]
        z = torch.zeros_like(y)
        z[::inc] = -0.75 * (y[::inc] + 1.5 * x[::inc])
        return {"z": z,
                "dot": np.float64(torch.dot(z[::inc], x[::inc]).item()),
                "asum": np.float64(z.abs().sum().item())}
    if kind == "lsq":
        m, n = case["m"], case["n"]
        A = _wide(s["A"])
        A = A.view(m, n) if case["order"] == hc.ROW_MAJOR else \
            A.view(n, m).t()
        r = _wide(s["b"]) - A.mv(_wide(s["x"]))
        return {"r": r, "g": A.t().mv(r)}
    if kind == "ger":
        x, y, A, W = (_wide(s[v]) for v in "xyAW")
        return {"out": A + 1.5 * torch.outer(x, y), "dx": 1.5 * W.mv(y),
                "dy": 1.5 * W.t().mv(x), "dA": W}
    if kind == "conv":
        p, f, c = case["pixels"], case["filters"], case["columns"]
        cols, weight = _wide(s["cols"]).view(c, p), _wide(s["weight"]).view(f, c)
        dout, bias = _wide(s["dout"]).view(f, p), _wide(s["bias"])
        return {"out": (weight @ cols + bias[:, None]).reshape(-1),
                "dcols": (weight.t() @ dout).reshape(-1),
                "dweight": (dout @ cols.t()).reshape(-1)}
    if kind in ("gemm", "split"):
        def op(t, o):
            t = _wide(t)
            t = t.mT if o != hc.OP_N else t
            return t.conj() if o == hc.OP_C else t

        A, B = op(s["A"], case["ta"]), op(s["B"], case["tb"])
        if case.get("order", hc.COL_MAJOR) == hc.COL_MAJOR:
            A, B = B, A  # storage holds the transposes
        return torch.matmul(A.resolve_conj().contiguous(),
                            B.resolve_conj().contiguous())
    if kind == "grouped":
        outs = [torch.zeros(t.numel(), device="cuda", dtype=torch.float64)
                for t in s["outputs"]]
        wide = [_wide(t) for t in s["inputs"]]
        for d, o, m, n, k, ao, bo, co in _table(case, _TABLE_SEED)[0]:
            A, B = wide[d][ao:ao + m * k], wide[d][bo:bo + k * n]
            out = outs[d][co:co + m * n]
            if o == hc.ROW_MAJOR:
                torch.mm(A.view(m, k), B.view(k, n), out=out.view(m, n))
            else:
                torch.mm(B.view(n, k), A.view(k, m), out=out.view(n, m))
        return outs
    A, B, W = _wide(s["A"]), _wide(s["B"]), _wide(s["W"])
    At, Bt = A.mT if case["ta"] else A, B.mT if case["tb"] else B

    def mm(a, b):
        return torch.matmul(a.contiguous(), b.contiguous())

    dA, dB = mm(W, Bt.mT), mm(At.mT, W)
    return {"out": mm(At, Bt), "dA": dA.mT if case["ta"] else dA,
            "dB": dB.mT if case["tb"] else dB}


def prepare_inputs(case, seed):
    """prepare()'s inputs without a plan over them."""
    if case["kind"] != "grouped":
        return prepare(case, seed)
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    _, used = _table(case, _TABLE_SEED)
    return {"inputs": [_uniform(gen, max(64, used[d][0]), dt)
                       for d, dt in ((0, "f32"), (1, "f16"))],
            "outputs": [torch.empty(max(64, used[d][1]), device="cuda")
                        for d in (0, 1)]}

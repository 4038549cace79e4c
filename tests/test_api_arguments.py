"""The generated Python entry points keep their arguments: what a call passes by
address (a temporary tensor among them) stays referenced by the call's own frame
while the C function runs, whoever called it and however the interpreter hands
arguments over."""
import sys

import pytest

import hcblas_amd as hc
from hcblas_amd import _lib
from hcblas_amd.api import _bind


class Buffer:
    def data_ptr(self):
        return 4096


@pytest.mark.parametrize("name", ["hcblas_sgemm", "hcblasSdot", "hcblasDaxpy",
                                  "hcblas_gemm_strided_batched", "hcblas_cgemm",
                                  "hcblas_sger_backward", "hcblasSgemmBatched"])
def test_arguments_live_through_the_call(name):
    proto = _lib.prototypes()[name]
    passed = {}
    seen = []

    def c_function(*args):
        frame = sys._getframe(1).f_locals
        for p, obj in passed.items():
            assert frame[p] is obj, p
        seen.append(args)
        return 0

    args = []
    for ctype, p in proto.args:
        if p == "dtype":
            args.append(hc.R_32F)
        elif "*" in ctype and p != "result":
            passed[p] = Buffer()
            args.append(passed[p])
        elif p == "result":
            args.append(None)
        else:
            args.append(7)
    got = _bind(name, proto, c_function)(*args)
    assert got == 0 or got[0] == 0
    (c_args,) = seen
    assert len(c_args) == len(proto.args)
    for (ctype, p), c in zip(proto.args, c_args):
        if p in passed:
            assert c == 4096, p
        elif p != "result" and p != "dtype":
            assert c == 7, p

"""Which kernel a projection of 2 and more rows takes, by the library's own dispatch
over a stand-in for the HIP runtime: the cases of tests/test_linear_mm_gpu.py that
name a kernel reach it, and they name every linear_mm_* kernel of the code object, so
that a change of the choice cannot leave one without a test."""
import re

import pytest

import g4a
import hip_standin as hip
from hip_standin import PTR
from test_linear_mm_gpu import EVERY_KERNEL


@pytest.fixture(scope="module")
def ctx():
    with hip.binding().Context(0) as c:
        yield c


@pytest.mark.parametrize("kernel,op,N,K,M,bits", EVERY_KERNEL)
def test_the_case_reaches_its_kernel(ctx, kernel, op, N, K, M, bits):
    w = hip.weight(N, K, bits, bits == 8 and N % 2 == 1)
    hip.launches()
    if op == "linear":
        ctx.linear_q(w, PTR, PTR, M)
    elif op == "geglu":
        ctx.linear_q_geglu(w, w, PTR, PTR, M)
    else:
        ctx.linear_q_gelu_mul_cols(w, PTR, PTR, N + 5, 3, PTR, M)
    split = [] if "few" in kernel else [f"g4a_split_x_b{bits}"]
    assert [x.name for x in hip.launches()] == split + [f"g4a_linear_mm_{kernel}"]


def test_the_cases_reach_every_kernel():
    built = set(re.findall(rb"g4a_linear_mm_(\w+?_mode\d)", g4a.HSACO_PATH.read_bytes()))
    assert {k.decode() for k in built} == {case[0] for case in EVERY_KERNEL}

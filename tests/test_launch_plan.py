"""Which main kernel a shape runs and how it is cut (launch_backward's rules,
through shaobo_fa3_ext_bwd_v2_plan; host only)."""
import ctypes

import pytest

import shaobo_fa3 as F
from gpu_util import launch_plan
from test_gpu_reg_kernel import CASES


def test_plan_arguments():
    lib = F.load()
    p = F.make_params(lib, batch=1, seqlen=128, heads_q=1)
    short = F.Plan(struct_size=ctypes.sizeof(F.Plan) - 1)
    assert lib.shaobo_fa3_ext_bwd_v2_plan(ctypes.byref(p), None) == F.INVALID_VALUE
    assert lib.shaobo_fa3_ext_bwd_v2_plan(ctypes.byref(p), ctypes.byref(short)) == F.INVALID_VALUE
    p.seqlen_q = p.seqlen_k = 64
    full = F.Plan(struct_size=ctypes.sizeof(F.Plan))
    assert lib.shaobo_fa3_ext_bwd_v2_plan(ctypes.byref(p), ctypes.byref(full)) == F.UNSUPPORTED


@pytest.mark.parametrize("row", CASES, ids=lambda r: "-".join(map(str, r[:6])))
def test_reg_kernel_rows_run_what_they_say(row):
    assert launch_plan(*row[:6]) == row[-1]

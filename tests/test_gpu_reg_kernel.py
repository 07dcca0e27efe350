"""The register-operand main kernel (bwd_reg_kernel) at the edges of the
shapes that reach it: a single 128-row tile, odd tile counts, group counts
without XCD-aligned parts, each way of cutting the jobs at each head dim and
mask (whole, some or all dKV halved, both roles halved), fp32 head-split
contributions, bf16, BSHD and a scale above ln 2.  Each case against the CPU oracle under the bar of gpu_util.check,
bitwise repeatable, and bit for bit equal to its race-check instantiation
(every job on an LDS of NaN bytes, a full wait and a barrier around every
phase)."""
import numpy as np
import pytest

import fa3_oracle as O
import shaobo_fa3 as F
from gpu_util import check, launch_plan, log, run_v2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, S, D, causal, dtype, bshd, scale, the plan (gpu_util.launch_plan);
    # longest dKV job / a CU's share
    (8, 25, 25, 128, 128, True, "fp16", False, None, "reg h0/1 q1 c1"),    # one tile (0.73)
    (4, 33, 33, 256, 128, True, "bf16", True, None, "reg h0/2 q1 c1"),     # BSHD (0.74)
    (2, 49, 49, 384, 128, True, "fp16", False, 1.0, "reg h0/3 q1 c1"),     # odd tiles and groups, unscaled range (0.75)
    (2, 33, 33, 384, 64, False, "bf16", False, None, "reg kv1 q1 c1"),     # D 64, full (0.74)
    (4, 64, 32, 128, 128, True, "bf16", False, None, "reg h1/1 q1 c1"),    # one tile, G 2 (1.14)
    (4, 16, 8, 1024, 128, True, "fp16", True, None, "reg h5/8 q1 c1"),     # BSHD (1.02)
    (4, 48, 12, 384, 64, False, "fp16", False, None, "reg kv2 q1 c1"),     # D 64, full (1.02)
    (4, 20, 5, 384, 128, True, "bf16", False, None, "reg h2/3 q1 c4"),     # head split (0.91)
    (3, 16, 2, 384, 64, False, "fp16", True, None, "reg kv2 q1 c8"),       # head split, D 64 (1.02)
    (1, 20, 5, 768, 64, False, "bf16", True, None, "reg kv2 q2 c4"),       # both halved, a chunk per head (1.22)
    (2, 12, 12, 1792, 128, False, "bf16", False, None, "reg kv2 q1 c1"),   # 1.3 rounds of workgroups (0.44)
    (3, 21, 21, 384, 64, True, "fp16", False, None, "reg kv2 q2 c1"),      # both roles halved, D 64 (1.16)
    (3, 43, 43, 384, 128, False, "fp16", False, None, "reg kv1 q1 c1"),    # full, whole jobs (0.38)
    (4, 64, 32, 512, 128, False, "bf16", True, None, "reg kv1 q1 c1"),     # ... G 2, BSHD (0.29)
    (5, 64, 32, 512, 128, True, "fp16", False, None, "reg h0/4 q1 c1"),    # causal, whole, G 2 (0.37)
    (7, 32, 32, 512, 64, True, "fp16", False, None, "reg h0/4 q1 c1"),     # ... D 64 (0.26)
    (4, 40, 20, 1408, 64, True, "bf16", True, None, "reg h0/11 q1 c1"),    # ... G 2, BSHD (0.30)
    (4, 32, 16, 512, 64, True, "bf16", True, None, "reg h3/4 q1 c1"),      # some halved, D 64, G 2 (0.91)
    (11, 57, 19, 256, 128, True, "bf16", False, None, "reg h0/2 q1 c1"),   # parts of one job: dealt across the groups (0.47)
    (3, 87, 29, 256, 64, False, "fp16", True, None, "reg kv1 q1 c1"),      # likewise, D 64, full (0.84)
    (3, 19, 19, 128, 64, True, "bf16", False, 1.0, "main c1"),             # few jobs (2.57)
]


@pytest.mark.parametrize("B,Hq,Hkv,S,D,causal,dtype,bshd,scale,plan", CASES)
def test_reg_kernel(B, Hq, Hkv, S, D, causal, dtype, bshd, scale, plan):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    log(f"[case] reg kernel B={B} Hq={Hq} Hkv={Hkv} S={S} D={D} causal={causal} {dtype} "
        f"bshd={bshd} scale={scale}: {plan}")
    lib = F.load()
    assert launch_plan(B, Hq, Hkv, S, D, causal) == plan
    kw = {} if scale is None else {"scale": scale}
    g = O.golden(B, Hq, Hkv, S, D, causal, dtype=dtype, **kw)
    res = run_v2(g, torch, bshd=bshd)
    assert res["status"] == F.SUCCESS, F.status_name(res["status"])
    check(res, g)
    again = run_v2(g, torch, bshd=bshd)
    lib.shaobo_fa3_ext_set_race_check(1)
    try:
        slow = run_v2(g, torch, bshd=bshd)
    finally:
        lib.shaobo_fa3_ext_set_race_check(0)
    for n in ("dq", "dk", "dv", "delta"):
        np.testing.assert_array_equal(again[n], res[n], err_msg=n)
        np.testing.assert_array_equal(slow[n], res[n], err_msg=n)

"""Which main kernel a shape runs and how it is cut (launch_backward's rules,
through shaobo_fa3_ext_bwd_v2_plan; host only)."""
import ctypes

import pytest

import shaobo_fa3 as F
from gpu_util import launch_plan
import test_gpu_parity
import test_gpu_race_check
import test_gpu_reg_kernel
import test_gpu_stages

CASES = [r[:6] + r[-1:] for rows in (test_gpu_reg_kernel.CASES, test_gpu_race_check.RACE_CASES,
                                     test_gpu_stages.CASES, test_gpu_parity.FULL_SIZE)
         for r in rows]
CASES += [(1, hq, hkv, s, 128, True, plan) for hq, hkv, s, plan in test_gpu_parity.MANY_JOBS]


def test_plan_arguments():
    lib = F.load()
    p = F.make_params(lib, batch=1, seqlen=128, heads_q=1)
    short = F.Plan(struct_size=ctypes.sizeof(F.Plan) - 1)
    assert lib.shaobo_fa3_ext_bwd_v2_plan(ctypes.byref(p), None) == F.INVALID_VALUE
    assert lib.shaobo_fa3_ext_bwd_v2_plan(ctypes.byref(p), ctypes.byref(short)) == F.INVALID_VALUE
    p.seqlen_q = p.seqlen_k = 64
    full = F.Plan(struct_size=ctypes.sizeof(F.Plan))
    assert lib.shaobo_fa3_ext_bwd_v2_plan(ctypes.byref(p), ctypes.byref(full)) == F.UNSUPPORTED


# The lines of the rule, each with a shape on either side of it.
RULES = [
    # B, Hq, Hkv, S, D, causal, plan; longest dKV job / a CU's share
    # one head per chunk: a dQ job is as long as a dKV job, as with G = 1
    (1, 4, 1, 3968, 128, False, "main c4 unscaled"),     # D 128 (1.18)
    (1, 20, 5, 768, 128, False, "main c4 unscaled"),     # (1.22)
    (1, 44, 11, 384, 128, False, "reg kv2 q1 c4"),       # (1.11)
    (1, 8, 2, 3584, 128, True, "main c4 unscaled"),      # causal, S >= 2048 (1.26)
    (2, 3, 1, 7808, 128, True, "main c3 unscaled"),      # (0.79)
    (2, 9, 3, 1536, 128, True, "main c3 unscaled"),      # S >= 1024 (1.25)
    (3, 8, 1, 1280, 128, True, "reg h6/10 q1 c8"),       # (1.11)
    (1, 18, 3, 1920, 128, True, "reg h8/15 q1 c6"),      # (1.05)
    (2, 60, 10, 128, 128, True, "main c6 unscaled"),     # S < 256 (1.22)
    (1, 36, 12, 768, 128, True, "reg h4/6 q1 c3"),       # between (1.16)
    (1, 20, 5, 768, 64, False, "reg kv2 q2 c4"),         # D 64 (1.22)
    (3, 24, 3, 256, 64, False, "reg kv2 q1 c8"),         # S < 512 (1.02)
    (1, 6, 2, 5632, 64, True, "reg kv2 q2 c3"),          # (1.08)
    # D 128 causal, one head per dKV job: none halved
    (1, 27, 27, 2560, 128, True, "reg h1/20 q1 c1"),     # (0.52)
    (10, 5, 5, 1280, 128, True, "reg h1/10 q1 c1"),      # (0.53)
    (3, 2, 2, 8832, 128, True, "reg h0/69 q1 c1"),       # (0.70)
    (1, 11, 11, 5376, 128, True, "reg h0/42 q1 c1"),     # (0.62)
    # D 64 causal, one head per dKV job: both halved from 0.6 on, S >= 512
    (3, 2, 2, 7424, 64, True, "reg kv2 q2 c1"),          # (0.83)
    (1, 5, 5, 8704, 64, True, "reg kv2 q2 c1"),          # (0.85)
    (2, 4, 4, 8064, 64, True, "reg h27/63 q1 c1"),       # (0.57)
    (6, 23, 23, 256, 64, True, "reg h2/2 q1 c1"),        # S < 512 (0.71)
    # D 64 full, more than one head per dKV job: halved from 0.7 on
    (2, 64, 4, 2816, 64, False, "reg kv2 q1 c1"),        # (0.83)
    (2, 6, 2, 6144, 64, False, "reg kv2 q1 c1"),         # (0.76)
    (3, 18, 6, 1664, 64, False, "reg kv1 q1 c1"),        # (0.63)
    (1, 18, 18, 1408, 64, False, "reg kv1 q1 c1"),       # one head (0.74)
    (13, 16, 8, 256, 64, False, "reg kv1 q1 c1"),        # S < 512 (0.70)
    # D 128 full: halved with two heads per dKV job from 1.14 on, with four from 0.8
    (8, 6, 3, 768, 128, False, "reg kv1 q1 c1"),         # two (1.02)
    (2, 16, 1, 1152, 128, False, "main c8 unscaled"),    # S >= 1024 (1.02)
    (1, 34, 17, 1024, 128, False, "main c1 unscaled"),   # (1.08)
    (5, 4, 2, 2304, 128, False, "reg kv1 q1 c1"),        # 1.05 rounds (0.81)
    (7, 14, 7, 512, 128, False, "reg kv2 q1 c1"),        # S < 1024 (0.75)
    (1, 32, 16, 1024, 128, False, "reg kv2 q1 c1"),      # (1.14)
    (1, 15, 5, 3712, 128, False, "reg kv2 q1 c1"),       # three (1.01)
    (2, 16, 4, 2688, 128, False, "reg kv2 q1 c1"),       # four (0.87)
    (1, 48, 8, 2944, 128, False, "reg kv1 q1 c1"),       # six (0.80)
    (4, 264, 44, 128, 128, False, "reg kv1 q1 c1"),      # S < 1024 (0.83)
    # D 64 full, two heads: from 0.76 on
    (4, 4, 2, 3328, 64, False, "reg kv1 q1 c1"),         # (0.70)
    (1, 32, 16, 1536, 64, False, "reg kv2 q1 c1"),       # (0.76)
]


@pytest.mark.parametrize("B,Hq,Hkv,S,D,causal,plan", RULES)
def test_rule(B, Hq, Hkv, S, D, causal, plan):
    assert launch_plan(B, Hq, Hkv, S, D, causal) == plan


@pytest.mark.parametrize("B,Hq,Hkv,S,D,causal,jobs,parts", [
    # jobs per group; the parts they are dealt to the XCDs in, 0: across all groups
    (11, 57, 19, 256, 128, True, 8, 0),    # eight parts would hold one job each
    (3, 33, 33, 512, 128, True, 8, 0),     # one head
    (3, 19, 19, 1024, 128, True, 16, 0),   # D 128 causal: two jobs each
    (5, 50, 50, 256, 128, True, 4, 4),     # S < 512
    (3, 19, 19, 1536, 128, True, 24, 8),   # three
    (9, 90, 30, 128, 128, False, 4, 0),    # four parts of one job, three heads
    (3, 87, 29, 256, 64, False, 8, 0),     # three heads
    (9, 87, 29, 512, 64, False, 16, 8),    # two jobs each
    (5, 45, 15, 512, 128, False, 16, 8),
    (3, 53, 53, 512, 64, False, 8, 8),     # one head: the parts stay
    (8, 25, 25, 128, 128, True, 2, 1),     # aligned group count
    (2, 49, 49, 384, 128, True, 6, 0),     # four parts do not divide six jobs
])
def test_job_map_parts(B, Hq, Hkv, S, D, causal, jobs, parts):
    p = F.plan_of(F.make_params(batch=B, seqlen=S, heads_q=Hq, heads_kv=Hkv, head_dim=D,
                                causal=causal))
    assert (p.kernel, p.jobs, p.xcd_parts) == (F.KERNEL_REG, jobs * B * Hkv, parts)


@pytest.mark.parametrize("row", CASES, ids=lambda r: "-".join(map(str, r[:6])))
def test_gpu_rows_run_what_they_say(row):
    assert launch_plan(*row[:6]) == row[-1]

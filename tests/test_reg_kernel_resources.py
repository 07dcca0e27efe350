"""CPU gate: bwd_reg_kernel is launched to keep two (D 128) or three (D 64)
4-wave workgroups on a CU, so its registers and LDS must allow that."""
import os

import pytest

import resource_gate as gate


def test_reg_kernel_workgroups_share_a_cu():
    if not os.path.exists(gate.LIB_PATH):
        pytest.fail(f"{gate.LIB_PATH} is not built (make -C flash-attention3_amd)")
    kernels, bad = gate.check(gate.LIB_PATH)
    assert bad == []
    regs = [k for k in kernels if "bwd_reg_kernel" in k[".name"]]
    assert regs
    for k in regs:
        n = 3 if "ILi64E" in k[".name"] else 2
        assert k[".max_flat_workgroup_size"] == 256
        assert k[".vgpr_count"] + k[".agpr_count"] <= 512 // n // 8 * 8, k[".name"]
        assert n * k[".group_segment_fixed_size"] <= gate.LDS_BYTES, k[".name"]

"""The PyTorch op's native body (csrc/fa3_torch_op.cpp) against the same body
in Python: bit-equal outputs over types, plans and the optional scale, and the
same exception for a shape that the library refuses."""
import pytest

import shaobo_fa3 as F

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    F.load()
    import shaobo_fa3_torch
    assert shaobo_fa3_torch._native(), "lib/_fa3_torch.so is not built"
    return shaobo_fa3_torch


def both(T, monkeypatch, *args):
    op = torch.ops.shaobo_fa3.flash_attn_backward
    got = op(*args)
    monkeypatch.setattr(T, "_NATIVE", False)
    want = op(*args)
    monkeypatch.undo()
    torch.cuda.synchronize()
    return got, want


@pytest.mark.parametrize("B,Hq,Hkv,S,D,causal,dtype,scale,det", [
    (1, 1, 1, 128, 128, True, torch.float16, None, False),
    (2, 4, 2, 256, 64, False, torch.bfloat16, 0.25, True),
    (1, 2, 2, 512, 128, True, torch.bfloat16, None, False),
])
def test_native_body_equals_python_body(T, monkeypatch, B, Hq, Hkv, S, D, causal, dtype, scale,
                                        det):
    print(f"[case] native body B{B} Hq{Hq} Hkv{Hkv} S{S} D{D} {dtype}", flush=True)
    torch.manual_seed(1)
    q, dout, out = (torch.randn(B, Hq, S, D, device="cuda").to(dtype) for _ in range(3))
    k, v = (torch.randn(B, Hkv, S, D, device="cuda").to(dtype) for _ in range(2))
    lse = torch.rand(B, Hq, S, device="cuda") + 8.0
    got, want = both(T, monkeypatch, dout, q, k, v, out, lse, causal, scale, det)
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and a.shape == b.shape and a.is_contiguous()
        assert torch.equal(a, b)


def test_refused_shape_raises_the_same(T, monkeypatch):
    q = torch.randn(1, 1, 64, 128, device="cuda").half()  # not a whole 128-row tile
    lse = torch.zeros(1, 1, 64, device="cuda")
    said = []
    for native in (True, False):
        if not native:
            monkeypatch.setattr(T, "_NATIVE", False)
        with pytest.raises(RuntimeError) as e:
            torch.ops.shaobo_fa3.flash_attn_backward(q, q, q, q, q, lse, True, None, False)
        said.append(str(e.value))
    monkeypatch.undo()
    assert said[0] == said[1] == "shaobo_fa3_bwd_v2: unsupported"

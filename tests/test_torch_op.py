"""PyTorch custom-op binding (flash-attention3_amd/shaobo_fa3_torch.py), host
side: registration, the fake implementation's shapes, argument checks.  The
GPU behaviour is in test_gpu_torch_op.py."""
import os
import shutil
import subprocess
import sys
import warnings

import pytest

torch = pytest.importorskip("torch")
from torch._subclasses.fake_tensor import FakeTensorMode  # noqa: E402

import shaobo_fa3_torch as T  # noqa: E402  (registers the op)


def tensors(B=2, Hq=4, Hkv=2, S=256, D=128, dtype=torch.float16):
    q = torch.empty(B, Hq, S, D, dtype=dtype, device="cuda")
    k = torch.empty(B, Hkv, S, D, dtype=dtype, device="cuda")
    v = torch.empty_like(k)
    out = torch.empty_like(q)
    dout = torch.empty_like(q)
    lse = torch.empty(B, Hq, S, dtype=torch.float32, device="cuda")
    return dout, q, k, v, out, lse


def test_op_is_registered():
    assert hasattr(torch.ops.shaobo_fa3, "flash_attn_backward")


def test_fake_shapes_bf16():
    with FakeTensorMode():
        args = tensors(dtype=torch.bfloat16)
        dq, dk, dv, delta = torch.ops.shaobo_fa3.flash_attn_backward(*args, False, 0.1, False)
        assert dq.dtype == torch.bfloat16 and dk.shape == args[2].shape


def test_fake_shapes():
    with FakeTensorMode():
        dout, q, k, v, out, lse = tensors()
        dq, dk, dv, delta = torch.ops.shaobo_fa3.flash_attn_backward(dout, q, k, v, out, lse, True,
                                                                     None, False)
        assert dq.shape == q.shape and dq.dtype == torch.float16
        assert dk.shape == k.shape and dv.shape == v.shape
        assert delta.shape == (2, 4, 256) and delta.dtype == torch.float32


@pytest.mark.parametrize("bad", ["dtype", "lse_shape", "heads", "noncontig"])
def test_fake_rejects_bad_arguments(bad):
    with FakeTensorMode():
        dout, q, k, v, out, lse = tensors()
        if bad == "dtype":
            q = q.to(torch.bfloat16)  # mixed with fp16 k / v / out / dout
        elif bad == "lse_shape":
            lse = lse[:, :, :128]
        elif bad == "heads":
            k = torch.empty(2, 3, 256, 128, dtype=torch.float16, device="cuda")
            v = torch.empty_like(k)
        elif bad == "noncontig":
            q = q.transpose(1, 2)
        with pytest.raises(ValueError):
            torch.ops.shaobo_fa3.flash_attn_backward(dout, q, k, v, out, lse, True, None, False)


def test_native_body_that_does_not_load_falls_back(tmp_path, monkeypatch):
    """A _fa3_torch.so built for another Python, torch or library leaves the op
    its Python body, with one warning that names the reason."""
    bad = tmp_path / "_fa3_torch.so"
    bad.write_bytes(b"not a shared object")
    monkeypatch.setattr(T, "_NATIVE", None)
    monkeypatch.setattr(T, "_NATIVE_PATH", str(bad))
    with pytest.warns(RuntimeWarning, match="_fa3_torch.so"):
        assert T._native() is False
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert T._native() is False
    monkeypatch.setattr(T, "_NATIVE", None)
    monkeypatch.setattr(T, "_NATIVE_PATH", str(tmp_path / "absent.so"))
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert T._native() is False


@pytest.mark.skipif(shutil.which("make") is None, reason="no make")
def test_build_keeps_the_native_body_in_step(monkeypatch):
    """`make all` rebuilds an op body that is there, and the body is built for
    the interpreter that build() runs in."""
    if not os.path.exists(T._NATIVE_PATH):
        pytest.skip("lib/_fa3_torch.so is not built")
    pkg = os.path.dirname(os.path.dirname(T._NATIVE_PATH))
    dry = lambda *a: subprocess.run(["make", "-n", "-B", "-C", pkg, *a], text=True,  # noqa: E731
                                    capture_output=True, check=True).stdout
    assert "_fa3_torch.so" in dry("all")
    monkeypatch.syspath_prepend(os.path.dirname(pkg))
    import __graft_entry__ as entry
    calls = []
    monkeypatch.setattr(entry, "_make", lambda path, *targets: calls.append((path, targets)))
    entry.build()
    targets = next(t for p, t in calls if p == pkg)
    assert f"{sys.executable} -c" in dry(*targets)

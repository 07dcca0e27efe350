"""What the FlashAttention-3 backward is measured on.

A case is one backward pass through a public entry point:

* "v2"    shaobo_fa3_bwd_v2, the C ABI, as a caller that keeps its parameters,
          its workspace and its gradient buffers calls it (fp16 or bf16, BHSD
          or BSHD);
* "op"    torch.ops.shaobo_fa3.flash_attn_backward, as a training step's
          autograd function calls it: outputs and workspace come from torch;
* "chain" the component entries, dot_do_o -> dkv -> dq, with fp32 gradients
          (fp16 BHSD, causal, one query head per KV head).

Inputs are N(0, 1) rounded to the tensors' type, O and the natural-log LSE
come from an fp32 forward, the softmax scale is 1 / sqrt(D): the recipe of
bench.py and of the tests.
"""
import ctypes
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "flash-attention3_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import shaobo_fa3 as F  # noqa: E402
import shaobo_fa3_torch  # noqa: E402,F401  (registers the op)

_LOG2E = 1.44269504088896340736


def _case(name, entry, batch, heads_q, heads_kv, seqlen, head_dim, causal, dtype="fp16",
          layout="bhsd"):
    return {"name": name, "entry": entry, "batch": batch, "heads_q": heads_q,
            "heads_kv": heads_kv, "seqlen": seqlen, "head_dim": head_dim, "causal": causal,
            "dtype": dtype, "layout": layout}


def listed():
    return [
        # the smallest call: four tiles, all latency (unit tests, toy models)
        _case("tiny_s128", "v2", 1, 1, 1, 128, 128, True),
        # a short-context training step's call through the framework binding
        _case("op_small_d64_bf16", "op", 2, 8, 8, 256, 64, True, "bf16"),
        # one head of a short sequence: one long causal chain, few workgroups
        _case("one_head_s1024", "v2", 1, 1, 1, 1024, 128, True),
        # the headline shape of bench.py: few heads, causal
        _case("headline_s2048", "v2", 1, 4, 4, 2048, 128, True),
        # odd counts: 7 heads, 15 tiles of 128
        _case("odd_h7_s1920_bf16", "op", 1, 7, 7, 1920, 128, True, "bf16"),
        # an ordinary training batch of short sequences
        _case("train_s1024_bf16", "op", 4, 16, 16, 1024, 128, True, "bf16"),
        # grouped-query training in the [B, S, H, D] layout
        _case("gqa_bshd_s2048_bf16", "v2", 2, 32, 8, 2048, 128, True, "bf16", "bshd"),
        # full attention over an odd number of tiles, small heads (encoders)
        _case("full_d64_s1664", "op", 2, 12, 12, 1664, 64, False),
        # multi-query attention: one KV head for all query heads
        _case("mqa_s4096", "op", 1, 32, 1, 4096, 128, True),
        # the component chain with fp32 gradients
        _case("chain_s2048", "chain", 1, 8, 8, 2048, 128, True),
        # bench.py's grouped-query shape
        _case("gqa_s4096", "v2", 2, 32, 8, 4096, 128, True),
        # the largest: bench.py's long full-attention shape
        _case("full_d64_s8192", "v2", 2, 16, 16, 8192, 64, False),
    ]


def draw(rng):
    """One case of the ranges above: S from 128 to 8192 and the (batch, head)
    count from 1 to 128 over their logarithms, no more costly than the
    largest listed ones."""
    while True:
        entry = rng.choice(["v2", "v2", "op", "op", "chain"])
        seqlen = 128 * max(1, round(2.0 ** rng.uniform(0.0, 6.0)))
        rows = max(1, round(2.0 ** rng.uniform(0.0, 7.0)))  # batch x query heads
        batch = max(1, min(8, round(2.0 ** rng.uniform(0.0, 3.0))))
        heads = max(1, rows // batch)
        group = 1 if entry == "chain" else rng.choice([1, 1, 2, 4, 8])
        heads_kv = max(1, heads // group)
        case = {"entry": entry, "batch": batch, "heads_q": heads_kv * group,
                "heads_kv": heads_kv, "seqlen": seqlen,
                "head_dim": rng.choice([128, 128, 64]),
                "causal": True if entry == "chain" else rng.random() < 0.65,
                "dtype": "fp16" if entry == "chain" else rng.choice(["fp16", "bf16"]),
                "layout": rng.choice(["bhsd", "bhsd", "bshd"]) if entry == "v2" else "bhsd"}
        w = work(case)
        if w["flops"] <= 1.3e12 and w["bytes"] <= 5e8:
            return case


def work(case):
    """FLOPs: five products of 2 S^2 D per query head, half of them causal;
    bytes: Q, K, V, O, dO and the row statistics read once, the gradients and
    delta written once."""
    B, Hq, Hkv, S, D = (case[n] for n in ("batch", "heads_q", "heads_kv", "seqlen", "head_dim"))
    flops = 10.0 * B * Hq * S * S * D * (0.5 if case["causal"] else 1.0)
    grad = 4 if case["entry"] == "chain" else 2
    rows = B * Hq * S
    stats = 4 + 4  # LSE in, delta out
    if case["entry"] == "chain":
        stats = 8 + 4  # max and sum in, delta out
    nbytes = rows * (D * (3 * 2 + grad) + stats) + B * Hkv * S * D * (2 * 2 + 2 * grad)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # P and dS are rounded to the tensors' 16-bit type before the gradient
    # products, and so are K c or Q c and the gradients: about 4x the error
    # measured against exact() (fp16 3.8e-4, bf16 3.0e-3 at most)
    if case["dtype"] == "bf16":
        return {"rel": 1.2e-2}
    return {"rel": 1.5e-3}


# ---------------------------------------------------------------------------
def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float16


def _inputs(case, seed):
    """q, k, v, dout, out (16-bit BHSD), lse, smax, ssum (fp32 [B, Hq, S])."""
    B, Hq, Hkv, S, D = (case[n] for n in ("batch", "heads_q", "heads_kv", "seqlen", "head_dim"))
    gen = torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1))
    dt = _dtype(case)

    def randn(h):
        return torch.randn(B, h, S, D, generator=gen, device="cuda").to(dt)

    q, k, v, dout = randn(Hq), randn(Hkv), randn(Hkv), randn(Hq)
    out = torch.empty_like(q)
    smax = torch.empty(B, Hq, S, dtype=torch.float32, device="cuda")
    ssum, lse = torch.empty_like(smax), torch.empty_like(smax)
    scale = 1.0 / math.sqrt(D)
    hidden = torch.ones(S, S, dtype=torch.bool, device="cuda").triu(1) if case["causal"] else None
    group = Hq // Hkv
    for b in range(B):
        for h in range(Hq):
            s = q[b, h].float() @ k[b, h // group].float().t().contiguous()
            if hidden is not None:
                s.masked_fill_(hidden, float("-inf"))
            m = s.amax(dim=1)
            s = torch.exp2((s - m[:, None]) * (scale * _LOG2E))
            z = s.sum(dim=1)
            smax[b, h], ssum[b, h] = m, z
            lse[b, h] = m * scale + torch.log(z)
            out[b, h] = ((s @ v[b, h // group].float()) / z[:, None]).to(dt)
    return q, k, v, dout, out, lse, smax, ssum


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


class _State:
    pass


def prepare(case, seed):
    q, k, v, dout, out, lse, smax, ssum = _inputs(case, seed)
    st = _State()
    st.entry = case["entry"]
    if st.entry == "op":
        st.args = (dout, q, k, v, out, lse, case["causal"], None, False)
        return st
    lib = F.load()
    p = F.make_params(lib, batch=case["batch"], seqlen=case["seqlen"], heads_q=case["heads_q"],
                      heads_kv=case["heads_kv"], head_dim=case["head_dim"],
                      causal=case["causal"])
    st.lib, st.params = lib, p
    if st.entry == "chain":
        p.softmax_scale, p.softmax_scale_is_set = 1.0 / math.sqrt(case["head_dim"]), 1
        p.softmax_aux_mode = F.AUX_SMAX_SSUM
        p.dkv_path, p.dq_path = F.DKV_PATH_CANONICAL, F.DQ_PATH_CANONICAL
        st.delta = torch.empty_like(lse)
        st.packed = torch.empty(lse.numel(), 3, dtype=torch.float32, device="cuda")
        p.reserved_ptr[0], p.reserved_ptr[3] = st.delta.data_ptr(), st.packed.data_ptr()
        st.dq, st.dk, st.dv = (torch.empty(t.shape, dtype=torch.float32, device="cuda")
                               for t in (q, k, v))
        st.keep = (q, k, v, dout, out, smax, ssum)
        st.dot_args = [_ptr(t) for t in (dout, out, smax, ssum, st.delta, st.packed)]
        st.in_args = [_ptr(t) for t in (dout, q, k, v, out, smax, ssum)]
        st.grads = [_ptr(t) for t in (st.dq, st.dk, st.dv)]
        return st
    if case["dtype"] == "bf16":
        p.dtype = F.DTYPE_BF16
    if case["layout"] == "bshd":
        p.layout = F.LAYOUT_BSHD
        q, k, v, dout, out = (t.transpose(1, 2).contiguous() for t in (q, k, v, dout, out))
    nbytes = lib.shaobo_fa3_bwd_v2_workspace_bytes(ctypes.byref(p))
    st.workspace = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    p.workspace, p.workspace_bytes = st.workspace.data_ptr(), nbytes
    st.dq, st.dk, st.dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    st.delta = torch.empty_like(lse)
    st.keep = (q, k, v, dout, out, lse)
    st.ptrs = [_ptr(t) for t in (dout, q, k, v, out, lse, st.dq, st.dk, st.dv, st.delta)]
    return st


def _ok(status):
    if status != F.SUCCESS:
        raise RuntimeError(F.status_name(status))


def run(st):
    if st.entry == "op":
        dq, dk, dv, delta = torch.ops.shaobo_fa3.flash_attn_backward(*st.args)
        return {"dq": dq, "dk": dk, "dv": dv, "delta": delta}
    p = ctypes.byref(st.params)
    if st.entry == "chain":
        _ok(st.lib.shaobo_fa3_bwd_dot_do_o(*st.dot_args, p))
        _ok(st.lib.shaobo_fa3_bwd_dkv(*st.in_args, None, st.grads[1], st.grads[2], p))
        _ok(st.lib.shaobo_fa3_bwd_dq(*st.in_args, st.grads[0], None, None, p))
    else:
        _ok(st.lib.shaobo_fa3_bwd_v2(*st.ptrs, p))
    return {"dq": st.dq, "dk": st.dk, "dv": st.dv, "delta": st.delta}


def exact(case, seed):
    """The gradients of the same inputs (O and LSE as given) in fp64."""
    q, k, v, dout, out, lse, smax, ssum = _inputs(case, seed)
    Hq, Hkv, S, D = (case[n] for n in ("heads_q", "heads_kv", "seqlen", "head_dim"))
    scale, group = 1.0 / math.sqrt(D), Hq // Hkv
    delta = (dout.double() * out.double()).sum(-1)
    dq = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    dk = torch.zeros(k.shape, dtype=torch.float64, device="cuda")
    dv = torch.zeros_like(dk)
    visible = torch.ones(S, S, dtype=torch.bool, device="cuda").tril() if case["causal"] else None
    for b in range(case["batch"]):
        for h in range(Hq):
            c = h // group
            qd, kd, vd, do = (t.double() for t in (q[b, h], k[b, c], v[b, c], dout[b, h]))
            s = qd @ kd.t().contiguous()
            if case["entry"] == "chain":  # the row statistics as the entries get them
                p = torch.exp((s - smax[b, h].double()[:, None]) * scale)
                p /= ssum[b, h].double()[:, None]
            else:
                p = torch.exp(s * scale - lse[b, h].double()[:, None])
            if visible is not None:
                p *= visible
            dv[b, c] += p.t().contiguous() @ do
            p *= do @ vd.t().contiguous() - delta[b, h][:, None]
            dq[b, h] = (p @ kd) * scale
            dk[b, c] += (p.t().contiguous() @ qd) * scale
    if case["entry"] == "v2" and case["layout"] == "bshd":
        dq, dk, dv = (t.transpose(1, 2).contiguous() for t in (dq, dk, dv))
    return {"dq": dq, "dk": dk, "dv": dv, "delta": delta}

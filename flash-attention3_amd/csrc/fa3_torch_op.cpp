// Native body of the PyTorch op (shaobo_fa3_torch.py): parameters, outputs,
// workspace and launch of one backward in C++.
//
// What bounds the op at small sizes is the host, not the GPU: B2 H8 S256 D64
// took 30.1 us a call, 7 of them in torch's dispatch and the rest in the
// Python body (three checks, five allocations, a device guard, a ctypes call),
// against ~9 us of GPU time.  With this body a call takes 21.1 us.  The op's
// registration, autograd behaviour, fake implementation and argument checks
// stay in Python; only the body below the checks moved.
//
// The arguments have been checked (_check): contiguous BHSD tensors of one
// 16-bit type on the GPU whose stream `stream` is, which is the current
// device.
#include <torch/extension.h>

#include <stdexcept>
#include <string>
#include <tuple>

#include "shaobo_fa3_ext.h"

namespace {

std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor> backward(
    const at::Tensor& dout, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
    const at::Tensor& out, const at::Tensor& lse, bool causal, c10::optional<double> scale,
    bool deterministic, int64_t stream) {
    ShaoboFa3Params p;
    shaobo_fa3_params_init(&p);
    p.batch = (int32_t)q.size(0);
    p.num_heads_q = (int32_t)q.size(1);
    p.num_heads_kv = (int32_t)k.size(1);
    p.seqlen_q = p.seqlen_k = (int32_t)q.size(2);
    p.head_dim_qk = p.head_dim_v = (int32_t)q.size(3);
    p.causal = causal ? 1 : 0;
    if (scale.has_value()) {
        p.softmax_scale = (float)*scale;
        p.softmax_scale_is_set = 1;
    }
    p.deterministic = deterministic ? 1 : 0;
    if (q.scalar_type() == at::kBFloat16) p.dtype = SHAOBO_FA3_DTYPE_BF16;
    const size_t nbytes = shaobo_fa3_bwd_v2_workspace_bytes(&p);
    if (nbytes == 0)
        throw std::runtime_error(std::string("shaobo_fa3_bwd_v2: ") +
                                 shaobo_fa3_status_string(shaobo_fa3_bwd_v2_validate(&p)));
    const at::Tensor ws = at::empty({(int64_t)nbytes}, q.options().dtype(at::kByte));
    at::Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    at::Tensor delta = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
    p.workspace = ws.data_ptr();
    p.workspace_bytes = nbytes;
    const int st = shaobo_fa3_bwd_v2_on_stream(
        dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr(),
        dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), delta.data_ptr(), &p,
        reinterpret_cast<void*>(stream));
    if (st != SHAOBO_FA3_STATUS_SUCCESS)
        throw std::runtime_error(std::string("shaobo_fa3_bwd_v2_on_stream: ") +
                                 shaobo_fa3_status_string(st));
    return {dq, dk, dv, delta};
}

// Out of memory stays torch.OutOfMemoryError, as from torch's own bindings.
template <typename... Args>
auto guarded(Args... args) {
    try {
        py::gil_scoped_release nogil;
        return backward(args...);
    } catch (const c10::OutOfMemoryError& e) {
        PyErr_SetString(py::module_::import("torch").attr("OutOfMemoryError").ptr(),
                        e.what_without_backtrace());
        throw py::error_already_set();
    }
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.def("backward",
          &guarded<const at::Tensor&, const at::Tensor&, const at::Tensor&, const at::Tensor&,
                   const at::Tensor&, const at::Tensor&, bool, c10::optional<double>, bool,
                   int64_t>);
}

// Python binding of the W4A16 AWQ entry point for torch tensors (host code
// only; the kernels are behind the C ABI of libawq_w4a16.so,
// include/awq_w4a16.h).
//
// awq_gemm_forward(x, qweight, qzeros, scales, group_size) replaces the
// reference's entry point of the same name (kernels/awq_gemm.py:237-284) on
// the eager path: operand checks, the [M, K] flattening
// (kernels/awq_gemm.py:244-246), the fp16 output allocation, the plan, the
// split-K workspace and the current stream are all handled here, so that an
// eager call costs one Python -> C++ transition and one kernel launch (the
// reference engine makes 112 of these calls per token and never replays a
// graph, inference/engine.py:114-139).  The checks and their messages are
// the Python mirror's (kernels/awq_gemm.py in this package): ValueError for
// a bad operand, AwqNativeError (kernels/_native.py) with the status for a
// refused plan or a failed launch.
//
// gemm is the same with the bias and residual adds (awq_gemm_forward_ex's AUTO
// path), qwen2_layer a whole decoder layer of the engine.  At M = 1 a kernel
// takes 5 - 17 us and a call through ctypes 10: 16 layers' projections issued
// eagerly took 612 us, 579 through here; eight eager decode steps of four
// layers 3.85 ms, 3.02.
//
// Workspace registry: one list of zero-filled float32 buffers per device,
// grown on demand and never shrunk; earlier buffers stay referenced so that
// graphs captured with them keep valid memory.  Counters and fixed-point
// slots are zero between calls (every call leaves them zero), as the C ABI
// requires.  Growing while the stream is being captured is refused.
#include <torch/extension.h>

#include <ATen/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <unordered_map>
#include <vector>

#include "../../include/awq_w4a16.h"

namespace {

constexpr int64_t kWorkspaceAlign = 1 << 20;
constexpr size_t kPlanCacheMax = 4096;

struct PlanKey {
    int64_t M, N, K;
    int32_t group_size, path;
    int dev;
    bool operator==(const PlanKey& o) const {
        return M == o.M && N == o.N && K == o.K && group_size == o.group_size && path == o.path && dev == o.dev;
    }
};
struct PlanKeyHash {
    size_t operator()(const PlanKey& k) const {
        uint64_t h = (uint64_t)k.M * 0x9E3779B97F4A7C15ull;
        h ^= (uint64_t)k.N + 0x7F4A7C159E3779B9ull + (h << 6) + (h >> 2);
        h ^= (uint64_t)k.K + 0x2545F4914F6CDD1Dull + (h << 6) + (h >> 2);
        h ^= (uint64_t)(k.group_size * 131 + k.path * 7 + k.dev) + (h << 6) + (h >> 2);
        return (size_t)h;
    }
};

// Called with the Python GIL held (pybind11's default), so the two maps need
// no lock of their own.
std::unordered_map<PlanKey, awq_w4a16_plan, PlanKeyHash> g_plans;
std::unordered_map<int, std::vector<at::Tensor>> g_workspaces;

// The Python class that check_status raises, called with (status, where); set
// when the module is loaded and held until the process ends.
PyObject* g_status_error = nullptr;

void check_status(int st, const char* where) {
    if (st == AWQ_OK) return;
    TORCH_CHECK(g_status_error != nullptr, where, ": status ", st, ": ", awq_w4a16_error_string(st));
    PyErr_SetObject(g_status_error, py::make_tuple(st, where).ptr());
    throw py::error_already_set();
}

// The plan for a shape on a device (the planner sizes grids by the device's
// compute units, so the device must be current when it plans).
const awq_w4a16_plan& plan_for(int64_t M, int64_t N, int64_t K, int32_t group_size, int32_t path, int dev) {
    const PlanKey key{M, N, K, group_size, path, dev};
    auto it = g_plans.find(key);
    if (it != g_plans.end()) return it->second;
    awq_w4a16_plan p;
    check_status(awq_w4a16_plan_for(M, N, K, group_size, path, &p), "awq_w4a16_plan_for");
    if (g_plans.size() >= kPlanCacheMax) g_plans.clear();
    return g_plans.emplace(key, p).first->second;
}

// The device's largest workspace buffer, grown to at least `bytes`.
at::Tensor& workspace_for(const at::Device& device, uint64_t bytes, hipStream_t stream) {
    auto& bufs = g_workspaces[device.index()];
    if (!bufs.empty() && (uint64_t)bufs.back().numel() * 4u >= bytes) return bufs.back();
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    TORCH_CHECK(hipStreamIsCapturing(stream, &cap) == hipSuccess, "hipStreamIsCapturing failed");
    TORCH_CHECK(cap == hipStreamCaptureStatusNone, "awq_gemm workspace must grow to ", bytes,
                " bytes during graph capture; run the largest shape once eagerly before capturing");
    const int64_t size = ((int64_t)bytes + kWorkspaceAlign - 1) / kWorkspaceAlign * kWorkspaceAlign;
    bufs.push_back(at::zeros({size / 4}, at::TensorOptions().dtype(at::kFloat).device(device)));
    return bufs.back();
}

// `t` when its data starts on a 16-byte boundary, else a copy (the kernels use
// 16-byte vector accesses; the reference's Triton path takes any view).
at::Tensor aligned16(const at::Tensor& t) {
    return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0 ? t : t.clone();
}

// The operands of one projection, checked: ValueError for a bad one.
struct Linear {
    at::Tensor qweight, qzeros, scales;  // dense, scales 16-byte aligned
    int64_t K, N;
};

Linear checked_linear(int64_t k_of_x, const at::Device& device, const at::Tensor& qweight, const at::Tensor& qzeros,
                      const at::Tensor& scales, int64_t group_size) {
    TORCH_CHECK_VALUE(qweight.scalar_type() == at::kInt && qzeros.scalar_type() == at::kInt,
                      "qweight/qzeros must be int32, got ", qweight.scalar_type(), "/", qzeros.scalar_type());
    TORCH_CHECK_VALUE(scales.scalar_type() == at::kHalf, "scales must be float16, got ", scales.scalar_type());
    TORCH_CHECK_VALUE(group_size == 128, "group_size ", group_size, " is not served (only 128)");
    TORCH_CHECK_VALUE(qweight.dim() == 2 && qzeros.dim() == 2 && scales.dim() == 2,
                      "qweight, qzeros and scales must be 2-D and x at least 1-D");
    const int64_t K = k_of_x;
    const int64_t N = scales.size(1);
    TORCH_CHECK_VALUE(N > 0 && N % 8 == 0, "N = scales.shape[1] = ", N, " must be a positive multiple of 8");
    TORCH_CHECK_VALUE(K > 0 && K % group_size == 0, "K = ", K, " must be a positive multiple of group_size ",
                      group_size);
    TORCH_CHECK_VALUE(qweight.size(0) == K && qweight.size(1) == N / 8, "qweight shape ", qweight.sizes(),
                      " != (K, N/8) = (", K, ", ", N / 8, ")");
    TORCH_CHECK_VALUE(qzeros.size(0) == K / group_size && qzeros.size(1) == N / 8, "qzeros shape ",
                      qzeros.sizes(), " != (K/G, N/8) = (", K / group_size, ", ", N / 8, ")");
    TORCH_CHECK_VALUE(scales.size(0) == K / group_size, "scales shape ", scales.sizes(), " != (K/G, N) = (",
                      K / group_size, ", ", N, ")");
    TORCH_CHECK_VALUE(device.is_cuda(), "operands must be on a ROCm device, got ", device);
    TORCH_CHECK_VALUE(qweight.device() == device && qzeros.device() == device && scales.device() == device,
                      "all operands must be on ", device);
    return Linear{qweight.contiguous(), qzeros.contiguous(), aligned16(scales.contiguous()), K, N};
}

struct Workspace {
    void* ptr = nullptr;
    size_t bytes = 0;
};
Workspace workspace_of(const awq_w4a16_plan& p, const at::Device& device, hipStream_t stream) {
    if (p.workspace_bytes == 0) return {};
    at::Tensor& w = workspace_for(device, p.workspace_bytes, stream);
    return {w.data_ptr(), (size_t)w.numel() * 4u};
}

const void* data_or_null(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// x2 [M, K] @ W (+ bias, + residual; undefined = none) -> [M, N], the AUTO
// plan, on the current stream of the current device (x2's).
at::Tensor run_linear(const at::Tensor& x2, const Linear& w, const at::Tensor& bias, const at::Tensor& residual) {
    const int64_t M = x2.size(0);
    at::Tensor out = at::empty({M, w.N}, x2.options());
    if (M == 0) return out;
    const at::Device device = x2.device();
    const awq_w4a16_plan& p = plan_for(M, w.N, w.K, 128, AWQ_PATH_AUTO, device.index());
    hipStream_t stream = c10::hip::getCurrentHIPStream(device.index()).stream();
    const Workspace ws = workspace_of(p, device, stream);
    const int st = awq_w4a16_gemm_epilogue(x2.data_ptr(), w.qweight.data_ptr<int32_t>(), w.qzeros.data_ptr<int32_t>(),
                                           w.scales.data_ptr(), data_or_null(bias), data_or_null(residual),
                                           out.data_ptr(), M, w.N, w.K, 128, ws.ptr, ws.bytes, &p, stream);
    check_status(st, "awq_w4a16_gemm_epilogue");
    return out;
}

at::Tensor gemm(const at::Tensor& x, const at::Tensor& qweight, const at::Tensor& qzeros, const at::Tensor& scales,
                int64_t group_size, const c10::optional<at::Tensor>& bias,
                const c10::optional<at::Tensor>& residual) {
    TORCH_CHECK_VALUE(x.scalar_type() == at::kHalf, "x must be float16, got ", x.scalar_type());
    TORCH_CHECK_VALUE(x.dim() >= 1, "qweight, qzeros and scales must be 2-D and x at least 1-D");
    const at::Device device = x.device();
    const Linear w = checked_linear(x.size(-1), device, qweight, qzeros, scales, group_size);
    const at::Tensor x2 = aligned16((x.dim() == 2 ? x : x.reshape({-1, w.K})).contiguous());
    const int64_t M = x2.size(0);
    at::Tensor b, r;
    if (bias.has_value()) {
        TORCH_CHECK_VALUE(bias->scalar_type() == at::kHalf && bias->numel() == w.N && bias->device() == device,
                          "bias must be an fp16 [N=", w.N, "] tensor on ", device);
        b = bias->contiguous();
    }
    if (residual.has_value()) {
        TORCH_CHECK_VALUE(residual->scalar_type() == at::kHalf && residual->numel() == M * w.N &&
                              residual->device() == device,
                          "residual must be an fp16 tensor of M*N = ", M * w.N, " elements on ", device);
        r = residual->contiguous();
    }
    const at::DeviceGuard guard(device);
    at::Tensor out = run_linear(x2, w, b, r);
    if (x.dim() == 2) return out;
    std::vector<int64_t> out_shape(x.sizes().begin(), x.sizes().end() - 1);
    out_shape.push_back(w.N);
    return out.view(out_shape);
}

at::Tensor awq_gemm_forward(const at::Tensor& x, const at::Tensor& qweight, const at::Tensor& qzeros,
                            const at::Tensor& scales, int64_t group_size) {
    return gemm(x, qweight, qzeros, scales, group_size, c10::nullopt, c10::nullopt);
}

at::Tensor half_operand(const at::Tensor& t, int64_t n, const at::Device& device, const char* what) {
    TORCH_CHECK_VALUE(t.scalar_type() == at::kHalf && t.numel() == n && t.device() == device, what,
                      " must be an fp16 tensor of ", n, " values on ", device);
    return t.contiguous();
}

// fp16(x * rsqrt(mean(x^2) + eps) * w) of every row.
at::Tensor run_rmsnorm(const at::Tensor& x, const at::Tensor& w, double eps, hipStream_t stream) {
    at::Tensor out = at::empty(x.sizes(), x.options());
    check_status(awq_fp16_rmsnorm(x.data_ptr(), w.data_ptr(), out.data_ptr(), x.size(0), x.size(1), (float)eps, stream),
                 "awq_fp16_rmsnorm");
    return out;
}

// The projection of RMSNorm(h): for one row in the projection's own prologue
// where its kernel has one.
at::Tensor normed_linear(const at::Tensor& h, const at::Tensor& norm_w, double eps, const Linear& w,
                         const at::Tensor& bias, hipStream_t stream) {
    if (h.size(0) != 1 || !awq_w4a16_decode_served(w.N, w.K, 128, AWQ_INPUT_RMSNORM))
        return run_linear(run_rmsnorm(h, norm_w, eps, stream), w, bias, at::Tensor());
    at::Tensor out = at::empty({1, w.N}, h.options());
    const Workspace ws = workspace_of(plan_for(1, w.N, w.K, 128, AWQ_PATH_AUTO, h.device().index()), h.device(), stream);
    check_status(awq_w4a16_gemm_decode(AWQ_INPUT_RMSNORM, h.data_ptr(), norm_w.data_ptr(), (float)eps,
                                       w.qweight.data_ptr<int32_t>(), w.qzeros.data_ptr<int32_t>(),
                                       w.scales.data_ptr(), data_or_null(bias), nullptr, out.data_ptr(), w.N, w.K, 128,
                                       ws.ptr, ws.bytes, stream),
                 "awq_w4a16_gemm_decode");
    return out;
}

// The projection of SiLU(gate) * up plus the residual, likewise.
at::Tensor silu_linear(const at::Tensor& gate_up, const Linear& w, const at::Tensor& residual, hipStream_t stream) {
    const int64_t S = gate_up.size(0);
    if (S != 1 || !awq_w4a16_decode_served(w.N, w.K, 128, AWQ_INPUT_SILU_MUL)) {
        at::Tensor x = at::empty({S, w.K}, gate_up.options());
        check_status(awq_silu_mul(gate_up.data_ptr(), x.data_ptr(), S, w.K, stream), "awq_silu_mul");
        return run_linear(x, w, at::Tensor(), residual);
    }
    at::Tensor out = at::empty({1, w.N}, gate_up.options());
    const Workspace ws = workspace_of(plan_for(1, w.N, w.K, 128, AWQ_PATH_AUTO, gate_up.device().index()),
                                      gate_up.device(), stream);
    check_status(awq_w4a16_gemm_decode(AWQ_INPUT_SILU_MUL, gate_up.data_ptr(), nullptr, 0.0f,
                                       w.qweight.data_ptr<int32_t>(), w.qzeros.data_ptr<int32_t>(),
                                       w.scales.data_ptr(), nullptr, residual.data_ptr(), out.data_ptr(), w.N, w.K, 128,
                                       ws.ptr, ws.bytes, stream),
                 "awq_w4a16_gemm_decode");
    return out;
}

// One decoder layer of the Qwen2 engine (engine/qwen2_decode.py _layer) over
// the rows of h: a prompt's positions 0 .. S - 1 (causal), or one decode
// position pos (int64 [1] on the device).  p: the layer's weights by name.
// Everything is issued here, so that a layer costs one transition from
// Python and its own launches.
at::Tensor qwen2_layer(const at::Tensor& h, const at::Tensor& pos, bool causal, const py::dict& p,
                       const at::Tensor& k_cache, const at::Tensor& v_cache, const at::Tensor& cos,
                       const at::Tensor& sin, int64_t num_heads, double eps) {
    TORCH_CHECK_VALUE(h.scalar_type() == at::kHalf && h.dim() == 2, "h must be a 2-D fp16 tensor");
    const at::Device device = h.device();
    const int64_t S = h.size(0), H = h.size(1);
    TORCH_CHECK_VALUE(k_cache.dim() == 3 && k_cache.sizes() == v_cache.sizes(),
                      "k_cache and v_cache must be equal 3-D shapes");
    const int64_t kvh = k_cache.size(0), max_seq = k_cache.size(1), hd = k_cache.size(2);
    for (const at::Tensor* t : {&k_cache, &v_cache})
        TORCH_CHECK_VALUE(t->scalar_type() == at::kHalf && t->is_contiguous() && t->device() == device,
                          "the caches must be contiguous fp16 tensors on ", device);
    for (const at::Tensor* t : {&cos, &sin})
        TORCH_CHECK_VALUE(t->scalar_type() == at::kFloat && t->is_contiguous() && t->device() == device &&
                              t->dim() == 2 && t->size(0) == max_seq && t->size(1) == hd,
                          "cos and sin must be contiguous fp32 tensors [", max_seq, ", ", hd, "] on ", device);
    TORCH_CHECK_VALUE(causal ? S <= max_seq
                             : S == 1 && pos.scalar_type() == at::kLong && pos.numel() == 1 && pos.device() == device,
                      "the positions do not fit the cache, or pos is not an int64 [1] tensor on ", device);
    auto linear = [&](const char* name, int64_t K) {
        const py::tuple op = p[name];
        TORCH_CHECK_VALUE(op.size() == 3, name, " must be (qweight, qzeros, scales)");
        return checked_linear(K, device, op[0].cast<at::Tensor>(), op[1].cast<at::Tensor>(), op[2].cast<at::Tensor>(),
                              128);
    };
    const int64_t att_width = num_heads * hd, qkv_width = (num_heads + 2 * kvh) * hd;
    const Linear qkv_w = linear("qkv", H), o_w = linear("o", att_width), gate_up_w = linear("gate_up", H),
                 down_w = linear("down", gate_up_w.N / 2);
    TORCH_CHECK_VALUE(qkv_w.N == qkv_width && o_w.N == H && down_w.N == H && gate_up_w.N % 16 == 0,
                      "the projections' widths do not fit each other");
    const at::Tensor ln1 = aligned16(half_operand(p["ln1"].cast<at::Tensor>(), H, device, "ln1"));
    const at::Tensor ln2 = aligned16(half_operand(p["ln2"].cast<at::Tensor>(), H, device, "ln2"));
    const at::Tensor bias = half_operand(p["qkv_bias"].cast<at::Tensor>(), qkv_width, device, "qkv_bias");

    const at::DeviceGuard guard(device);
    hipStream_t stream = c10::hip::getCurrentHIPStream(device.index()).stream();
    const at::Tensor x = aligned16(h.contiguous());
    const at::Tensor qkv = normed_linear(x, ln1, eps, qkv_w, bias, stream);
    at::Tensor att = at::empty({S, att_width}, x.options());
    const size_t bytes = causal ? awq_fp16_attention_prefill_workspace(S, kvh, hd)
                                : awq_fp16_attention_decode_workspace(num_heads, kvh, hd, max_seq);
    const at::Tensor ws = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte));
    const int st =
        causal ? awq_fp16_attention_prefill(qkv.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), cos.data_ptr(),
                                            sin.data_ptr(), att.data_ptr(), S, num_heads, kvh, hd, max_seq,
                                            ws.data_ptr(), bytes, stream)
               : awq_fp16_attention_decode(qkv.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), cos.data_ptr(),
                                           sin.data_ptr(), pos.data_ptr<int64_t>(), att.data_ptr(), num_heads, kvh,
                                           hd, max_seq, ws.data_ptr(), bytes, stream);
    check_status(st, "awq_fp16_attention");
    const at::Tensor h2 = run_linear(att, o_w, at::Tensor(), x);
    const at::Tensor gate_up = normed_linear(h2, ln2, eps, gate_up_w, at::Tensor(), stream);
    return silu_linear(gate_up, down_w, h2, stream);
}

// The registry's buffer for `device_index` holding at least `nbytes` (grown
// if needed, refused during capture), for the Python entry points that pass
// a workspace through the C ABI themselves.
at::Tensor workspace(int64_t device_index, int64_t nbytes) {
    const at::Device device(at::kCUDA, (c10::DeviceIndex)device_index);
    const at::DeviceGuard guard(device);
    hipStream_t stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device_index).stream();
    return workspace_for(device, (uint64_t)nbytes, stream);
}

// Every buffer the registry holds for `device_index`, oldest first.
std::vector<at::Tensor> workspace_buffers(int64_t device_index) {
    auto it = g_workspaces.find((int)device_index);
    return it == g_workspaces.end() ? std::vector<at::Tensor>{} : it->second;
}

}  // namespace

PYBIND11_MODULE(_awq_torch, m) {
    m.doc() = "torch binding of the W4A16 AWQ GEMM C ABI (eager entry point, plan cache, workspace registry)";
    m.def("awq_gemm_forward", &awq_gemm_forward, "x @ dequant(qweight, qzeros, scales), fp16 (AUTO plan)",
          py::arg("x"), py::arg("qweight"), py::arg("qzeros"), py::arg("scales"), py::arg("group_size") = 128);
    m.def("gemm", &gemm, "awq_gemm_forward with the bias and residual adds fused into the store", py::arg("x"),
          py::arg("qweight"), py::arg("qzeros"), py::arg("scales"), py::arg("group_size"), py::arg("bias"),
          py::arg("residual"));
    m.def("qwen2_layer", &qwen2_layer, "one decoder layer of the Qwen2 engine", py::arg("h"), py::arg("pos"),
          py::arg("causal"), py::arg("p"), py::arg("k_cache"), py::arg("v_cache"), py::arg("cos"), py::arg("sin"),
          py::arg("num_heads"), py::arg("eps"));
    m.def("workspace", &workspace, "the device's workspace buffer, at least nbytes", py::arg("device_index"),
          py::arg("nbytes"));
    m.def("workspace_buffers", &workspace_buffers, "every workspace buffer of a device", py::arg("device_index"));
    m.def("set_status_error", [](const py::object& type) { g_status_error = type.inc_ref().ptr(); },
          "the exception class for a status of the C ABI", py::arg("type"));
    m.def("abi_version", [] { return awq_w4a16_abi_version(); });
}

// The host path of the three products between torch and the C ABI of pbs_hip.h: a CPython module (no pybind11) whose
// functions take torch tensors, allocate results and workspaces, build and keep the plans, launch on the current stream
// and record the autograd node.
//
// Why native: a product of a small layer runs 4 us on the GPU.  Issued from Python (autograd.Function, ctypes, the
// checks and the plan cache in Python) a call took 21 us of host time and a training step of one layer 160 us, so every
// case below some thousand tokens was bound by it; the same calls take 7.7 us and 70 us here (most of the latter in torch's
// autograd engine).
#include <Python.h>

#include <chrono>
#include <cstdlib>
#include <memory>
#include <mutex>
#include <unordered_map>

#include <ATen/core/Tensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/dynamo/compiled_autograd.h>
#include <torch/library.h>

#include "../../include/pbs_hip.h"

namespace {

using at::Tensor;

void check(int code, const char* what) {
    TORCH_CHECK(code == PBS_OK, what, " failed with code ", code, ": ", pbs_error_string(code));
}

// With PBS_DEBUG set (read at every call: tests switch it): raise if a bounded wait of a barrier-free kernel has run out
// since the last check.  The kernel marks the affected results NaN and counts the event; without this the call reports success.
void check_protocol(const char* what, int device) {
    const char* e = std::getenv("PBS_DEBUG");
    if (!e || !*e) return;
    static std::mutex lock;
    static unsigned seen[64];
    unsigned count = 0;
    check(pbs_protocol_failures(&count), "pbs_protocol_failures");
    std::lock_guard<std::mutex> hold(lock);
    const unsigned before = seen[device & 63];
    seen[device & 63] = count;
    TORCH_CHECK(count == before, what, ": ", count - before,
                " wait(s) of the kernel's progress protocol ran into their bound; the results of the affected tiles are NaN");
}

int dtype_code(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return PBS_DTYPE_F32;
        case at::kBFloat16: return PBS_DTYPE_BF16;
        default: TORCH_CHECK(false, "unsupported dtype ", t.dtype(), "; supported: float32, bfloat16");
    }
}

void check_gpu(const Tensor& t) {
    TORCH_CHECK(!t.defined() || t.is_cuda(),
                "pytorch_block_sparse_amd: the block-sparse matmuls run only on a GPU through libpbs_hip.so; got a tensor on ", t.device());
}

void* current_stream(const Tensor& t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }

// An index tensor as it was when the plans were made.
struct Seen {
    Tensor t;
    const void* data = nullptr;
    uint32_t version = 0;

    static uint32_t version_of(const Tensor& t) {   // (tensors made in inference mode do not count)
        const auto& v = t.unsafeGetTensorImpl()->version_counter();
        return v.enabled() ? v.current_version() : 0;
    }
    void take(const Tensor& now) {
        t = now;
        data = now.const_data_ptr();
        version = version_of(now);
    }
    bool still(const Tensor& now) const {
        return now.unsafeGetTensorImpl() == t.unsafeGetTensorImpl() && now.const_data_ptr() == data && version_of(now) == version;
    }
};

bool capturing(void* stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    const hipError_t e = hipStreamIsCapturing(static_cast<hipStream_t>(stream), &status);
    TORCH_CHECK(e == hipSuccess, "hipStreamIsCapturing: ", hipGetErrorString(e));
    return status != hipStreamCaptureStatusNone;
}

// A buffer that kernels on one stream fill and products on any stream read: each other stream waits for the filling once, and
// the allocator learns of it.  A stream that is being captured cannot wait for work outside its graph: whoever captures
// has the earlier work finished first (torch.cuda.graph waits for the device).
struct Derived {
    Tensor t;
    void* filled_on = nullptr;
    hipEvent_t event = nullptr;
    c10::SmallVector<void*, 4> waited;

    Derived() = default;
    Derived(const Derived&) = delete;
    Derived& operator=(const Derived&) = delete;
    ~Derived() {
        if (event) (void)hipEventDestroy(event);
    }
    void use_on(void* stream) {
        if (!t.defined() || stream == filled_on || capturing(stream)) return;
        for (void* w : waited)
            if (w == stream) return;
        const hipError_t e = hipStreamWaitEvent(static_cast<hipStream_t>(stream), event, 0);
        TORCH_CHECK(e == hipSuccess, "hipStreamWaitEvent: ", hipGetErrorString(e));
        t.record_stream(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).unwrap());
        waited.push_back(stream);
    }
    // after the kernels that fill `now` were launched on `stream`, which has waited for what was in it before
    void filled(const Tensor& now, void* stream) {
        hipError_t e = event ? hipSuccess : hipEventCreateWithFlags(&event, hipEventDisableTiming);
        if (e == hipSuccess) e = hipEventRecord(event, static_cast<hipStream_t>(stream));
        TORCH_CHECK(e == hipSuccess, "hipEventRecord: ", hipGetErrorString(e));
        t = now;
        filled_on = stream;
        waited.clear();
    }
};

// One pattern: its index arrays and the plans of both directions.  Never changed once made, except that parts of
// the plans are added when a product first needs them; a matrix whose index arrays change gets a new one, and autograd
// nodes keep the one of their forward product.  A part that is first needed while a graph is captured exists only
// when the graph has run: it is built inside the graph, for the graph, and not kept.
struct Pattern {
    Seen row_ptr, cols, col_ptr, rows;
    int out_features = 0, in_features = 0, nnz = 0;
    std::mutex lock;
    Derived plan[2];     // [transpose]
    int parts[2] = {0, 0};
    Derived units;       // of the weight gradient
    int64_t trained_tokens = 0;   // of the last training step's forward product, and its type
    int trained_code = 0;
    int64_t number = 0;  // that graphs of torch know it by (pattern_number)

    ~Pattern();
    bool still(const Tensor& rp, const Tensor& c, const Tensor& cp, const Tensor& r) const {
        return row_ptr.still(rp) && cols.still(c) && col_ptr.still(cp) && rows.still(r);
    }

    Tensor plan_for(bool transpose, int n, int k, int part, void* stream) {
        std::lock_guard<std::mutex> hold(lock);
        Derived& kept = plan[transpose];
        kept.use_on(stream);
        part |= PBS_PLAN_LIST;
        if ((parts[transpose] & part) == part) return kept.t;
        const Tensor& ptr = transpose ? row_ptr.t : col_ptr.t;
        const Tensor& idx = transpose ? cols.t : rows.t;
        TORCH_CHECK(ptr.is_cuda() && idx.is_cuda(), "the index buffers are not on the GPU");
        const bool keep = !capturing(stream);
        const size_t bytes = pbs_blocksparse_matmul_plan_part_bytes(n, k);
        const Tensor t = keep && kept.t.defined() ? kept.t : at::empty({(int64_t)bytes}, ptr.options().dtype(at::kByte));
        check(pbs_blocksparse_matmul_plan_part(ptr.const_data_ptr<int>(), idx.const_data_ptr<int>(), n, k, nnz,
                                               keep ? part & ~parts[transpose] : part, t.mutable_data_ptr(), bytes, stream),
              "pbs_blocksparse_matmul_plan_part");
        if (keep) {
            kept.filled(t, stream);
            parts[transpose] |= part;
        }
        return t;
    }
    // a training step's plans in one launch, if there is none yet
    void train(int64_t tokens, int code, void* stream) {
        std::lock_guard<std::mutex> hold(lock);
        derive_all(tokens, code, stream);
        trained_tokens = tokens;
        trained_code = code;
    }
    void derive_all(int64_t tokens, int code, void* stream) {
        if (parts[0] || parts[1] || units.t.defined() || !row_ptr.t.is_cuda() || !cols.t.is_cuda() || !col_ptr.t.is_cuda() ||
            !rows.t.is_cuda() || capturing(stream))
            return;
        const auto bytes = row_ptr.t.options().dtype(at::kByte);
        const size_t forward_bytes = pbs_blocksparse_matmul_plan_part_bytes(out_features, in_features),
                     input_bytes = pbs_blocksparse_matmul_plan_part_bytes(in_features, out_features),
                     units_bytes = pbs_blocksparse_matmul_back_units_bytes(tokens, out_features, in_features, nnz, code);
        const Tensor forward = at::empty({(int64_t)forward_bytes}, bytes), input = at::empty({(int64_t)input_bytes}, bytes);
        const Tensor table = units_bytes ? at::empty({(int64_t)units_bytes}, bytes) : Tensor();
        const int* no_blocks = nullptr;
        check(pbs_blocksparse_derive(row_ptr.t.const_data_ptr<int>(), nnz ? cols.t.const_data_ptr<int>() : no_blocks,
                                     col_ptr.t.const_data_ptr<int>(), nnz ? rows.t.const_data_ptr<int>() : no_blocks, out_features, in_features,
                                     nnz, forward.mutable_data_ptr(), forward_bytes, input.mutable_data_ptr(), input_bytes,
                                     units_bytes ? table.mutable_data_ptr() : nullptr, units_bytes, stream),
              "pbs_blocksparse_derive");
        plan[1].filled(forward, stream);
        plan[0].filled(input, stream);
        parts[0] = parts[1] = PBS_PLAN_LIST;
        if (units_bytes) units.filled(table, stream);
    }
    Tensor units_for(int64_t tokens, int code, void* stream) {
        const size_t bytes = pbs_blocksparse_matmul_back_units_bytes(tokens, out_features, in_features, nnz, code);
        if (!bytes) return Tensor();
        std::lock_guard<std::mutex> hold(lock);
        units.use_on(stream);
        if (units.t.defined()) return units.t;
        TORCH_CHECK(row_ptr.t.is_cuda() && cols.t.is_cuda(), "the index buffers are not on the GPU");
        const Tensor t = at::empty({(int64_t)bytes}, row_ptr.t.options().dtype(at::kByte));
        check(pbs_blocksparse_matmul_back_units(row_ptr.t.const_data_ptr<int>(), nnz ? cols.t.const_data_ptr<int>() : nullptr, out_features,
                                                in_features, nnz, t.mutable_data_ptr(), bytes, stream),
              "pbs_blocksparse_matmul_back_units");
        if (!capturing(stream)) units.filled(t, stream);
        return t;
    }
};
using PatternPtr = std::shared_ptr<Pattern>;

const void* data_or_null(const Tensor& t) { return t.defined() && t.numel() ? t.const_data_ptr() : nullptr; }

// what matmul asks of its operands; the sizes (n, k) of the product
std::pair<int, int> check_matmul(const Pattern& p, const Tensor& a_any, const Tensor& data, const Tensor& bias, bool transpose) {
    check_gpu(a_any);
    check_gpu(data);
    check_gpu(bias);
    dtype_code(a_any);
    TORCH_CHECK(data.scalar_type() == a_any.scalar_type(), "dense operand is ", a_any.dtype(), " but the block data is ", data.dtype());
    TORCH_CHECK(!bias.defined() || bias.scalar_type() == a_any.scalar_type(), "bias is ", bias.dtype(), ", expected ", a_any.dtype());
    TORCH_CHECK(data.is_contiguous(), "block data must be contiguous");
    TORCH_CHECK(data.device() == a_any.device() && (!bias.defined() || bias.device() == a_any.device()),
                "the operands are on different devices");
    const int n = transpose ? p.out_features : p.in_features, k = transpose ? p.in_features : p.out_features;
    TORCH_CHECK(a_any.dim() >= 2, "Invalid dimensions for dense_a ", a_any.sizes(), " : dense_a should have at least 2 dimensions.");
    TORCH_CHECK(a_any.size(-1) == k, "Invalid matrices sizes ", a_any.sizes(), " x (", k, ", ", n, ")");
    TORCH_CHECK(data.numel() == (int64_t)p.nnz * 1024, "the block data does not match the index buffers");
    TORCH_CHECK(!bias.defined() || (bias.numel() == n && bias.is_contiguous()), "bias should be contiguous and hold ", n, " values");
    return {n, k};
}

// a [..., k] -> [..., n]; `training`: the products of a backward pass will follow
Tensor matmul(Pattern& p, const Tensor& a_any, const Tensor& data, const Tensor& bias, bool transpose, bool training = false) {
    const auto [n, k] = check_matmul(p, a_any, data, bias, transpose);
    const int code = dtype_code(a_any);
    const Tensor a = a_any.is_contiguous() ? a_any : a_any.contiguous();
    const int64_t tokens = a.numel() / k;
    c10::DeviceGuard guard(a.device());
    void* stream = current_stream(a);
    c10::SmallVector<int64_t, 6> sizes(a.sizes().begin(), a.sizes().end());
    sizes.back() = n;
    Tensor out = at::empty(sizes, a.options());
    if (tokens == 0) return out;
    if (training) p.train(tokens, code, stream);
    const int part = pbs_blocksparse_matmul_part(tokens, n, k, p.nnz, transpose, code, 1);
    const Tensor plan = p.plan_for(transpose, n, k, part, stream);
    // the transposed copy of the blocks that the bf16 column kernel's forward product works from, or the blocks in bf16 parts for larger fp32 products
    size_t ws_bytes = 0;
    if (code == PBS_DTYPE_F32) ws_bytes = pbs_blocksparse_matmul_parts_bytes(tokens, n, k, p.nnz, transpose, code);
    else if (transpose && part == PBS_PLAN_COLUMN) ws_bytes = pbs_blocksparse_matmul_workspace_bytes(tokens, n, k, p.nnz, 1, code);
    Tensor ws;
    if (ws_bytes) ws = at::empty({(int64_t)ws_bytes}, a.options().dtype(at::kByte));
    check(pbs_blocksparse_matmul_ws(a.const_data_ptr(), data_or_null(data), plan.const_data_ptr(), data_or_null(bias), out.mutable_data_ptr(), tokens, n, k,
                                    p.nnz, transpose, code, ws_bytes ? ws.mutable_data_ptr() : nullptr, ws_bytes, stream),
          "pbs_blocksparse_matmul_ws");
    check_protocol("pbs_blocksparse_matmul_ws", a.device().index());
    return out;
}

void check_matmul_back(const Pattern& p, const Tensor& a_any, const Tensor& b_any, const Tensor& out) {
    check_gpu(a_any);
    check_gpu(b_any);
    check_gpu(out);
    dtype_code(a_any);
    TORCH_CHECK(b_any.scalar_type() == a_any.scalar_type() && out.scalar_type() == a_any.scalar_type(), "operands and result must share one dtype");
    TORCH_CHECK(b_any.device() == a_any.device() && out.device() == a_any.device() && p.cols.t.device() == a_any.device(),
                "the operands are on different devices");
    TORCH_CHECK(a_any.size(-1) == p.out_features && b_any.size(-1) == p.in_features && out.numel() == (int64_t)p.nnz * 1024 && out.is_contiguous(),
                "Invalid matrices sizes ", a_any.sizes(), "^T x ", b_any.sizes());
    TORCH_CHECK(b_any.numel() / p.in_features == a_any.numel() / p.out_features, "Invalid matrices sizes ", a_any.sizes(), "^T x ", b_any.sizes());
}

// packed blocks of a^T b on the pattern, into `out`, and the sums of a's columns, into `sums` (if defined)
void matmul_back(Pattern& p, const Tensor& a_any, const Tensor& b_any, const Tensor& out, const Tensor& sums = Tensor()) {
    check_matmul_back(p, a_any, b_any, out);
    const int code = dtype_code(a_any);
    const Tensor a = a_any.is_contiguous() ? a_any : a_any.contiguous();
    const Tensor b = b_any.is_contiguous() ? b_any : b_any.contiguous();
    const int64_t tokens = a.numel() / p.out_features;
    c10::DeviceGuard guard(a.device());
    void* stream = current_stream(a);
    const Tensor units = p.units_for(tokens, code, stream);
    const size_t ws_bytes = pbs_blocksparse_matmul_back_bias_workspace_bytes(tokens, p.out_features, p.in_features, p.nnz, code);
    Tensor ws;
    if (ws_bytes) ws = at::empty({(int64_t)ws_bytes}, a.options().dtype(at::kByte));
    check(pbs_blocksparse_matmul_back_bias(data_or_null(a), data_or_null(b), p.row_ptr.t.const_data_ptr<int>(),
                                           static_cast<const int*>(data_or_null(p.cols.t)), data_or_null(units), out.numel() ? out.mutable_data_ptr() : nullptr,
                                           sums.defined() ? sums.mutable_data_ptr() : nullptr, tokens, p.out_features, p.in_features, p.nnz, code,
                                           ws_bytes ? ws.mutable_data_ptr() : nullptr, ws_bytes, stream),
          "pbs_blocksparse_matmul_back_bias");
}

// both, of a contiguous dy: dx = dy W, and the blocks of dy^T x with the sums of dy's columns (if defined)
Tensor both_gradients(Pattern& p, const Tensor& dy, const Tensor& x_any, const Tensor& data, const Tensor& out, const Tensor& sums) {
    const auto [n, k] = check_matmul(p, dy, data, Tensor(), false);
    check_matmul_back(p, dy, x_any, out);
    const int code = dtype_code(dy);
    const int64_t tokens = dy.numel() / k;
    if (tokens == 0) {
        matmul_back(p, dy, x_any, out, sums);
        return matmul(p, dy, data, Tensor(), false);
    }
    const Tensor x = x_any.is_contiguous() ? x_any : x_any.contiguous();
    c10::DeviceGuard guard(dy.device());
    void* stream = current_stream(dy);
    c10::SmallVector<int64_t, 6> sizes(dy.sizes().begin(), dy.sizes().end());
    sizes.back() = n;
    Tensor dx = at::empty(sizes, dy.options());
    const Tensor plan = p.plan_for(false, n, k, pbs_blocksparse_matmul_part(tokens, n, k, p.nnz, 0, code, 1), stream);
    const Tensor units = p.units_for(tokens, code, stream);
    const size_t ws_bytes = pbs_blocksparse_linear_back_workspace_bytes(tokens, p.out_features, p.in_features, p.nnz, code);
    Tensor ws;
    if (ws_bytes) ws = at::empty({(int64_t)ws_bytes}, dy.options().dtype(at::kByte));
    check(pbs_blocksparse_linear_back(data_or_null(dy), data_or_null(x), data_or_null(data), plan.const_data_ptr(), p.row_ptr.t.const_data_ptr<int>(),
                                      static_cast<const int*>(data_or_null(p.cols.t)), data_or_null(units), dx.mutable_data_ptr(),
                                      out.numel() ? out.mutable_data_ptr() : nullptr, sums.defined() ? sums.mutable_data_ptr() : nullptr, tokens,
                                      p.out_features, p.in_features, p.nnz, code, ws_bytes ? ws.mutable_data_ptr() : nullptr, ws_bytes, stream),
          "pbs_blocksparse_linear_back");
    check_protocol("pbs_blocksparse_linear_back", dy.device().index());
    return dx;
}

// The gradients of x (dx = dy W), of the blocks and of the bias (the sum of dy over the tokens) that are wanted, others undefined.
std::array<Tensor, 3> linear_backward(Pattern& p, const Tensor& dy_any, const Tensor& x, const Tensor& data, std::array<bool, 3> wanted) {
    at::NoGradGuard no_grad;
    std::array<Tensor, 3> out;
    const Tensor dy = dy_any.is_contiguous() ? dy_any : dy_any.contiguous();
    if (wanted[0] && !wanted[1]) out[0] = matmul(p, dy, data, Tensor(), false);
    if (wanted[1]) {
        out[1] = at::empty({(int64_t)p.nnz * 32, 32}, x.options());
        if (wanted[2]) out[2] = at::empty({p.out_features}, x.options());
        if (wanted[0]) out[0] = both_gradients(p, dy, x, data, out[1], out[2]);
        else matmul_back(p, dy, x, out[1], out[2]);
    } else if (wanted[2]) {
        out[2] = dy.reshape({-1, dy.size(-1)}).sum(0);
    }
    return out;
}

// Patterns that graphs of torch refer to, by a number that is never given out again; a graph does not keep its pattern.
std::mutex numbered_lock;
std::unordered_map<int64_t, std::weak_ptr<Pattern>>& numbered() {   // (outlives every pattern)
    static auto* all = new std::unordered_map<int64_t, std::weak_ptr<Pattern>>();
    return *all;
}
int64_t pattern_number(const PatternPtr& p) {
    static int64_t last = 0;
    std::lock_guard<std::mutex> hold(numbered_lock);
    if (!p->number) {
        p->number = ++last;
        numbered()[p->number] = p;
    }
    return p->number;
}
PatternPtr numbered_pattern(int64_t number) {
    std::lock_guard<std::mutex> hold(numbered_lock);
    const auto at = numbered().find(number);
    const PatternPtr p = at == numbered().end() ? nullptr : at->second.lock();
    TORCH_CHECK(p, "the block-sparse pattern of this graph does not exist any more");
    return p;
}
Pattern::~Pattern() {
    if (!number) return;
    std::lock_guard<std::mutex> hold(numbered_lock);
    numbered().erase(number);
}

// The same as an operator that a graph of torch can hold, for compiled autograd, which calls the node below with tensors that have no
// data.  Returns the wanted gradients alone.
std::vector<Tensor> linear_backward_op(const Tensor& dy, const std::optional<Tensor>& x, const std::optional<Tensor>& data, int64_t pattern, bool dx,
                                       bool dw, bool db) {
    std::vector<Tensor> out;
    for (Tensor& t : linear_backward(*numbered_pattern(pattern), dy, x.value_or(Tensor()), data.value_or(Tensor()), {dx, dw, db}))
        if (t.defined()) out.push_back(std::move(t));
    return out;
}
std::vector<Tensor> linear_backward_shapes(const Tensor& dy, const std::optional<Tensor>&, const std::optional<Tensor>&, int64_t pattern, bool dx,
                                           bool dw, bool db) {
    const PatternPtr p = numbered_pattern(pattern);
    std::vector<Tensor> out;
    auto sizes = dy.sym_sizes().vec();
    sizes.back() = p->in_features;
    if (dx) out.push_back(at::empty_symint(sizes, dy.options()));
    if (dw) out.push_back(at::empty({(int64_t)p->nnz * 32, 32}, dy.options()));
    if (db) out.push_back(at::empty({p->out_features}, dy.options()));
    return out;
}
TORCH_LIBRARY(pytorch_block_sparse_amd, m) {
    m.def("linear_backward(Tensor dy, Tensor? x, Tensor? data, int pattern, bool dx, bool dw, bool db) -> Tensor[]");
}
TORCH_LIBRARY_IMPL(pytorch_block_sparse_amd, CUDA, m) { m.impl("linear_backward", linear_backward_op); }
TORCH_LIBRARY_IMPL(pytorch_block_sparse_amd, Meta, m) { m.impl("linear_backward", linear_backward_shapes); }

// y = x W^T + bias
struct BlockSparseLinearBackward : public torch::autograd::Node {
    PatternPtr pattern;
    torch::autograd::SavedVariable x, data;
    bool has_bias = false;

    std::string name() const override { return "BlockSparseLinearBackward"; }
    void release_variables() override {
        x.reset_data();
        data.reset_data();
    }
    torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
        torch::autograd::variable_list out(3);
        const Tensor& g = grads[0];
        if (!g.defined()) return out;
        std::array<bool, 3> wanted = wants();
        // under create_graph the sum of dy is recorded, as the operator it is; the products have no second derivative
        if (c10::GradMode::is_enabled() && wanted[2]) {
            out[2] = g.reshape({-1, g.size(-1)}).sum(0);
            wanted[2] = false;
        }
        auto made = linear_backward(*pattern, g, wanted[1] ? x.unpack(shared_from_this()) : Tensor(), wanted[0] ? data.unpack(shared_from_this()) : Tensor(),
                                    wanted);
        for (int i = 0; i < 3; ++i)
            if (wanted[i]) out[i] = std::move(made[i]);
        return out;
    }

    void compiled_args(torch::dynamo::autograd::CompiledNodeArgs& args) const override {
        args.collect(x, false);
        args.collect(data, false);
        args.collect(has_bias);
        args.collect(pattern_number(pattern));   // a graph is made for one pattern
    }
    torch::autograd::variable_list apply_with_saved(const torch::autograd::variable_list& grads, torch::dynamo::autograd::SwapSavedVariables& saved) override {
        saved.before(x);
        saved.before(data);
        torch::autograd::variable_list out(3);
        if (grads[0].defined()) {
            static const auto op = c10::Dispatcher::singleton()
                                       .findSchemaOrThrow("pytorch_block_sparse_amd::linear_backward", "")
                                       .typed<std::vector<Tensor>(const Tensor&, const std::optional<Tensor>&, const std::optional<Tensor>&, int64_t, bool, bool, bool)>();
            const std::array<bool, 3> wanted = wants();
            const auto maybe = [&](bool want, torch::autograd::SavedVariable& v) {
                return want ? std::optional<Tensor>(v.unpack(shared_from_this())) : std::nullopt;
            };
            auto made = op.call(grads[0], maybe(wanted[1], x), maybe(wanted[0], data), pattern_number(pattern), wanted[0], wanted[1], wanted[2]);
            size_t at = 0;
            for (int i = 0; i < 3; ++i)
                if (wanted[i]) out[i] = std::move(made[at++]);
        }
        saved.after(x);
        saved.after(data);
        return out;
    }

  private:
    std::array<bool, 3> wants() const {
        return {task_should_compute_output(0), task_should_compute_output(1), has_bias && task_should_compute_output(2)};
    }
};

Tensor linear(const PatternPtr& p, const Tensor& x, const Tensor& data, const Tensor& bias) {
    for (const Tensor* t : {&x, &data, &bias})
        TORCH_CHECK_NOT_IMPLEMENTED(!t->defined() || !t->_fw_grad(0).defined(), "the block-sparse linear layer has no forward-mode derivative");
    const bool training = torch::autograd::compute_requires_grad(x, data, bias);
    Tensor y;
    {
        at::NoGradGuard no_grad;
        y = matmul(*p, x, data, bias, true, training && x.requires_grad() && data.requires_grad());
    }
    if (training) {
        auto node = std::shared_ptr<BlockSparseLinearBackward>(new BlockSparseLinearBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(x, data, bias));
        node->pattern = p;
        node->has_bias = bias.defined();
        if (data.requires_grad()) node->x = torch::autograd::SavedVariable(x, false);
        if (x.requires_grad()) node->data = torch::autograd::SavedVariable(data, false);
        torch::autograd::set_history(y, node);
    }
    return y;
}

// ---------------------------------------------------------------------------------------------------------------
// Python side
// ---------------------------------------------------------------------------------------------------------------

// Where a matrix keeps its Pattern.
struct Schedule {
    PyObject_HEAD
    PatternPtr* pattern;
    std::mutex* lock;
};

PyObject* schedule_new(PyTypeObject* type, PyObject*, PyObject*) {
    Schedule* self = reinterpret_cast<Schedule*>(type->tp_alloc(type, 0));
    if (self) {
        self->pattern = new PatternPtr();
        self->lock = new std::mutex();
    }
    return reinterpret_cast<PyObject*>(self);
}
void schedule_dealloc(PyObject* o) {
    Schedule* self = reinterpret_cast<Schedule*>(o);
    delete self->pattern;
    delete self->lock;
    Py_TYPE(o)->tp_free(o);
}
PyTypeObject ScheduleType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject *s_row_ptr, *s_cols, *s_col_ptr, *s_rows;   // buffer names, interned

Tensor tensor_arg(PyObject* o, const char* what) {
    TORCH_CHECK_TYPE(THPVariable_Check(o), what, " should be a tensor, not ", Py_TYPE(o)->tp_name);
    return THPVariable_Unpack(o);
}
Tensor optional_tensor(PyObject* o, const char* what) { return o == Py_None ? Tensor() : tensor_arg(o, what); }

const Tensor& buffer(PyObject* buffers, PyObject* name) {
    PyObject* o = PyDict_GetItem(buffers, name);   // borrowed
    TORCH_CHECK(o && THPVariable_Check(o), "the matrix has no index buffer ", PyUnicode_AsUTF8(name));
    return THPVariable_Unpack(o);
}

PatternPtr pattern_of(const Tensor& rp, const Tensor& c, const Tensor& cp, const Tensor& r) {
    for (const Tensor* t : {&rp, &c, &cp, &r})
        TORCH_CHECK(t->scalar_type() == at::kInt && t->is_contiguous(), "index buffers should be contiguous int32 tensors");
    auto q = std::make_shared<Pattern>();
    q->row_ptr.take(rp);
    q->cols.take(c);
    q->col_ptr.take(cp);
    q->rows.take(r);
    q->out_features = (int)(rp.numel() - 1) * 32;
    q->in_features = (int)(cp.numel() - 1) * 32;
    q->nnz = (int)(c.numel() / 2);
    TORCH_CHECK(r.numel() == c.numel(), "cols_a and rows_b differ in length");
    return q;
}

// The pattern of a matrix, from its `_buffers` and its Schedule; a new one if the buffers are not those it was made from.
PatternPtr pattern_arg(PyObject* buffers, PyObject* schedule) {
    TORCH_CHECK_TYPE(PyDict_Check(buffers) && Py_TYPE(schedule) == &ScheduleType, "expected a matrix's buffers and Schedule");
    Schedule* s = reinterpret_cast<Schedule*>(schedule);
    const Tensor &rp = buffer(buffers, s_row_ptr), &c = buffer(buffers, s_cols), &cp = buffer(buffers, s_col_ptr), &r = buffer(buffers, s_rows);
    std::lock_guard<std::mutex> hold(*s->lock);
    PatternPtr& p = *s->pattern;
    if (!p || !p->still(rp, c, cp, r)) p = pattern_of(rp, c, cp, r);
    return p;
}

void need(Py_ssize_t got, Py_ssize_t want, const char* what) { TORCH_CHECK_TYPE(got == want, what, " takes ", want, " arguments, got ", got); }

struct NoGil {
    PyThreadState* s = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(s); }
};

// linear(x, data, bias or None, buffers, schedule) -> y, recorded for autograd
PyObject* py_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need(n, 5, "linear");
    const Tensor x = tensor_arg(args[0], "x"), data = tensor_arg(args[1], "data"), bias = optional_tensor(args[2], "bias");
    const PatternPtr p = pattern_arg(args[3], args[4]);
    Tensor y;
    {
        NoGil no_gil;
        y = linear(p, x, data, bias);
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// matmul(a, data, bias or None, transpose, buffers, schedule) -> a W^T or a W, outside autograd
PyObject* py_matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need(n, 6, "matmul");
    const Tensor a = tensor_arg(args[0], "dense_a"), data = tensor_arg(args[1], "data"), bias = optional_tensor(args[2], "bias");
    const bool transpose = PyObject_IsTrue(args[3]) == 1;
    const PatternPtr p = pattern_arg(args[4], args[5]);
    Tensor y;
    {
        NoGil no_gil;
        at::NoGradGuard no_grad;
        y = matmul(*p, a, data, bias, transpose);
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// matmul_back(a, b, out, buffers, schedule): packed blocks of a^T b into out
PyObject* py_matmul_back(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need(n, 5, "matmul_back");
    const Tensor a = tensor_arg(args[0], "dense_a"), b = tensor_arg(args[1], "dense_b"), out = tensor_arg(args[2], "out");
    const PatternPtr p = pattern_arg(args[3], args[4]);
    {
        NoGil no_gil;
        at::NoGradGuard no_grad;
        matmul_back(*p, a, b, out);
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// One status word that the GPU writes once, in memory that the host sees at once.  The host looks for it for a millisecond, so that it is back
// within a microsecond or two and not when the stream's signal has arrived and what was launched behind the word is done; then it waits
// for the stream, as it does for a word that cannot come (an error, a stream that is being captured).
constexpr int STATUS_PENDING = -1;
Tensor status_word() {
    Tensor word = at::empty({1}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    *word.mutable_data_ptr<int>() = STATUS_PENDING;
    return word;
}
int read_status(const Tensor& status, void* stream) {
    const volatile int* word = static_cast<const volatile int*>(status.const_data_ptr());
    if (!capturing(stream)) {
        const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
        while (*word == STATUS_PENDING && std::chrono::steady_clock::now() < until) {
        }
        if (*word != STATUS_PENDING) return *word;
    }
    const hipError_t e = hipStreamSynchronize(static_cast<hipStream_t>(stream));
    TORCH_CHECK(e == hipSuccess, "hipStreamSynchronize: ", hipGetErrorString(e));
    return *word;
}
Tensor workspace(size_t bytes, const Tensor& like) { return at::empty({(int64_t)(bytes ? bytes : 16)}, like.options().dtype(at::kByte)); }
const int* ints(const Tensor& t) { return static_cast<const int*>(data_or_null(t)); }
int* ints_out(Tensor& t) { return t.numel() ? t.mutable_data_ptr<int>() : nullptr; }

// replace_blocks(blocks, moves [n, 3] int64, X, Y, Schedule or None) -> (status, (blocks, cols_a, row_start_ends_a, rows_b, col_start_ends_b), Schedule or
// None).  Where the pattern of the given Schedule has been trained, the new one will be: its plans are made behind the arrays, while the host is still
// waiting for the status, and come in a Schedule.  (768 -> 3072 density 0.5, 1024 tokens, fp32: block_replace and a step 130 -> 112 us, of which the step is 85.)
PyObject* py_replace_blocks(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need(n, 5, "replace_blocks");
    const Tensor old = tensor_arg(args[0], "blocks"), moves_any = tensor_arg(args[1], "moves");
    const int X = (int)PyLong_AsLong(args[2]), Y = (int)PyLong_AsLong(args[3]);
    check_gpu(old);
    TORCH_CHECK(old.scalar_type() == at::kInt && old.is_contiguous() && moves_any.scalar_type() == at::kLong && moves_any.device() == old.device() &&
                    moves_any.dim() == 2 && moves_any.size(1) == 3,
                "moves should be a [n, 3] int64 tensor on the device of the matrix");
    const int nnz = (int)(old.numel() / 2);
    PatternPtr before, after;
    if (args[4] != Py_None) {
        TORCH_CHECK_TYPE(Py_TYPE(args[4]) == &ScheduleType, "expected a Schedule");
        const Schedule* s = reinterpret_cast<Schedule*>(args[4]);
        std::lock_guard<std::mutex> hold(*s->lock);
        before = *s->pattern;
    }
    Tensor made[5];
    int status = 0;
    {
        NoGil no_gil;
        at::NoGradGuard no_grad;
        const Tensor moves = moves_any.contiguous();
        c10::DeviceGuard guard(old.device());
        void* stream = current_stream(old);
        const int64_t sizes[5][2] = {{2 * (int64_t)nnz, 0}, {nnz, 2}, {X + 1, 0}, {nnz, 2}, {Y + 1, 0}};
        for (int i = 0; i < 5; ++i) made[i] = at::empty(at::IntArrayRef(sizes[i], sizes[i][1] ? 2 : 1), old.options());
        const size_t bytes = pbs_replace_blocks_workspace_bytes(X, Y, nnz);
        Tensor ws = workspace(bytes, old), word = status_word();
        check(pbs_replace_blocks(ints(old), moves.numel() ? moves.const_data_ptr<int64_t>() : nullptr, (int)moves.size(0), X, Y, nnz,
                                 ints_out(made[1]), ints_out(made[2]), ints_out(made[3]), ints_out(made[4]), ints_out(made[0]),
                                 word.mutable_data_ptr<int>(), ws.mutable_data_ptr(), bytes, stream),
              "pbs_replace_blocks");
        int64_t tokens = 0;
        int code = 0;
        if (before) {
            std::lock_guard<std::mutex> hold(before->lock);
            tokens = before->trained_tokens;
            code = before->trained_code;
        }
        if (tokens && before->out_features == 32 * X && before->in_features == 32 * Y) {
            // (arrays of rejected moves hold anything: the kernels that read them clamp what they find.  The moves need no plans: without room for these, the next
            // product makes its own or says why not.  The status is waited for in any case, as the kernel that writes it is under way.)
            try {
                after = pattern_of(made[2], made[1], made[4], made[3]);
                std::lock_guard<std::mutex> hold(after->lock);
                after->derive_all(tokens, code, stream);
            } catch (const std::exception&) {
                after.reset();
            }
        }
        status = read_status(word, stream);
    }
    PyObject* schedule = Py_None;
    if (after && status == 0) {
        schedule = schedule_new(&ScheduleType, nullptr, nullptr);
        if (!schedule) return nullptr;
        *reinterpret_cast<Schedule*>(schedule)->pattern = std::move(after);
    } else {
        Py_INCREF(Py_None);
    }
    PyObject* arrays = PyTuple_New(5);
    for (int i = 0; i < 5; ++i) PyTuple_SET_ITEM(arrays, i, THPVariable_Wrap(std::move(made[i])));
    return Py_BuildValue("(iNN)", status, arrays, schedule);
    END_HANDLE_TH_ERRORS
}

// validate(cols_a, row_start_ends_a, rows_b, col_start_ends_b, blocks) -> status
PyObject* py_validate(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need(n, 5, "validate");
    Tensor t[5];
    for (int i = 0; i < 5; ++i) {
        t[i] = tensor_arg(args[i], "index buffer");
        check_gpu(t[i]);
        TORCH_CHECK(t[i].scalar_type() == at::kInt && t[i].device() == t[0].device(), "index buffers should be int32 and on one device");
    }
    TORCH_CHECK(t[0].numel() == t[2].numel() && t[0].numel() == t[4].numel() && t[1].numel() >= 2 && t[3].numel() >= 2, "index buffers differ in length");
    int status = 0;
    {
        NoGil no_gil;
        at::NoGradGuard no_grad;
        for (Tensor& x : t) x = x.contiguous();
        c10::DeviceGuard guard(t[0].device());
        void* stream = current_stream(t[0]);
        const int nnz = (int)(t[0].numel() / 2);
        const size_t bytes = pbs_validate_indices_workspace_bytes(nnz);
        Tensor ws = workspace(bytes, t[0]), word = status_word();
        check(pbs_validate_indices(ints(t[0]), ints(t[1]), ints(t[2]), ints(t[3]), ints(t[4]), (int)t[1].numel() - 1, (int)t[3].numel() - 1, nnz,
                                   word.mutable_data_ptr<int>(), ws.mutable_data_ptr(), bytes, stream),
              "pbs_validate_indices");
        status = read_status(word, stream);
    }
    return PyLong_FromLong(status);
    END_HANDLE_TH_ERRORS
}

// check_protocol(what): with PBS_DEBUG set, raise if a bounded wait has run out on the current device since the last check
PyObject* py_check_protocol(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need(n, 1, "check_protocol");
    const char* what = PyUnicode_AsUTF8(args[0]);
    if (!what) return nullptr;
    {
        NoGil no_gil;
        check_protocol(what, c10::hip::current_device());
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"check_protocol", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_check_protocol)), METH_FASTCALL, nullptr},
                         {"replace_blocks", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_replace_blocks)), METH_FASTCALL, nullptr},
                         {"validate", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_validate)), METH_FASTCALL, nullptr},
                         {"linear", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_linear)), METH_FASTCALL, nullptr},
                         {"matmul", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_matmul)), METH_FASTCALL, nullptr},
                         {"matmul_back", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_matmul_back)), METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pbs_torch", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__pbs_torch() {
    if (pbs_abi_version() != PBS_ABI_VERSION)
        return PyErr_Format(PyExc_ImportError, "_pbs_torch.so was built for version %d of libpbs_hip.so, which is version %d: build both again",
                            PBS_ABI_VERSION, pbs_abi_version());
    ScheduleType.tp_name = "pytorch_block_sparse_amd.csrc._pbs_torch.Schedule";
    ScheduleType.tp_basicsize = sizeof(Schedule);
    ScheduleType.tp_flags = Py_TPFLAGS_DEFAULT;
    ScheduleType.tp_new = schedule_new;
    ScheduleType.tp_dealloc = schedule_dealloc;
    if (PyType_Ready(&ScheduleType) < 0) return nullptr;
    s_row_ptr = PyUnicode_InternFromString("row_start_ends_a");
    s_cols = PyUnicode_InternFromString("cols_a");
    s_col_ptr = PyUnicode_InternFromString("col_start_ends_b");
    s_rows = PyUnicode_InternFromString("rows_b");
    PyObject* m = PyModule_Create(&module);
    if (!m) return nullptr;
    Py_INCREF(&ScheduleType);
    if (PyModule_AddObject(m, "Schedule", reinterpret_cast<PyObject*>(&ScheduleType)) < 0) return nullptr;
    return m;
}

// _oeq_torch-*.so: the torch ops over the C ABI of include/oeq_amd.h, as the Python module _torch/ops.py loads it.
//
// Stands in for the reference's native op library (openequivariance/openequivariance/extension/torch_core.hpp:274-644):
// argument checks (torch_core.hpp:109-134), allocation of results and scratch memory, launches on
// torch's current stream, and autograd. An op carries the id of its kernel set and, for processes that have not
// seen it, the set's description; what is rare or needs the code generator stays in Python and is called from here:
// building a kernel set, building the index of an edge list that is not kept from an earlier call, the convolutions
// without a fused kernel, and the second-order routes by composition.
//
// The host side of a call is what a small product or graph costs: forward and backward of 777 rows take 8 us on the
// GPU and took 111 to 196 us, by machine, through Python ops (64 to 67 now). What runs in the backward pass matters
// most: it runs in the autograd engine's thread, where Python code finds neither its interpreter state nor its data in
// the caches. Looking up the kept index and choosing the second-order route in Python cost, per pass, before / now:
// MACE-medium, 192 nodes, new edges, forward and backward 157 / 96 us; 16 molecules with second order 281 / 192.
#include "oeq_amd.h"

#include <ATen/ATen.h>
#include <ATen/Context.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/grad_mode.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cstdlib>
#include <memory>
#include <mutex>
#include <shared_mutex>
#include <tuple>
#include <unordered_map>
#include <vector>

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;
using Tensor3 = std::tuple<Tensor, Tensor, Tensor>;
using Tensor4 = std::tuple<Tensor, Tensor, Tensor, Tensor>;

namespace {

struct Entry {
    oeq_kernels* k = nullptr;
    int64_t L1 = 0, L2 = 0, L3 = 0, WN = 0;
    bool shared = false, deterministic = false;
    at::ScalarType dtype = at::kFloat;
    int mode = 0, dx_mode = 0;  // oeq_conv_mode, oeq_dx_mode
    std::array<int64_t, 3> index_dims{};  // what an index depends on besides the mode: order_hops, order_min_nodes, hub_limit
    bool native = true;         // false: a convolution without fused kernels, see Callbacks::conv_*
    bool alert_forward = false, alert_backward = false;  // uses float atomics
    bool direct_loads = false;  // has kernels that bring operands into LDS 16 bytes at a time, see operand()
    bool fused_second_order = false;  // has the second-order kernels (of its own: not second_order_kid's)
    int64_t second_order_kid = 0;
    py::object owner;  // keeps the kernel set alive
};
using EntryRef = std::shared_ptr<const Entry>;

// (never destroyed: the entries hold Python objects)
auto& g_entries = *new std::unordered_map<int64_t, EntryRef>();
std::shared_mutex g_entries_mu;

// Python functions of _torch/ops.py; held until the process ends (no destructor runs after the interpreter's).
struct Callbacks {
    py::object resolve, without_terms, check_edges, build_index, conv_forward, conv_backward, conv_double_backward, tp_second_order,
        conv_second_order, error_type;
};
Callbacks* g_py = nullptr;

EntryRef entry_of(int64_t kid, const OptTensor& spec) {
    for (int attempt = 0; attempt < 2; ++attempt) {
        {
            std::shared_lock<std::shared_mutex> lock(g_entries_mu);
            auto it = g_entries.find(kid);
            if (it != g_entries.end()) return it->second;
        }
        py::gil_scoped_acquire gil;
        g_py->resolve(kid, spec.has_value() ? py::cast(*spec) : py::object(py::none()));
    }
    TORCH_CHECK(false, "kernel id ", kid, " could not be registered");
}

// The kernel set of the same problem whose backward pass keeps no terms per edge in scratch memory, for a call that has
// no room for them; 0: none.
int64_t without_terms(int64_t kid) {
    py::gil_scoped_acquire gil;
    return g_py->without_terms(kid).cast<int64_t>();
}

void check(int rc, const char* what) {
    if (rc == OEQ_OK) return;
    const char* msg = oeq_last_error();
    const std::string text = std::string(what) + " failed (" + std::to_string(rc) + "): " + (msg ? msg : "");
    py::gil_scoped_acquire gil;
    PyErr_SetString(g_py->error_type.ptr(), text.c_str());
    python_error err;
    err.persist();
    throw err;
}

int dtype_code(at::ScalarType t) {  // the reference's codes
    switch (t) {
        case at::kFloat: return 1;
        case at::kDouble: return 2;
        case at::kInt: return 3;
        case at::kLong: return 4;
        case at::kByte: return 5;
        default: return 0;
    }
}

std::string dtype_text(at::ScalarType t) {
    const int code = dtype_code(t);
    return code ? std::to_string(code) : std::string(at::toString(t));
}

void check_tensor(const Tensor& t, at::IntArrayRef shape, at::ScalarType dtype, const char* name) {
    TORCH_CHECK(t.sizes() == shape, "Shape mismatch for tensor '", name, "'. Expected: ", shape, ". Got: ", t.sizes());
    TORCH_CHECK(t.is_cuda(), "Tensor '", name, "' is not on the GPU.");
    TORCH_CHECK(t.scalar_type() == dtype, "Dtype mismatch for tensor '", name, "'. Expected: ", dtype_text(dtype),
                ". Got: ", dtype_text(t.scalar_type()));
}

void check_weights(const Entry& e, const Tensor& w, int64_t rows, const char* name) {
    if (e.shared)
        check_tensor(w, {e.WN}, e.dtype, name);
    else
        check_tensor(w, {rows, e.WN}, e.dtype, name);
}

int64_t rows_of(const Tensor& t) { return t.dim() > 0 ? t.size(0) : -1; }

// The device of a call's operands made current, and torch's stream on it.
struct OnDevice {
    c10::hip::OptionalHIPGuardMasqueradingAsCUDA guard;
    void* stream;
    explicit OnDevice(const Tensor& t) : guard(t.device()) {
        stream = (void*)(hipStream_t)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index());
    }
};

Tensor scratch(const Tensor& like, size_t bytes) {
    return at::empty({(int64_t)(bytes ? bytes : 1)}, like.options().dtype(at::kByte));
}

// An operand as the kernels read it: its rows one after the other and, where they are brought into LDS 16 bytes at a time,
// from a multiple of 16 on. A view into a larger tensor can begin anywhere (plain loads of any width want no more than
// the alignment of an element).
Tensor operand(const Entry& e, const Tensor& t) {
    const Tensor c = t.contiguous();
    return e.direct_loads && ((uintptr_t)c.data_ptr() & 15) ? c.clone() : c;
}

// ---------------------------------------------------------------------------
// batch tensor product
// ---------------------------------------------------------------------------

Tensor tp_forward_gpu(const Tensor& L1_in, const Tensor& L2_in, const Tensor& W, int64_t kid, const OptTensor& spec) {
    const EntryRef ref = entry_of(kid, spec);
    const Entry& e = *ref;
    const int64_t n = rows_of(L1_in);
    check_tensor(L1_in, {n, e.L1}, e.dtype, "L1_in");
    check_tensor(L2_in, {n, e.L2}, e.dtype, "L2_in");
    check_weights(e, W, n, "W");
    const Tensor x = operand(e, L1_in), y = operand(e, L2_in), w = operand(e, W);
    OnDevice dev(x);
    Tensor out = at::empty({n, e.L3}, x.options());
    check(oeq_tp_forward(e.k, n, x.data_ptr(), y.data_ptr(), w.data_ptr(), out.data_ptr(), dev.stream), "oeq_tp_forward");
    return out;
}

Tensor3 tp_backward_gpu(const Tensor& L1_in, const Tensor& L2_in, const Tensor& W, const Tensor& L3_grad, int64_t kid,
                        const OptTensor& spec) {
    const EntryRef ref = entry_of(kid, spec);
    const Entry& e = *ref;
    const int64_t n = rows_of(L1_in);
    check_tensor(L1_in, {n, e.L1}, e.dtype, "L1_in");
    check_tensor(L2_in, {n, e.L2}, e.dtype, "L2_in");
    check_weights(e, W, n, "W");
    check_tensor(L3_grad, {n, e.L3}, e.dtype, "L3_grad");
    const Tensor x = operand(e, L1_in), y = operand(e, L2_in), w = operand(e, W), g = operand(e, L3_grad);
    OnDevice dev(x);
    Tensor dx = at::empty_like(x), dy = at::empty_like(y), dw = at::empty_like(w);
    const size_t nb = oeq_tp_backward_workspace_bytes(e.k, n);
    Tensor ws;
    if (nb) ws = scratch(x, nb);
    check(oeq_tp_backward(e.k, n, x.data_ptr(), dx.data_ptr(), y.data_ptr(), dy.data_ptr(), w.data_ptr(), dw.data_ptr(),
                          g.data_ptr(), nb ? ws.data_ptr() : nullptr, nb, dev.stream),
          "oeq_tp_backward");
    return {dx, dy, dw};
}

Tensor4 tp_double_backward_gpu(const Tensor& L1_in, const Tensor& L2_in, const Tensor& W, const Tensor& L3_grad,
                               const Tensor& L1_dgrad, const Tensor& L2_dgrad, const Tensor& W_dgrad, int64_t kid,
                               const OptTensor& spec) {
    const EntryRef ref = entry_of(kid, spec);
    const Entry& e = *ref;
    const int64_t n = rows_of(L1_in);
    check_tensor(L1_in, {n, e.L1}, e.dtype, "L1_in");
    check_tensor(L1_dgrad, {n, e.L1}, e.dtype, "L1_dgrad");
    check_tensor(L2_in, {n, e.L2}, e.dtype, "L2_in");
    check_tensor(L2_dgrad, {n, e.L2}, e.dtype, "L2_dgrad");
    check_weights(e, W, n, "W");
    check_weights(e, W_dgrad, n, "W_dgrad");
    check_tensor(L3_grad, {n, e.L3}, e.dtype, "L3_grad");
    const Tensor x = operand(e, L1_in), y = operand(e, L2_in), w = operand(e, W), g = operand(e, L3_grad);
    const Tensor a = operand(e, L1_dgrad), b = operand(e, L2_dgrad), c = operand(e, W_dgrad);
    OnDevice dev(x);
    Tensor dx = at::empty_like(x), dy = at::empty_like(y), dw = at::empty_like(w), gg = at::empty_like(g);
    const size_t nb = oeq_tp_double_backward_workspace_bytes(e.k, n);
    const Tensor ws = scratch(x, nb);
    check(oeq_tp_double_backward(e.k, n, x.data_ptr(), y.data_ptr(), w.data_ptr(), g.data_ptr(), a.data_ptr(),
                                 b.data_ptr(), c.data_ptr(), dx.data_ptr(), dy.data_ptr(), dw.data_ptr(), gg.data_ptr(),
                                 ws.data_ptr(), nb, dev.stream),
          "oeq_tp_double_backward");
    return {dx, dy, dw, gg};
}

// ---------------------------------------------------------------------------
// fused convolution
// ---------------------------------------------------------------------------

struct GraphSize {
    int64_t nodes, edges;
};

GraphSize conv_checks(const Entry& e, const Tensor& L1_in, const Tensor& L2_in, const Tensor& W, const Tensor& rows,
                      const Tensor& cols, const Tensor& perm, const Tensor* L3_grad) {
    const int64_t nodes = rows_of(L1_in), nnz = rows_of(rows);
    check_tensor(L1_in, {nodes, e.L1}, e.dtype, "L1_in");
    check_tensor(L2_in, {nnz, e.L2}, e.dtype, "L2_in");
    check_weights(e, W, nnz, "W");
    if (L3_grad) check_tensor(*L3_grad, {nodes, e.L3}, e.dtype, "L3_grad");
    check_tensor(rows, {nnz}, at::kLong, "rows");
    check_tensor(cols, {nnz}, at::kLong, "cols");
    if (e.deterministic) check_tensor(perm, {nnz}, at::kLong, "transpose perm");
    // counterpart of at::globalContext().alertNotDeterministic (torch_core.hpp:448) for the calls that use float
    // atomics: the backward of deterministic=False (sender gradients), and both directions of the float-atomics
    // kernels. The grouped forward sums in a fixed order and needs no alert.
    if ((e.alert_forward || (L3_grad && e.alert_backward)) && at::globalContext().deterministicAlgorithms()) {
        const char* msg =
            "OpenEquivariance_conv_atomic does not have a deterministic implementation, but you set "
            "'torch.use_deterministic_algorithms(True)'. Use TensorProductConv(..., deterministic=True).";
        TORCH_CHECK(at::globalContext().deterministicAlgorithmsWarnOnly(), msg);
        // (a Python warning: TORCH_WARN from an op called directly would only print)
        py::gil_scoped_acquire gil;
        if (PyErr_WarnEx(PyExc_UserWarning, msg, 1) < 0) throw py::error_already_set();
    }
    return {nodes, nnz};
}

// What _torch/ops.py lets a program set (its module attributes of these names).
std::atomic<bool> g_check_indices{false}, g_fused_double_backward{true};
std::atomic<int64_t> g_index_cache_entries{4};

bool check_indices() {
    if (g_check_indices) return true;
    // (Python's os.environ writes the environment under the interpreter lock, and may move it)
    py::gil_scoped_acquire gil;
    const char* env = std::getenv("OEQ_AMD_CHECK_INDICES");
    return env && *env && !(env[0] == '0' && !env[1]);
}

void check_edges(const Entry& e, GraphSize n, const Tensor& rows, const Tensor& cols, const Tensor& perm) {
    if (!check_indices()) return;
    py::gil_scoped_acquire gil;
    g_py->check_edges(n.nodes, rows, cols, e.deterministic ? py::cast(perm) : py::object(py::none()), e.deterministic);
}

struct Index {
    Tensor data;
    bool sender_side = false;
};

// A walk-mode convolution first derives an index from the edge list (CSR pointers, edge grouping, walk order;
// oeq_conv_index_build). The layers of a model, and the forward and backward of each, usually run over the same edge
// tensors, so the last few indices are kept and one is used again when a call brings the same tensors (same storage,
// same version counters, i.e. not written to since), on the same stream, for a kernel set that indexes the same way.
// The list holds references to the edge tensors, so their memory cannot be handed to different data while an entry
// exists.
struct IndexKey {
    std::array<int64_t, 13> v{};
    bool operator==(const IndexKey& o) const { return v == o.v; }
};

struct KeptIndex {
    IndexKey key;
    std::array<uint32_t, 3> versions;
    Index index;
    Tensor rows, cols, perm;
};

auto& g_indices = *new std::vector<KeptIndex>();  // least recently used first
std::mutex g_indices_mu;

struct IndexQuery {
    IndexKey key;
    std::array<uint32_t, 3> versions{};
    bool sender_side, keep;

    // perm is undefined where the caller's edges are not sorted
    IndexQuery(int mode, const std::array<int64_t, 3>& dims, GraphSize n, const Tensor& rows, const Tensor& cols,
               const Tensor& perm, bool need_sender_side) {
        const bool sorted = perm.defined() && mode != OEQ_CONV_GROUPED;
        // the sender side is cheap to add when the caller brings the sender-major permutation, costly when the
        // library has to group the edges by sender itself: then only the calls that need it build it
        sender_side = need_sender_side || (sorted && perm.numel() == n.edges);
        const auto stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA();
        key.v = {mode, dims[0], dims[1], dims[2], n.nodes, n.edges, (int64_t)rows.data_ptr(), (int64_t)cols.data_ptr(),
                 sorted ? (int64_t)perm.data_ptr() : 0, (int64_t)(hipStream_t)stream, rows.device().index(), sorted, 0};
        // an edge tensor without a version counter could be rewritten unnoticed: such a call builds its index and
        // keeps nothing. Nor does one that is being captured.
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        keep = g_index_cache_entries > 0 && !rows.is_inference() && !cols.is_inference() &&
               !(sorted && perm.is_inference()) &&
               hipStreamIsCapturing((hipStream_t)stream, &capture) == hipSuccess && capture == hipStreamCaptureStatusNone;
        if (keep) versions = {(uint32_t)rows._version(), (uint32_t)cols._version(), sorted ? (uint32_t)perm._version() : 0u};
    }

    int64_t stream() const { return key.v[9]; }

    std::optional<Index> find() const {
        if (!keep) return std::nullopt;
        std::lock_guard<std::mutex> lock(g_indices_mu);
        for (auto it = g_indices.begin(); it != g_indices.end(); ++it) {
            if (!(it->key == key) || it->versions != versions || (sender_side && !it->index.sender_side)) continue;
            std::rotate(it, it + 1, g_indices.end());
            return g_indices.back().index;
        }
        return std::nullopt;
    }

    void store(const Tensor& data, const Tensor& rows, const Tensor& cols, const Tensor& perm) const {
        if (!keep) return;
        std::vector<KeptIndex> gone;  // (freed after the lock is released)
        std::lock_guard<std::mutex> lock(g_indices_mu);
        std::vector<KeptIndex> kept;
        for (auto& k : g_indices) (k.key == key ? gone : kept).push_back(std::move(k));
        kept.push_back({key, versions, {data, sender_side}, rows, cols, perm});
        const size_t limit = (size_t)std::max<int64_t>(1, g_index_cache_entries);
        while (kept.size() > limit) {
            gone.push_back(std::move(kept.front()));
            kept.erase(kept.begin());
        }
        g_indices.swap(kept);
    }
};

// The index of the edge list, kept from an earlier call over the same tensors or built now (_torch/ops.py), after the
// opt-in check of the list itself.
Index conv_index(const Entry& e, int64_t kid, GraphSize n, const Tensor& rows, const Tensor& cols, const Tensor& perm,
                 bool sender_side) {
    const Tensor order = e.deterministic ? perm : Tensor();
    check_edges(e, n, rows, cols, order);
    const IndexQuery q(e.mode, e.index_dims, n, rows, cols, order, sender_side);
    if (auto kept = q.find()) return *kept;
    const size_t nb = oeq_conv_index_bytes(e.k, n.nodes, n.edges, q.sender_side);
    const Tensor data = scratch(rows, nb);
    {
        py::gil_scoped_acquire gil;
        const int64_t list = order.defined() && e.mode != OEQ_CONV_GROUPED ? (int64_t)order.data_ptr() : 0;
        g_py->build_index(kid, n.nodes, n.edges, (int64_t)rows.data_ptr(), (int64_t)cols.data_ptr(), list, q.sender_side,
                          (int64_t)data.data_ptr(), nb, q.stream());
    }
    q.store(data, rows, cols, order);
    return {data, q.sender_side};
}

py::object none_or(const OptTensor& t) { return t.has_value() ? py::cast(*t) : py::object(py::none()); }

Tensor conv_forward_gpu(const Tensor& L1_in, const Tensor& L2_in, const Tensor& W, const Tensor& rows,
                        const Tensor& cols, const Tensor& transpose_perm, int64_t kid, const OptTensor& spec) {
    const EntryRef ref = entry_of(kid, spec);
    const Entry& e = *ref;
    const GraphSize n = conv_checks(e, L1_in, L2_in, W, rows, cols, transpose_perm, nullptr);
    const Tensor x = operand(e, L1_in), y = operand(e, L2_in), w = operand(e, W);
    const Tensor r = rows.contiguous(), c = cols.contiguous();
    if (!e.native) {
        py::gil_scoped_acquire gil;
        return py::cast<Tensor>(g_py->conv_forward(x, y, w, r, c, transpose_perm, kid));
    }
    OnDevice dev(x);
    Tensor out = at::empty({n.nodes, e.L3}, x.options());
    if (e.mode == OEQ_CONV_ATOMIC || n.nodes == 0 || n.edges == 0) {
        check_edges(e, n, rows, cols, transpose_perm);
        check(oeq_conv_forward(e.k, n.nodes, n.edges, x.data_ptr(), y.data_ptr(), w.data_ptr(), out.data_ptr(),
                               r.data_ptr<int64_t>(), c.data_ptr<int64_t>(), nullptr, 0, dev.stream),
              "oeq_conv_forward");
        return out;
    }
    // the forward walk needs the receiver side only; where the backward pass will want the edges grouped by sender as
    // well, both are built now, so that one index serves the whole step
    const bool both = e.mode == OEQ_CONV_GROUPED && e.dx_mode != OEQ_DX_ATOMIC;
    const Tensor p = e.deterministic ? transpose_perm.contiguous() : Tensor();
    const Index ix = conv_index(e, kid, n, r, c, p, both);
    const size_t nb = oeq_conv_forward_scratch_bytes(e.k, n.nodes, n.edges);
    Tensor ws;
    if (nb) ws = scratch(x, nb);
    check(oeq_conv_forward_indexed(e.k, n.nodes, n.edges, x.data_ptr(), y.data_ptr(), w.data_ptr(), out.data_ptr(),
                                   r.data_ptr<int64_t>(), c.data_ptr<int64_t>(), ix.data.data_ptr(), ix.data.numel(),
                                   ix.sender_side, nb ? ws.data_ptr() : nullptr, nb, dev.stream),
          "oeq_conv_forward_indexed");
    return out;
}

Tensor3 conv_backward_gpu(const Tensor& L1_in, const Tensor& L2_in, const Tensor& W, const Tensor& L3_grad,
                          const Tensor& rows, const Tensor& cols, const Tensor& transpose_perm, int64_t kid,
                          const OptTensor& spec) {
    const EntryRef ref = entry_of(kid, spec);
    const Entry& e = *ref;
    const GraphSize n = conv_checks(e, L1_in, L2_in, W, rows, cols, transpose_perm, &L3_grad);
    const Tensor x = operand(e, L1_in), y = operand(e, L2_in), w = operand(e, W), g = operand(e, L3_grad);
    const Tensor r = rows.contiguous(), c = cols.contiguous(), p = transpose_perm.contiguous();
    if (!e.native) {
        py::gil_scoped_acquire gil;
        return py::cast<Tensor3>(g_py->conv_backward(x, y, w, g, r, c, p, kid));
    }
    OnDevice dev(x);
    Tensor dx = at::empty_like(x), dy = at::empty_like(y), dw = at::empty_like(w);
    const int64_t* pp = e.deterministic ? p.data_ptr<int64_t>() : nullptr;
    if (e.mode == OEQ_CONV_ATOMIC || n.nodes == 0 || n.edges == 0) {
        check_edges(e, n, rows, cols, transpose_perm);
        check(oeq_conv_backward(e.k, n.nodes, n.edges, x.data_ptr(), dx.data_ptr(), y.data_ptr(), dy.data_ptr(),
                                w.data_ptr(), dw.data_ptr(), g.data_ptr(), r.data_ptr<int64_t>(),
                                c.data_ptr<int64_t>(), pp, nullptr, 0, dev.stream),
              "oeq_conv_backward");
        return {dx, dy, dw};
    }
    const Index ix = conv_index(e, kid, n, r, c, p, e.dx_mode != OEQ_DX_ATOMIC);
    const size_t nb = oeq_conv_backward_scratch_bytes(e.k, n.nodes, n.edges);
    Tensor ws;
    try {
        if (nb) ws = scratch(x, nb);
    } catch (const c10::OutOfMemoryError&) {
        const int64_t other = e.dx_mode == OEQ_DX_TERMS ? without_terms(kid) : 0;
        if (!other) throw;
        dx = dy = dw = Tensor();
        return conv_backward_gpu(L1_in, L2_in, W, L3_grad, rows, cols, transpose_perm, other, std::nullopt);
    }
    check(oeq_conv_backward_indexed(e.k, n.nodes, n.edges, x.data_ptr(), dx.data_ptr(), y.data_ptr(), dy.data_ptr(),
                                    w.data_ptr(), dw.data_ptr(), g.data_ptr(), r.data_ptr<int64_t>(),
                                    c.data_ptr<int64_t>(), pp, ix.data.data_ptr(), ix.data.numel(), ix.sender_side,
                                    nb ? ws.data_ptr() : nullptr, nb, dev.stream),
          "oeq_conv_backward_indexed");
    return {dx, dy, dw};
}

Tensor4 conv_double_backward_gpu(const Tensor& L1_in, const Tensor& L2_in, const Tensor& W, const Tensor& L3_grad,
                                 const Tensor& L1_dgrad, const Tensor& L2_dgrad, const Tensor& W_dgrad,
                                 const Tensor& rows, const Tensor& cols, const Tensor& transpose_perm, int64_t kid,
                                 const OptTensor& spec) {
    EntryRef ref = entry_of(kid, spec);
    // float-atomics kernel sets have no pair of their own: the grouped-walk set of the same problem
    if (ref->second_order_kid) {
        kid = ref->second_order_kid;
        ref = entry_of(kid, std::nullopt);
    }
    const Entry& e = *ref;
    const GraphSize n = conv_checks(e, L1_in, L2_in, W, rows, cols, transpose_perm, &L3_grad);
    check_tensor(L1_dgrad, {n.nodes, e.L1}, e.dtype, "L1_in");
    check_tensor(L2_dgrad, {n.edges, e.L2}, e.dtype, "L2_in");
    check_weights(e, W_dgrad, n.edges, "W");
    const Tensor x = operand(e, L1_in), y = operand(e, L2_in), w = operand(e, W), g = operand(e, L3_grad);
    const Tensor a = operand(e, L1_dgrad), b = operand(e, L2_dgrad), c = operand(e, W_dgrad);
    const Tensor r = rows.contiguous(), cc = cols.contiguous(), p = transpose_perm.contiguous();
    if (!e.native) {
        py::gil_scoped_acquire gil;
        return py::cast<Tensor4>(g_py->conv_double_backward(x, y, w, g, a, b, c, r, cc, p, kid));
    }
    OnDevice dev(x);
    Tensor dx = at::empty_like(x), dy = at::empty_like(y), dw = at::empty_like(w), gg = at::empty_like(g);
    const int64_t* pp = e.deterministic ? p.data_ptr<int64_t>() : nullptr;
    if (n.nodes == 0 || n.edges == 0) {
        check_edges(e, n, rows, cols, transpose_perm);
        check(oeq_conv_double_backward(e.k, n.nodes, n.edges, x.data_ptr(), y.data_ptr(), w.data_ptr(), g.data_ptr(),
                                       a.data_ptr(), b.data_ptr(), c.data_ptr(), dx.data_ptr(), dy.data_ptr(),
                                       dw.data_ptr(), gg.data_ptr(), r.data_ptr<int64_t>(), cc.data_ptr<int64_t>(), pp,
                                       nullptr, 0, dev.stream),
              "oeq_conv_double_backward");
        return {dx, dy, dw, gg};
    }
    const Index ix = conv_index(e, kid, n, r, cc, p, true);
    const size_t nb = oeq_conv_double_backward_scratch_bytes(e.k, n.nodes, n.edges);
    Tensor ws;
    if (nb) ws = scratch(x, nb);
    check(oeq_conv_double_backward_indexed(
              e.k, n.nodes, n.edges, x.data_ptr(), y.data_ptr(), w.data_ptr(), g.data_ptr(), a.data_ptr(),
              b.data_ptr(), c.data_ptr(), dx.data_ptr(), dy.data_ptr(), dw.data_ptr(), gg.data_ptr(),
              r.data_ptr<int64_t>(), cc.data_ptr<int64_t>(), pp, ix.data.data_ptr(), ix.data.numel(),
              nb ? ws.data_ptr() : nullptr, nb, dev.stream),
          "oeq_conv_double_backward_indexed");
    return {dx, dy, dw, gg};
}

// ---------------------------------------------------------------------------
// autograd
// ---------------------------------------------------------------------------

template <typename Sig>
c10::TypedOperatorHandle<Sig> find_op(const char* name) {
    return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Sig>();
}

Tensor call_tp_forward(const Tensor& x, const Tensor& y, const Tensor& w, int64_t kid, const OptTensor& spec) {
    static const auto op = find_op<decltype(tp_forward_gpu)>("oeq_amd::tp_forward");
    return op.call(x, y, w, kid, spec);
}
Tensor3 call_tp_backward(const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& g, int64_t kid,
                         const OptTensor& spec) {
    static const auto op = find_op<decltype(tp_backward_gpu)>("oeq_amd::tp_backward");
    return op.call(x, y, w, g, kid, spec);
}
Tensor4 call_tp_double_backward(const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& g, const Tensor& a,
                                const Tensor& b, const Tensor& c, int64_t kid, const OptTensor& spec) {
    static const auto op = find_op<decltype(tp_double_backward_gpu)>("oeq_amd::tp_double_backward");
    return op.call(x, y, w, g, a, b, c, kid, spec);
}
Tensor4 call_conv_double_backward(const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& g, const Tensor& a,
                                  const Tensor& b, const Tensor& c, const Tensor& rows, const Tensor& cols,
                                  const Tensor& p, int64_t kid, const OptTensor& spec) {
    static const auto op = find_op<decltype(conv_double_backward_gpu)>("oeq_amd::conv_double_backward");
    return op.call(x, y, w, g, a, b, c, rows, cols, p, kid, spec);
}
Tensor call_conv_forward(const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& r, const Tensor& c,
                         const Tensor& p, int64_t kid, const OptTensor& spec) {
    static const auto op = find_op<decltype(conv_forward_gpu)>("oeq_amd::conv_forward");
    return op.call(x, y, w, r, c, p, kid, spec);
}
Tensor3 call_conv_backward(const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& g, const Tensor& r,
                           const Tensor& c, const Tensor& p, int64_t kid, const OptTensor& spec) {
    static const auto op = find_op<decltype(conv_backward_gpu)>("oeq_amd::conv_backward");
    return op.call(x, y, w, g, r, c, p, kid, spec);
}

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void keep_id(AutogradContext* ctx, int64_t kid, const OptTensor& spec) {
    ctx->saved_data["kid"] = kid;
    if (spec.has_value()) ctx->saved_data["spec"] = *spec;
}
int64_t kid_of(AutogradContext* ctx) { return ctx->saved_data["kid"].toInt(); }
OptTensor spec_of(AutogradContext* ctx) {
    auto it = ctx->saved_data.find("spec");
    return it == ctx->saved_data.end() ? OptTensor() : OptTensor(it->second.toTensor());
}

py::object defined_or_none(const Tensor& t) { return t.defined() ? py::cast(t) : py::object(py::none()); }
Tensor tensor_or_none(py::handle h) { return h.is_none() ? Tensor() : py::cast<Tensor>(h); }

// The backward of a backward op. The fused second-order op, called here, is for calls that record nothing for a third
// derivative (then the composition of differentiable first-order ops is needed) and bring at least two of the three
// cotangents (a missing one is passed as zeros; with a single one the two first-order calls of the composition read
// less). The compositions, and kernel sets that borrow another's second-order kernels, are in Python.
variable_list second_order(const py::object& fn, const variable_list& saved, const variable_list& grads, int64_t kid,
                           const OptTensor& spec, size_t n_inputs) {
    variable_list out(n_inputs);
    const int present = (int)grads[0].defined() + (int)grads[1].defined() + (int)grads[2].defined();
    if (!present) return out;
    if (present >= 2 && g_fused_double_backward && !at::GradMode::is_enabled() && entry_of(kid, spec)->fused_second_order) {
        std::array<Tensor, 3> d;
        for (size_t i = 0; i < 3; ++i) d[i] = grads[i].defined() ? grads[i] : at::zeros_like(saved[i]);
        const Tensor4 got = saved.size() == 4
            ? call_tp_double_backward(saved[0], saved[1], saved[2], saved[3], d[0], d[1], d[2], kid, spec)
            : call_conv_double_backward(saved[0], saved[1], saved[2], saved[3], d[0], d[1], d[2], saved[4], saved[5],
                                        saved[6], kid, spec);
        std::tie(out[0], out[1], out[2], out[3]) = got;
        return out;
    }
    py::gil_scoped_acquire gil;
    py::tuple ts(saved.size()), gs(3);
    for (size_t i = 0; i < saved.size(); ++i) ts[i] = py::cast(saved[i]);
    for (size_t i = 0; i < 3; ++i) gs[i] = defined_or_none(grads[i]);
    py::tuple got = fn(ts, gs, kid, none_or(spec));
    for (size_t i = 0; i < 4; ++i) out[i] = tensor_or_none(got[i]);
    return out;
}

struct TpForward : public torch::autograd::Function<TpForward> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& y, const Tensor& w, int64_t kid,
                          const OptTensor& spec) {
        at::AutoDispatchBelowADInplaceOrView below;
        ctx->save_for_backward({x, y, w});
        ctx->set_materialize_grads(false);
        keep_id(ctx, kid, spec);
        return call_tp_forward(x, y, w, kid, spec);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        variable_list out(5);
        if (!grads[0].defined()) return out;
        const auto s = ctx->get_saved_variables();
        std::tie(out[0], out[1], out[2]) = call_tp_backward(s[0], s[1], s[2], grads[0], kid_of(ctx), spec_of(ctx));
        return out;
    }
};

struct TpBackward : public torch::autograd::Function<TpBackward> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& y, const Tensor& w,
                                 const Tensor& g, int64_t kid, const OptTensor& spec) {
        at::AutoDispatchBelowADInplaceOrView below;
        ctx->save_for_backward({x, y, w, g});
        ctx->set_materialize_grads(false);
        keep_id(ctx, kid, spec);
        auto [dx, dy, dw] = call_tp_backward(x, y, w, g, kid, spec);
        return {dx, dy, dw};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        return second_order(g_py->tp_second_order, ctx->get_saved_variables(), grads, kid_of(ctx), spec_of(ctx), 6);
    }
};

struct ConvForward : public torch::autograd::Function<ConvForward> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& r,
                          const Tensor& c, const Tensor& p, int64_t kid, const OptTensor& spec) {
        at::AutoDispatchBelowADInplaceOrView below;
        ctx->save_for_backward({x, y, w, r, c, p});
        ctx->set_materialize_grads(false);
        keep_id(ctx, kid, spec);
        return call_conv_forward(x, y, w, r, c, p, kid, spec);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        variable_list out(8);
        if (!grads[0].defined()) return out;
        const auto s = ctx->get_saved_variables();
        std::tie(out[0], out[1], out[2]) =
            call_conv_backward(s[0], s[1], s[2], grads[0], s[3], s[4], s[5], kid_of(ctx), spec_of(ctx));
        return out;
    }
};

struct ConvBackward : public torch::autograd::Function<ConvBackward> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& y, const Tensor& w,
                                 const Tensor& g, const Tensor& r, const Tensor& c, const Tensor& p, int64_t kid,
                                 const OptTensor& spec) {
        at::AutoDispatchBelowADInplaceOrView below;
        ctx->save_for_backward({x, y, w, g, r, c, p});
        ctx->set_materialize_grads(false);
        keep_id(ctx, kid, spec);
        auto [dx, dy, dw] = call_conv_backward(x, y, w, g, r, c, p, kid, spec);
        return {dx, dy, dw};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        return second_order(g_py->conv_second_order, ctx->get_saved_variables(), grads, kid_of(ctx), spec_of(ctx), 9);
    }
};

// The fused second-order ops are not differentiated themselves: a call that records returns outputs whose backward is
// an error (without a kernel for the Autograd key torch would warn and leave their part of the gradient out). Third
// derivatives go through the first-order ops: _tp_second_order and _conv_second_order in _torch/ops.py.
template <typename Sig, const char* const& name>
struct NotDifferentiated : public torch::autograd::Function<NotDifferentiated<Sig, name>> {
    template <typename... Args>
    static variable_list forward(AutogradContext* ctx, const Args&... args) {
        at::AutoDispatchBelowADInplaceOrView below;
        ctx->set_materialize_grads(false);
        static const auto op = find_op<Sig>(name);
        auto [dx, dy, dw, gg] = op.call(args...);
        return {dx, dy, dw, gg};
    }
    static variable_list backward(AutogradContext*, variable_list) {
        TORCH_CHECK(false, "Trying to backward through ", name, " but no autograd formula was registered. Differentiate ",
                    "the first-order ops with create_graph=True instead.");
    }
};

const char* const kTpDoubleBackward = "oeq_amd::tp_double_backward";
const char* const kConvDoubleBackward = "oeq_amd::conv_double_backward";

template <typename... Ts>
bool records(const Ts&... ts) {
    return at::GradMode::is_enabled() && (ts.requires_grad() || ...);
}

Tensor tp_forward_autograd(const Tensor& x, const Tensor& y, const Tensor& w, int64_t kid, const OptTensor& spec) {
    if (records(x, y, w)) return TpForward::apply(x, y, w, kid, spec);
    at::AutoDispatchBelowADInplaceOrView below;
    return call_tp_forward(x, y, w, kid, spec);
}
Tensor3 tp_backward_autograd(const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& g, int64_t kid,
                             const OptTensor& spec) {
    if (records(x, y, w, g)) {
        const auto out = TpBackward::apply(x, y, w, g, kid, spec);
        return {out[0], out[1], out[2]};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    return call_tp_backward(x, y, w, g, kid, spec);
}
Tensor conv_forward_autograd(const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& r, const Tensor& c,
                             const Tensor& p, int64_t kid, const OptTensor& spec) {
    if (records(x, y, w)) return ConvForward::apply(x, y, w, r, c, p, kid, spec);
    at::AutoDispatchBelowADInplaceOrView below;
    return call_conv_forward(x, y, w, r, c, p, kid, spec);
}
Tensor3 conv_backward_autograd(const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& g, const Tensor& r,
                               const Tensor& c, const Tensor& p, int64_t kid, const OptTensor& spec) {
    if (records(x, y, w, g)) {
        const auto out = ConvBackward::apply(x, y, w, g, r, c, p, kid, spec);
        return {out[0], out[1], out[2]};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    return call_conv_backward(x, y, w, g, r, c, p, kid, spec);
}

Tensor4 tp_double_backward_autograd(const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& g,
                                    const Tensor& a, const Tensor& b, const Tensor& c, int64_t kid,
                                    const OptTensor& spec) {
    if (records(x, y, w, g, a, b, c)) {
        const auto out =
            NotDifferentiated<decltype(tp_double_backward_gpu), kTpDoubleBackward>::apply(x, y, w, g, a, b, c, kid, spec);
        return {out[0], out[1], out[2], out[3]};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    return call_tp_double_backward(x, y, w, g, a, b, c, kid, spec);
}
Tensor4 conv_double_backward_autograd(const Tensor& x, const Tensor& y, const Tensor& w, const Tensor& g,
                                      const Tensor& a, const Tensor& b, const Tensor& c, const Tensor& rows,
                                      const Tensor& cols, const Tensor& p, int64_t kid, const OptTensor& spec) {
    if (records(x, y, w, g, a, b, c)) {
        const auto out = NotDifferentiated<decltype(conv_double_backward_gpu), kConvDoubleBackward>::apply(
            x, y, w, g, a, b, c, rows, cols, p, kid, spec);
        return {out[0], out[1], out[2], out[3]};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    return call_conv_double_backward(x, y, w, g, a, b, c, rows, cols, p, kid, spec);
}

}  // namespace

// (schemas, fake kernels and autocast: _torch/ops.py)
TORCH_LIBRARY_IMPL(oeq_amd, CUDA, m) {
    m.impl("tp_forward", tp_forward_gpu);
    m.impl("tp_backward", tp_backward_gpu);
    m.impl("tp_double_backward", tp_double_backward_gpu);
    m.impl("conv_forward", conv_forward_gpu);
    m.impl("conv_backward", conv_backward_gpu);
    m.impl("conv_double_backward", conv_double_backward_gpu);
}

TORCH_LIBRARY_IMPL(oeq_amd, Autograd, m) {
    m.impl("tp_forward", tp_forward_autograd);
    m.impl("tp_backward", tp_backward_autograd);
    m.impl("conv_forward", conv_forward_autograd);
    m.impl("conv_backward", conv_backward_autograd);
    m.impl("tp_double_backward", tp_double_backward_autograd);
    m.impl("conv_double_backward", conv_double_backward_autograd);
}

PYBIND11_MODULE(_oeq_torch, m) {
    m.def("abi_version", [] { return OEQ_ABI_VERSION; });
    m.def("set_callbacks", [](py::dict fns) {
        auto* c = new Callbacks();
        c->resolve = fns["resolve"];
        c->without_terms = fns["without_terms"];
        c->check_edges = fns["check_edges"];
        c->build_index = fns["build_index"];
        c->conv_forward = fns["conv_forward"];
        c->conv_backward = fns["conv_backward"];
        c->conv_double_backward = fns["conv_double_backward"];
        c->tp_second_order = fns["tp_second_order"];
        c->conv_second_order = fns["conv_second_order"];
        c->error_type = fns["error_type"];
        g_py = c;
    });
    m.def("register_entry", [](int64_t kid, py::dict d) {
        std::shared_ptr<Entry> e(new Entry(), [](Entry* p) {
            py::gil_scoped_acquire gil;
            delete p;
        });
        e->k = (oeq_kernels*)d["handle"].cast<uintptr_t>();
        e->L1 = d["L1"].cast<int64_t>();
        e->L2 = d["L2"].cast<int64_t>();
        e->L3 = d["L3"].cast<int64_t>();
        e->WN = d["WN"].cast<int64_t>();
        e->shared = d["shared"].cast<bool>();
        e->deterministic = d["deterministic"].cast<bool>();
        e->dtype = d["double"].cast<bool>() ? at::kDouble : at::kFloat;
        e->mode = d["mode"].cast<int>();
        e->dx_mode = d["dx_mode"].cast<int>();
        e->index_dims = d["index_dims"].cast<std::array<int64_t, 3>>();
        e->direct_loads = d["direct_loads"].cast<bool>();
        e->fused_second_order = d["fused_second_order"].cast<bool>();
        e->native = d["native"].cast<bool>();
        e->alert_forward = d["alert_forward"].cast<bool>();
        e->alert_backward = d["alert_backward"].cast<bool>();
        e->second_order_kid = d["second_order_kid"].cast<int64_t>();
        e->owner = d["owner"];
        EntryRef old = std::move(e);  // (what it replaces, if anything, goes after the lock is released)
        std::unique_lock<std::shared_mutex> lock(g_entries_mu);
        std::swap(g_entries[kid], old);
    });
    m.def("set_check_indices", [](bool on) { g_check_indices = on; });
    m.def("set_fused_double_backward", [](bool on) { g_fused_double_backward = on; });
    m.def("set_index_cache_entries", [](int64_t n) { g_index_cache_entries = n; });
    m.def("check_indices", check_indices);
    m.def("index_cache_size", [] {
        std::lock_guard<std::mutex> lock(g_indices_mu);
        return g_indices.size();
    });
    m.def("clear_index_cache", [] {
        std::vector<KeptIndex> gone;
        std::lock_guard<std::mutex> lock(g_indices_mu);
        gone.swap(g_indices);
    });
    // (index, sender_side) of the edge list: the kept one, or what build(sender_side) returns, which is kept if it may be
    m.def("kept_index", [](int mode, std::array<int64_t, 3> dims, int64_t nodes, int64_t edges, const Tensor& rows,
                           const Tensor& cols, const OptTensor& perm, bool need_sender_side, py::function build) {
        const Tensor order = perm.has_value() ? *perm : Tensor();
        const IndexQuery q(mode, dims, {nodes, edges}, rows, cols, order, need_sender_side);
        if (auto kept = q.find()) return std::make_pair(kept->data, kept->sender_side);
        const Tensor data = py::cast<Tensor>(build(q.sender_side));
        q.store(data, rows, cols, order);
        return std::make_pair(data, q.sender_side);
    });
    m.def("forget_entry", [](int64_t kid) {
        EntryRef old;
        std::unique_lock<std::shared_mutex> lock(g_entries_mu);
        auto it = g_entries.find(kid);
        if (it == g_entries.end()) return;
        old = std::move(it->second);
        g_entries.erase(it);
    });
}

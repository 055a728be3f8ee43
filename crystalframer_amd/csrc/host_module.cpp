// Host side of the whole-model pass and of the optimizer, as a Python extension module: what stands between the framework's
// tensors and the entry points of the library for every pass, in native code.
//
// A pass of the library is 30 (inference) to 80 launches; around them Python spent 90 us on looking the model and the batch
// over, 190 us on the gradients' tensors and the bookkeeping of the autograd function and 100 us on the optimizer's job
// table, per training step of the 4-layer model with its 65 parameters, as long as the GPU takes for a step on 13 crystals.
//
// The entry points are called through addresses that the Python side hands over: the module does not link the library.
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SavedTensorHooks.h>

#include <mutex>

#include "../../include/crystalframer_hip.h"

namespace py = pybind11;

namespace {

struct Library {
    int64_t (*sizes)(const cfh_model*, const cfh_model_batch*, size_t*) = nullptr;
    int (*forward)(const cfh_model*, const cfh_model_batch*, float*) = nullptr;
    int (*backward)(const cfh_model*, const cfh_model_batch*, const float*, void*, size_t, float*) = nullptr;
    const char* (*last_error)() = nullptr;
} g_lib;

void check(int rc, const char* what) {
    TORCH_CHECK(rc == 0, what, " failed (", rc, "): ", g_lib.last_error ? g_lib.last_error() : "");
}

// The launches of a pass share the scratch of their stream, and a backward pass is enqueued by a thread of the autograd engine
// without the interpreter's lock: no other thread's launches come between those of a pass.  (Nothing that is done with this
// held waits for the interpreter.)
std::mutex g_enqueue;

at::Tensor bytes(size_t n, const c10::Device& dev) {
    return at::empty({(int64_t)n}, at::TensorOptions().dtype(at::kByte).device(dev));
}
// Memory of a pass.  Sizes are rounded up to an eighth of their power of two: the batches of an epoch differ a little from each
// other, and the framework's allocator then finds a block to use again.
at::Tensor arena(size_t n, const c10::Device& dev) {
    size_t step = 512;
    int bits = 0;
    for (size_t v = n; v; v >>= 1) bits++;
    if (bits > 4 && ((size_t)1 << (bits - 4)) > step) step = (size_t)1 << (bits - 4);
    return bytes((n + step - 1) / step * step, dev);
}

// Memory whose address the library was given: kept, and still where it was.
struct Held {
    c10::Storage storage;
    const void* base;
    explicit Held(const at::Tensor& t) : storage(t.storage()), base(storage.data()) {}
    bool there() const { return storage.data() == base; }
};

// What a plan's passes share (see model_pass._Plan).
struct Shared {
    std::vector<at::Tensor> params;            // in the order of the library's gradients
    std::vector<at::Tensor> gauss;
    std::vector<Held> held;                    // of params and gauss as the plan was made
    std::vector<std::vector<int64_t>> sizes;   // of params
    std::vector<int64_t> offset;               // of a parameter's gradient, in floats
    c10::Device device{c10::kCPU};
    int64_t feat = 0, D = 0, H = 0, out_features = 0;
};

// Structures of the library call, kept alive by the Python object that made them.
struct Model {
    const cfh_model* m;
    std::shared_ptr<void> owner;               // drops a reference to the Python object, with the GIL held
};
std::shared_ptr<void> hold(py::object o) {
    return std::shared_ptr<void>(o.release().ptr(), [](void* p) {
        if (!Py_IsInitialized()) return;
        py::gil_scoped_acquire gil;
        Py_DECREF(reinterpret_cast<PyObject*>(p));
    });
}

struct ModelPassBackward : public torch::autograd::Node {
    std::shared_ptr<Shared> plan;
    Model model;
    cfh_model_batch b;
    int64_t total;
    size_t scratch_bytes;
    std::vector<uint64_t> seeds;
    at::Tensor arena_, workspace_;
    std::vector<torch::autograd::SavedVariable> data;
    std::vector<Held> held;                    // of the batch
    std::vector<at::Tensor> first;
    std::vector<int64_t> versions;
    bool released = false;

    std::string name() const override { return "ModelPassHIPBackward"; }
    void release_variables() override {
        released = true;
        arena_.reset();
        workspace_.reset();
        data.clear();
        held.clear();
        first.clear();
    }
    static std::vector<int64_t> current_versions(const Shared& P) {
        std::vector<int64_t> v;
        v.reserve(P.params.size() + P.gauss.size());
        for (auto& p : P.params) v.push_back((int64_t)p._version());
        for (auto& p : P.gauss) v.push_back((int64_t)p._version());
        return v;
    }
    torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
        TORCH_CHECK(!released, "the backward pass of this model output has been made and what its forward pass kept is given back; to "
                    "make it a second time, make the first one with retain_graph=True");
        // The .data of a parameter or of the batch was exchanged since the forward pass: the addresses are those of the storages
        // before, which are held, and the gradients those of what the forward pass computed.
        const size_t n = plan->params.size();
        torch::autograd::variable_list out(n);
        if (!grads[0].defined()) return out;
        TORCH_CHECK(current_versions(*plan) == versions,
                    "a parameter of the model was modified by an inplace operation between its forward and its backward pass");
        for (auto& s : data) s.unpack(shared_from_this());       // (says so if an input was changed in place)
        for (auto* list : {&plan->held, &held})
            for (auto& h : *list)
                TORCH_CHECK(h.there(), "the memory of a parameter of the model or of the batch was resized or given back between the "
                            "forward and the backward pass");
        const at::Tensor gout = grads[0].detach().to(at::kFloat).contiguous();
        c10::DeviceGuard guard(plan->device);
        const at::Tensor flat = at::empty({total}, at::TensorOptions().dtype(at::kFloat).device(plan->device));
        const at::Tensor scratch = arena(scratch_bytes, plan->device);
        cfh_model_batch q = b;
        q.workspace = workspace_.data_ptr();
        q.workspace_bytes = (size_t)workspace_.numel();
        q.stream = (void*)c10::hip::getCurrentHIPStream(plan->device.index()).stream();
        int rc;
        {
            std::lock_guard<std::mutex> lock(g_enqueue);
            rc = g_lib.backward(model.m, &q, gout.data_ptr<float>(), scratch.data_ptr(), (size_t)scratch.numel(),
                                flat.data_ptr<float>());
        }
        check(rc, "cfh_model_backward");
        // a tensor of its own per parameter over the common storage (autograd adopts it as .grad: nobody else holds it)
        const c10::Storage& storage = flat.storage();
        for (size_t i = 0; i < n; i++) {
            if (!task_should_compute_output(i)) continue;
            auto t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(storage), flat.key_set(), flat.dtype());
            c10::TensorImpl* impl = t.unsafeGetTensorImpl();
            impl->set_storage_offset(plan->offset[i]);
            impl->set_sizes_contiguous(plan->sizes[i]);
            out[i] = std::move(t);
        }
        return out;
    }
};

struct Plan {
    std::shared_ptr<Shared> S = std::make_shared<Shared>();
    // Borrowed: the Python object that owns the plan keeps them (a reference from here would close a cycle that the garbage
    // collector cannot see).
    struct Link { PyObject *dict, *key, *value; };
    std::vector<Link> links;
    struct Walked { PyObject* dict; Py_ssize_t entries; };
    std::vector<Walked> walked;
    struct Layout { void* ptr; std::vector<int64_t> sizes; };
    std::vector<Layout> layout;                // of params, then gauss; all of them contiguous float32

    Plan(py::list links_, py::list walked_, std::vector<at::Tensor> params, std::vector<at::Tensor> gauss, int64_t feat, int64_t D,
         int64_t H, int64_t out_features) {
        for (auto l : links_) {
            auto t = py::reinterpret_borrow<py::tuple>(l);
            links.push_back({PyTuple_GET_ITEM(t.ptr(), 0), PyTuple_GET_ITEM(t.ptr(), 1), PyTuple_GET_ITEM(t.ptr(), 2)});
        }
        for (auto w : walked_) {
            auto t = py::reinterpret_borrow<py::tuple>(w);
            walked.push_back({PyTuple_GET_ITEM(t.ptr(), 0), PyLong_AsSsize_t(PyTuple_GET_ITEM(t.ptr(), 1))});
        }
        S->params = std::move(params);
        S->gauss = std::move(gauss);
        int64_t off = 0;
        for (auto& p : S->params) {
            S->offset.push_back(off);
            off += p.numel();
        }
        for (auto* list : {&S->params, &S->gauss})
            for (auto& p : *list) {
                layout.push_back({p.data_ptr(), p.sizes().vec()});
                S->held.emplace_back(p);
            }
        for (auto& p : S->params) S->sizes.push_back(p.sizes().vec());
        S->device = S->params[0].device();
        S->feat = feat; S->D = D; S->H = H; S->out_features = out_features;
    }
    // Whether the modules and parameters are still those the plan was made from, no more and no fewer, in the same storages
    // and with the same layout.
    bool current() const {
        for (auto& w : walked)
            if (PyDict_GET_SIZE(w.dict) != w.entries) return false;
        for (auto& l : links) {
            PyObject* v = PyDict_GetItemWithError(l.dict, l.key);
            if (v != l.value) {
                if (!v && PyErr_Occurred()) throw py::error_already_set();
                if (v || l.value != Py_None) return false;
            }
        }
        const Layout* l = layout.data();
        for (auto* list : {&S->params, &S->gauss})
            for (auto& p : *list) {
                if (p.data_ptr() != l->ptr || p.scalar_type() != at::kFloat || !p.is_contiguous() || p.sizes() != l->sizes)
                    return false;
                l++;
            }
        return true;
    }
    // The batch is one that the library call takes: it reads as many words of each tensor as x and trans have rows.
    bool accepts(const at::Tensor& x, const at::Tensor& pos, const at::Tensor& batch, const at::Tensor& trans,
                 const at::Tensor& sizes) const {
        auto good = [&](const at::Tensor& t, at::ScalarType ty) {
            return t.scalar_type() == ty && t.device() == S->device && t.is_contiguous();
        };
        return good(x, at::kFloat) && good(pos, at::kFloat) && good(trans, at::kFloat) && good(batch, at::kLong) &&
               good(sizes, at::kLong) && x.dim() == 2 && x.size(1) == S->feat && x.size(0) > 0 &&
               pos.dim() == 2 && pos.size(0) == x.size(0) && pos.size(1) == 3 && batch.dim() == 1 && batch.size(0) == x.size(0) &&
               trans.dim() == 3 && trans.size(1) == 3 && trans.size(2) == 3 && sizes.dim() == 1 && sizes.size(0) == trans.size(0);
    }
    // How many of the parameters want a gradient: 0 none, 1 some, 2 all.
    int wanted() const {
        size_t n = 0;
        for (auto& p : S->params) n += p.requires_grad() ? 1 : 0;
        return n == 0 ? 0 : (n == S->params.size() ? 2 : 1);
    }
    // out (B, features).  workspace: called with a size, gives the scratch of the current stream.  x0, qkv0: see
    // cfh_model_batch (undefined: made by the library).  noise: seeds of the layers' frame searches, or empty.
    at::Tensor forward(uintptr_t model, py::object owner, const at::Tensor& x, const at::Tensor& pos, const at::Tensor& batch,
                       const at::Tensor& trans, const at::Tensor& sizes, int64_t E, bool keep, py::function workspace,
                       std::vector<uint64_t> noise, std::vector<at::Tensor> first) {
        const cfh_model* m = reinterpret_cast<const cfh_model*>(model);
        cfh_model_batch b;
        std::memset(&b, 0, sizeof(b));
        b.x = x.data_ptr<float>(); b.pos = pos.data_ptr<float>(); b.batch = batch.data_ptr<int64_t>();
        b.tvecs = trans.data_ptr<float>(); b.sizes = sizes.data_ptr<int64_t>();
        b.N = x.size(0); b.B = trans.size(0); b.E = E;
        b.keep = keep ? 1 : 0;
        if (!first.empty()) { b.x0 = first[0].data_ptr<float>(); b.qkv0 = first[1].data_ptr<float>(); }
        if (!noise.empty()) b.noise_seeds = noise.data();
        size_t nbytes[4] = {0, 0, 0, 0};
        const int64_t total = g_lib.sizes(m, &b, nbytes);
        if (total < 0) check((int)total, "cfh_model_sizes");
        at::Tensor arena_ = arena(nbytes[0], S->device);
        at::Tensor ws = py::cast<at::Tensor>(workspace(keep ? std::max(nbytes[1], nbytes[3]) : nbytes[1]));
        at::Tensor out = at::empty({b.B, S->out_features}, at::TensorOptions().dtype(at::kFloat).device(S->device));
        b.arena = arena_.data_ptr(); b.arena_bytes = (size_t)arena_.numel();
        b.workspace = ws.data_ptr(); b.workspace_bytes = (size_t)ws.numel();
        b.stream = (void*)c10::hip::getCurrentHIPStream(S->device.index()).stream();
        int rc;
        {
            std::lock_guard<std::mutex> lock(g_enqueue);
            rc = g_lib.forward(m, &b, out.data_ptr<float>());
        }
        check(rc, "cfh_model_forward");
        if (!keep) return out;
        auto node = std::shared_ptr<ModelPassBackward>(new ModelPassBackward(), torch::autograd::deleteNode);
        node->plan = S;
        node->model = Model{m, hold(std::move(owner))};
        node->seeds = std::move(noise);            // (the vector's memory moves along: b.noise_seeds stays right)
        node->b = b;
        node->total = total;
        node->scratch_bytes = nbytes[2];
        node->arena_ = std::move(arena_);
        node->workspace_ = std::move(ws);
        node->first = std::move(first);
        node->versions = ModelPassBackward::current_versions(*S);
        for (const at::Tensor* t : {&x, &pos, &batch, &trans, &sizes}) {
            node->data.emplace_back(*t, false);
            node->held.emplace_back(*t);
        }
        torch::autograd::edge_list edges;
        edges.reserve(S->params.size());
        for (auto& p : S->params) edges.push_back(torch::autograd::impl::gradient_edge(p));
        node->set_next_edges(std::move(edges));
        torch::autograd::set_history(out, node);
        return out;
    }
};

// Who would see the framework's operations in this thread beside autograd's backward pass.
enum : int { WATCHED = 1, FUNCTION_MODE = 2, SAVED_TENSOR_HOOKS = 4 };
int watchers() {
    int seen = 0;
    if (torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::stack_len() > 0 ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        seen |= WATCHED;
    if (at::impl::PythonTorchFunctionTLS::stack_len() > 0) seen |= FUNCTION_MODE;
    if (at::SavedTensorDefaultHooks::get_hooks().has_value()) seen |= SAVED_TENSOR_HOOKS;
    return seen;
}

// Addresses of an optimizer's launch: fills the jobs of the parameters that have a gradient.  Returns how many, or -1 when a
// gradient is one that the Python side has to look at (not contiguous, sparse, another type) or does not fit the moments:
// the kernel goes over as many words of parameter, gradient and moments as the parameter had when these were made.
struct Updates {
    std::vector<at::Tensor> params;
    std::vector<int64_t> offset;               // of a parameter's moments, in floats (-1: none)
    std::vector<int64_t> numel;                // of a parameter's moments
    c10::Device device;                        // of the moments
    Updates(std::vector<at::Tensor> p, std::vector<int64_t> o, std::vector<int64_t> n, const at::Tensor& moments)
        : params(std::move(p)), offset(std::move(o)), numel(std::move(n)), device(moments.device()) {}
    // Whether these are the tensors of the list, in its order.
    bool of(py::object list) const {
        py::object seq = py::reinterpret_steal<py::object>(PySequence_Fast(list.ptr(), "the parameters of a group"));
        if (!seq) throw py::error_already_set();
        if (PySequence_Fast_GET_SIZE(seq.ptr()) != (Py_ssize_t)params.size()) return false;
        PyObject** const items = PySequence_Fast_ITEMS(seq.ptr());
        for (size_t i = 0; i < params.size(); i++)
            if (!THPVariable_Check(items[i]) || THPVariable_Unpack(items[i]).unsafeGetTensorImpl() != params[i].unsafeGetTensorImpl())
                return false;
        return true;
    }
    int64_t fill(uintptr_t jobs, uintptr_t m, uintptr_t v) const {
        cfh_adamw_job* const J = reinterpret_cast<cfh_adamw_job*>(jobs);
        int64_t n = 0;
        for (size_t i = 0; i < params.size(); i++) {
            const at::Tensor& p = params[i];
            const at::Tensor& g = p.grad();
            if (!g.defined()) continue;
            if (offset[i] < 0 || g.layout() != at::kStrided || g.scalar_type() != at::kFloat || !g.is_contiguous() ||
                !p.is_contiguous() || p.scalar_type() != at::kFloat || p.numel() != numel[i] || g.numel() != numel[i] ||
                p.device() != device || g.device() != device)
                return -1;
            cfh_adamw_job& j = J[n++];
            j.param = reinterpret_cast<float*>(p.data_ptr());
            j.grad = reinterpret_cast<const float*>(g.data_ptr());
            j.exp_avg = reinterpret_cast<float*>(m) + offset[i];
            j.exp_avg_sq = reinterpret_cast<float*>(v) + offset[i];
            j.n = p.numel();
        }
        return n;
    }
    // every .grad becomes None
    void drop() {
        for (auto& p : params) p.mutable_grad().reset();
    }
};

}  // namespace

PYBIND11_MODULE(_host, mod) {
    mod.def("bind", [](uintptr_t sizes, uintptr_t forward, uintptr_t backward, uintptr_t last_error) {
        g_lib.sizes = reinterpret_cast<decltype(g_lib.sizes)>(sizes);
        g_lib.forward = reinterpret_cast<decltype(g_lib.forward)>(forward);
        g_lib.backward = reinterpret_cast<decltype(g_lib.backward)>(backward);
        g_lib.last_error = reinterpret_cast<decltype(g_lib.last_error)>(last_error);
    });
    mod.attr("abi") = CFH_ABI_VERSION;
    mod.attr("WATCHED") = (int)WATCHED;
    mod.attr("FUNCTION_MODE") = (int)FUNCTION_MODE;
    mod.attr("SAVED_TENSOR_HOOKS") = (int)SAVED_TENSOR_HOOKS;
    mod.def("watchers", &watchers);
    py::class_<Plan>(mod, "Plan")
        .def(py::init<py::list, py::list, std::vector<at::Tensor>, std::vector<at::Tensor>, int64_t, int64_t, int64_t, int64_t>())
        .def("current", &Plan::current)
        .def("accepts", &Plan::accepts)
        .def("wanted", &Plan::wanted)
        .def("forward", &Plan::forward);
    py::class_<Updates>(mod, "Updates")
        .def(py::init<std::vector<at::Tensor>, std::vector<int64_t>, std::vector<int64_t>, const at::Tensor&>())
        .def("of", &Updates::of)
        .def("fill", &Updates::fill)
        .def("drop", &Updates::drop);
}

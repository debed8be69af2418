// Layers' forward passes with their adjoints as native autograd nodes.  A training
// step of a small layer waits for the host: a torch.autograd.Function costs some 10 us
// in each direction on top of what its methods do, and its backward, on the
// engine's thread, needs the interpreter lock that the caller has just given up.
// These nodes run without it, and call Python for what only Python can do: a
// gather through the transport, and forms that the native adjoint does not take (a
// gradient that is not contiguous, say), which go to the same function as the
// torch.autograd.Function of the layer.
//
// Every function answers None where torch wants to see what happens or where the
// node would drop something: under a tracer, a dispatch mode or a functorch transform, for
// tensors with tangents, for subclasses of torch.Tensor (but for parameters), which
// may want their own type back.  The callers then
// apply their torch.autograd.Function.  Tensors are saved as SavedVariables: hooks on
// saved tensors, checks of versions and of a second pass work as for any node.
#include "front.h"

#include <ATen/core/PythonFallbackKernel.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/dynamo/compiled_autograd.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include <atomic>

namespace ddl_front {
namespace {

namespace py = pybind11;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

bool unobserved() {
    return !torch::jit::tracer::isTracing() && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

bool ordinary(const Tensor& t) {
    constexpr c10::DispatchKeySet kSeen({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::FuncTorchBatched,
                                         c10::DispatchKey::Functionalize});
    const PyObject* const object = t.unsafeGetTensorImpl()->pyobj_slot()->load_pyobj();   // the caller's reference keeps it
    return !t.key_set().has_any(kSeen) && !t._fw_grad(0).defined() && (!object || THPVariable_CheckExact(const_cast<PyObject*>(object)));
}
bool ordinary(const MaybeTensor& t) { return !t || ordinary(*t); }

bool wanted(const Tensor& t) { return t.requires_grad(); }
bool wanted(const MaybeTensor& t) { return t && t->requires_grad(); }

// A Python callable that nodes share; the last owner may be a node that dies on a thread without the interpreter lock.
class Callback {
public:
    explicit Callback(py::object f) : f_(std::move(f)) {}
    Callback(const Callback&) = delete;
    ~Callback() {
        if (!Py_IsInitialized()) {
            f_.release();
            return;
        }
        py::gil_scoped_acquire gil;
        f_ = py::object();
    }
    template <typename R, typename... Args>
    R call(Args&&... args) const {
        py::gil_scoped_acquire gil;
        try {
            return f_(std::forward<Args>(args)...).template cast<R>();
        } catch (py::error_already_set& e) {   // as torch's own nodes throw it: the engine hands it to its caller as it is
            e.restore();
            python_error error;
            error.persist();
            throw error;
        }
    }

private:
    py::object f_;
};
typedef std::shared_ptr<Callback> Shared;

typedef std::tuple<MaybeTensor, MaybeTensor, MaybeTensor> Three;

// The gradients that a pass asks for, and those that a node was made for: bit i for input i.
struct Asked {
    uint32_t now = 0, ever = 0;
};
inline bool has(uint32_t bits, int i) { return (bits >> i) & 1; }

// What tells two adjoints apart, for a compiled pass that is used again.
class Key {
public:
    Key& operator()(int64_t v) {
        bytes_.append(reinterpret_cast<const char*>(&v), sizeof(v));
        return *this;
    }
    Key& operator()(at::IntArrayRef v) {
        (*this)(static_cast<int64_t>(v.size()));
        for (const int64_t n : v) (*this)(n);
        return *this;
    }
    Key& operator()(const MaybeShape& v) { return v ? (*this)(at::IntArrayRef(*v)) : (*this)(int64_t{-1}); }
    template <typename T>
    Key& operator()(const std::shared_ptr<T>& v) {   // a compiled pass holds it, so no other object has its address
        return (*this)(static_cast<int64_t>(reinterpret_cast<intptr_t>(v.get())));
    }
    const std::string& bytes() const { return bytes_; }

private:
    std::string bytes_;
};

// The node of an adjoint A: `A::run(saved tensors, gradient, asked)` computes the gradients, `A::identify(key)` adds all that A
// holds.  Unpacking runs hooks on saved tensors under the lock, as torch's nodes do; the adjoint runs without it.
//
// A compiled pass (torch's compiled autograd) keeps the adjoint as one opaque call: it copies A, and hands in the saved
// tensors and the gradient of the pass it runs in.
template <typename A>
struct ShardNode final : Node {
    A adjoint;
    std::vector<SavedVariable> saved;
    uint32_t present = 0;   // saved tensors that are there
    void save(const Tensor& t) {
        present |= (t.defined() ? 1u : 0u) << saved.size();
        saved.emplace_back(t, false);
    }
    std::string name() const override { return A::kName; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable& s : saved) s.reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        return adjoint.run(unpacked(), grads[0].defined() ? grads[0] : input_metadata(0).zeros_like(), asked());
    }
    void compiled_args(torch::dynamo::autograd::CompiledNodeArgs& args) const override {
        const auto& meta = input_metadata(0);
        Key key;
        key(int64_t{present})(int64_t{asked().now})(int64_t{asked().ever});
        key(static_cast<int64_t>(c10::typeMetaToScalarType(meta.dtype())))(int64_t{meta.device().index()});
        for (const c10::SymInt& n : meta.shape_as_dim_vector()) key(n.expect_int());
        adjoint.identify(key);
        args.collect(key.bytes());
        for (const SavedVariable& s : saved) args.collect(s, false);
    }
    variable_list apply_with_saved(const variable_list& grads, torch::dynamo::autograd::SwapSavedVariables& swap) override {
        namespace compiled = torch::dynamo::autograd;
        for (SavedVariable& s : saved) swap.before(s);
        std::vector<Tensor> there;
        for (const Tensor& t : unpacked())
            if (t.defined()) there.push_back(t);
        compiled::PackedArgs packed;
        packed.pack(there);
        compiled::functional_apply_t call = [adjoint = adjoint, present = present, count = saved.size(), asked = asked(), meta = input_metadata(0)](
                                                const variable_list& given, const compiled::ivalue_list& packed_args) {
            compiled::PackedArgs args(packed_args);
            const auto tensors = args.template unpack<std::vector<Tensor>>();
            std::vector<Tensor> kept(count);
            for (size_t i = 0, k = 0; i < count; ++i)
                if (has(present, static_cast<int>(i))) kept[i] = tensors.at(k++);
            return adjoint.run(kept, given[0].defined() ? given[0] : meta.zeros_like(), asked);
        };
        const auto& compiler = compiled::getPyCompilerInterface();
        const std::string bound = compiler->bind_function(swap.get_py_compiler(), name(), std::move(call), {compiled::IValuePacker<std::vector<Tensor>>::packed_type()},
                                                          /*is_custom_function=*/true, /*is_traceable=*/false);
        auto results = compiler->call_function(swap.get_py_compiler(), "apply_functional", bound, grads, packed.vec(),
                                               compiled::IValuePacker<std::vector<std::optional<torch::autograd::InputMetadata>>>::pack(compiled::get_input_metadata(next_edges())));
        for (SavedVariable& s : saved) swap.after(s);
        return results;
    }

private:
    std::vector<Tensor> unpacked() {
        std::lock_guard<std::mutex> lock(mutex_);
        std::vector<Tensor> tensors;
        for (SavedVariable& s : saved) tensors.push_back(s.unpack());
        return tensors;
    }
    Asked asked() const {
        Asked a;
        for (int i = 0; i < static_cast<int>(num_outputs()); ++i) {
            a.now |= (task_should_compute_output(i) ? 1u : 0u) << i;
            a.ever |= (should_compute_output(i) ? 1u : 0u) << i;
        }
        return a;
    }
};

// y's node, for the inputs given.
template <typename A>
std::shared_ptr<ShardNode<A>> make_node(A adjoint, std::initializer_list<MaybeTensor> inputs) {
    std::shared_ptr<ShardNode<A>> node(new ShardNode<A>, torch::autograd::deleteNode);
    node->adjoint = std::move(adjoint);
    torch::autograd::edge_list edges;
    for (const MaybeTensor& t : inputs) edges.push_back(t ? torch::autograd::impl::gradient_edge(*t) : torch::autograd::Edge());
    node->set_next_edges(std::move(edges));
    return node;
}

MaybeTensor defined(const Tensor& t) { return t.defined() ? MaybeTensor(t) : std::nullopt; }
variable_list listed(const Three& t) {
    auto one = [](const MaybeTensor& v) { return v ? *v : Tensor(); };
    return {one(std::get<0>(t)), one(std::get<1>(t)), one(std::get<2>(t))};
}

// ---------------------------------------------------------------- linear --

struct LinearShard {
    static constexpr const char* kName = "LinearShardBackward";
    std::vector<int64_t> bias_shape;
    Shared general;
    void identify(Key& key) const { key(at::IntArrayRef(bias_shape))(general); }
    variable_list run(const std::vector<Tensor>& kept, const Tensor& dy, const Asked& asked) const {
        const Tensor &x = kept[0], &w = kept[1];
        const bool need_x = has(asked.now, 0), need_w = has(asked.now, 1), need_b = has(asked.now, 2);
        auto res = product_backward(x, w, dy, need_x, need_w, need_b ? MaybeShape(bias_shape) : std::nullopt);
        if (res) return {std::get<0>(*res), std::get<1>(*res), std::get<2>(*res)};
        return listed(general->call<Three>(x, w, dy, need_x, need_w, need_b ? MaybeShape(bias_shape) : std::nullopt));
    }
};

MaybeTensor linear_shard(const Tensor& x, const Tensor& w, const MaybeTensor& bias, const Shared& general) {
    if (!unobserved() || !ordinary(x) || !ordinary(w) || !ordinary(bias)) return std::nullopt;
    MaybeTensor y;
    {
        at::NoGradGuard no_grad;
        y = product(x, w, bias);
    }
    if (!y || !at::GradMode::is_enabled() || !(wanted(x) || wanted(w) || wanted(bias))) return y;
    auto node = make_node(LinearShard{bias ? bias->sizes().vec() : std::vector<int64_t>(), general}, {x, w, bias});
    node->save(x);
    node->save(w);
    torch::autograd::create_gradient_edge(*y, node);
    return y;
}

// ------------------------------------------------------------ layer norm --

struct LayerNormShard {
    static constexpr const char* kName = "LayerNormShardBackward";
    MaybeShape gamma_shape, beta_shape;
    int64_t workers = 1;
    Shared gather, general;   // gather: this worker's row sums -> those of all workers
    void identify(Key& key) const { key(gamma_shape)(beta_shape)(workers)(gather)(general); }
    variable_list run(const std::vector<Tensor>& kept, const Tensor& dy, const Asked& asked) const {
        const Tensor &x2d = kept[0], &mean = kept[1], &rstd = kept[2];
        const MaybeTensor gamma = defined(kept[3]);
        // Those that require gradients, whether or not this pass asks for them: the order of the sums hangs on it.
        const bool need_x = has(asked.ever, 0);
        const MaybeShape for_gamma = has(asked.ever, 1) ? gamma_shape : std::nullopt, for_beta = has(asked.ever, 2) ? beta_shape : std::nullopt;
        std::optional<std::tuple<Tensor, Tensor, Tensor>> res;
        if (need_x && workers == 1) {
            res = ln_backward_whole(dy, x2d, mean, rstd, gamma, for_gamma, for_beta);
        }
        if (!res && need_x && (for_gamma || for_beta) && plain(dy)) {
            const Tensor rows = dy.detach().view(x2d.sizes());
            if (auto partial = ln_backward_partial_params(rows, x2d, mean, rstd, gamma)) {
                const Tensor sums = workers == 1 ? std::get<0>(*partial).unsqueeze(0) : gather->call<Tensor>(std::get<0>(*partial));
                res = ln_backward_input_params(rows, x2d, mean, rstd, gamma, sums, 1.0 / static_cast<double>(workers * x2d.size(1)), std::get<1>(*partial),
                                               for_gamma, for_beta);
                if (!res) throw std::runtime_error("layer norm: row sums of the workers do not fit the rows");
                std::get<0>(*res) = std::get<0>(*res).view(dy.sizes());
            }
        }
        if (res) return {std::get<0>(*res), std::get<1>(*res), std::get<2>(*res)};
        return listed(general->call<Three>(dy, x2d, mean, rstd, gamma, need_x, for_gamma, for_beta));
    }
};

MaybeTensor normalized(const Tensor& x, const MaybeTensor& gamma, const MaybeTensor& beta, const std::optional<Normalized>& res, int64_t workers,
                       const Shared& gather, const Shared& general) {
    if (!res) return std::nullopt;
    Tensor y = std::get<0>(*res);
    auto shape = [](const MaybeTensor& t) { return t ? MaybeShape(t->sizes().vec()) : std::nullopt; };
    auto node = make_node(LayerNormShard{shape(gamma), shape(beta), workers, gather, general}, {x, gamma, beta});
    node->save(std::get<1>(*res));
    node->save(std::get<2>(*res));
    node->save(std::get<3>(*res));
    node->save(std::get<4>(*res));
    torch::autograd::create_gradient_edge(y, node);
    return y;
}

// For callers that want a gradient: y with its node.
MaybeTensor layer_norm_shard(const Tensor& x, const MaybeTensor& gamma, const MaybeTensor& beta, int64_t cols, double eps, const Shared& general) {
    if (!unobserved() || !ordinary(x) || !ordinary(gamma) || !ordinary(beta)) return std::nullopt;
    std::optional<Normalized> res;
    {
        at::NoGradGuard no_grad;
        res = layer_norm(x, gamma, beta, cols, eps);
    }
    return normalized(x, gamma, beta, res, 1, nullptr, general);
}

// The node for rows shared with other workers, whose y, mean and reciprocal deviation the caller has computed.
Tensor layer_norm_node(const Tensor& x, const MaybeTensor& gamma, const MaybeTensor& beta, const Tensor& y, const Tensor& mean, const Tensor& rstd,
                       int64_t workers, const Shared& gather, const Shared& general) {
    if (x.dim() < 1 || mean.numel() == 0 || x.numel() % mean.numel() != 0) throw std::invalid_argument("layer_norm_node: rows and their means disagree");
    const int64_t cols = x.numel() / mean.numel();
    const Normalized res(y, x.detach().view({mean.numel(), cols}), mean, rstd, gamma ? gamma->detach().view({cols}) : Tensor());
    return *normalized(x, gamma, beta, res, workers, gather, general);
}

// ------------------------------------------------------------- embedding --

struct EmbeddingShard {
    static constexpr const char* kName = "EmbeddingShardBackward";
    int64_t lo = 0, hi = 0;
    std::optional<int64_t> padding_idx;
    bool by_freq = false;
    Shared general;
    void identify(Key& key) const { key(lo)(hi)(int64_t{padding_idx.has_value()})(padding_idx.value_or(0))(int64_t{by_freq})(general); }
    variable_list run(const std::vector<Tensor>& kept, const Tensor& dy, const Asked& asked) const {
        const Tensor& ids = kept[0];
        if (!has(asked.now, 0)) return {Tensor()};
        const MaybeTensor dw = embedding_backward(dy, ids, lo, hi, padding_idx.value_or(-1), by_freq);
        if (dw) return {*dw};
        return {general->call<Tensor>(dy, ids, lo, hi, padding_idx, by_freq)};
    }
};

MaybeTensor embedding_shard(const Tensor& weight, const Tensor& ids, int64_t lo, int64_t hi, std::optional<int64_t> padding_idx, bool by_freq,
                            const Shared& general) {
    if (!unobserved() || !ordinary(weight) || !ordinary(ids) || !float_code(weight)) return std::nullopt;
    MaybeTensor y = embedding_gather(weight, ids, lo, hi);
    if (!y || !at::GradMode::is_enabled() || !wanted(weight)) return y;
    auto node = make_node(EmbeddingShard{lo, hi, padding_idx, by_freq, general}, {weight});
    node->save(ids);
    torch::autograd::create_gradient_edge(*y, node);
    return y;
}

// ----------------------------------------------------------------- moves --

// Pooled communication buffers that have been reallocated since this extension was loaded.
std::atomic<int64_t> reallocated{0};

// The launches of one direction of a data movement that needs no message in between, for one structure of its input: boxes
// between the input (base address 0), the output (1) and buffers (2, ...), and the staging of a convolution (pad, ghosts, bulk
// strips) as a launch of its own kind.  `out_shape` empty: the input itself is worked on.  Calls only read the object.  It
// keeps its buffers alive, and takes no call any more once some buffer has been reallocated since `epoch`, which its maker asked
// for before it took the buffers: the layer has others then.
class Moves {
public:
    typedef std::tuple<std::shared_ptr<Boxes>, int, int> Step;                                                        // boxes, operation, element type
    typedef std::tuple<std::vector<int64_t>, std::vector<int64_t>, std::vector<int64_t>, std::vector<MaybeTensor>, std::vector<MaybeTensor>> Staging;

    Moves(std::vector<int64_t> shape, std::vector<int64_t> strides, at::ScalarType dtype, MaybeShape out_shape, std::vector<Step> steps,
          std::vector<MaybeTensor> buffers, std::optional<Staging> staging, Shared general, int64_t epoch)
        : shape_(std::move(shape)), strides_(std::move(strides)), dtype_(dtype), out_shape_(std::move(out_shape)), steps_(std::move(steps)),
          buffers_(std::move(buffers)), staging_(std::move(staging)), general_(std::move(general)), epoch_(epoch) {
        if (staging_ && !out_shape_) throw std::invalid_argument("Moves: staging needs an output");
        if (staging_) {
            const size_t nd = shape_.size();
            if (std::get<0>(*staging_).size() != 2 * nd || std::get<1>(*staging_).size() != 2 * nd || std::get<2>(*staging_).size() != 2 * nd ||
                std::get<3>(*staging_).size() != 2 * nd || std::get<4>(*staging_).size() != 2 * nd)
                throw std::invalid_argument("Moves: staging of another number of dimensions");
        }
    }
    bool takes(const Tensor& t) const {
        return t.is_cuda() && t.scalar_type() == dtype_ && t.sizes() == at::IntArrayRef(shape_) && t.strides() == at::IntArrayRef(strides_) &&
               epoch_ == reallocated.load();
    }
    Tensor run(const Tensor& t) const {
        Tensor out = out_shape_ ? at::empty(*out_shape_, t.options()) : t;
        auto address = [](const void* p) { return static_cast<int64_t>(reinterpret_cast<intptr_t>(p)); };
        std::vector<int64_t> bases{out_shape_ ? address(t.data_ptr()) : 0, address(out.data_ptr())};
        for (const MaybeTensor& b : buffers_) bases.push_back(address(pointer(b)));
        if (staging_) {
            std::vector<const void*> ghosts;
            std::vector<void*> bulk;
            for (const MaybeTensor& b : std::get<3>(*staging_)) ghosts.push_back(pointer(b));
            for (const MaybeTensor& b : std::get<4>(*staging_)) bulk.push_back(const_cast<void*>(pointer(b)));
            check(ddl_halo_pad_exchange(t.data_ptr(), out.data_ptr(), shape_.data(), static_cast<int>(shape_.size()), static_cast<int>(t.element_size()),
                                        std::get<0>(*staging_).data(), std::get<1>(*staging_).data(), std::get<2>(*staging_).data(), ghosts.data(), bulk.data(),
                                        DDL_HALO_AUTO, current_stream()),
                  "ddl_halo_pad_exchange");
        }
        for (const Step& s : steps_) std::get<0>(s)->run(bases, std::get<1>(s), std::get<2>(s));
        return out;
    }
    // The way through Python, for a tensor that run() does not take.
    Tensor general(const Tensor& t) const { return general_->call<Tensor>(t); }

private:
    std::vector<int64_t> shape_, strides_;
    at::ScalarType dtype_;
    MaybeShape out_shape_;
    std::vector<Step> steps_;
    std::vector<MaybeTensor> buffers_;
    std::optional<Staging> staging_;
    Shared general_;
    int64_t epoch_;
};

struct Move {
    static constexpr const char* kName = "MoveBackward";
    std::shared_ptr<Moves> moves;
    void identify(Key& key) const { key(moves); }
    variable_list run(const std::vector<Tensor>&, const Tensor& dy, const Asked&) const { return {moves->takes(dy) ? moves->run(dy) : moves->general(dy)}; }
};

MaybeTensor move(const Tensor& x, const std::shared_ptr<Moves>& forward, const std::shared_ptr<Moves>& adjoint) {
    const bool graph = at::GradMode::is_enabled() && wanted(x);
    if (!forward->takes(x) || (graph && !adjoint) || !unobserved() || !ordinary(x)) return std::nullopt;
    Tensor y = forward->run(x);
    if (graph) torch::autograd::create_gradient_edge(y, make_node(Move{adjoint}, {x}));
    return y;
}

// ----------------------------------------------------------------- alias --

// What a rank that is alone hands to itself: a result of its own on the same memory.
struct Alias {
    static constexpr const char* kName = "AliasBackward";
    void identify(Key&) const {}
    // No layer's adjoint has a history of its own, so a second derivative does not go through this one either.
    variable_list run(const std::vector<Tensor>&, const Tensor& dy, const Asked&) const { return {at::GradMode::is_enabled() ? dy.detach() : dy}; }
};

MaybeTensor alias(const Tensor& x) {
    if (!unobserved() || !ordinary(x)) return std::nullopt;
    Tensor y = x.detach();
    if (at::GradMode::is_enabled() && wanted(x)) torch::autograd::create_gradient_edge(y, make_node(Alias{}, {x}));
    return y;
}

// ---------------------------------------------------------------- Python --

// y, computed from x in Python, with an adjoint in Python.
struct Call {
    static constexpr const char* kName = "CallBackward";
    Shared function;
    void identify(Key& key) const { key(function); }
    variable_list run(const std::vector<Tensor>&, const Tensor& dy, const Asked&) const { return {function->call<Tensor>(dy)}; }
};

bool attachable(const Tensor& x) { return at::GradMode::is_enabled() && wanted(x) && unobserved() && ordinary(x); }

Tensor attach(Tensor y, const Tensor& x, const Shared& adjoint) {
    if (y.requires_grad() || !at::isFloatingType(y.scalar_type())) throw std::invalid_argument("attach: a result with a history of its own");
    torch::autograd::create_gradient_edge(y, make_node(Call{adjoint}, {x}));
    return y;
}

}  // namespace

void define_nodes(py::module_& m) {
    typedef py::call_guard<py::gil_scoped_release> unlocked;
    py::class_<Callback, Shared>(m, "Callback").def(py::init<py::object>());
    py::class_<Moves, std::shared_ptr<Moves>>(m, "Moves")
        .def(py::init<std::vector<int64_t>, std::vector<int64_t>, at::ScalarType, MaybeShape, std::vector<Moves::Step>, std::vector<MaybeTensor>,
                      std::optional<Moves::Staging>, Shared, int64_t>());
    m.def("linear_shard", &linear_shard, unlocked());
    m.def("layer_norm_shard", &layer_norm_shard, unlocked());
    m.def("layer_norm_node", &layer_norm_node, unlocked());
    m.def("embedding_shard", &embedding_shard, unlocked());
    m.def("move", &move, unlocked());
    m.def("alias", &alias, unlocked());
    m.def("attachable", &attachable);
    m.def("unobserved", [](const Tensor& x, const MaybeTensor& a, const MaybeTensor& b) { return unobserved() && ordinary(x) && ordinary(a) && ordinary(b); });
    m.def("attach", &attach);
    m.def("buffers_moved", [] { ++reallocated; });
    m.def("buffers_epoch", [] { return reallocated.load(); });
}

}  // namespace ddl_front

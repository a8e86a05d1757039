// The host side of the MoE block in C++: allocations, launches of the C-ABI entry points and the
// autograd nodes around them, as the Python module `optimus_torch_host`.
//
// What bounded the small calls was the interpreter: a training step of the tiny layer was 22 launches
// (10 now) of 2-14 us each, and enqueueing them through ctypes and Python autograd functions took 510 us.  Here a
// layer is two autograd nodes (router, experts) whose forward and backward run without the interpreter:
// each reads the three run-time switches of the Python modules once (launch log, profiler, in-place
// weight gradients) and then only allocates and launches.
//
// The nodes are plain torch::autograd::Node objects: outputs nobody differentiates arrive as undefined
// tensors (nothing is filled or added for them), and a weight whose gradient already lives in a flat
// buffer gets it added there by the GEMM and an undefined gradient returned.
#include <torch/extension.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/engine.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <c10/hip/HIPStream.h>
#include <unordered_set>

#include "../../../include/optimus_mi355x.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

namespace {

struct NativeError : std::runtime_error {
    using std::runtime_error::runtime_error;
};

// ---- the Python modules' run-time switches --------------------------------------------------------

PyObject *module_attr(const char *module, const char *name) {   // new reference; GIL held
    PyObject *m = PyImport_ImportModule(module);
    if (!m) throw py::error_already_set();
    PyObject *v = PyObject_GetAttrString(m, name);
    Py_DECREF(m);
    if (!v) throw py::error_already_set();
    return v;
}
// A module-level switch, read at every call.  The module object and the name are looked up once and kept (reloading a module
// keeps its object): importing it by name each time took most of the 2.4 us that a call spent on its three switches.
struct ModuleSwitch {
    const char *module_name, *name;
    PyObject *module = nullptr, *key = nullptr;
    bool is(PyObject *what) {                       // GIL held
        if (!module) {
            PyObject *m = PyImport_ImportModule(module_name);   // (may let another thread run)
            if (!m) throw py::error_already_set();
            if (!module) module = m;
            else Py_DECREF(m);
        }
        if (!key) key = PyUnicode_InternFromString(name);
        PyObject *v = key ? PyObject_GetAttr(module, key) : nullptr;
        if (!v) throw py::error_already_set();
        const bool same = v == what;
        Py_DECREF(v);
        return same;
    }
};

struct Call {
    bool log = false;        // optimus._native.launch_log is a list: time every launch
    bool profile = false;    // optimus.globals.profiler is set
    bool in_place = true;    // moe.accumulate_weight_grads_in_place
    void *stream = nullptr;
};

Call begin_call() {
    static ModuleSwitch log{"optimus._native", "launch_log"}, profiler{"optimus.globals", "profiler"},
        in_place{"optimus.models.common.moe", "accumulate_weight_grads_in_place"};
    Call c;
    {
        py::gil_scoped_acquire gil;
        c.log = !log.is(Py_None);
        c.profile = !profiler.is(Py_None);
        c.in_place = in_place.is(Py_True);
    }
    c.stream = c10::hip::getCurrentHIPStream().stream();
    return c;
}

void check(int code, const char *what) {
    if (code != 0)
        throw NativeError(std::string(what) + " failed with code " + std::to_string(code) + ": " + om_strerror(code));
}

// A Python object that may be dropped without the GIL, also while an exception passes.
struct PyRef {
    py::object object;
    ~PyRef() {
        if (!object) return;
        py::gil_scoped_acquire gil;
        object = py::object();
    }
};

template <typename F> void launch(const Call &c, const char *name, F &&fn) {
    if (!c.log) {
        check(fn(), name);
        return;
    }
    PyRef start;
    {
        py::gil_scoped_acquire gil;
        start.object = py::module_::import("optimus._native").attr("timed_begin")(name);
    }
    const int code = fn();
    {
        py::gil_scoped_acquire gil;
        py::module_::import("optimus._native").attr("timed_end")(name, start.object);
    }
    check(code, name);
}
#define OM(c, fn, ...) launch(c, #fn, [&] { return fn(__VA_ARGS__); })
// the form of fn that takes a bound and the rows to expect, logged as fn
#define OM_BOUND(c, fn, ...) launch(c, #fn, [&] { return fn##_bound(__VA_ARGS__); })

// optimus.profilers.record_pcl_function(name) around a scope, when a profiler is set.  What the profiler raises
// at the scope's end reaches the caller, as from a `with` block; while another exception passes it is reported
// and dropped.
struct ProfiledScope {
    PyRef context;
    int exceptions = std::uncaught_exceptions();
    ProfiledScope(const Call &c, const char *name) {
        if (!c.profile) return;
        py::gil_scoped_acquire gil;
        py::object entered = py::module_::import("optimus.profilers").attr("record_pcl_function")(name);
        entered.attr("__enter__")();
        context.object = std::move(entered);
    }
    ProfiledScope(const ProfiledScope &) = delete;
    ~ProfiledScope() noexcept(false) {
        if (!context.object) return;
        py::gil_scoped_acquire gil;
        const py::object entered = std::move(context.object);
        try {
            entered.attr("__exit__")(py::none(), py::none(), py::none());
        } catch (py::error_already_set &e) {
            if (std::uncaught_exceptions() == exceptions) throw;
            e.discard_as_unraisable("the end of a profiled scope");
        }
    }
};

// ---- tensor helpers -------------------------------------------------------------------------------

void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
const int32_t *iptr(const Tensor &t) { return t.defined() ? t.data_ptr<int32_t>() : nullptr; }
int dtype_code(const Tensor &t) {
    if (t.scalar_type() == at::kFloat) return OM_F32;
    TORCH_CHECK_TYPE(t.scalar_type() == at::kBFloat16, "unsupported dtype ", t.scalar_type(),
                     ": the HIP kernels take float32 or bfloat16");
    return OM_BF16;
}
int index_code(const Tensor &t) {
    if (t.scalar_type() == at::kLong) return OM_I64;
    TORCH_CHECK_TYPE(t.scalar_type() == at::kInt, "expert indices must be int64 or int32, got ", t.scalar_type());
    return OM_I32;
}
void require_device(const Tensor &t) {
    if (!t.defined()) return;
    if (!t.is_cuda())
        throw NativeError("the HIP kernels need device tensors (got a CPU tensor); there is no CPU fallback");
    if (!t.is_contiguous()) throw NativeError("the HIP kernels need contiguous row-major tensors");
}
void require_bf16(const Tensor &t) {
    TORCH_CHECK_TYPE(t.scalar_type() == at::kBFloat16, "the fused expert kernels run in bfloat16 (got ",
                     t.scalar_type(), "); cast the module with .to(torch.bfloat16)");
}
Tensor make(at::IntArrayRef size, const Tensor &like) { return at::empty(size, like.options()); }
Tensor make(at::IntArrayRef size, const Tensor &like, at::ScalarType dt) { return at::empty(size, like.options().dtype(dt)); }

// Elements between consecutive experts of a [G, out, in] weight whose inner two dims are dense; 0 for
// the packed layout.
int64_t expert_stride(const Tensor &w) {
    const int64_t o = w.size(1), i = w.size(2);
    if (w.stride(2) != 1 || w.stride(1) != i) throw NativeError("expert weights must be dense [out, in] matrices");
    const int64_t s = w.size(0) > 1 ? w.stride(0) : o * i;
    return s == o * i ? 0 : s;
}

// [G, out, in] over per-expert matrices that lie at a constant pitch in one storage; undefined when
// they do not.
Tensor strided_view_or_undefined(const Tensor *w, size_t step, int64_t G) {
    const Tensor &w0 = w[0];
    if (w0.dim() != 2) return Tensor();
    const int64_t o = w0.size(0), i = w0.size(1);
    if (G == 1) return w0.unsqueeze(0);
    const int64_t esz = w0.element_size();
    const char *p0 = static_cast<const char *>(w0.data_ptr());
    const int64_t pitch = static_cast<const char *>(w[step].data_ptr()) - p0;
    if (pitch <= 0 || pitch % esz != 0 || pitch < o * i * esz) return Tensor();
    for (int64_t n = 0; n < G; n++) {
        const Tensor &t = w[n * step];
        if (!t.is_contiguous() || t.dim() != 2 || t.size(0) != o || t.size(1) != i ||
            t.scalar_type() != w0.scalar_type() || static_cast<const char *>(t.data_ptr()) != p0 + n * pitch ||
            !t.storage().is_alias_of(w0.storage()))
            return Tensor();
    }
    return w0.as_strided({G, o, i}, {pitch / esz, i, 1});
}
Tensor strided_view(const Tensor *w, size_t step, int64_t G) {
    Tensor v = strided_view_or_undefined(w, step, G);
    if (!v.defined())
        throw NativeError("per-expert weights must lie at a constant pitch inside one buffer (merge them with "
                          "pack_expert_weights, or build the optimizer first so they alias flat_param)");
    return v;
}

// ---- weight gradients that live in a flat buffer ----------------------------------------------------

// Whether a hook on the parameter would have to see the incoming gradient.  A hook that was registered and
// removed leaves its (empty) Python dictionary behind, and so does a deepcopy or a load: asked in Python then.
bool has_grad_hooks(const Tensor &param) {
    const size_t n = torch::autograd::impl::hooks(param).size();
    const bool post = torch::autograd::impl::post_acc_grad_hooks(param) != nullptr;
    if (n == 0 && !post) return false;
    py::gil_scoped_acquire gil;
    const py::object p = py::cast(param), hooks = p.attr("_backward_hooks"), posts = p.attr("_post_accumulate_grad_hooks");
    return n > (hooks.is_none() ? 0u : 1u) || (post && posts.is_none()) ||   // (the rest: registered from C++)
           (!hooks.is_none() && py::len(hooks) > 0) || (!posts.is_none() && py::len(posts) > 0);
}

// Whether the running backward pass accumulates into param.grad: torch.autograd.grad() returns gradients instead,
// and backward(inputs=...) leaves the parameters alone that it does not name.
bool accumulates_into(const Tensor &param) {
    const auto *tasks = torch::autograd::get_current_graph_task_exec_info();
    if (!tasks || tasks->empty()) return true;            // backward() of everything
    const auto accumulator = torch::autograd::impl::try_get_grad_accumulator(param);
    const auto it = tasks->find(accumulator.get());
    return it != tasks->end() && it->second.needed_ && !it->second.captures_;
}

// param.grad if the weight-gradient kernels may add into it in place: a leaf parameter whose gradient
// already exists as a dense view of a larger buffer, same dtype and shape, in a pass that accumulates into it
// and with no hooks that would have to see the incoming gradient; else undefined.
Tensor live_grad(const Tensor &param) {
    if (!param.defined() || !param.is_leaf() || !param.requires_grad()) return Tensor();
    const Tensor &grad = param.grad();
    if (!grad.defined() || !grad.is_view() || grad.scalar_type() != param.scalar_type() ||
        grad.sizes() != param.sizes() || !grad.is_cuda() || !grad.is_contiguous() || grad.requires_grad())
        return Tensor();
    return !accumulates_into(param) || has_grad_hooks(param) ? Tensor() : grad;
}

// At the end of the running backward pass: order the caller's stream behind what this stream has been given.  A
// gradient that a GEMM adds into its live buffer never reaches autograd, which orders the caller's stream only
// behind gradients that it accumulates itself; the forward may have run on another stream than its caller's.
void order_live_gradients() {
    if (!torch::autograd::get_current_graph_task_exec_info()) return;   // (not in a backward pass)
    const auto stream = c10::hip::getCurrentHIPStream();
    torch::autograd::Engine::get_default_engine().queue_callback([stream] {
        const auto caller = c10::hip::getCurrentHIPStream(stream.device_index());
        if (caller.stream() == stream.stream()) return;
        const c10::DeviceGuard device(stream.device());
        hipEvent_t done = nullptr;
        const bool ok = hipEventCreateWithFlags(&done, hipEventDisableTiming) == hipSuccess &&
                        hipEventRecord(done, stream.stream()) == hipSuccess &&
                        hipStreamWaitEvent(caller.stream(), done, 0) == hipSuccess;
        if (done) (void)hipEventDestroy(done);
        if (!ok) throw NativeError("ordering the caller's stream behind the weight gradients failed");
    });
}

// One projection's gradient: where the GEMM writes it.
struct Sink {
    Tensor grad;          // [G, out, in]: the live buffer, or a fresh tensor
    int64_t pitch = 0;
    bool accumulate = false;
};
// `leaves`: the parameter itself, or the G per-expert parameters `step` apart
Sink grad_sink(const Call &c, const Tensor *leaves, size_t step, int64_t n_leaves, const Tensor &view) {
    Sink s;
    if (c.in_place && !at::GradMode::is_enabled()) {
        if (n_leaves == 1) {
            s.grad = live_grad(leaves[0]);
            if (s.grad.defined() && s.grad.dim() == 2) s.grad = s.grad.unsqueeze(0);
        } else {
            std::vector<Tensor> grads;
            grads.reserve(n_leaves);
            for (int64_t n = 0; n < n_leaves; n++) {
                grads.push_back(live_grad(leaves[n * step]));
                if (!grads.back().defined()) break;
            }
            if (grads.back().defined()) s.grad = strided_view_or_undefined(grads.data(), 1, n_leaves);
        }
    }
    if (s.grad.defined()) {
        s.pitch = expert_stride(s.grad);
        s.accumulate = true;
    } else {
        s.grad = make(view.sizes(), view);
    }
    return s;
}

// ---- index construction ---------------------------------------------------------------------------

// The arrays of om_moe_sort and the tensors that own them.
struct Index {
    std::vector<Tensor> owners;     // one buffer that holds them all, or five tensors (cum, cum_ep, in, out, sel)
    int64_t NR = 0, T = 0, TK = 0;  // the one buffer's parts
    void resolve() {
        if (owners.size() == 1) {
            int32_t *p = owners[0].data_ptr<int32_t>();
            cum = p; cum_ep = p + NR + 1; in = cum_ep + T + 1; out = in + TK; sel = out + TK;
            row_weights = reinterpret_cast<const float *>(sel + TK);
        } else {
            cum = iptr(owners[0]); cum_ep = iptr(owners[1]); in = iptr(owners[2]); out = iptr(owners[3]); sel = iptr(owners[4]);
            row_weights = nullptr;
        }
    }
    Index without_arrays() const {  // what a node keeps beside the saved owners: no pointer outlives the forward pass
        Index ix;
        ix.NR = NR; ix.T = T; ix.TK = TK; ix.rows = rows; ix.bound = bound; ix.expected = expected;
        return ix;
    }
    const int32_t *cum = nullptr, *cum_ep = nullptr, *in = nullptr, *out = nullptr, *sel = nullptr;
    const float *row_weights = nullptr;   // the routing weight of every sorted row (one-buffer form only)
    int64_t rows = 0;               // entries of the three last: the routed rows, or an upper bound of them
    bool bound = false;
    int64_t expected = -1;          // with a bound: the rows to expect, where they can be told
    int64_t to_choose_by() const { return bound && expected >= 0 ? expected : rows; }
};

std::vector<Tensor> sort_tensors(const Call &c, const Tensor &experts, int64_t start, int64_t end) {
    require_device(experts);
    const int64_t T = experts.size(0), K = experts.size(1), NR = end - start;
    const auto opt = experts.options().dtype(at::kInt);
    std::vector<Tensor> r = {at::empty({NR + 1}, opt), at::empty({T + 1}, opt), at::empty({T * K}, opt),
                             at::empty({T * K}, opt), at::empty({T * K}, opt)};
    const int64_t ws_bytes = om_moe_sort_workspace_bytes(T, K, NR);
    Tensor ws = at::empty({std::max<int64_t>(ws_bytes / 4, 1)}, opt);
    OM(c, om_moe_sort, ptr(experts), index_code(experts), T, K, start, end, r[0].data_ptr<int32_t>(),
       r[1].data_ptr<int32_t>(), r[2].data_ptr<int32_t>(), r[3].data_ptr<int32_t>(), r[4].data_ptr<int32_t>(),
       ptr(ws), ws_bytes, c.stream);
    return r;
}

// The one-buffer form for T tokens of K selections, its arrays in `buffer` or, where that is undefined, in a new one with
// `more` words behind them.
int64_t index_words(int64_t T, int64_t K, int64_t NR) { return NR + 1 + T + 1 + 4 * T * K; }
Index one_buffer_index(int64_t T, int64_t K, int64_t NR, Tensor buffer, const Tensor &like = Tensor(), int64_t more = 0) {
    Index ix;
    ix.T = T;
    ix.NR = NR;
    ix.TK = ix.rows = T * K;
    if (!buffer.defined()) buffer = at::empty({index_words(T, K, NR) + more}, like.options().dtype(at::kInt));
    ix.owners = {std::move(buffer)};
    ix.resolve();
    return ix;
}
template <typename T> T *rwp(const T *p) { return const_cast<T *>(p); }

Index sort_index(const Call &c, const Tensor &experts, int64_t start, int64_t end, const Tensor &rw) {
    require_device(experts);
    require_device(rw);
    const int64_t K = experts.size(1), T = experts.size(0), NR = end - start;
    const int64_t ws_bytes = om_moe_sort_workspace_bytes(T, K, NR), ws_at = index_words(T, K, NR);
    Index ix = one_buffer_index(T, K, NR, Tensor(), experts, std::max<int64_t>(ws_bytes / 4, 1));
    int32_t *p = ix.owners[0].data_ptr<int32_t>();
    OM(c, om_moe_sort_weighted, ptr(experts), index_code(experts), ix.T, K, start, end, rwp(ix.cum), rwp(ix.cum_ep),
       rwp(ix.in), rwp(ix.out), rwp(ix.sel), ptr(rw), dtype_code(rw), rwp(ix.row_weights), p + ws_at, ws_bytes, c.stream);
    return ix;
}

// ---- the expert MLP ---------------------------------------------------------------------------------

struct MlpWeights {
    Tensor gate, up, down;   // [G, I, H], [G, I, H], [G, H, I]
    int64_t G() const { return gate.size(0); }
    int64_t I() const { return gate.size(1); }
    int64_t H() const { return gate.size(2); }
};
struct MlpState {
    Tensor cum, g, u, h;     // cum undefined: the caller's index holds the offsets
};

int64_t shared_pitch(const MlpWeights &w) {
    const int64_t s = expert_stride(w.gate);
    if (expert_stride(w.up) != s) throw NativeError("gate and up expert weights must share one expert pitch");
    return s;
}

// Operands that the expert kernels would misread: they trust shapes and device.
void require_mlp_operands(const Tensor &x, const MlpWeights &w) {
    const auto gate = w.gate.sizes();
    if (gate.size() != 3 || x.dim() != 2 || x.size(1) != gate[2] || w.up.sizes() != gate ||
        w.down.sizes() != at::IntArrayRef({gate[0], gate[2], gate[1]}))
        throw NativeError("expert MLP: expected activations [rows, hidden], gate and up weights [experts, ffn, hidden] and down "
                          "weights [experts, hidden, ffn]");
    for (const Tensor *t : {&w.gate, &w.up, &w.down})
        if (!t->is_cuda())
            throw NativeError("the HIP kernels need device tensors (got CPU expert weights); there is no CPU fallback");
}

void gemm_dtype(const Tensor &a, const Tensor &b, const Tensor &c) {
    const auto dt = a.scalar_type();
    TORCH_CHECK_TYPE((dt == at::kBFloat16 || dt == at::kFloat) && b.scalar_type() == dt && c.scalar_type() == dt,
                     "the grouped expert GEMMs take operands that are all bfloat16 or all float32 (got ", dt, ", ",
                     b.scalar_type(), ", ", c.scalar_type(), ")");
}

const float *fp(const Tensor &t) { return static_cast<const float *>(ptr(t)); }
float *fpm(const Tensor &t) { return static_cast<float *>(ptr(t)); }

// y = (silu(x Wg^T) * (x Wu^T)) Wd^T per expert segment; with x_rows the MLP input is x[x_rows].  `keep`: whether a backward may
// follow, which needs g and u.
Tensor merged_forward(const Call &c, const Tensor &x, const MlpWeights &w, const int32_t *cum, const int32_t *x_rows,
                      int64_t rows, MlpState &s, bool keep = true) {
    require_mlp_operands(x, w);
    require_device(x);
    gemm_dtype(x, w.gate, w.up);
    gemm_dtype(x, w.gate, w.down);
    const int64_t G = w.G(), I = w.I(), H = w.H();
    keep = keep || x.scalar_type() == at::kFloat;
    if (keep) {
        s.g = make({rows, I}, x);
        s.u = make({rows, I}, x);
    }
    s.h = make({rows, I}, x);
    Tensor y = make({rows, H}, x);
    ProfiledScope scope(c, "1moeblock--7gmlp_fwd");
    if (x.scalar_type() == at::kFloat) {
        OM(c, om_merged_mlp_gate_up_fwd_f32, fp(x), rows ? x_rows : nullptr, x.size(0), fp(w.gate), fp(w.up), fpm(s.g),
           fpm(s.u), fpm(s.h), cum, rows, G, I, H, expert_stride(w.gate), expert_stride(w.up), c.stream);
        OM(c, om_grouped_gemm_fwd_f32, fp(s.h), fp(w.down), fpm(y), cum, rows, G, H, I, expert_stride(w.down), c.stream);
        return y;
    }
    const int64_t pitch = shared_pitch(w);
    if (!keep)
        OM(c, om_merged_mlp_hidden_fwd, ptr(x), rows ? x_rows : nullptr, x.size(0), ptr(w.gate), ptr(w.up), nullptr, ptr(s.h), cum, rows,
           rows, G, I, H, pitch, nullptr, c.stream);
    else if (x_rows && rows > 0)
        OM(c, om_merged_mlp_gate_up_fwd_gathered, ptr(x), x_rows, x.size(0), ptr(w.gate), ptr(w.up), ptr(s.g), ptr(s.u),
           ptr(s.h), cum, rows, G, I, H, pitch, c.stream);
    else
        OM(c, om_merged_mlp_gate_up_fwd, ptr(x), ptr(w.gate), ptr(w.up), ptr(s.g), ptr(s.u), ptr(s.h), cum, rows, G, I, H,
           pitch, c.stream);
    OM(c, om_grouped_gemm_fwd, ptr(s.h), ptr(w.down), ptr(y), cum, rows, G, H, I, expert_stride(w.down), c.stream);
    return y;
}

enum class WgradRows { PLAIN, INPUT, OUTPUT_GRAD };

// One of the bf16 weight-gradient entry points: plain, or with the rows of `input` or of
// `output_grad` taken through an index, writing or (accumulate) adding into the sink.
void wgrad(const Call &c, const Tensor &output_grad, const Tensor &input, const Sink &s, const int32_t *cum,
           int64_t rows, int64_t G, int64_t N, int64_t K, WgradRows kind = WgradRows::PLAIN,
           const int32_t *index = nullptr, int64_t src_rows = 0) {
    void *out = ptr(s.grad);
#define OM_W(fn, ...)                                                                    \
    do {                                                                                 \
        if (s.accumulate) OM(c, fn##_accumulate, __VA_ARGS__);                           \
        else OM(c, fn, __VA_ARGS__);                                                     \
    } while (0)
    if (kind == WgradRows::INPUT)
        OM_W(om_grouped_gemm_wgrad_gathered, ptr(output_grad), ptr(input), index, src_rows, out, cum, rows, G, N, K,
             s.pitch, c.stream);
    else if (kind == WgradRows::OUTPUT_GRAD)
        OM_W(om_grouped_gemm_wgrad_gathered_out, ptr(output_grad), index, src_rows, ptr(input), out, cum, rows, G, N, K,
             s.pitch, c.stream);
    else
        OM_W(om_grouped_gemm_wgrad, ptr(output_grad), ptr(input), out, cum, rows, G, N, K, s.pitch, c.stream);
#undef OM_W
}
void wgrad_f32(const Call &c, const Tensor &output_grad, const Tensor &input, const Sink &s, const int32_t *cum,
               int64_t rows, int64_t G, int64_t N, int64_t K) {
    if (s.accumulate)
        OM(c, om_grouped_gemm_wgrad_f32_accumulate, fp(output_grad), fp(input), fpm(s.grad), cum, rows, G, N, K, s.pitch, c.stream);
    else
        OM(c, om_grouped_gemm_wgrad_f32, fp(output_grad), fp(input), fpm(s.grad), cum, rows, G, N, K, s.pitch, c.stream);
}

struct Sinks {
    Sink gate, up, down;
    static Tensor fresh(const Sink &s) { return s.accumulate ? Tensor() : s.grad; }
};

// All three weight gradients of a bf16 merged MLP: one call where all are written or all are added into their sinks.
// dout_rows / x_rows: rows of dout / x taken through an index.  `expected`: the rows to choose launches by, where `rows` is a bound.
void wgrads(const Call &c, const Tensor &dout, const int32_t *dout_rows, const Tensor &h, const Tensor &dg, const Tensor &du,
            const Tensor &x, const int32_t *x_rows, const Sinks &k, const int32_t *cum, int64_t rows, int64_t expected, int64_t G,
            int64_t I, int64_t H) {
    if (k.gate.accumulate == k.up.accumulate && k.gate.accumulate == k.down.accumulate) {
        const int64_t src_rows = dout_rows ? dout.size(0) : x.size(0);
#define OM_W(fn)                                                                                                        \
    OM_BOUND(c, fn, ptr(dout), dout_rows, ptr(h), ptr(dg), ptr(du), ptr(x), x_rows, src_rows, ptr(k.down.grad), ptr(k.gate.grad), \
             ptr(k.up.grad), cum, rows, expected, G, I, H, k.down.pitch, k.gate.pitch, k.up.pitch, c.stream)
        if (k.gate.accumulate) OM_W(om_grouped_gemm_wgrad_merged_accumulate);
        else OM_W(om_grouped_gemm_wgrad_merged);
#undef OM_W
        return;
    }
    wgrad(c, dout, h, k.down, cum, rows, G, H, I, dout_rows ? WgradRows::OUTPUT_GRAD : WgradRows::PLAIN, dout_rows, dout.size(0));
    const WgradRows kind = x_rows ? WgradRows::INPUT : WgradRows::PLAIN;
    wgrad(c, dg, x, k.gate, cum, rows, G, I, H, kind, x_rows, x.size(0));
    wgrad(c, du, x, k.up, cum, rows, G, I, H, kind, x_rows, x.size(0));
}

// Backward of merged_forward: returns dx (of the gathered matrix when x_rows is set); the weight
// gradients go into the sinks.
Tensor merged_backward(const Call &c, Tensor dy, const Tensor &x, const MlpWeights &w, const int32_t *cum,
                       const MlpState &s, const int32_t *x_rows, const Sinks &k) {
    dy = dy.contiguous();
    const int64_t rows = dy.size(0), H = dy.size(1), G = w.G(), I = w.I();
    Tensor dg = make({rows, I}, x), du = make({rows, I}, x), dx = make({rows, H}, x);
    ProfiledScope scope(c, "1moeblock--7gmlp_bwd");
    if (x.scalar_type() == at::kFloat) {
        OM(c, om_merged_mlp_down_dgrad_f32, fp(dy), fp(w.down), fp(s.g), fp(s.u), fpm(dg), fpm(du), cum, rows, G, I, H,
           expert_stride(w.down), c.stream);
        const int32_t *rows_of_x = rows ? x_rows : nullptr;
        if (k.gate.accumulate == k.up.accumulate && k.gate.accumulate == k.down.accumulate) {
#define OM_W(fn)                                                                                                           \
    OM(c, fn, fp(dy), fp(s.h), fp(dg), fp(du), fp(x), rows_of_x, x.size(0), fp(w.gate), fp(w.up), fpm(dx), fpm(k.down.grad), \
       fpm(k.gate.grad), fpm(k.up.grad), cum, rows, G, I, H, expert_stride(w.gate), expert_stride(w.up), k.down.pitch,         \
       k.gate.pitch, k.up.pitch, c.stream)
            if (k.gate.accumulate) OM_W(om_grouped_gemm_wgrad_merged_dgrad_f32_accumulate);
            else OM_W(om_grouped_gemm_wgrad_merged_dgrad_f32);
#undef OM_W
            return dx;
        }
        wgrad_f32(c, dy, s.h, k.down, cum, rows, G, H, I);
        OM(c, om_merged_mlp_gate_up_wgrad_f32, fp(dg), fp(du), fp(x), rows_of_x, x.size(0), fpm(k.gate.grad), fpm(k.up.grad), cum,
           rows, G, I, H, k.gate.pitch, k.up.pitch, k.gate.accumulate | k.up.accumulate << 1, c.stream);
        OM(c, om_merged_mlp_gate_up_dgrad_f32, fp(dg), fp(du), fp(w.gate), fp(w.up), fpm(dx), cum, rows, G, I, H,
           expert_stride(w.gate), expert_stride(w.up), c.stream);
        return dx;
    }
    OM(c, om_merged_mlp_down_dgrad, ptr(dy), ptr(w.down), ptr(s.g), ptr(s.u), ptr(dg), ptr(du), cum, rows, G, I, H,
       expert_stride(w.down), c.stream);
    wgrads(c, dy, nullptr, s.h, dg, du, x, rows > 0 ? x_rows : nullptr, k, cum, rows, rows, G, I, H);
    OM(c, om_merged_mlp_gate_up_dgrad, ptr(dg), ptr(du), ptr(w.gate), ptr(w.up), ptr(dx), cum, rows, G, I, H,
       expert_stride(w.gate), c.stream);
    return dx;
}

// The shared expert of a block as it goes along with the routed ones, whose extents it has (om_dense_expert).
struct Alongside {
    const MlpWeights &w;
    MlpState &s;             // the forward's; its cum: device {0, tokens}
    Tensor y;                // its output
    static bool fits(const MlpWeights &w, int64_t I, int64_t H) {
        return w.I() == I && w.H() == H && w.gate.is_contiguous() && w.up.is_contiguous() && w.down.is_contiguous();
    }
    // Whether one of `products` (OM_DENSE_...) would run in a routed launch.  Where none would, the shared expert goes first, all of
    // it: what it computes with in between (64 MB of dg and du with 8192 tokens of intermediate size 2048) is used at once and given back.
    static bool rides(const MlpWeights &w, const MlpWeights &routed, int64_t expected, int64_t tokens, int products) {
        if (!fits(w, routed.I(), routed.H()) || tokens < 1) return false;
        const int which = om_merged_mlp_dense_products(expected, static_cast<int>(routed.G()), static_cast<int>(routed.I()),
                                                       static_cast<int>(routed.H()), tokens);
        return which > 0 && (which & products);
    }
};
om_dense_expert dense_expert(std::array<const Tensor *, 2> a, std::array<const Tensor *, 2> w, std::array<const Tensor *, 3> cs,
                             const MlpState &s, int64_t rows) {
    auto p = [](const Tensor *t) { return t ? ptr(*t) : nullptr; };
    return {{p(a[0]), p(a[1])}, {p(w[0]), p(w[1])}, {p(cs[0]), p(cs[1]), p(cs[2])}, ptr(s.g), ptr(s.u), iptr(s.cum), rows};
}

// The routed half of a bf16 block: gather, weighted SwiGLU MLP, unweighted sum of a token's rows.  `along`: and the shared
// expert, whose output is the residual.
Tensor routed_forward(const Call &c, const Tensor &x, const Tensor &rw, const Index &ix, const MlpWeights &w,
                      Tensor residual, MlpState &s, Tensor &row_weights, Alongside *along = nullptr, bool keep = true) {
    require_mlp_operands(x, w);
    if (rw.dim() != 2 || rw.size(0) != x.size(0)) throw NativeError("routing weights: expected [tokens, top_k]");
    if (residual.defined()) {
        if (residual.sizes() != x.sizes()) throw NativeError("residual: expected the shape of the hidden states");
        require_bf16(residual);
    }
    require_device(x);
    require_device(rw);
    require_device(residual);
    require_bf16(x);
    require_bf16(w.gate);
    require_bf16(w.up);
    require_bf16(w.down);
    const int64_t T = x.size(0), H = x.size(1), K = rw.size(1), rows = ix.rows, G = w.G(), I = w.I();
    const int64_t pitch = shared_pitch(w);
    if (keep) {
        s.g = make({rows, I}, x);
        s.u = make({rows, I}, x);
    }
    s.h = make({rows, I}, x);
    Tensor y = make({rows, H}, x), final = make({T, H}, x);
    {
        ProfiledScope scope(c, "1moeblock--7gmlp_fwd");
        const float *weights = ix.row_weights;
        if (!weights) {
            row_weights = make({rows}, x, at::kFloat);
            weights = fp(row_weights);
            OM(c, om_moe_row_weights, ptr(rw), ix.sel, ix.in, ix.out, fpm(row_weights), rows, K, dtype_code(rw), c.stream);
        }
        if (along) {
            MlpState &d = along->s;
            if (keep) {
                d.g = make({T, I}, x);
                d.u = make({T, I}, x);
            }
            d.h = make({T, I}, x);
            residual = along->y = make({T, H}, x);
            const om_dense_expert up = dense_expert({&x, nullptr}, {&along->w.gate, &along->w.up}, {&d.g, &d.u, &d.h}, d, T);
            if (!keep)
                OM(c, om_merged_mlp_hidden_fwd, ptr(x), ix.in, T, ptr(w.gate), ptr(w.up), weights, ptr(s.h), ix.cum, rows,
                   ix.to_choose_by(), G, I, H, pitch, &up, c.stream);
            else OM(c, om_merged_mlp_gate_up_fwd_weighted_dense, ptr(x), ix.in, T, ptr(w.gate), ptr(w.up), weights, ptr(s.g), ptr(s.u),
               ptr(s.h), ix.cum, rows, ix.to_choose_by(), G, I, H, pitch, &up, c.stream);
            const om_dense_expert down = dense_expert({&d.h, nullptr}, {&along->w.down, nullptr}, {&along->y, nullptr, nullptr}, d, T);
            OM(c, om_grouped_gemm_fwd_dense, ptr(s.h), ptr(w.down), ptr(y), ix.cum, rows, ix.to_choose_by(), G, H, I,
               expert_stride(w.down), &down, c.stream);
        } else {
            if (!keep)
                OM(c, om_merged_mlp_hidden_fwd, ptr(x), ix.in, T, ptr(w.gate), ptr(w.up), weights, ptr(s.h), ix.cum, rows,
                   ix.to_choose_by(), G, I, H, pitch, nullptr, c.stream);
            else OM_BOUND(c, om_merged_mlp_gate_up_fwd_weighted, ptr(x), ix.in, T, ptr(w.gate), ptr(w.up), weights, ptr(s.g),
                     ptr(s.u), ptr(s.h), ix.cum, rows, ix.to_choose_by(), G, I, H, pitch, c.stream);
            OM_BOUND(c, om_grouped_gemm_fwd, ptr(s.h), ptr(w.down), ptr(y), ix.cum, rows, ix.to_choose_by(), G, H, I,
                     expert_stride(w.down), c.stream);
        }
    }
    ProfiledScope scope(c, "1moeblock--8gmlp_output_reduction_fwd");
    OM(c, om_sum_ggemm_output, ptr(y), ix.cum_ep, ix.out, ptr(residual), ptr(final), T, H, OM_BF16, c.stream);
    return final;
}

// -> (dx, d routing_weights); `base` [T,H]: another gradient of the same hidden states, added to dx
// inside the per-token sum.  `along`: the shared expert's backward as well, whose input gradient is that base; its weight
// gradients go into `along_sinks`.
std::pair<Tensor, Tensor> routed_backward(const Call &c, const Tensor &dfinal, const Tensor &x, const Tensor &rw,
                                          const Index &ix, const MlpWeights &w, const MlpState &s,
                                          const Tensor &row_weights, const Sinks &k, Tensor base, Alongside *along = nullptr,
                                          const Sinks *along_sinks = nullptr) {
    const int64_t T = x.size(0), H = x.size(1), K = rw.size(1), rows = ix.rows, G = w.G(), I = w.I();
    Tensor dg = make({rows, I}, x), du = make({rows, I}, x), dx_rows = make({rows, H}, x);
    Tensor drw = rows > 0 ? make(rw.sizes(), rw) : at::zeros(rw.sizes(), rw.options());
    Tensor row_dot;
    const int parts = om_merged_mlp_row_dot_parts(I);
    if (parts < 1) check(parts, "om_merged_mlp_row_dot_parts");
    Tensor dx = make(x.sizes(), x);
    {
        ProfiledScope scope(c, "1moeblock--7gmlp_bwd");
        if (rows > 0) {
            row_dot = make({parts, rows}, x, at::kFloat);
            const float *row_w = ix.row_weights ? ix.row_weights : fp(row_weights);
            Tensor dense_dg, dense_du;
            if (along) {
                dense_dg = make({T, I}, x);
                dense_du = make({T, I}, x);
                base = make({T, H}, x);
                const om_dense_expert d = dense_expert({&dfinal, nullptr}, {&along->w.down, nullptr}, {&dense_dg, &dense_du, nullptr}, along->s, T);
                OM(c, om_merged_mlp_down_dgrad_weighted_dense, ptr(dfinal), ix.in, T, ptr(w.down), ptr(s.g), ptr(s.u), row_w, ptr(dg),
                   ptr(du), fpm(row_dot), ix.cum, rows, ix.to_choose_by(), G, I, H, expert_stride(w.down), &d, c.stream);
                wgrads(c, dfinal, nullptr, along->s.h, dense_dg, dense_du, x, nullptr, *along_sinks, iptr(along->s.cum), T, T, 1, I, H);
            } else {
                OM_BOUND(c, om_merged_mlp_down_dgrad_weighted, ptr(dfinal), ix.in, T, ptr(w.down), ptr(s.g), ptr(s.u), row_w, ptr(dg),
                         ptr(du), fpm(row_dot), ix.cum, rows, ix.to_choose_by(), G, I, H, expert_stride(w.down), c.stream);
            }
            const bool joined = !along && k.gate.accumulate == k.up.accumulate && k.gate.accumulate == k.down.accumulate &&
                                om_merged_mlp_backward_joins(ix.to_choose_by(), G, I, H) == 1;
#define OM_JOINED(fn)                                                                                                                 \
    OM(c, fn, ptr(dfinal), ix.in, ptr(s.h), ptr(dg), ptr(du), ptr(x), ix.in, T, ptr(w.gate), ptr(w.up), ptr(dx_rows), ptr(k.down.grad), \
       ptr(k.gate.grad), ptr(k.up.grad), ix.cum, rows, ix.to_choose_by(), G, I, H, expert_stride(w.gate), k.down.pitch, k.gate.pitch,   \
       k.up.pitch, c.stream)
            if (joined && k.gate.accumulate) OM_JOINED(om_grouped_gemm_wgrad_merged_dgrad_accumulate);
            else if (joined) OM_JOINED(om_grouped_gemm_wgrad_merged_dgrad);
#undef OM_JOINED
            else wgrads(c, dfinal, ix.in, s.h, dg, du, x, ix.in, k, ix.cum, rows, ix.to_choose_by(), G, I, H);
            if (along) {
                const om_dense_expert d = dense_expert({&dense_dg, &dense_du}, {&along->w.gate, &along->w.up}, {&base, nullptr, nullptr}, along->s, T);
                OM(c, om_merged_mlp_gate_up_dgrad_dense, ptr(dg), ptr(du), ptr(w.gate), ptr(w.up), ptr(dx_rows), ix.cum, rows,
                   ix.to_choose_by(), G, I, H, expert_stride(w.gate), &d, c.stream);
            } else if (!joined) {
                OM_BOUND(c, om_merged_mlp_gate_up_dgrad, ptr(dg), ptr(du), ptr(w.gate), ptr(w.up), ptr(dx_rows), ix.cum, rows,
                         ix.to_choose_by(), G, I, H, expert_stride(w.gate), c.stream);
            }
        } else {   // nothing routed to these experts: fresh weight gradients are zero, live ones stay as they are
            for (const Sink *sk : {&k.down, &k.gate, &k.up})
                if (!sk->accumulate) {
                    const int64_t n = sk->grad.size(1), kk = sk->grad.size(2);
                    OM(c, om_grouped_gemm_wgrad, nullptr, nullptr, ptr(sk->grad), ix.cum, 0, G, n, kk, 0, c.stream);
                }
        }
    }
    ProfiledScope scope(c, "1moeblock--6gmlp_input_prep_bwd");
    require_device(base);
    if (rows > 0)
        OM(c, om_sum_ggemm_output_row_weights_grad, ptr(dx_rows), ix.cum_ep, ix.out, ptr(base), ptr(dx), T, H, OM_BF16, fp(row_dot),
           parts, rows, ix.sel, ptr(drw), K, dtype_code(drw), c.stream);
    else
        OM(c, om_sum_ggemm_output, ptr(dx_rows), ix.cum_ep, ix.out, ptr(base), ptr(dx), T, H, OM_BF16, c.stream);
    return {dx, drw};
}

// What merged_forward checks of a shared expert, for one that goes along with the routed experts.
void require_shared_operands(const Tensor &x, const MlpWeights &w, const Tensor &one, MlpState &s) {
    require_mlp_operands(x, w);
    require_device(x);
    gemm_dtype(x, w.gate, w.up);
    gemm_dtype(x, w.gate, w.down);
    s.cum = one;
}

// ---- autograd plumbing --------------------------------------------------------------------------------

// The nodes below have no forward-mode formula and no batching rule, and their forward runs below the
// dispatch keys that would ask for one: without this a tangent or a batch dimension is dropped unnoticed.
// Called first by every entry point with a differentiable input.  (NotImplementedError: what a Python
// autograd function without `jvp` raises.)
void refuse_transforms(at::ArrayRef<Tensor> ts) {
    static constexpr c10::DispatchKeySet functorch({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper});
    for (const Tensor &t : ts) {
        if (!t.defined()) continue;
        TORCH_CHECK_NOT_IMPLEMENTED(!t._fw_grad(/*level=*/0).defined(),
                                    "the fused MoE functions have no forward-mode derivative (jvp): use reverse mode");
        TORCH_CHECK(!t.key_set().has_any(functorch),
                    "the fused MoE functions cannot run under torch.func transforms (vmap, grad, jvp): use torch.autograd");
    }
}

bool any_requires_grad(at::ArrayRef<Tensor> ts) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor &t : ts)
        if (t.defined() && t.requires_grad()) return true;
    return false;
}

template <typename N> std::shared_ptr<N> make_node(const variable_list &inputs) {
    std::shared_ptr<N> node(new N(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(inputs));
    return node;
}

MlpWeights weights_of(at::ArrayRef<Tensor> leaves, bool merged, int64_t n_groups) {
    if (!merged)
        return {strided_view(&leaves[0], 3, n_groups), strided_view(&leaves[1], 3, n_groups),
                strided_view(&leaves[2], 3, n_groups)};
    if (leaves[0].dim() == 2) return {leaves[0].unsqueeze(0), leaves[1].unsqueeze(0), leaves[2].unsqueeze(0)};
    return {leaves[0], leaves[1], leaves[2]};
}

// What a node keeps of one set of expert weights.  The weights themselves are three saved variables (the merged
// tensors, or the views over the per-expert matrices), and the backward computes with what those unpack to.
// The parameters are kept beside them only to find a live gradient buffer, so only where they can have one.
struct ExpertWeights {
    bool merged = false, single = false;   // single: one MLP's [out, in] matrices
    int64_t G = 0;
    size_t n_leaves = 0, at = 0;           // the caller's weight tensors; position of the saved variables
    std::vector<Tensor> params;
    // of the per-expert matrices: a view over them has a counter of its own
    std::vector<std::pair<c10::VariableVersion, uint32_t>> versions;

    static ExpertWeights of(at::ArrayRef<Tensor> leaves, bool merged) {
        ExpertWeights e;
        e.merged = merged;
        e.single = merged && leaves[0].dim() == 2;
        e.G = merged ? (e.single ? 1 : leaves[0].size(0)) : static_cast<int64_t>(leaves.size() / 3);
        e.n_leaves = leaves.size();
        for (const Tensor &t : leaves) e.params.push_back(t.is_leaf() && t.requires_grad() ? t : Tensor());
        return e;
    }
};

// A node's backward: kernel errors become the package's own exception type in the thread that called
// backward(), and Python's own (a profiler's) arrive there as they are.
struct HostNode : Node {
    virtual variable_list run(variable_list &&grads) = 0;
    // (one thread at a time unpacks and releases the saved variables, as in the nodes that PyTorch generates)
    variable_list apply(variable_list &&grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        try {
            return run(std::move(grads));
        } catch (const NativeError &e) {
            py::gil_scoped_acquire gil;
            PyObject *cls = module_attr("optimus._native", "NativeLibraryError");
            PyErr_SetString(cls, e.what());
            Py_DECREF(cls);
            throw_python_error();
        } catch (py::error_already_set &e) {
            py::gil_scoped_acquire gil;
            e.restore();
            throw_python_error();
        }
    }
    [[noreturn]] static void throw_python_error() {   // the one that is set; GIL held
        python_error err;
        err.persist();
        throw std::move(err);
    }
    // Everything the backward needs is saved through SavedVariable, so that saved-tensor hooks (activation
    // checkpointing, offloading) see all of it and a second backward is refused.
    std::vector<SavedVariable> vars;
    void save(const Tensor &t) { vars.emplace_back(t, false); }
    // (to be called where autograd records: a hook may run a whole forward pass, as checkpointing does)
    std::vector<Tensor> saved() {
        std::vector<Tensor> out;
        out.reserve(vars.size());
        for (auto &v : vars) {
            out.push_back(v.unpack(shared_from_this()));
            if (v.has_hooks() && out.back().defined() && !out.back().is_cuda())
                throw NativeError("a saved-tensor hook unpacked a tensor that is not on the device it was packed from");
        }
        return out;
    }
    ExpertWeights save_weights(at::ArrayRef<Tensor> leaves, bool merged, const MlpWeights &w) {
        ExpertWeights e = ExpertWeights::of(leaves, merged);
        e.at = vars.size();
        if (merged) {
            for (const Tensor &t : leaves) save(t);
            return e;
        }
        for (const Tensor &t : {w.gate, w.up, w.down}) save(t);
        for (const Tensor &t : leaves) {
            const auto &counter = torch::autograd::impl::version_counter(t);
            e.versions.emplace_back(counter, counter.current_version());
        }
        return e;
    }
    MlpWeights weights(const ExpertWeights &e, const std::vector<Tensor> &kept) {
        if (e.merged) return weights_of(at::ArrayRef<Tensor>(&kept[e.at], 3), true, e.G);
        if (!vars[e.at].has_hooks())       // (what a hook packed is its own: autograd tracks no versions through it either)
            for (const auto &[counter, saved_version] : e.versions)
                TORCH_CHECK(counter.current_version() == saved_version,
                            "one of the variables needed for gradient computation has been modified by an inplace "
                            "operation: an expert's weight, at version ", counter.current_version(), ", expected ", saved_version);
        return {kept[e.at], kept[e.at + 1], kept[e.at + 2]};
    }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (auto &v : vars) v.reset_data();
    }
};

Sinks sinks_of(const Call &c, const ExpertWeights &e, const MlpWeights &w) {
    const int64_t n = e.merged ? 1 : e.G;
    Sinks k = {grad_sink(c, &e.params[0], 3, n, w.gate), grad_sink(c, &e.params[1], 3, n, w.up),
               grad_sink(c, &e.params[2], 3, n, w.down)};
    if (k.gate.accumulate || k.up.accumulate || k.down.accumulate) order_live_gradients();
    return k;
}
// gradients in the order of the leaves; undefined for a projection whose gradient went into its live buffer
void push_grads(variable_list &out, const Sinks &k, const ExpertWeights &e) {
    const Tensor g[3] = {Sinks::fresh(k.gate), Sinks::fresh(k.up), Sinks::fresh(k.down)};
    if (e.merged) {
        for (const Tensor &t : g) out.push_back(e.single && t.defined() ? t.select(0, 0) : t);
        return;
    }
    for (int64_t n = 0; n < e.G; n++)
        for (const Tensor &t : g) out.push_back(t.defined() ? t.select(0, n) : t);
}

// ---- router nodes -------------------------------------------------------------------------------------

void require_gate_shape(const Tensor &weight, const char *what) {
    const int64_t N = weight.size(0), H = weight.size(1);
    if (N > 256 || H % 8 != 0)
        throw NativeError(std::string(what) + ": the gate kernels take at most 256 experts and hidden sizes that are "
                          "multiples of 8 (got " + std::to_string(N) + " experts, hidden " + std::to_string(H) +
                          "); there is no library fallback");
}

// Operands that the gate's kernels would misread: they take both in one type and trust the shapes.
void require_gate_operands(const Tensor &x, const Tensor &weight) {
    TORCH_CHECK_TYPE(x.scalar_type() == weight.scalar_type() && (x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kFloat),
                     "router gate: activations and weight must both be bfloat16 or both float32 (got ", x.scalar_type(), ", ",
                     weight.scalar_type(), ")");
    if (x.dim() != 2 || weight.dim() != 2 || x.size(1) != weight.size(1))
        throw NativeError("router gate: expected activations [tokens, hidden] and a weight [experts, hidden]");
}

Tensor gate_weight_grad(const Call &c, const Tensor &x, const Tensor &weight, Tensor dlogits) {
    require_gate_shape(weight, "gate weight gradient");
    const int64_t T = x.size(0), N = weight.size(0), H = weight.size(1);
    const int64_t ws_bytes = om_router_gate_wgrad_workspace_bytes(T, H, N);
    if (ws_bytes < 0) check(static_cast<int>(ws_bytes), "om_router_gate_wgrad_workspace_bytes");
    Tensor ws = make({std::max<int64_t>(ws_bytes, 16)}, x, at::kByte), dw = make(weight.sizes(), weight);
    dlogits = dlogits.contiguous();
    OM(c, om_router_gate_wgrad, ptr(x), fp(dlogits), T, H, N, ptr(dw), dtype_code(dw), ptr(ws), ws_bytes, c.stream);
    return dw;
}

// dx = bf16(dlogits) @ weight (+ other_grad, the gradient that reached the same hidden states through
// the experts, with autograd's two roundings)
Tensor gate_input_grad(const Call &c, const Tensor &weight, Tensor dlogits, Tensor other_grad) {
    require_gate_shape(weight, "gate input gradient");
    const int64_t T = dlogits.size(0), N = weight.size(0), H = weight.size(1);
    dlogits = dlogits.contiguous();
    if (other_grad.defined()) {
        other_grad = other_grad.contiguous();
        require_bf16(other_grad);
    }
    Tensor dx = make({T, H}, dlogits, at::kBFloat16);
    OM(c, om_router_gate_dgrad, fp(dlogits), ptr(weight), ptr(other_grad), ptr(dx), T, H, N, c.stream);
    return dx;
}

// (dx, dweight) of logits = x @ weight.T from the gradient of the logits; float32 modules run the plain
// float32 gate kernels.
std::pair<Tensor, Tensor> gate_backward(const Call &c, const Tensor &x, const Tensor &weight, Tensor dlogits, bool need_x,
                                        bool need_w, const Tensor &other_grad) {
    dlogits = dlogits.to(at::kFloat).contiguous();
    Tensor dx, dw;
    if (x.scalar_type() == at::kFloat) {
        const int64_t T = x.size(0), N = weight.size(0), H = weight.size(1);
        const Tensor base = other_grad.defined() ? other_grad.contiguous() : Tensor();
        if (need_x && need_w && T > 0) {
            dx = make(x.sizes(), x);
            dw = make(weight.sizes(), weight);
            OM(c, om_router_gate_bwd_f32, fp(x), fp(dlogits), fp(weight), fp(base), T, H, N, fpm(dx), fpm(dw), c.stream);
            return {dx, dw};
        }
        if (need_x) {
            dx = make(x.sizes(), x);
            OM(c, om_router_gate_dgrad_f32_add, fp(dlogits), fp(weight), fp(base), T, H, N, fpm(dx), c.stream);
        }
        if (need_w) {
            dw = make(weight.sizes(), weight);
            OM(c, om_router_gate_wgrad_f32, fp(x), fp(dlogits), T, H, N, fpm(dw), c.stream);
        }
        return {dx, dw};
    }
    require_bf16(x);
    require_bf16(weight);
    if (need_x) dx = gate_input_grad(c, weight, dlogits, other_grad);
    if (need_w) dw = gate_weight_grad(c, x, weight, dlogits);
    return {dx, dw};
}

Tensor gate_logits_forward(const Call &c, const Tensor &x, const Tensor &weight) {
    require_device(x);
    require_device(weight);
    const int64_t T = x.size(0), N = weight.size(0), H = weight.size(1);
    Tensor logits = make({T, N}, x, at::kFloat);
    if (x.scalar_type() == at::kFloat) {
        OM(c, om_router_gate_logits_f32, fp(x), fp(weight), T, H, N, fpm(logits), c.stream);
        return logits;
    }
    require_gate_shape(weight, "gate projection");
    if (N > 64 || H % 512 != 0) {
        // many experts: the weight no longer fits a block's re-reads; split over H instead (also the
        // form for hidden sizes the one-pass kernel does not take)
        const int64_t ws_bytes = om_router_gate_logits_split_workspace_bytes(T, H, N);
        if (ws_bytes < 0) check(static_cast<int>(ws_bytes), "om_router_gate_logits_split_workspace_bytes");
        Tensor ws = make({std::max<int64_t>(ws_bytes, 16)}, x, at::kByte);
        OM(c, om_router_gate_logits_split, ptr(x), ptr(weight), T, H, N, fpm(logits), ptr(ws), ws_bytes, c.stream);
    } else {
        OM(c, om_router_gate_logits, ptr(x), ptr(weight), T, H, N, fpm(logits), c.stream);
    }
    return logits;
}

// Gate projection and routing.  Outputs: the logits and the selection that follows from them, and x
// itself: experts fed from that output make their input gradient arrive here, where the gate's own is
// added to it inside its kernel.
struct RouterNode : HostNode {       // saves x, weight, and (selecting) logits as the selection saw them, experts
    bool renorm = false, sigmoid = false;
    double scale = 1.0;
    int out_logits = -1, out_weights = -1, out_x = -1;   // positions of the differentiable outputs
    std::string name() const override { return "OptimusRouterBackward"; }
    variable_list run(variable_list &&grads) override {
        auto grad = [&](int at) { return at >= 0 && at < static_cast<int>(grads.size()) ? grads[at] : Tensor(); };
        Tensor logits_grad = grad(out_logits), weights_grad = grad(out_weights), x_grad = grad(out_x);
        if (!logits_grad.defined() && !weights_grad.defined()) return {x_grad, Tensor()};
        const std::vector<Tensor> kept = saved();
        at::AutoDispatchBelowADInplaceOrView below;
        const Call c = begin_call();
        const Tensor &xs = kept[0], &ws = kept[1];
        Tensor dlogits = logits_grad;
        if (weights_grad.defined()) {
            const Tensor &logits = kept[2], &experts = kept[3];
            const int64_t T = logits.size(0), N = logits.size(1), K = experts.size(1);
            const bool both = !sigmoid && xs.scalar_type() == at::kBFloat16 && task_should_compute_output(0) && task_should_compute_output(1) &&
                              (!logits_grad.defined() || logits_grad.scalar_type() == logits.scalar_type());
            // (negative for sizes that it does not take: more than 64 experts, no tokens)
            const int64_t ws_bytes = both ? om_router_softmax_bwd_workspace_bytes(T, xs.size(1), N) : -1;
            if (ws_bytes > 0) return softmax_backward(c, xs, ws, logits, experts, weights_grad, logits_grad, x_grad, ws_bytes);
            dlogits = make(logits.sizes(), logits);
            if (sigmoid) {
                weights_grad = weights_grad.contiguous().to(at::kFloat);
                OM(c, om_route_sigmoid_topk_bwd, fp(logits), experts.data_ptr<int64_t>(), fp(weights_grad), T, N, K, renorm,
                   scale, fpm(dlogits), c.stream);
            } else {
                weights_grad = weights_grad.contiguous();
                OM(c, om_route_softmax_topk_bwd, ptr(logits), dtype_code(logits), experts.data_ptr<int64_t>(),
                   ptr(weights_grad), dtype_code(weights_grad), T, N, K, renorm, ptr(dlogits), c.stream);
            }
            if (logits_grad.defined()) dlogits = dlogits.add(logits_grad);
        }
        auto d = gate_backward(c, xs, ws, dlogits, task_should_compute_output(0), task_should_compute_output(1), x_grad);
        return {d.first, d.second};
    }
    // Both gradients of the gate behind a softmax router in one call.
    variable_list softmax_backward(const Call &c, const Tensor &x, const Tensor &weight, const Tensor &logits, const Tensor &experts,
                                   Tensor weights_grad, Tensor logits_grad, Tensor x_grad, int64_t ws_bytes) const {
        const int64_t T = x.size(0), H = x.size(1), N = weight.size(0), K = experts.size(1);
        weights_grad = weights_grad.contiguous();
        if (logits_grad.defined()) logits_grad = logits_grad.contiguous();
        if (x_grad.defined()) {
            x_grad = x_grad.contiguous();
            require_bf16(x_grad);
        }
        Tensor ws = make({ws_bytes}, x, at::kByte), dx = make(x.sizes(), x), dw = make(weight.sizes(), weight);
        OM(c, om_router_softmax_bwd, ptr(x), ptr(weight), ptr(logits), dtype_code(logits), experts.data_ptr<int64_t>(),
           ptr(weights_grad), dtype_code(weights_grad), ptr(logits_grad), ptr(x_grad), ptr(dx), ptr(dw), dtype_code(dw), T, H, N, K,
           renorm, ptr(ws), ws_bytes, c.stream);
        return {dx, dw};
    }
};

// x as an output: a view of it made where autograd sees views, so that it shares x's version counter (an
// in-place change of either between forward and backward is noticed by whatever saved the other).
Tensor pass_through(const Tensor &x) {
    at::NoGradGuard no_grad;
    return x.view_as(x);
}

void set_outputs(const std::shared_ptr<RouterNode> &node, Tensor *logits, Tensor *weights, Tensor &x) {
    int at = 0;
    if (weights) { node->out_weights = at++; torch::autograd::set_history(*weights, node); }
    if (logits) { node->out_logits = at++; torch::autograd::set_history(*logits, node); }
    // (an in-place change of a view that is one of several outputs would bypass the node: refused by autograd)
    if (auto *view = torch::autograd::impl::get_view_autograd_meta(x); view && view->has_bw_view())
        view->set_creation_meta(torch::autograd::CreationMeta::MULTI_OUTPUT_NODE);
    node->out_x = at++;
    torch::autograd::set_history(x, node);
}

std::shared_ptr<RouterNode> router_node(const Tensor &x, const Tensor &weight) {
    auto node = make_node<RouterNode>({x, weight});
    node->save(x);
    node->save(weight);
    return node;
}

// (logits float32, x)
std::tuple<Tensor, Tensor> gate_logits(const Tensor &x, const Tensor &weight) {
    refuse_transforms({x, weight});
    require_gate_operands(x, weight);
    Tensor logits;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        logits = gate_logits_forward(begin_call(), x, weight);
    }
    Tensor x_out = pass_through(x);
    if (any_requires_grad({x, weight})) {
        auto node = router_node(x, weight);
        set_outputs(node, &logits, nullptr, x_out);
    }
    return {logits, x_out};
}

Tensor route_workspace(const Tensor &x, int64_t T, int64_t H, int64_t N) {
    const int64_t bytes = om_router_gate_route_workspace_bytes(T, H, N);
    if (bytes < 0) check(static_cast<int>(bytes), "om_router_gate_route_workspace_bytes");
    return make({std::max<int64_t>(bytes, 16)}, x, at::kByte);
}

// softmax top-K router -> (routing_weights, selected_experts int64, logits, x).  `one_pass`: one launch for
// projection and routing (shapes of om_router_gate_softmax_topk).  `bf16_logits`: the logits are rounded
// to bf16 before the softmax, as a bf16 linear layer returns them.
// start, end (end > start): the experts that the selections are to be sorted by, where the router's launch can do that too; the
// fifth result is then moe_experts' `index`, else undefined.
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> route_softmax(const Tensor &x, const Tensor &weight, int64_t top_k, bool renorm,
                                                                 at::ScalarType out_dtype, bool one_pass, bool bf16_logits,
                                                                 int64_t start, int64_t end) {
    refuse_transforms({x, weight});
    require_gate_operands(x, weight);
    const int64_t T = x.size(0), N = weight.size(0), H = weight.size(1);
    // Few tokens: one CU would take in all of the gate weight, the projection split over the chip and a launch behind it
    // are sooner; with many selections it depends (om_router_gate_split_softmax_topk, which has the figures and decides).
    if (one_pass && N <= 64 && H % 512 == 0 && (top_k > 16 || (T <= 512 && H >= 1024))) one_pass = false;
    Tensor logits, weights, experts, index;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const Call c = begin_call();
        require_device(x);
        require_device(weight);
        weights = make({T, top_k}, x, out_dtype);
        experts = make({T, top_k}, x, at::kLong);
        if (x.scalar_type() == at::kFloat && N <= 64) {
            logits = make({T, N}, x, at::kFloat);
            OM(c, om_router_gate_softmax_topk_f32, fp(x), fp(weight), T, H, N, top_k, renorm, fpm(logits), ptr(weights),
               dtype_code(weights), experts.data_ptr<int64_t>(), c.stream);
        } else if (x.scalar_type() == at::kFloat) {
            logits = gate_logits_forward(c, x, weight);
            OM(c, om_route_softmax_topk, ptr(logits), dtype_code(logits), T, N, top_k, renorm, ptr(weights),
               dtype_code(weights), experts.data_ptr<int64_t>(), c.stream);
        } else if (one_pass) {
            logits = make({T, N}, x, at::kFloat);
            OM(c, om_router_gate_softmax_topk, ptr(x), ptr(weight), T, H, N, top_k, renorm, fpm(logits), ptr(weights),
               dtype_code(weights), experts.data_ptr<int64_t>(), c.stream);
        } else {
            require_gate_shape(weight, "gate projection");
            logits = make({T, N}, x, bf16_logits ? at::kBFloat16 : at::kFloat);
            const Tensor ws = route_workspace(x, T, H, N);
            if (end > start && om_router_gate_softmax_topk_sort_fits(T, static_cast<int>(H), static_cast<int>(N), static_cast<int>(top_k))) {
                const Index ix = one_buffer_index(T, top_k, end - start, Tensor(), x);
                index = ix.owners[0];
                OM(c, om_router_gate_softmax_topk_sort, ptr(x), ptr(weight), T, H, N, top_k, renorm, ptr(logits), dtype_code(logits),
                   ptr(weights), dtype_code(weights), experts.data_ptr<int64_t>(), start, end, rwp(ix.cum), rwp(ix.cum_ep), rwp(ix.in),
                   rwp(ix.out), rwp(ix.sel), rwp(ix.row_weights), ptr(ws), ws.numel(), c.stream);
            } else
                OM(c, om_router_gate_split_softmax_topk, ptr(x), ptr(weight), T, H, N, top_k, renorm, ptr(logits),
               dtype_code(logits), ptr(weights), dtype_code(weights), experts.data_ptr<int64_t>(), ptr(ws), ws.numel(), c.stream);
        }
    }
    Tensor x_out = pass_through(x);
    if (any_requires_grad({x, weight})) {
        auto node = router_node(x, weight);
        // (a detached alias: saving an output itself would tie the node to itself)
        node->save(logits.detach());
        node->save(experts);
        node->renorm = renorm;
        set_outputs(node, &logits, &weights, x_out);
    }
    return {weights, experts, logits, x_out, index};
}

// sigmoid / group-limited router -> (selected_experts int64, routing_weights float32, x)
std::tuple<Tensor, Tensor, Tensor> route_sigmoid(const Tensor &x, const Tensor &weight, const Tensor &bias, int64_t n_group,
                                                 int64_t topk_group, int64_t top_k, bool renorm, double scale) {
    refuse_transforms({x, weight, bias});
    require_gate_operands(x, weight);
    const int64_t T = x.size(0), N = weight.size(0);
    TORCH_CHECK_TYPE(bias.scalar_type() == at::kFloat || bias.scalar_type() == at::kBFloat16,
                     "router bias must be float32 or bfloat16 (got ", bias.scalar_type(), ")");
    if (bias.numel() != N) throw NativeError("router bias: expected one value per expert");
    Tensor logits, weights, experts;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const Call c = begin_call();
        require_device(bias);
        require_device(x);
        require_device(weight);
        weights = make({T, top_k}, x, at::kFloat);
        experts = make({T, top_k}, x, at::kLong);
        if (x.scalar_type() == at::kFloat) {
            logits = gate_logits_forward(c, x, weight);
            const Tensor bias_f32 = bias.to(at::kFloat);
            OM(c, om_route_sigmoid_group_topk, fp(logits), fp(bias_f32), T, N, n_group, topk_group, top_k, renorm, scale,
               experts.data_ptr<int64_t>(), fpm(weights), c.stream);
        } else {
            require_gate_shape(weight, "gate projection");
            logits = make({T, N}, x, at::kFloat);
            const Tensor ws = route_workspace(x, T, x.size(1), N);
            OM(c, om_router_gate_split_sigmoid_group_topk_bias, ptr(x), ptr(weight), ptr(bias), dtype_code(bias), T, x.size(1), N, n_group, topk_group,
               top_k, renorm, scale, fpm(logits), experts.data_ptr<int64_t>(), fpm(weights), ptr(ws), ws.numel(), c.stream);
        }
    }
    Tensor x_out = pass_through(x);
    if (any_requires_grad({x, weight})) {
        auto node = router_node(x, weight);
        node->save(logits);
        node->save(experts);
        node->renorm = renorm;
        node->sigmoid = true;
        node->scale = scale;
        set_outputs(node, nullptr, &weights, x_out);
    }
    return {experts, weights, x_out};
}

// ---- expert nodes -------------------------------------------------------------------------------------

// The expert half of a bf16 block (see routed_forward), with an optional residual or shared expert.
// Inputs in order: hidden_states, routing_weights, residual, routed leaves, shared leaves.
struct RoutedNode : HostNode {
    Index ix;                        // (without its arrays)
    ExpertWeights routed, shared;
    bool has_residual = false, has_shared = false;
    std::string name() const override { return "OptimusRoutedExpertsBackward"; }
    variable_list run(variable_list &&grads) override {
        const size_t n_in = 3 + routed.n_leaves + shared.n_leaves;
        if (!grads[0].defined()) return variable_list(n_in);
        // x, rw, row_weights, g, u, h [, shared g, u, h, cum], the index arrays' owners, the weights [, the shared ones]
        const std::vector<Tensor> kept = saved();
        at::AutoDispatchBelowADInplaceOrView below;
        const Call c = begin_call();
        const Tensor dfinal = grads[0].contiguous();
        const MlpWeights w = weights(routed, kept), ws = has_shared ? weights(shared, kept) : MlpWeights();
        const MlpState s{Tensor(), kept[3], kept[4], kept[5]};
        size_t at = 6;
        MlpState ss;
        if (has_shared) {
            ss = {kept[9], kept[6], kept[7], kept[8]};
            at = 10;
        }
        Index index = ix;
        index.owners.assign(kept.begin() + at, kept.begin() + routed.at);
        index.resolve();
        Tensor base;
        Sinks ks;
        Alongside along{ws, ss, Tensor()};
        const bool together = has_shared && index.rows > 0 && Alongside::rides(ws, w, index.to_choose_by(), dfinal.size(0), OM_DENSE_DOWN_DGRAD | OM_DENSE_GATE_UP_DGRAD);
        if (has_shared) {   // first: its input gradient is the base of the routed experts' per-token sum
            ks = sinks_of(c, shared, ws);
            if (!together) base = merged_backward(c, dfinal, kept[0], ws, iptr(ss.cum), ss, nullptr, ks);
        }
        const Sinks k = sinks_of(c, routed, w);
        auto d = routed_backward(c, dfinal, kept[0], kept[1], index, w, s, kept[2], k, base, together ? &along : nullptr, &ks);
        variable_list out = {d.first, d.second, has_residual ? grads[0] : Tensor()};
        out.reserve(n_in);
        push_grads(out, k, routed);
        if (has_shared) push_grads(out, ks, shared);
        return out;
    }
};

Tensor routed_experts(const Call &c, Tensor x, Tensor rw, Index ix, const Tensor &residual_in, bool merged,
                      const std::vector<Tensor> &leaves, bool has_shared, const Tensor &one,
                      const std::function<void(Index &)> &after_shared = nullptr) {
    variable_list inputs = {x, rw, residual_in};
    inputs.insert(inputs.end(), leaves.begin(), leaves.end());
    const at::ArrayRef<Tensor> all(leaves);
    const at::ArrayRef<Tensor> routed = all.slice(0, leaves.size() - (has_shared ? 3 : 0)), shared = all.slice(routed.size());
    const int64_t G = merged ? leaves[0].size(0) : static_cast<int64_t>(routed.size() / 3);
    MlpWeights w, ws;
    MlpState s, ss;
    Tensor row_weights, final, xc, rwc;
    const bool keep = any_requires_grad(inputs);
    {
        at::AutoDispatchBelowADInplaceOrView below;
        w = weights_of(routed, merged, G);
        xc = x.contiguous();
        rwc = rw.contiguous();
        Tensor residual = residual_in.defined() ? residual_in.contiguous() : Tensor();
        Alongside along{ws, ss, Tensor()};
        bool together = false;
        if (has_shared) {
            ws = weights_of(shared, true, 1);
            // (the host waits for the rows behind the shared expert's kernels, where it has to)
            together = !after_shared && Alongside::rides(ws, w, ix.to_choose_by(), xc.size(0), OM_DENSE_GATE_UP | OM_DENSE_DOWN);
            if (together) require_shared_operands(xc, ws, one, ss);
            else residual = merged_forward(c, xc, ws, iptr(one), nullptr, xc.size(0), ss, keep);
        }
        if (after_shared) after_shared(ix);
        final = routed_forward(c, xc, rwc, ix, w, residual, s, row_weights, together ? &along : nullptr, keep);
    }
    if (keep) {
        auto node = make_node<RoutedNode>(inputs);
        node->vars.reserve(21);
        node->save(xc.is_same(x) ? x : xc);
        node->save(rwc.is_same(rw) ? rw : rwc);
        for (const Tensor &t : {row_weights, s.g, s.u, s.h}) node->save(t);
        if (has_shared)
            for (const Tensor &t : {ss.g, ss.u, ss.h, one}) node->save(t);
        for (const Tensor &t : ix.owners) node->save(t);
        node->routed = node->save_weights(routed, merged, w);
        if (has_shared) node->shared = node->save_weights(shared, true, ws);
        node->ix = ix.without_arrays();
        node->has_residual = residual_in.defined();
        node->has_shared = has_shared;
        torch::autograd::set_history(final, node);
    }
    return final;
}

// The kernels of RoutedMLPFunction / RoutedAndSharedMLPFunction, for the Python autograd functions: index arrays
// that the caller has built, weights as [G, out, in] tensors or views.
Index caller_index(const Tensor &x, const Tensor &in, const Tensor &cum_ep, const Tensor &out, const Tensor &sel, Tensor cum,
                   bool bound) {
    for (const Tensor *t : {&in, &cum_ep, &out, &sel}) require_device(*t);
    if (!cum.is_cuda()) cum = cum.to(x.device(), /*non_blocking=*/true);
    Index ix;
    ix.owners = {cum.to(at::kInt).contiguous(), cum_ep, in, out, sel};
    ix.resolve();
    ix.rows = in.size(0);
    ix.bound = bound;
    return ix;
}
// -> final, cum, row_weights, g, u, h
std::vector<Tensor> routed_mlp_forward(const Tensor &x, const Tensor &rw, const Tensor &in, const Tensor &cum_ep,
                                       const Tensor &out, const Tensor &sel, const Tensor &cum,
                                       const std::optional<Tensor> &residual, const std::vector<Tensor> &w) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Index ix = caller_index(x, in, cum_ep, out, sel, cum, false);
    MlpState s;
    Tensor row_weights;
    const Tensor res = residual ? residual->contiguous() : Tensor();
    Tensor final = routed_forward(begin_call(), x, rw, ix, weights_of(w, true, 0), res, s, row_weights);
    return {final, ix.owners[0], row_weights, s.g, s.u, s.h};
}
// -> dx, d routing_weights, the gradients of the leaves (undefined: added into a live buffer)
variable_list routed_mlp_backward(const Tensor &dfinal, const Tensor &x, const Tensor &rw, const Tensor &in,
                                  const Tensor &cum_ep, const Tensor &out, const Tensor &sel, const Tensor &cum,
                                  const Tensor &row_weights, const Tensor &g, const Tensor &u, const Tensor &h,
                                  const std::vector<Tensor> &w, const std::vector<Tensor> &leaves, bool merged, bool bound,
                                  const std::optional<Tensor> &base) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Call c = begin_call();
    const ExpertWeights e = ExpertWeights::of(leaves, merged);
    const MlpWeights mw = weights_of(w, true, 0);
    const Sinks k = sinks_of(c, e, mw);
    auto d = routed_backward(c, dfinal.contiguous(), x, rw, caller_index(x, in, cum_ep, out, sel, cum, bound), mw,
                             {Tensor(), g, u, h}, row_weights, k, base.value_or(Tensor()));
    variable_list grads = {d.first, d.second};
    push_grads(grads, k, e);
    return grads;
}

// Activations of the expert MLP sized by the upper bound T*K instead of the routed rows of an expert window cost
// expert_parallelism times their memory, and save the host the wait for the count.  What the wait costs, whole
// passes, us, count read -> bound: forward of 1024/256 experts 64 tokens 89.6 -> 82.5, 1000 tokens 109 -> 104, of
// 7168/2048 16 tokens 255 -> 254, 512 tokens 583 -> 576; training steps of 1024/256 16 tokens 412 -> 402, of 7168/2048
// 64 tokens 2435 -> 2432.
// Without gradients the memory lives for the call only: 64 MB, 0.02 % of the card.  Where a backward follows every
// layer keeps it, so there the limit is also a 32nd of the layer's own expert weights: whatever the depth of a model,
// at most 3 % of what its weights take.
constexpr int64_t BOUND_ROWS_BYTES = 64 << 20, BOUND_ROWS_WEIGHTS = 32;
bool sized_by_bound(int64_t rows, int64_t G, int64_t I, int64_t H, bool needs_grad) {
    const int64_t activations = rows * (3 * I + H) * 2, weights = 3 * G * I * H * 2;
    return activations <= BOUND_ROWS_BYTES && (!needs_grad || activations <= weights / BOUND_ROWS_WEIGHTS);
}

// One device integer on its way to the host.
struct CountReadback {
    Tensor value = at::empty({1}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    hipEvent_t copied = nullptr;
    CountReadback(const int32_t *device, void *stream) {
        hipStream_t st = static_cast<hipStream_t>(stream);
        if (hipEventCreateWithFlags(&copied, hipEventDisableTiming) != hipSuccess ||
            hipMemcpyAsync(value.data_ptr(), device, 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipEventRecord(copied, st) != hipSuccess)
            throw NativeError("reading the routed row count back failed");
    }
    CountReadback(const CountReadback &) = delete;
    int64_t wait() {
        if (hipEventSynchronize(copied) != hipSuccess) throw NativeError("reading the routed row count back failed");
        return value.data_ptr<int32_t>()[0];
    }
    ~CountReadback() {
        if (copied) {
            (void)hipEventSynchronize(copied);   // the pinned word may be handed out again
            (void)hipEventDestroy(copied);
        }
    }
};

// Whether the host waits for the row count ahead of the shared expert's kernels: where they are those of the routed experts and,
// alone, too few for the chip (fewer tiles than three quarters of its CUs) that saves more than the wait costs.  Forward passes, us, behind
// them -> together: 7168/2048 of 600 tokens (160 tiles) 566 -> 516, 3000/1000 of 1000 (128) 248 -> 234; but 1200/1000 of 3000 (384)
// 187 -> 191, 1024/256 of 8000 (252) 146 -> 155.
bool waits_ahead_of_shared(int64_t expected, int64_t G, int64_t I, int64_t H, int64_t tokens, const std::vector<Tensor> &shared) {
    int device = 0, cus = 0;
    if (hipGetDevice(&device) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1)
        cus = 256;
    at::AutoDispatchBelowADInplaceOrView below;
    const int64_t tiles = (tokens + 127) / 128 * ((I + 63) / 64);
    return tiles * 4 < cus * 3 && Alongside::fits(weights_of(shared, true, 1), I, H) &&
           om_merged_mlp_dense_rides(expected, static_cast<int>(G), static_cast<int>(I), static_cast<int>(H), tokens) == 1;
}

// Sort (with the routing weights laid out per sorted row) and experts in one call: hidden_states [T,H], the experts [start, end) of n_total.
// sync_free: never read the routed-row count of an expert window back (else up to a limit: sized_by_bound).  `sorted`: the index that
// route_softmax made of these selections and weights.
Tensor moe_experts(const Tensor &x, Tensor rw, const Tensor &experts, int64_t start, int64_t end, int64_t n_total,
                   bool sync_free, const std::optional<Tensor> &residual, bool merged, const std::vector<Tensor> &leaves,
                   bool has_shared, const std::optional<Tensor> &one, const std::optional<Tensor> &sorted) {
    refuse_transforms({x, rw, residual.value_or(Tensor())});
    refuse_transforms(leaves);
    if (experts.dim() != 2 || x.dim() != 2 || experts.size(0) != x.size(0) || rw.sizes() != experts.sizes())
        throw NativeError("expected hidden states [tokens, hidden], and routing weights and expert indices [tokens, top_k]");
    const Call c = begin_call();
    Index ix;
    rw = rw.contiguous();
    {
        at::AutoDispatchBelowADInplaceOrView below;
        ProfiledScope scope(c, "1moeblock--3index_calculation");
        if (sorted) {
            if (sorted->scalar_type() != at::kInt || sorted->numel() != index_words(x.size(0), experts.size(1), end - start))
                throw NativeError("expert MLP: the sorted index is of other sizes");
            require_device(*sorted);
            ix = one_buffer_index(x.size(0), experts.size(1), end - start, *sorted);
        } else {
            ix = sort_index(c, experts, start, end, rw);
        }
    }
    const bool windowed = !(start == 0 && end == n_total);
    if (windowed) {
        const int64_t I = leaves[0].size(-2), H = x.size(1);
        const Tensor res = residual.value_or(Tensor());
        if (sync_free || sized_by_bound(ix.rows, end - start, I, H, any_requires_grad({x, rw, res}) || any_requires_grad(leaves))) {
            ix.bound = true;
            // the kernels are chosen by the window's share of the pairs, not by all of them
            ix.expected = std::max<int64_t>(1, ix.rows * (end - start) / n_total);
            ix.expected = std::min(ix.expected, ix.rows);
        } else {
            // read the count back (as the reference does), behind the shared expert's kernels: they do not
            // need it, and while the GPU runs them the host waits for a copy that was enqueued before them
            auto count = std::make_shared<CountReadback>(ix.cum + (end - start), c.stream);
            if (has_shared && one && waits_ahead_of_shared(ix.rows * (end - start) / n_total, end - start, I, H, x.size(0),
                                                           std::vector<Tensor>(leaves.end() - 3, leaves.end()))) {
                ix.rows = count->wait();
                return routed_experts(c, x, rw, ix, residual.value_or(Tensor()), merged, leaves, has_shared, *one);
            }
            return routed_experts(c, x, rw, ix, residual.value_or(Tensor()), merged, leaves, has_shared,
                                  one.value_or(Tensor()), [count](Index &index) { index.rows = count->wait(); });
        }
    }
    return routed_experts(c, x, rw, ix, residual.value_or(Tensor()), merged, leaves, has_shared, one.value_or(Tensor()));
}

// Gradients of the expert MLPs without routing weights: dx, then the leaves'.  `x_rows` (with the two arrays
// of the per-token sum): the MLPs read x through it.
variable_list merged_mlp_grads(const Call &c, const Tensor &dy, const Tensor &x, const MlpWeights &w, const MlpState &s,
                               const Tensor &x_rows, const Tensor &cum_ep, const Tensor &out_rows, const ExpertWeights &e) {
    const Sinks k = sinks_of(c, e, w);
    Tensor dx = merged_backward(c, dy, x, w, iptr(s.cum), s, iptr(x_rows), k);
    if (x_rows.defined()) {
        ProfiledScope scope(c, "1moeblock--6gmlp_input_prep_bwd");
        Tensor sum = make(x.sizes(), x);
        OM(c, om_shuffle_sub_matrix_reduce, ptr(dx), iptr(cum_ep), iptr(out_rows), ptr(sum), x.size(0), x.size(1),
           dtype_code(x), c.stream);
        dx = sum;
    }
    variable_list grads = {dx};
    grads.reserve(1 + e.n_leaves);
    push_grads(grads, k, e);
    return grads;
}

// Inputs in order: x, leaves.
struct MergedNode : HostNode {
    ExpertWeights experts;
    std::string name() const override { return "OptimusExpertMlpBackward"; }
    variable_list run(variable_list &&grads) override {
        if (!grads[0].defined()) return variable_list(1 + experts.n_leaves);
        // x, cum, g, u, h, the gathered forms' index arrays (x_rows, cum_ep, out_rows), the weights
        const std::vector<Tensor> kept = saved();
        at::AutoDispatchBelowADInplaceOrView below;
        return merged_mlp_grads(begin_call(), grads[0], kept[0], weights(experts, kept), {kept[1], kept[2], kept[3], kept[4]},
                                kept[5], kept[6], kept[7], experts);
    }
};

// (y, cum, g, u, h) of the expert MLPs; `x_rows`: they read x through it
std::vector<Tensor> merged_mlp_state(const Tensor &x, Tensor cum, const MlpWeights &w, const Tensor &x_rows) {
    require_mlp_operands(x, w);
    const Call c = begin_call();
    MlpState s;
    require_device(x);
    require_device(x_rows);
    if (!cum.is_cuda()) cum = cum.to(x.device(), /*non_blocking=*/true);
    s.cum = cum.to(at::kInt).contiguous();
    Tensor y = merged_forward(c, x, w, iptr(s.cum), iptr(x_rows), x_rows.defined() ? x_rows.size(0) : x.size(0), s);
    return {y, s.cum, s.g, s.u, s.h};
}

// The kernels of MergedMLPFunction, GroupMLPFunction and their gathered forms, for the Python autograd functions.
std::vector<Tensor> merged_mlp_forward(const Tensor &x, const Tensor &cum, const std::vector<Tensor> &w,
                                       const std::optional<Tensor> &x_rows) {
    at::AutoDispatchBelowADInplaceOrView below;
    return merged_mlp_state(x, cum, weights_of(w, true, 0), x_rows.value_or(Tensor()));
}
variable_list merged_mlp_backward(const Tensor &dy, const Tensor &x, const Tensor &cum, const Tensor &g, const Tensor &u,
                                  const Tensor &h, const std::vector<Tensor> &w, const std::vector<Tensor> &leaves, bool merged,
                                  const std::optional<Tensor> &x_rows, const std::optional<Tensor> &cum_ep,
                                  const std::optional<Tensor> &out_rows) {
    at::AutoDispatchBelowADInplaceOrView below;
    for (const auto *t : {&cum_ep, &out_rows}) require_device(t->value_or(Tensor()));
    return merged_mlp_grads(begin_call(), dy, x, weights_of(w, true, 0), {cum, g, u, h}, x_rows.value_or(Tensor()),
                            cum_ep.value_or(Tensor()), out_rows.value_or(Tensor()), ExpertWeights::of(leaves, merged));
}

// The expert MLPs without routing weights as one autograd node.
Tensor merged_mlp(const Tensor &x, const Tensor &cum, bool merged, const std::vector<Tensor> &leaves,
                  const std::optional<Tensor> &x_rows, const std::optional<Tensor> &cum_ep,
                  const std::optional<Tensor> &out_rows) {
    variable_list inputs = {x};
    inputs.insert(inputs.end(), leaves.begin(), leaves.end());
    refuse_transforms(inputs);
    MlpWeights w;
    std::vector<Tensor> state;
    Tensor xc = x;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        if (x_rows) xc = x.contiguous();
        for (const auto *t : {&cum_ep, &out_rows}) require_device(t->value_or(Tensor()));
        w = weights_of(leaves, merged, static_cast<int64_t>(leaves.size() / 3));
        state = merged_mlp_state(xc, cum, w, x_rows.value_or(Tensor()));
    }
    Tensor y = state[0];
    if (any_requires_grad(inputs)) {
        auto node = make_node<MergedNode>(inputs);
        node->vars.reserve(11);
        node->save(xc.is_same(x) ? x : xc);
        for (size_t i = 1; i < state.size(); i++) node->save(state[i]);
        for (const auto *t : {&x_rows, &cum_ep, &out_rows}) node->save(t->value_or(Tensor()));
        node->experts = node->save_weights(leaves, merged, w);
        torch::autograd::set_history(y, node);
    }
    return y;
}

// K6 (GroupGemmOutputReduction[Residual]Function): final[t] = (residual[t] +) sum_k w[t,k] y[pos(t,k)].
std::pair<Tensor, Tensor> combine_backward(const Tensor &dfinal_in, const Tensor &y, const Tensor &rw, const Tensor &sel,
                                           const Tensor &in, const Tensor &out) {
    at::AutoDispatchBelowADInplaceOrView below;
    const Call c = begin_call();
    const Tensor dfinal = dfinal_in.contiguous();
    Tensor dy = make(y.sizes(), y);
    // the kernel writes the entry of every routed (token, k) pair; pairs outside the expert window
    // stay zero (the reference pre-zeroes the whole tensor, moe.py:336)
    Tensor drw = out.size(0) == rw.numel() ? make(rw.sizes(), rw) : at::zeros(rw.sizes(), rw.options());
    ProfiledScope scope(c, "1moeblock--8gmlp_output_reduction_bwd");
    OM(c, om_reduce_ggemm_output_backward, ptr(dfinal), ptr(y), ptr(rw), iptr(sel), iptr(in), iptr(out), ptr(dy), ptr(drw),
       out.size(0), rw.size(1), dfinal.size(1), dtype_code(y), dtype_code(rw), c.stream);
    return {dy, drw};
}

struct CombineNode : HostNode {      // saves y, rw, sel, in, out
    bool has_residual = false;
    std::string name() const override { return "OptimusCombineBackward"; }
    variable_list run(variable_list &&grads) override {
        if (!grads[0].defined()) return variable_list(3);
        const std::vector<Tensor> kept = saved();
        auto d = combine_backward(grads[0], kept[0], kept[1], kept[2], kept[3], kept[4]);
        return {d.first, d.second, has_residual ? grads[0] : Tensor()};
    }
};

Tensor combine(const Tensor &y, const Tensor &rw_in, const Tensor &cum_ep, const Tensor &sel, const Tensor &in,
               const Tensor &out, const std::optional<Tensor> &residual) {
    refuse_transforms({y, rw_in, residual.value_or(Tensor())});
    if (y.dim() != 2 || rw_in.dim() != 2 || cum_ep.numel() != rw_in.size(0) + 1)
        throw NativeError("combine: expected expert outputs [rows, hidden], routing weights [tokens, top_k], tokens + 1 offsets");
    if (residual) {
        if (residual->sizes() != at::IntArrayRef({rw_in.size(0), y.size(1)})) throw NativeError("combine: expected a residual [tokens, hidden]");
        TORCH_CHECK_TYPE(residual->scalar_type() == y.scalar_type(), "combine: the residual must have the expert outputs' type");
    }
    Tensor final, rw = rw_in;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const Call c = begin_call();
        rw = rw_in.contiguous();
        for (const Tensor *t : std::initializer_list<const Tensor *>{&y, &rw, &cum_ep, &sel, &in, &out}) require_device(*t);
        const int64_t T = rw.size(0), K = rw.size(1), H = y.size(1);
        ProfiledScope scope(c, "1moeblock--8gmlp_output_reduction_fwd");
        final = make({T, H}, y);
        if (residual) {
            const Tensor res = residual->contiguous();
            require_device(res);
            OM(c, om_reduce_ggemm_output_residual, ptr(y), ptr(rw), iptr(cum_ep), iptr(sel), iptr(out), ptr(res), ptr(final),
               T, K, H, dtype_code(y), dtype_code(rw), c.stream);
        } else {
            OM(c, om_reduce_ggemm_output, ptr(y), ptr(rw), iptr(cum_ep), iptr(sel), iptr(out), ptr(final), T, K, H,
               dtype_code(y), dtype_code(rw), 0, c.stream);
        }
    }
    if (any_requires_grad({y, rw_in, residual.value_or(Tensor())})) {
        auto node = make_node<CombineNode>({y, rw_in, residual.value_or(Tensor())});
        node->save(y);
        node->save(rw.is_same(rw_in) ? rw_in : rw);
        for (const Tensor &t : {sel, in, out}) node->save(t);
        node->has_residual = residual.has_value();
        torch::autograd::set_history(final, node);
    }
    return final;
}

// ---- optimizer ----------------------------------------------------------------------------------------
// A step of a small optimizer is two launches of 7 to 10 us; through ctypes, with the operands looked over in Python, they
// took the host 29 us (19 now).

bool flat_buffer(const Tensor &t, int64_t n) { return t.is_cuda() && t.is_contiguous() && t.numel() == n; }

// The update of adamw_step_; false: operands that its Python part refuses (it raises).
bool adamw_step(const Tensor &param, const Tensor &grad, const Tensor &master, const Tensor &exp_avg, const Tensor &exp_avg_sq,
                int64_t step, double lr, double beta1, double beta2, double eps, double weight_decay,
                const std::optional<Tensor> &grad_scale, bool store_scaled_grad) {
    const int64_t n = master.numel();
    for (const Tensor *t : {&param, &grad, &master, &exp_avg, &exp_avg_sq})
        if (!flat_buffer(*t, n)) return false;
    for (const Tensor *t : {&master, &exp_avg, &exp_avg_sq})
        if (t->scalar_type() != at::kFloat) return false;
    const auto dt = param.scalar_type();
    if (grad.scalar_type() != dt || (dt != at::kBFloat16 && (dt != at::kFloat || param.data_ptr() != master.data_ptr()))) return false;
    if (grad_scale && (!flat_buffer(*grad_scale, 1) || grad_scale->scalar_type() != at::kFloat)) return false;
    const Call c = begin_call();
    if (grad_scale)
        OM(c, om_adamw_step_clipped, ptr(param), ptr(grad), fpm(master), fpm(exp_avg), fpm(exp_avg_sq), n, lr, beta1, beta2, eps,
           weight_decay, step, dtype_code(param), fp(*grad_scale), store_scaled_grad, c.stream);
    else
        OM(c, om_adamw_step, ptr(param), ptr(grad), fpm(master), fpm(exp_avg), fpm(exp_avg_sq), n, lr, beta1, beta2, eps,
           weight_decay, step, dtype_code(param), c.stream);
    return true;
}

// GradNormPlan's one-launch form; words: total norm, clip coefficient, the kernel's block count.
void grad_norm(const Tensor &grad, const Tensor &chunk_offsets, int64_t n_chunks, const Tensor &seg_first_chunk, int64_t n_segs,
               double max_norm, const Tensor &partials, const Tensor &seg_norms, const Tensor &words,
               const std::optional<Tensor> &norm_out) {
    require_device(grad);
    const Call c = begin_call();
    float *w = fpm(words);
    OM(c, om_grad_norm, ptr(grad), dtype_code(grad), chunk_offsets.data_ptr<int64_t>(), n_chunks, seg_first_chunk.data_ptr<int64_t>(),
       n_segs, max_norm, fpm(partials), fpm(seg_norms), w, w + 1, norm_out ? ptr(*norm_out) : nullptr,
       reinterpret_cast<unsigned *>(w + 2), c.stream);
}

// ---- Python module ----------------------------------------------------------------------------------

PyObject *module_base() {   // torch.nn.Module (kept for good)
    static PyObject *base = py::object(py::module_::import("torch.nn").attr("Module")).release().ptr();
    return base;
}

// Attributes of nn.Module objects, one name: out of the module's `dictionary` (_parameters or _modules) where that is
// what attribute access would end at, which costs a microsecond each; as an attribute where the class or the object
// has the name itself (a property, a tensor put there) or the class brings its own attribute access.
struct ModuleAttribute {
    PyObject *name, *dictionary;
    PyTypeObject *type = nullptr;   // the last type seen, and whether it leaves the name to the dictionaries
    bool plain = false;
    ModuleAttribute(const char *n, const char *d) : name(PyUnicode_InternFromString(n)), dictionary(PyUnicode_InternFromString(d)) {}
    py::object of(py::handle owner) {
        PyObject *o = owner.ptr();
        if (Py_TYPE(o) != type) {
            type = Py_TYPE(o);
            auto *base = reinterpret_cast<PyTypeObject *>(module_base());
            plain = PyType_IsSubtype(type, base) && !_PyType_Lookup(type, name);
            for (const char *hook : {"__getattr__", "__getattribute__"}) {
                const py::str h(hook);
                plain = plain && _PyType_Lookup(type, h.ptr()) == _PyType_Lookup(base, h.ptr());
            }
        }
        if (plain) {
            PyObject **own = _PyObject_GetDictPtr(o);
            if (own && *own && !PyDict_GetItemWithError(*own, name)) {
                PyObject *d = PyDict_GetItemWithError(*own, dictionary);      // borrowed, as all of these
                PyObject *value = d && PyDict_Check(d) ? PyDict_GetItemWithError(d, name) : nullptr;
                if (value) return py::reinterpret_borrow<py::object>(value);
            }
            if (PyErr_Occurred()) throw py::error_already_set();
        }
        py::object value = py::reinterpret_steal<py::object>(PyObject_GetAttr(o, name));
        if (!value) throw py::error_already_set();
        return value;
    }
};

// The (gate, up, down) weights of a ModuleList of expert MLPs in GroupMLPFunction's order (a DeepSeek-V3 share has 96).
std::vector<Tensor> expert_parameters(py::handle experts) {
    ModuleAttribute projections[3] = {{"gate_proj", "_modules"}, {"up_proj", "_modules"}, {"down_proj", "_modules"}};
    ModuleAttribute weight("weight", "_parameters");
    std::vector<Tensor> out;
    const py::object children = experts.attr("_modules");
    for (auto item : py::cast<py::dict>(children))
        for (ModuleAttribute &projection : projections) out.push_back(weight.of(projection.of(item.second)).cast<Tensor>());
    return out;
}

// The .grad of every parameter of `model` whose id() is not in `owned` and that has one, each parameter
// once.  For a plain nn.Module tree this walks the modules' dictionaries (a step of a small optimizer spent
// 20 us in the generator behind model.parameters()); where anything overrides the traversal, on the model's class,
// on the model itself or on the class of a module inside it, model.parameters() is asked.
bool walk_parameters(PyObject *module, std::unordered_set<PyObject *> &modules, const std::function<void(PyObject *)> &visit) {
    if (!modules.insert(module).second) return true;
    static PyObject *named_modules = PyUnicode_InternFromString("named_modules");
    const py::object ours = py::reinterpret_steal<py::object>(PyObject_GetAttr(reinterpret_cast<PyObject *>(Py_TYPE(module)), named_modules));
    const py::object base = py::reinterpret_steal<py::object>(PyObject_GetAttr(module_base(), named_modules));
    if (!ours || !base) { PyErr_Clear(); return false; }
    if (ours.ptr() != base.ptr()) return false;
    for (const char *name : {"_parameters", "_modules"}) {
        py::object d = py::reinterpret_steal<py::object>(PyObject_GetAttrString(module, name));
        if (!d) throw py::error_already_set();
        PyObject *key, *value;
        Py_ssize_t at = 0;
        if (!PyDict_Check(d.ptr())) return false;
        while (PyDict_Next(d.ptr(), &at, &key, &value)) {
            if (value == Py_None) continue;
            if (name[1] == 'p') visit(value);
            else if (!walk_parameters(value, modules, visit)) return false;
        }
    }
    return true;
}
py::list foreign_grads(py::object model, py::set owned) {
    py::list out;
    std::unordered_set<PyObject *> modules, seen;
    auto visit = [&](PyObject *p) {
        if (!seen.insert(p).second) return;
        py::object id = py::reinterpret_steal<py::object>(PyLong_FromVoidPtr(p));
        if (owned.contains(id)) return;
        py::object grad = py::reinterpret_steal<py::object>(PyObject_GetAttrString(p, "grad"));
        if (!grad) throw py::error_already_set();
        if (!grad.is_none()) out.append(grad);
    };
    const py::handle base(module_base());
    bool plain = py::isinstance(model, base);
    if (plain) {
        const py::dict own = model.attr("__dict__");
        for (const char *name : {"parameters", "named_parameters", "_named_members", "named_modules"})
            plain = plain && !own.contains(name) && py::type::of(model).attr(name).ptr() == base.attr(name).ptr();
    }
    if (plain && walk_parameters(model.ptr(), modules, visit)) return out;
    out = py::list();
    seen.clear();
    for (py::handle p : model.attr("parameters")()) visit(p.ptr());
    return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    py::register_local_exception_translator([](std::exception_ptr p) {
        try {
            if (p) std::rethrow_exception(p);
        } catch (const NativeError &e) {
            PyObject *cls = module_attr("optimus._native", "NativeLibraryError");
            PyErr_SetString(cls, e.what());
            Py_DECREF(cls);
        }
    });
    // These only allocate and launch: other Python threads run meanwhile (the switches are read under the GIL).
    const py::call_guard<py::gil_scoped_release> no_gil;
    m.def("build_token_permutation", [](const Tensor &experts, int64_t start, int64_t end) {
        at::AutoDispatchBelowADInplaceOrView below;
        auto r = sort_tensors(begin_call(), experts, start, end);
        return std::make_tuple(r[0], r[1], r[2], r[3], r[4]);
    }, no_gil);
    m.def("gate_logits", &gate_logits, no_gil);
    m.def("gate_weight_grad", [](const Tensor &x, const Tensor &w, const Tensor &dlogits) {
        return gate_weight_grad(begin_call(), x, w, dlogits);
    }, no_gil);
    m.def("gate_input_grad", [](const Tensor &w, const Tensor &dlogits, const std::optional<Tensor> &other) {
        return gate_input_grad(begin_call(), w, dlogits, other.value_or(Tensor()));
    }, no_gil);
    m.def("gate_backward", [](const Tensor &x, const Tensor &w, const Tensor &dlogits, bool need_x, bool need_w,
                              const std::optional<Tensor> &other) {
        return gate_backward(begin_call(), x, w, dlogits, need_x, need_w, other.value_or(Tensor()));
    }, no_gil);
    m.def("route_softmax", [](const Tensor &x, const Tensor &w, int64_t top_k, bool renorm, py::object dtype, bool fused,
                              bool bf16_logits) {
        const at::ScalarType dt = torch::python::detail::py_object_to_dtype(dtype);
        py::gil_scoped_release nogil;
        auto r = route_softmax(x, w, top_k, renorm, dt, fused, bf16_logits, 0, 0);
        return std::make_tuple(std::get<0>(r), std::get<1>(r), std::get<2>(r), std::get<3>(r));
    });
    // with the index for moe_experts of the experts [start, end), or None
    m.def("route_softmax_sorted", [](const Tensor &x, const Tensor &w, int64_t top_k, bool renorm, py::object dtype, bool fused,
                                     bool bf16_logits, int64_t start, int64_t end) {
        const at::ScalarType dt = torch::python::detail::py_object_to_dtype(dtype);
        py::gil_scoped_release nogil;
        auto r = route_softmax(x, w, top_k, renorm, dt, fused, bf16_logits, start, end);
        return std::make_tuple(std::get<0>(r), std::get<1>(r), std::get<2>(r), std::get<3>(r),
                               std::get<4>(r).defined() ? std::optional<Tensor>(std::get<4>(r)) : std::nullopt);
    });
    m.def("route_sigmoid", &route_sigmoid, no_gil);
    m.def("routed_mlp_forward", &routed_mlp_forward, no_gil);
    m.def("routed_mlp_backward", &routed_mlp_backward, no_gil);
    m.def("moe_experts", &moe_experts, no_gil, py::arg(), py::arg(), py::arg(), py::arg(), py::arg(), py::arg(), py::arg(), py::arg(), py::arg(),
          py::arg(), py::arg(), py::arg(), py::arg("sorted") = std::optional<Tensor>());
    m.def("merged_mlp", &merged_mlp, no_gil);
    m.def("merged_mlp_forward", &merged_mlp_forward, no_gil);
    m.def("merged_mlp_backward", &merged_mlp_backward, no_gil);
    m.def("combine", &combine, no_gil);
    m.def("combine_backward", &combine_backward, no_gil);
    m.def("expert_view", [](const std::vector<Tensor> &weights) {
        if (weights.empty()) throw NativeError("no expert weights");
        at::NoGradGuard no_grad;
        return strided_view(weights.data(), 1, static_cast<int64_t>(weights.size()));
    });
    m.def("adamw_step", &adamw_step, no_gil);
    m.def("grad_norm", &grad_norm, no_gil);
    m.def("sized_by_bound", &sized_by_bound);
    m.def("waits_ahead_of_shared", &waits_ahead_of_shared);
    m.def("live_grad", [](const Tensor &param) {
        Tensor grad = live_grad(param);
        if (grad.defined()) order_live_gradients();
        return grad;
    });
    m.def("expert_parameters", &expert_parameters);
    m.def("foreign_grads", &foreign_grads);
    m.def("constant_pitch", [](const std::vector<Tensor> &weights) {
        at::NoGradGuard no_grad;
        return weights.empty() || strided_view_or_undefined(weights.data(), 1, static_cast<int64_t>(weights.size())).defined();
    });
}

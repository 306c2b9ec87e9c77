// The convolution operator's host side for the common call, in one native call each way.
//
// A pass over a small graph is host work: 1 000 atoms at 32 channels keep the GPU busy for 82 us, while
// the Python operator and its autograd function took 250 (argument conversion for a dozen library calls,
// twenty tensor allocations, and the interpreter's hand-over to and from autograd's thread).  Here a
// `Plan` holds what is fixed for a module, value type and channel count; a call prepares the adjacency (or
// takes a handle's), launches the forward pass and records one node, whose backward builds the schedule and
// launches the VJP without the interpreter.  1 000 atoms, forward and VJP: 150 to 250 us (as the host was busy) -> 95;
// 21 atoms, forward: 69 -> 15 us, three launches of 2 to 7.
//
// It takes calls whose route is the plain one (the conditions of `call`, `Plan::operands` and e3j_amd/native.py); every
// other call, every error and every derivative of a derivative goes to the Python operators, which stay the
// only place where those are decided: the caller gets None, or the node calls `Plan::fallback`.

#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/Event.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <memory>
#include <mutex>
#include <optional>

#include "../../../include/e3j_amd.h"

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// the library's entry points, bound by address: the library instance the ctypes side has loaded
struct Library {
    decltype(&e3j_amd_prepare_rows) prepare_rows = nullptr;
    decltype(&e3j_amd_prepare_rows_workspace_bytes) prepare_rows_workspace_bytes = nullptr;
    decltype(&e3j_amd_row_segments_max) row_segments_max = nullptr;
    decltype(&e3j_amd_row_partials_bytes) row_partials_bytes = nullptr;
    decltype(&e3j_amd_convolution_fwd) fwd = nullptr;
    decltype(&e3j_amd_convolution_fwd_whole) fwd_whole = nullptr;
    decltype(&e3j_amd_convolution_bwd_receiver) bwd_receiver = nullptr;
    decltype(&e3j_amd_convolution_bwd_tiled) bwd_tiled = nullptr;
    decltype(&e3j_amd_convolution_bwd_tiled_edges) bwd_tiled_edges = nullptr;
    decltype(&e3j_amd_convolution_bwd_tiled_f64) bwd_tiled_f64 = nullptr;
    decltype(&e3j_amd_tile_schedule_num_work) tile_schedule_num_work = nullptr;
    decltype(&e3j_amd_tile_schedule_workspace_bytes) tile_schedule_workspace_bytes = nullptr;
    decltype(&e3j_amd_tile_schedule_build) tile_schedule_build = nullptr;
} lib;

// the number of the settings in force (`options.config.number`)
const int64_t *settings_number = nullptr;
int64_t settings_now() { return __atomic_load_n(settings_number, __ATOMIC_RELAXED); }

// A Python object that may be dropped from any thread, with or without the interpreter's lock.
class Held {
public:
    Held() = default;
    explicit Held(py::object o) : o_(o.release().ptr()) {}
    Held(const Held &) = delete;
    Held &operator=(const Held &) = delete;
    ~Held() {
        if (o_ == nullptr || !Py_IsInitialized()) return;
        const PyGILState_STATE state = PyGILState_Ensure();
        Py_DECREF(o_);
        PyGILState_Release(state);
    }
    explicit operator bool() const { return o_ != nullptr; }
    py::object get() const { return py::reinterpret_borrow<py::object>(o_); }  // (with the lock held)
    void set(py::object o) { o_ = o.release().ptr(); }                          // (once, with the lock held)

private:
    PyObject *o_ = nullptr;
};

int64_t padded(int64_t count) { return (count + 3) / 4 * 4; }  // 16-byte boundaries of int32 arrays

c10::Stream current_stream(c10::Device device) { return c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getStream(device); }
void *raw_stream(c10::Device device) { return static_cast<void *>(c10::hip::getCurrentHIPStream(device.index()).stream()); }

// A prepared adjacency: the arrays of a call's own preparation, or those of a `PreparedGraph` handle.
struct Adjacency {
    int32_t num_nodes = 0;
    int64_t num_edges = 0;
    std::vector<at::Tensor> keep;          // the memory behind the pointers
    const int32_t *other = nullptr, *row_ptr = nullptr, *perm = nullptr, *order = nullptr;
    bool shared_rows = false;              // long rows are shared between waves (their list may be empty)
    int32_t row_cap = 0, row_piece = 0, max_segments = 0;
    const int32_t *segments = nullptr;
    at::Tensor partials;
    // its own preparation: positions in keep[0], the stream it ran on, and an event after it
    int64_t at_row_ptr = 0, at_order = 0, at_perm = 0, at_segments = 0;
    std::mutex lock;                       // guards what follows
    std::optional<c10::Stream> stream;
    std::optional<c10::Event> event;
    at::Tensor schedule_memory;
    e3j_amd_tile_schedule schedule{};

    void mark(const c10::Stream &s) {
        stream = s;
        if (!event) event.emplace(c10::DeviceType::CUDA);
        event->record(s);
    }
    void wait_on(const c10::Stream &s) {
        if (event && *stream != s) event->block(s);
    }
};

at::TensorOptions on(c10::Device device, at::ScalarType type) { return at::TensorOptions().device(device).dtype(type); }

struct Plan {
    e3j_amd_conv_params params{};          // sizes, signature, layout; nodes, edges and pointers per call
    at::ScalarType type = at::kFloat;
    c10::Device device = c10::Device(c10::DeviceType::CUDA, 0);
    at::Tensor coef;                       // the packed table in GPU memory
    bool trailing = true, sorted = true;
    int32_t rounds = 0, unordered_rows = 0;             // sweeps of the row order, rows that need none
    bool share_rows = false;                            // long rows of the forward pass (float32, trailing)
    int32_t row_cap = -1, min_row_cap = 0, piece = 0;
    int64_t partials_budget = 0;
    int32_t tile_rows = 0, max_work_edges = 0;          // backward over tiles, from that many dx values on
    int64_t tile_values = 0, tile_values_kept = 0;
    Held fallback, make_graph, classes;                 // (classes: memory behind params.coef_classes)

    int64_t x_at(int i) const { return trailing ? (i == 0 ? params.num_x : params.channels) : (i == 0 ? params.channels : params.num_x); }
    int64_t s_at(int i) const { return trailing ? (i == 0 ? params.num_scalars : params.channels) : (i == 0 ? params.channels : params.num_scalars); }

    bool plain(const at::Tensor &t, at::ScalarType want) const {
        static const c10::DispatchKeySet unusual({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                                  c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                                  c10::DispatchKey::ZeroTensor, c10::DispatchKey::FuncTorchBatched,
                                                  c10::DispatchKey::BatchedNestedTensor,
                                                  c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                                  c10::DispatchKey::Batched});
        return t.defined() && t.layout() == c10::kStrided && t.device() == device && t.scalar_type() == want &&
               !t.key_set().has_any(unusual) && t.is_contiguous() && reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
    }
    bool operands(const at::Tensor &x, const at::Tensor &y, const at::Tensor &s) const {
        return plain(x, type) && plain(y, type) && plain(s, type) && x.dim() == 3 && y.dim() == 2 && s.dim() == 3 &&
               x.size(1) == x_at(0) && x.size(2) == x_at(1) && y.size(1) == params.num_y && s.size(1) == s_at(0) &&
               s.size(2) == s_at(1) && y.size(0) == s.size(0) && x.size(0) >= 1 && x.size(0) < INT32_MAX &&
               y.size(0) >= 1;
    }
    bool tiles(int64_t num_edges, bool kept) const {
        return tile_rows >= 1 && num_edges * params.num_x * params.channels >= (kept ? tile_values_kept : tile_values);
    }
    e3j_amd_conv_params with(const Adjacency &g) const {
        e3j_amd_conv_params p = params;
        p.num_nodes = g.num_nodes;
        p.num_edges = g.num_edges;
        p.row_order = g.order;
        return p;
    }
};

// No transform, mode or tracer is at work that has to see the operator's tensors.
bool plain_context() {
    static const c10::DispatchKeySet modes({c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                            c10::DispatchKey::FuncTorchDynamicLayerBackMode, c10::DispatchKey::FuncTorchVmapMode,
                                            c10::DispatchKey::VmapMode, c10::DispatchKey::Python,
                                            c10::DispatchKey::Functionalize, c10::DispatchKey::PreDispatch});
    return !c10::impl::tls_local_dispatch_key_set().included_.has_any(modes) && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !at::impl::torch_function_mode_enabled() && !torch::jit::tracer::isTracing() &&
           !torch::autograd::ForwardADLevel::try_get_by_idx(0);
}

// The sizes of the list of long rows for a graph (as `RowSegments` and the operators choose them).
void size_pieces(const Plan &plan, Adjacency &g) {
    const int64_t n = g.num_nodes, e = g.num_edges;
    const int64_t cap = plan.row_cap < 0 ? std::max<int64_t>(plan.min_row_cap, (int64_t)(2 * ((double)e / (double)n))) : plan.row_cap;
    if (!plan.share_rows || cap <= 0) return;
    const int64_t bytes = e * (int64_t)plan.params.num_out * plan.params.channels * 4;
    const int64_t piece = std::max<int64_t>(plan.piece, (bytes + plan.partials_budget - 1) / plan.partials_budget);
    g.shared_rows = true;
    g.row_cap = (int32_t)(piece > plan.piece ? std::max(cap, piece) : cap);
    g.row_piece = (int32_t)std::min<int64_t>(piece, g.row_cap);
    g.max_segments = (int32_t)lib.row_segments_max(e, g.row_piece);
}

// Null where the library refuses the call.
std::shared_ptr<Adjacency> prepare(const Plan &plan, const at::Tensor &sender, const at::Tensor &receiver, int64_t n,
                                   bool for_backward) {
    auto g = std::make_shared<Adjacency>();
    const int64_t e = receiver.numel();
    g->num_nodes = (int32_t)n;
    g->num_edges = e;
    size_pieces(plan, *g);
    const int32_t rounds = n < 2 || plan.rounds <= 0 || n <= plan.unordered_rows ? 0 : plan.rounds;
    g->at_row_ptr = padded(e);
    g->at_order = g->at_row_ptr + padded(n + 1);
    g->at_perm = g->at_order + (rounds > 0 ? padded(n) : 0);
    g->at_segments = g->at_perm + (plan.sorted ? 0 : padded(e));
    const int64_t total = g->at_segments + (g->shared_rows ? 4 + 3 * (int64_t)g->max_segments : 0);
    const c10::Stream stream = current_stream(plan.device);
    g->keep.push_back(at::empty({total}, on(plan.device, at::kInt)));
    int32_t *base = g->keep[0].data_ptr<int32_t>();
    const at::Tensor workspace = at::empty({(int64_t)lib.prepare_rows_workspace_bytes((int32_t)n, e, plan.sorted)},
                                           on(plan.device, at::kByte));
    int32_t *order = rounds > 0 ? base + g->at_order : nullptr, *perm = plan.sorted ? nullptr : base + g->at_perm;
    int32_t *segments = g->shared_rows ? base + g->at_segments : nullptr;
    if (lib.prepare_rows(receiver.const_data_ptr<int32_t>(), sender.const_data_ptr<int32_t>(), e, (int32_t)n, plan.sorted,
                         rounds, perm, base, base + g->at_row_ptr, order, g->row_cap, g->row_piece, g->max_segments, segments,
                         workspace.data_ptr(), raw_stream(plan.device)) != E3J_AMD_OK)
        return nullptr;
    g->other = base;
    g->row_ptr = base + g->at_row_ptr;
    g->order = order;
    g->perm = perm;
    g->segments = segments;
    if (segments != nullptr && g->max_segments > 0)
        g->partials = at::empty({std::max<int64_t>(16, (int64_t)lib.row_partials_bytes(g->max_segments, plan.params.num_out, plan.params.channels))},
                                on(plan.device, at::kByte));
    if (for_backward) g->mark(stream);
    return g;
}

// Undefined where the library refuses the call.
at::Tensor forward_pass(const Plan &plan, const Adjacency &g, const at::Tensor &x, const at::Tensor &y, const at::Tensor &s) {
    const int64_t n = x.size(0);
    at::Tensor out = plan.trailing ? at::empty({n, plan.params.num_out, plan.params.channels}, x.options())
                                   : at::empty({n, plan.params.channels, plan.params.num_out}, x.options());
    e3j_amd_conv_params p = plan.with(g);
    auto call = lib.fwd;
    if (g.shared_rows) {
        p.row_cap = g.row_cap;
        p.row_piece = g.row_piece;
        if (g.max_segments > 0) {
            p.segments = g.segments;
            p.max_segments = g.max_segments;
            p.partials = static_cast<float *>(g.partials.data_ptr());
            call = lib.fwd_whole;
        }
    }
    const int rc = call(&p, plan.coef.data_ptr(), x.data_ptr(), y.data_ptr(), s.data_ptr(), g.other, g.row_ptr, g.perm,
                        out.data_ptr(), raw_stream(plan.device));
    return rc == E3J_AMD_OK ? out : at::Tensor();
}

bool build_schedule(const Plan &plan, Adjacency &g, const c10::Stream &stream) {  // with g.lock held
    const int64_t e = g.num_edges;
    const int64_t num_work = lib.tile_schedule_num_work(g.num_nodes, e, plan.tile_rows, plan.max_work_edges);
    const int64_t work = padded(4 * std::max<int64_t>(num_work, 1)), list = padded(e);
    at::Tensor memory = at::empty({work + 3 * list}, on(plan.device, at::kInt));
    const at::Tensor workspace = at::empty(
        {std::max<int64_t>(256, (int64_t)lib.tile_schedule_workspace_bytes(g.num_nodes, e, plan.tile_rows))}, on(plan.device, at::kByte));
    int32_t *base = memory.data_ptr<int32_t>();
    if (lib.tile_schedule_build(g.other, g.row_ptr, g.perm, g.order, g.num_nodes, e, plan.tile_rows, plan.max_work_edges, base,
                                base + work, base + work + list, base + work + 2 * list, workspace.data_ptr(),
                                raw_stream(plan.device)) != E3J_AMD_OK)
        return false;
    g.schedule.tile_rows = plan.tile_rows;
    g.schedule.num_work = (int32_t)num_work;
    g.schedule.work = base;
    g.schedule.sender = base + work;
    g.schedule.edge = base + work + list;
    g.schedule.local = base + work + 2 * list;
    g.schedule_memory = memory;
    g.mark(stream);
    return true;
}

// What a node keeps of its forward call.
struct Call : torch::CustomClassHolder {
    std::shared_ptr<Plan> plan;
    std::shared_ptr<Adjacency> graph;
    at::Tensor sender, receiver;
    int64_t settings = 0;               // of the forward call: its plan's
    Held handle;                        // the caller's `PreparedGraph`, if there is one
    std::optional<e3j_amd_tile_schedule> handle_schedule;  // its schedule, if it was built before the call
    Held schedule_owner;                // (the memory of that schedule)
    std::optional<c10::Stream> stream;  // of the forward call: a handle's work is waited for there
    at::Tensor out;                     // on its way to the node
    Held python_graph;                  // the call's own adjacency for the Python operators, once asked for
};

py::object python_graph(Call &call) {  // with the interpreter's lock held
    if (call.handle) return call.handle.get();
    if (call.python_graph) return call.python_graph.get();
    const Adjacency &g = *call.graph;
    const at::Tensor &all = g.keep[0];
    auto part = [&](bool there, int64_t at, int64_t count) -> py::object {
        return there ? py::cast(all.narrow(0, at, count)) : py::none();
    };
    py::object made = call.plan->make_graph.get()(
        part(true, 0, g.num_edges), part(true, g.at_row_ptr, g.num_nodes + 1), part(g.perm != nullptr, g.at_perm, g.num_edges),
        part(g.order != nullptr, g.at_order, g.num_nodes), g.num_nodes,
        part(g.shared_rows, g.at_segments, 4 + 3 * (int64_t)g.max_segments), g.row_cap, g.row_piece);
    call.python_graph.set(made);
    return made;
}

// The Python operators' backward: for derivatives of derivatives, under transforms, under other settings than the
// forward call's (a backward follows the settings it runs under), and wherever something is unusual
// or failed (the call is then made again there and raises what it raises).
variable_list python_backward(Call &call, const at::Tensor &x, const at::Tensor &y, const at::Tensor &s, const at::Tensor &dm,
                              bool need_dx) {
    if (!call.handle) {
        std::lock_guard<std::mutex> guard(call.graph->lock);
        call.graph->wait_on(current_stream(call.plan->device));
    }
    py::gil_scoped_acquire gil;
    try {
        const py::tuple r = call.plan->fallback.get()(x, y, s, dm, call.sender, call.receiver, python_graph(call), need_dx);
        return {r[0].is_none() ? at::Tensor() : r[0].cast<at::Tensor>(), r[1].cast<at::Tensor>(), r[2].cast<at::Tensor>()};
    } catch (py::error_already_set &e) {
        e.restore();
        python_error error;
        error.persist();
        throw error;
    }
}

struct Convolution : torch::autograd::Function<Convolution> {
    static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x, const at::Tensor &y, const at::Tensor &s,
                              const c10::intrusive_ptr<Call> &call) {
        ctx->save_for_backward({x, y, s});
        ctx->saved_data["call"] = c10::IValue::make_capsule(call);
        return std::move(call->out);
    }

    static variable_list backward(AutogradContext *ctx, const variable_list &cotangents) {
        auto call = c10::static_intrusive_pointer_cast<Call>(ctx->saved_data["call"].toCapsule());
        const variable_list saved = ctx->get_saved_variables();
        const at::Tensor &x = saved[0], &y = saved[1], &s = saved[2];
        const Plan &plan = *call->plan;
        Adjacency &g = *call->graph;
        c10::OptionalDeviceGuard on_device(plan.device);
        const std::vector<int64_t> out_shape = plan.trailing ? std::vector<int64_t>{g.num_nodes, plan.params.num_out, plan.params.channels}
                                                             : std::vector<int64_t>{g.num_nodes, plan.params.channels, plan.params.num_out};
        at::Tensor dm = cotangents[0].defined() ? cotangents[0] : at::zeros(out_shape, on(plan.device, plan.type));
        variable_list grads;
        const bool plain = !c10::GradMode::is_enabled() && settings_now() == call->settings && plain_context();
        if (!plain || !native(plan, g, *call, x, y, s, dm, out_shape, ctx->needs_input_grad(0), grads))
            grads = python_backward(*call, x, y, s, dm, ctx->needs_input_grad(0));
        return {grads[0], grads[1], grads[2], at::Tensor()};
    }

    static bool native(const Plan &plan, Adjacency &g, const Call &call, const at::Tensor &x, const at::Tensor &y,
                       const at::Tensor &s, const at::Tensor &dm_in, const std::vector<int64_t> &out_shape, bool need_dx,
                       variable_list &grads) {
        // (saved tensors may come back changed from hooks)
        if (!plan.operands(x, y, s) || x.size(0) != g.num_nodes || y.size(0) != g.num_edges || dm_in.sizes() != out_shape) return false;
        const at::Tensor dm = dm_in.contiguous();
        if (!plan.plain(dm, plan.type)) return false;
        const c10::Stream stream = current_stream(plan.device);
        e3j_amd_tile_schedule schedule{};
        const bool tiles = plan.tiles(g.num_edges, (bool)call.handle);
        if (call.handle) {
            // what a handle prepares is ordered by the Python side; the forward call's stream has waited for it
            if (stream != *call.stream || (tiles && !call.handle_schedule)) return false;
            if (tiles) schedule = *call.handle_schedule;
        } else {
            std::lock_guard<std::mutex> guard(g.lock);
            g.wait_on(stream);
            if (tiles) {
                if (!g.schedule_memory.defined() && !build_schedule(plan, g, stream)) return false;
                schedule = g.schedule;
            }
        }
        // dx is left out where nobody asks for it (unrolled_bwd_tile_part has the figures)
        const bool edges_only = tiles && plan.type == at::kFloat && !need_dx;
        const at::Tensor dx = edges_only ? at::Tensor() : at::empty(x.sizes(), x.options());
        const at::Tensor dy = at::empty(y.sizes(), y.options()), ds = at::empty(s.sizes(), s.options());
        const e3j_amd_conv_params p = plan.with(g);
        int rc;
        if (edges_only) {
            rc = lib.bwd_tiled_edges(&p, x.data_ptr(), y.data_ptr(), s.data_ptr(), dm.data_ptr(), g.other, g.row_ptr, g.perm,
                                     &schedule, dy.data_ptr(), ds.data_ptr(), raw_stream(plan.device));
        } else if (tiles) {
            const auto run = plan.type == at::kDouble ? lib.bwd_tiled_f64 : lib.bwd_tiled;
            rc = run(&p, x.data_ptr(), y.data_ptr(), s.data_ptr(), dm.data_ptr(), g.other, g.row_ptr, g.perm, &schedule,
                     dx.data_ptr(), dy.data_ptr(), ds.data_ptr(), raw_stream(plan.device));
        } else {
            rc = lib.bwd_receiver(&p, plan.coef.data_ptr(), x.data_ptr(), y.data_ptr(), s.data_ptr(), dm.data_ptr(), g.other,
                                  g.row_ptr, g.perm, dx.data_ptr(), dy.data_ptr(), ds.data_ptr(), raw_stream(plan.device));
        }
        if (rc != E3J_AMD_OK) return false;
        grads = {dx, dy, ds};
        return true;
    }
};

// torch's own tensor types: a subclass may change what an operation on it means.
bool is_tensor(const py::object &o) {
    const PyObject *type = reinterpret_cast<const PyObject *>(Py_TYPE(o.ptr()));
    return type == THPVariableClass || type == ParameterClass;
}

// One call of the operator; None where it is not the plain one.  `kept`: the adjacency of `handle`, both None
// for a call that prepares its own; `settings`: the number of those that `plan` is for.
py::object call(const std::shared_ptr<Plan> &plan, const py::object &x_, const py::object &y_, const py::object &s_,
                const py::object &sender_, const py::object &receiver_, const std::shared_ptr<Adjacency> &kept,
                const py::object &handle, const py::object &schedule, int64_t settings) {
    for (const py::object *o : {&x_, &y_, &s_, &sender_, &receiver_})
        if (!is_tensor(*o)) return py::none();
    const at::Tensor &x = THPVariable_Unpack(x_.ptr()), &y = THPVariable_Unpack(y_.ptr()), &s = THPVariable_Unpack(s_.ptr());
    const at::Tensor &sender = THPVariable_Unpack(sender_.ptr()), &receiver = THPVariable_Unpack(receiver_.ptr());
    const int64_t n = x.dim() > 0 ? x.size(0) : 0, e = y.dim() > 0 ? y.size(0) : 0;
    if (!plain_context() || !plan->operands(x, y, s)) return py::none();
    auto index = [&](const at::Tensor &t) {
        return t.device() == plan->device && t.scalar_type() == at::kInt && t.dim() == 1 && t.numel() == e && t.is_contiguous();
    };
    // (a handle's call does not read the endpoints; the operators refuse those outside GPU memory all the same)
    if (kept ? kept->num_nodes != n || kept->num_edges != e || !sender.is_cuda() || !receiver.is_cuda()
             : !index(sender) || !index(receiver))
        return py::none();
    const bool record = c10::GradMode::is_enabled() && (x.requires_grad() || y.requires_grad() || s.requires_grad());
    c10::intrusive_ptr<Call> state;
    if (record) {
        state = c10::make_intrusive<Call>();
        state->settings = settings;
        if (!handle.is_none()) state->handle.set(handle);
        if (!schedule.is_none()) {
            e3j_amd_tile_schedule t{};
            t.tile_rows = schedule.attr("tile_rows").cast<int32_t>();
            t.num_work = schedule.attr("num_work").cast<int32_t>();
            auto pointer = [&](const char *name) {
                return THPVariable_Unpack(py::object(schedule.attr(name)).ptr()).data_ptr<int32_t>();
            };
            t.work = pointer("work");
            t.sender = pointer("sender");
            t.edge = pointer("edge");
            t.local = pointer("local");
            state->handle_schedule = t;
            state->schedule_owner.set(schedule);
        }
    }
    at::Tensor out;
    {
        py::gil_scoped_release no_gil;
        c10::OptionalDeviceGuard on_device(plan->device);
        const std::shared_ptr<Adjacency> g = kept ? kept : prepare(*plan, sender, receiver, n, record);
        if (g) out = forward_pass(*plan, *g, x, y, s);
        if (out.defined() && record) {
            state->plan = plan;
            state->graph = g;
            state->sender = sender;
            state->receiver = receiver;
            state->stream = current_stream(plan->device);
            state->out = std::move(out);
            out = Convolution::apply(x, y, s, state);
        }
    }
    return out.defined() ? py::cast(out) : py::none();
}

const int32_t *int_pointer(const std::optional<at::Tensor> &t) { return t ? t->data_ptr<int32_t>() : nullptr; }

std::shared_ptr<Adjacency> adjacency(int32_t num_nodes, const at::Tensor &other, const at::Tensor &row_ptr,
                                     const std::optional<at::Tensor> &perm, const std::optional<at::Tensor> &order,
                                     bool shared_rows, int32_t row_cap, int32_t row_piece, int32_t max_segments,
                                     const std::optional<at::Tensor> &segments, const std::optional<at::Tensor> &partials) {
    auto g = std::make_shared<Adjacency>();
    g->num_nodes = num_nodes;
    g->num_edges = other.numel();
    for (const auto &t : {std::optional<at::Tensor>(other), std::optional<at::Tensor>(row_ptr), perm, order, segments})
        if (t) g->keep.push_back(*t);
    g->other = other.data_ptr<int32_t>();
    g->row_ptr = row_ptr.data_ptr<int32_t>();
    g->perm = int_pointer(perm);
    g->order = int_pointer(order);
    g->shared_rows = shared_rows;
    g->row_cap = row_cap;
    g->row_piece = row_piece;
    g->max_segments = max_segments;
    g->segments = int_pointer(segments);
    if (partials) g->partials = *partials;
    return g;
}

template <typename F>
void take(const py::dict &d, const char *name, F &slot) {
    slot = reinterpret_cast<F>(d[name].cast<uintptr_t>());
}

}  // namespace

PYBIND11_MODULE(_operators, m) {
    m.def("bind", [](const py::dict &d, uintptr_t number) {
        settings_number = reinterpret_cast<const int64_t *>(number);
        take(d, "e3j_amd_prepare_rows", lib.prepare_rows);
        take(d, "e3j_amd_prepare_rows_workspace_bytes", lib.prepare_rows_workspace_bytes);
        take(d, "e3j_amd_row_segments_max", lib.row_segments_max);
        take(d, "e3j_amd_row_partials_bytes", lib.row_partials_bytes);
        take(d, "e3j_amd_convolution_fwd", lib.fwd);
        take(d, "e3j_amd_convolution_fwd_whole", lib.fwd_whole);
        take(d, "e3j_amd_convolution_bwd_receiver", lib.bwd_receiver);
        take(d, "e3j_amd_convolution_bwd_tiled", lib.bwd_tiled);
        take(d, "e3j_amd_convolution_bwd_tiled_edges", lib.bwd_tiled_edges);
        take(d, "e3j_amd_convolution_bwd_tiled_f64", lib.bwd_tiled_f64);
        take(d, "e3j_amd_tile_schedule_num_work", lib.tile_schedule_num_work);
        take(d, "e3j_amd_tile_schedule_workspace_bytes", lib.tile_schedule_workspace_bytes);
        take(d, "e3j_amd_tile_schedule_build", lib.tile_schedule_build);
    });
    py::class_<Adjacency, std::shared_ptr<Adjacency>>(m, "Adjacency");
    m.def("adjacency", torch::wrap_pybind_function(adjacency));
    py::class_<Plan, std::shared_ptr<Plan>>(m, "Plan")
        .def(py::init([](const py::bytes &params, const at::Tensor &coef, int64_t type, const py::dict &d, py::object fallback,
                         py::object make_graph, py::object classes) {
            auto plan = std::make_shared<Plan>();
            const std::string bytes = params;
            TORCH_CHECK(bytes.size() == sizeof(plan->params), "e3j_amd_conv_params: ", bytes.size(), " bytes");
            std::memcpy(&plan->params, bytes.data(), bytes.size());
            plan->type = type == E3J_AMD_F64 ? at::kDouble : type == E3J_AMD_F16 ? at::kHalf : at::kFloat;
            plan->coef = coef;
            plan->device = coef.device();
            plan->trailing = plan->params.layout == E3J_AMD_LAYOUT_TRAILING;
            plan->sorted = d["sorted"].cast<bool>();
            plan->rounds = d["rounds"].cast<int32_t>();
            plan->unordered_rows = d["unordered_rows"].cast<int32_t>();
            plan->share_rows = d["share_rows"].cast<bool>();
            plan->row_cap = d["row_cap"].cast<int32_t>();
            plan->min_row_cap = d["min_row_cap"].cast<int32_t>();
            plan->piece = d["piece"].cast<int32_t>();
            plan->partials_budget = d["partials_budget"].cast<int64_t>();
            plan->tile_rows = d["tile_rows"].cast<int32_t>();
            plan->max_work_edges = d["max_work_edges"].cast<int32_t>();
            plan->tile_values = d["tile_values"].cast<int64_t>();
            plan->tile_values_kept = d["tile_values_kept"].cast<int64_t>();
            plan->fallback.set(std::move(fallback));
            plan->make_graph.set(std::move(make_graph));
            plan->classes.set(std::move(classes));
            return plan;
        }))
        .def_readonly("tile_rows", &Plan::tile_rows)
        .def("tiles", &Plan::tiles);
    m.def("call", torch::wrap_pybind_function(call));
}

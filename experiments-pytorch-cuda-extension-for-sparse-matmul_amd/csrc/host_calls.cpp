// The host side of sparse.matmul, sparse.softmax and sparse.attention in native code: what a call decides from the shapes,
// types and device of its operands (checks, walk, schedule, workspace) is decided once, by sparse/_ops.py, and kept with the
// layout as a plan; a call that finds its plan allocates the result, launches, and leaves one autograd node behind whose
// backward does the same without the interpreter.
//
// Whatever a plan does not cover takes the Python functions it was made from: the first call of a shape, operands that
// are not plain contiguous tensors of the current device, functorch transforms, forward-mode AD, tracing, dispatch modes, and a
// split group's workspace while a graph is captured.
//
// What bounds it: per call an allocation, a launch and a node.  us a pass, by the Python functions -> by plans (both in turn on
// one box; where two figures stand on the left, the backward thread's wake-ups decide which a process gets): one fp32 product of
// 512 tokens 17.4 -> 6.5, one of 16 heads of 2048 17.4 -> 6.6, fused attention of 3 x 5 heads of 2976 17.4 -> 12.0 (its
// kernel), softmax forward and backward of 16 heads of 4096 48 or 94 -> 48, three-call training pass of the same 155 or 250
// -> 144, of 2048 in fp32 166 or 250 -> 150, sparse linear layer 100 or 132 -> 100.
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/grad_mode.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <atomic>
#include <memory>
#include <mutex>
#include <vector>

#include "../../include/bsa.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

enum Op : int { MATMUL = 0, WEIGHT_GRAD = 1, SOFTMAX_FORWARD = 2, SOFTMAX_BACKWARD = 3, ATTENTION_FORWARD = 4, ATTENTION_BACKWARD = 5 };
enum Route : int { GENERAL = 0, RUNS = 1, PANELS = 2 };

// Filled once by setup(): the library's entry points as ctypes loaded them, and the Python functions behind this file.
struct Entry {
    decltype(&bsa_matmul) matmul;
    decltype(&bsa_matmul_dsd_runs) runs;
    decltype(&bsa_matmul_dds_panels) panels;
    decltype(&bsa_weight_grad) weight_grad;
    decltype(&bsa_softmax_forward) softmax_forward;
    decltype(&bsa_softmax_backward) softmax_backward;
    decltype(&bsa_attention_forward) attention_forward;
    decltype(&bsa_attention_gradients) attention_gradients;
} lib;
struct PythonSide {
    PyObject *matmul, *softmax, *attention;                                     // autograd Functions' apply
    PyObject *plan_matmul, *plan_weight, *plan_softmax, *plan_softmax_backward, *plan_attention, *plan_attention_backward;
    PyObject *run_matmul, *run_weight, *run_softmax_backward, *run_attention_backward;      // without a plan
    PyObject *failed;
    PyDictObject *settings[2];               // of the modules whose globals decide routes
    PyObject *name_plans, *name_row, *name_col, *modes[3];
} python;

// ---- plans ------------------------------------------------------------------------------------------
// A value that is released under the interpreter's lock, wherever its owner goes away.
struct PythonRef {
    PyObject *object = nullptr;
    explicit PythonRef(PyObject *o) : object(o) { Py_XINCREF(o); }
    PythonRef(const PythonRef &) = delete;
    PythonRef &operator=(const PythonRef &) = delete;
    ~PythonRef()
    {
        if (object == nullptr || !Py_IsInitialized()) return;
        py::gil_scoped_acquire gil;
        Py_DECREF(object);
    }
};

// The zeroed workspace of a schedule's split groups, as the plans that launch with it share it.  The schedule owns it (_ops.Schedule)
// and says when it is theirs no more: a launch that failed, the schedule's bound, a spare to be put back.
struct Space {
    std::mutex mutex;
    Tensor buffer;
    Tensor get()
    {
        std::lock_guard<std::mutex> lock(mutex);
        return buffer;
    }
    void drop()
    {
        Tensor gone;                         // released behind the lock
        std::lock_guard<std::mutex> lock(mutex);
        std::swap(gone, buffer);
    }
};
typedef std::shared_ptr<Space> SpacePtr;
constexpr const char *SPACE = "bsa.space";

struct Plan {
    int op, flags;
    at::ScalarType dtype;
    int device;
    std::vector<int64_t> a, b;               // shapes it holds for
    int route, bsa_dtype;
    bool aligned;                            // operands must start at a multiple of 16 bytes
    std::vector<int> n;                      // sizes and schedule figures in the order of the launch below
    std::vector<Tensor> tables;
    std::vector<int64_t> out;
    SpacePtr space;                          // of split groups: zero between launches, which one stream orders
    size_t workspace_bytes = 0;
    hipStream_t stream = nullptr;            // of the workspace
    std::unique_ptr<PythonRef> schedule;     // the schedule and the key its workspace is kept under there
    std::unique_ptr<PythonRef> workspace_key;
    template <class T = int32_t>
    T *table(int i) const { return tables[i].defined() ? static_cast<T *>(tables[i].data_ptr()) : nullptr; }
};
typedef std::shared_ptr<const Plan> PlanPtr;

// A plan to launch by, with its workspace held until the launch is in the stream
struct Found {
    PlanPtr plan;
    Tensor workspace;
    const Plan *operator->() const { return plan.get(); }
    explicit operator bool() const { return plan != nullptr; }
    void *ws() const { return workspace.defined() ? workspace.data_ptr() : nullptr; }
};

uint64_t settings_version()
{
    // bumped by every assignment to a global of either module; read without the lock by backward threads
    return reinterpret_cast<volatile PyDictObject *>(python.settings[0])->ma_version_tag +
           reinterpret_cast<volatile PyDictObject *>(python.settings[1])->ma_version_tag;
}

// The plans of one layout.  At most MOST: the oldest goes first (a launch in flight keeps the stream order of its workspace:
// the allocator gives it out again on the same stream only).
struct Plans {
    static constexpr size_t MOST = 64;
    std::mutex mutex;
    std::vector<PlanPtr> plans;
    uint64_t version = 0;
    PyObject *row_layout, *col_layout;       // the tuples the plans were made from
    Found find(int op, int flags, const Tensor &a, const Tensor &b, hipStream_t stream)
    {
        const uint64_t now = settings_version();
        Found found;
        std::vector<PlanPtr> gone;           // released behind the lock
        std::lock_guard<std::mutex> lock(mutex);
        if (version != now) return found;
        for (size_t i = 0; i < plans.size(); ++i) {
            const PlanPtr p = plans[i];
            if (p->op != op || p->flags != flags || p->dtype != a.scalar_type() || p->device != a.get_device() ||
                !a.sizes().equals(p->a) || (p->space && p->stream != stream))
                continue;
            if (b.defined() && !(b.sizes().equals(p->b) && b.scalar_type() == p->dtype && b.get_device() == p->device)) continue;
            if (p->space) {
                found.workspace = p->space->get();
                if (!found.workspace.defined()) {
                    gone.push_back(p);
                    plans.erase(plans.begin() + i--);
                    continue;
                }
            }
            found.plan = p;
            return found;
        }
        return found;
    }
    void add(PlanPtr plan)
    {
        const uint64_t now = settings_version();
        std::vector<PlanPtr> gone;           // released behind the lock
        std::lock_guard<std::mutex> lock(mutex);
        if (version != now) {
            gone.swap(plans);
            version = now;
        }
        if (plans.size() >= MOST) {
            gone.push_back(plans.front());
            plans.erase(plans.begin());
        }
        plans.push_back(std::move(plan));
    }
    void drop(const PlanPtr &plan)
    {
        std::lock_guard<std::mutex> lock(mutex);
        for (size_t i = 0; i < plans.size(); ++i)
            if (plans[i] == plan) {
                plans.erase(plans.begin() + i);
                return;
            }
    }
};
typedef std::shared_ptr<Plans> PlansPtr;
constexpr const char *CAPSULE = "bsa.plans";

PyObject *new_space(PyObject *, PyObject *workspace)
{
    HANDLE_TH_ERRORS
    SpacePtr space = std::make_shared<Space>();
    space->buffer = THPVariable_Unpack(workspace);
    return PyCapsule_New(new SpacePtr(std::move(space)), SPACE,
                         [](PyObject *c) { delete static_cast<SpacePtr *>(PyCapsule_GetPointer(c, SPACE)); });
    END_HANDLE_TH_ERRORS
}

PyObject *drop_space(PyObject *, PyObject *capsule)
{
    HANDLE_TH_ERRORS
    auto *space = static_cast<SpacePtr *>(PyCapsule_GetPointer(capsule, SPACE));
    if (space == nullptr) return nullptr;
    (*space)->drop();
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// Address of each plan's workspace, 0 where it has none
PyObject *plan_workspaces(PyObject *, PyObject *capsule)
{
    HANDLE_TH_ERRORS
    auto *plans = static_cast<PlansPtr *>(PyCapsule_GetPointer(capsule, CAPSULE));
    if (plans == nullptr) return nullptr;
    py::list result;
    std::lock_guard<std::mutex> lock((*plans)->mutex);
    for (const PlanPtr &p : (*plans)->plans) {
        const Tensor ws = p->space ? p->space->get() : Tensor();
        result.append(ws.defined() ? reinterpret_cast<uintptr_t>(ws.data_ptr()) : 0);
    }
    return result.release().ptr();
    END_HANDLE_TH_ERRORS
}

PyObject *new_plans(PyObject *, PyObject *args)
{
    HANDLE_TH_ERRORS
    PyObject *row, *col;
    if (!PyArg_ParseTuple(args, "OO", &row, &col)) return nullptr;
    PlansPtr plans = std::make_shared<Plans>();
    plans->row_layout = row;                 // compared, never followed: the capsule's context keeps both alive
    plans->col_layout = col;
    PyObject *capsule = PyCapsule_New(new PlansPtr(std::move(plans)), CAPSULE, [](PyObject *c) {
        delete static_cast<PlansPtr *>(PyCapsule_GetPointer(c, CAPSULE));
        Py_XDECREF(static_cast<PyObject *>(PyCapsule_GetContext(c)));
    });
    if (capsule != nullptr) {
        Py_INCREF(args);
        PyCapsule_SetContext(capsule, args);
    }
    return capsule;
    END_HANDLE_TH_ERRORS
}

// plans, op, flags, a, b, route, dtype, aligned, ints, tables, out, space, workspace bytes, stream, schedule, key
PyObject *add_plan(PyObject *, PyObject *args)
{
    HANDLE_TH_ERRORS
    PyObject *capsule, *a, *b, *ints, *tables, *out, *space, *schedule, *key;
    int op, flags, route, dtype, aligned;
    unsigned long long bytes, stream;
    if (!PyArg_ParseTuple(args, "OiiOOiipO!O!O!OKKOO", &capsule, &op, &flags, &a, &b, &route, &dtype, &aligned, &PyTuple_Type, &ints,
                          &PyTuple_Type, &tables, &PyTuple_Type, &out, &space, &bytes, &stream, &schedule, &key))
        return nullptr;
    auto *plans = static_cast<PlansPtr *>(PyCapsule_GetPointer(capsule, CAPSULE));
    if (plans == nullptr) return nullptr;
    auto plan = std::make_shared<Plan>();
    const Tensor &ta = THPVariable_Unpack(a);
    plan->op = op;
    plan->flags = flags;
    plan->dtype = ta.scalar_type();
    plan->device = ta.get_device();
    plan->a = ta.sizes().vec();
    if (b != Py_None) plan->b = THPVariable_Unpack(b).sizes().vec();
    plan->route = route;
    plan->bsa_dtype = dtype;
    plan->aligned = aligned;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(ints); ++i) plan->n.push_back((int)PyLong_AsLong(PyTuple_GET_ITEM(ints, i)));
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(tables); ++i) {
        PyObject *t = PyTuple_GET_ITEM(tables, i);
        plan->tables.push_back(t == Py_None ? Tensor() : THPVariable_Unpack(t));
    }
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(out); ++i) plan->out.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(out, i)));
    if (PyErr_Occurred()) return nullptr;
    if (space != Py_None) {
        auto *shared = static_cast<SpacePtr *>(PyCapsule_GetPointer(space, SPACE));
        if (shared == nullptr) return nullptr;
        plan->space = *shared;
        plan->workspace_bytes = bytes;
        plan->stream = reinterpret_cast<hipStream_t>(stream);
        plan->schedule = std::make_unique<PythonRef>(schedule);
        plan->workspace_key = std::make_unique<PythonRef>(key);
    }
    (*plans)->add(std::move(plan));
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// the interpreter's pending error, kept for whichever thread reports it; the lock is held
[[noreturn]] void raise_pending()
{
    python_error error;
    error.persist();
    throw error;
}

// ---- calls ------------------------------------------------------------------------------------------
// A dense CUDA tensor and nothing else: no subclass, no functorch wrapper, no lazily negated view
bool plain(const Tensor &t)
{
    static const uint64_t allowed = c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA,
                                                         c10::DispatchKey::AutocastCUDA, c10::DispatchKey::ADInplaceOrView}).raw_repr();
    return t.defined() && (t.key_set().raw_repr() & ~allowed) == 0 && t.is_contiguous();
}
bool on_current_device(const Tensor &t) { return t.get_device() == c10::hip::current_device(); }
bool at_16_bytes(const Tensor &t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }
bool forward_mode(const Tensor &t) { return t._fw_grad(0).defined(); }
// modes that see a Python autograd Function or the operators inside it
bool plain_thread()
{
    static const c10::DispatchKeySet modes({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::PythonDispatcher,
                                            c10::DispatchKey::Tracer, c10::DispatchKey::Functionalize,
                                            c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::FuncTorchDynamicLayerBackMode});
    return (c10::impl::tls_local_dispatch_key_set().included_ & modes).empty();
}
hipStream_t current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }
// Whether Python would make a plan of a call on these operands (_ops._plans): to ask takes 2 us
bool plannable(std::initializer_list<const Tensor *> operands)
{
    for (const Tensor *t : operands)
        if (!at_16_bytes(*t)) return false;
    return !capturing();
}

// The plan of a call on these operands, if the call can go by one here and now
Found find_plan(Plans &plans, int op, int flags, const Tensor &a, const Tensor &b)
{
    Found p = plans.find(op, flags, a, b, current_stream());
    if (p && p->space && capturing()) return Found();
    return p;
}
void check(int status, Plans &plans, const Found &p)
{
    if (status == 0) return;
    // the launch may have left counters of the workspace non-zero: its schedule forgets it and takes it from every plan
    plans.drop(p.plan);
    py::gil_scoped_acquire gil;
    PyObject *none = PyObject_CallFunction(python.failed, "iOO", status, p->schedule ? p->schedule->object : Py_None,
                                           p->workspace_key ? p->workspace_key->object : Py_None);
    if (none != nullptr) {                   // it raises
        Py_DECREF(none);
        TORCH_CHECK(false, "bsa status ", status);
    }
    raise_pending();
}

Tensor run_matmul(Plans &plans, const Found &p, const Tensor &a, const Tensor &b)
{
    Tensor c = at::empty(p->out, a.options());
    const int *n = p->n.data();
    const hipStream_t st = current_stream();
    int status;
    if (p->route == RUNS)                    // runs, strips, pairs, waves, rows, cols, nnz, batches, sparse batches, N
        status = lib.runs(p->bsa_dtype, a.data_ptr(), b.data_ptr(), c.data_ptr(), p->table(0), p->table(1), p->table<void>(2), n[0], n[1], n[2],
                          n[3], n[4], n[5], n[6], n[7], n[8], n[9], st);
    else if (p->route == PANELS)             // rows, cols, nnz, batches, sparse batches, M, trans_b
        status = lib.panels(p->bsa_dtype, a.data_ptr(), b.data_ptr(), c.data_ptr(), p->table(0), p->table(1), n[0], n[1], n[2], n[3], n[4],
                            n[5], n[6], st);
    else                                     // mode, groups, wgs, waves, tiles, splits, rows, cols, nnz, batches, sparse batches, M, N, K, ta, tb
        status = lib.matmul(n[0], p->bsa_dtype, a.data_ptr(), b.data_ptr(), c.data_ptr(), p->table(0), p->table(1), n[1], p->table(2), n[2],
                            n[3], n[4], n[5], p.ws(), p->workspace_bytes, n[6], n[7], n[8], n[9], n[10], n[11], n[12], n[13], n[14], n[15],
                            st);
    check(status, plans, p);
    return c;
}

struct Borrow {                              // a new reference to a tensor's Python object, released behind the call
    py::object held;
    explicit Borrow(const Tensor &t) : held(py::reinterpret_steal<py::object>(THPVariable_Wrap(t))) {}
    PyObject *get() const { return held.ptr(); }
};

PyObject *py_bool(bool x) { return x ? Py_True : Py_False; }

Tensor unwrap_new(PyObject *result)          // steals
{
    if (result == nullptr) raise_pending();
    Tensor t = THPVariable_Unpack(result);
    Py_DECREF(result);
    return t;
}

// One product of a backward pass: by its plan, or as Python does it
Tensor product(Plans &plans, PyObject *layout, const Tensor &a, const Tensor &b, int mode, bool ta, bool tb)
{
    const int flags = mode << 2 | ta << 1 | tb;
    const bool direct = plain(a) && plain(b) && on_current_device(a);
    Found p = direct ? find_plan(plans, MATMUL, flags, a, b) : Found();
    if (!p || (p->aligned && !(at_16_bytes(a) && at_16_bytes(b)))) {
        py::gil_scoped_acquire gil;
        Borrow pa(a), pb(b);
        if (direct && plannable({&a, &b})) {
            PyObject *made = PyObject_CallFunctionObjArgs(python.plan_matmul, pa.get(), pb.get(), python.modes[mode], layout, py_bool(ta),
                                                          py_bool(tb), nullptr);
            if (made == nullptr) raise_pending();
            const bool planned = made == Py_True;
            Py_DECREF(made);
            p = planned ? find_plan(plans, MATMUL, flags, a, b) : Found();
        }
        if (!p || (p->aligned && !(at_16_bytes(a) && at_16_bytes(b))))
            return unwrap_new(PyObject_CallFunctionObjArgs(python.run_matmul, pa.get(), pb.get(), python.modes[mode], layout, py_bool(ta),
                                                           py_bool(tb), nullptr));
    }
    return run_matmul(plans, p, a, b);
}

Tensor weight_gradient(Plans &plans, PyObject *layout, const Tensor &a, const Tensor &b, bool ta, bool tb)
{
    auto by_plan = [&]() -> Found {
        if (!(plain(a) && plain(b) && on_current_device(a) && at_16_bytes(a) && at_16_bytes(b))) return Found();
        return find_plan(plans, WEIGHT_GRAD, ta << 1 | tb, a, b);
    };
    Found p = by_plan();
    if (!p) {
        py::gil_scoped_acquire gil;
        Borrow pa(a), pb(b);
        if (plain(a) && plain(b) && plannable({&a, &b})) {
            PyObject *made = PyObject_CallFunctionObjArgs(python.plan_weight, pa.get(), pb.get(), layout, py_bool(ta), py_bool(tb), nullptr);
            if (made == nullptr) raise_pending();
            const bool planned = made == Py_True;
            Py_DECREF(made);
            p = planned ? by_plan() : Found();
        }
        if (!p)
            return unwrap_new(PyObject_CallFunctionObjArgs(python.run_weight, pa.get(), pb.get(), layout, py_bool(ta), py_bool(tb), nullptr));
    }
    const int *n = p->n.data();              // rows, cols, nnz, tokens, shares, floats of the parts
    Tensor out = at::empty(p->out, a.options());
    Tensor parts = at::empty({(int64_t)n[5]}, a.options().dtype(at::kFloat));
    check(lib.weight_grad(p->bsa_dtype, a.data_ptr(), b.data_ptr(), out.data_ptr(), p->table(0), p->table(1), n[0], n[1], n[2], n[3], n[4],
                          parts.data_ptr<float>(), 4 * (size_t)n[5], current_stream()), plans, p);
    return out;
}

Tensor first_gradient(const variable_list &grads, const Node &node)
{
    return grads[0].defined() ? grads[0].contiguous() : node.input_metadata(0).zeros_like();
}

// ---- autograd nodes -----------------------------------------------------------------------------------
// sparse/matmul.py, SparseMatMul.backward
struct MatMulNode : public Node {
    SavedVariable a_, b_;
    int mode[3], mode_id;
    bool ta, tb;
    PlansPtr plans;
    std::unique_ptr<PythonRef> layout;
    std::string name() const override { return "SparseMatMulBackward"; }
    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        a_.reset_data();
        b_.reset_data();
    }
    static int mode_of(int x, int y, int z)  // 0 sparse, 1 dense: of the result and the two operands
    {
        return x == 0 ? 0 : y == 0 ? 1 : 2;  // sdd, dsd, dds
    }
    variable_list apply(variable_list &&grads) override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        const Tensor a = a_.unpack(), b = b_.unpack(), dc = first_gradient(grads, *this);
        const int *m = mode;
        PyObject *lay = layout->object;
        Tensor da, db;
        if (task_should_compute_output(0)) { // d op(a) = dc op(b)^T, stored in a's orientation
            const Tensor &lhs = ta ? b : dc, &rhs = ta ? dc : b;
            if (m[1] == 0 && a.dim() == 3) da = weight_gradient(*plans, lay, lhs, rhs, ta && tb, ta || !tb);
            else da = product(*plans, lay, lhs, rhs, ta ? mode_of(m[1], m[2], m[0]) : mode_of(m[1], m[0], m[2]), ta && tb, ta || !tb);
        }
        if (task_should_compute_output(1)) { // d op(b) = op(a)^T dc, stored in b's orientation
            const Tensor &lhs = tb ? dc : a, &rhs = tb ? a : dc;
            if (m[2] == 0 && b.dim() == 3) db = weight_gradient(*plans, lay, lhs, rhs, !ta || tb, ta && tb);
            else db = product(*plans, lay, lhs, rhs, tb ? mode_of(m[2], m[0], m[1]) : mode_of(m[2], m[1], m[0]), !ta || tb, ta && tb);
        }
        return {da, db};
    }
};

// sparse/softmax.py, SparseSoftmax.backward
struct SoftmaxNode : public Node {
    SavedVariable y_;
    double scale;
    PlansPtr plans;
    std::unique_ptr<PythonRef> layout;
    std::string name() const override { return "SparseSoftmaxBackward"; }
    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        y_.reset_data();
    }
    variable_list apply(variable_list &&grads) override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        const Tensor y = y_.unpack(getptr()), dy = first_gradient(grads, *this);
        if (!task_should_compute_output(0)) return {Tensor()};
        auto by_plan = [&]() -> Found {
            if (!(plain(y) && plain(dy) && on_current_device(y) && y.sizes() == dy.sizes() && y.scalar_type() == dy.scalar_type()))
                return Found();
            return find_plan(*plans, SOFTMAX_BACKWARD, 0, y, Tensor());
        };
        Found p = by_plan();
        if (!p) {
            py::gil_scoped_acquire gil;
            Borrow py_y(y), py_dy(dy);
            if (plain(y) && plannable({&y})) {
                PyObject *made = PyObject_CallFunctionObjArgs(python.plan_softmax_backward, py_y.get(), layout->object, nullptr);
                if (made == nullptr) raise_pending();
                const bool planned = made == Py_True;
                Py_DECREF(made);
                p = planned ? by_plan() : Found();
            }
            if (!p) {
                py::object s = py::float_(scale);
                return {unwrap_new(PyObject_CallFunctionObjArgs(python.run_softmax_backward, py_y.get(), py_dy.get(), layout->object, s.ptr(), nullptr))};
            }
        }
        const int *n = p->n.data();          // wgs, waves, rows, cols, nnz, batches
        Tensor dx = at::empty(y.sizes(), y.options());
        check(lib.softmax_backward(p->bsa_dtype, y.data_ptr(), dy.data_ptr(), dx.data_ptr(), p->table(0), p->table(1), p->table(2), n[0], n[1],
                                   n[2], n[3], n[4], n[5], (float)scale, current_stream()), *plans, p);
        return {dx};
    }
};

// sparse/attention.py, SparseAttention.backward
struct AttentionNode : public Node {
    SavedVariable q_, k_, v_, out_, lse_;
    double scale;
    bool causal;
    PlansPtr plans;
    std::unique_ptr<PythonRef> layout;
    std::string name() const override { return "SparseAttentionBackward"; }
    void release_variables() override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable *s : {&q_, &k_, &v_, &out_, &lse_}) s->reset_data();
    }
    variable_list apply(variable_list &&grads) override
    {
        std::lock_guard<std::mutex> lock(mutex_);
        const Tensor q = q_.unpack(), k = k_.unpack(), v = v_.unpack(), out = out_.unpack(getptr()), lse = lse_.unpack();
        const Tensor dout = first_gradient(grads, *this);
        const bool dkdv = task_should_compute_output(1) || task_should_compute_output(2);
        auto by_plan = [&]() -> Found {
            for (const Tensor *t : {&q, &k, &v, &dout, &out, &lse})
                if (!plain(*t) || t->get_device() != q.get_device()) return Found();
            if (!(on_current_device(q) && at_16_bytes(q) && at_16_bytes(k) && at_16_bytes(v) && at_16_bytes(dout))) return Found();
            if (dout.sizes() != q.sizes() || out.sizes() != q.sizes() || v.sizes() != k.sizes() || lse.scalar_type() != at::kFloat ||
                lse.sizes() != q.sizes().slice(0, q.dim() - 1))
                return Found();
            for (const Tensor *t : {&k, &v, &dout, &out})
                if (t->scalar_type() != q.scalar_type()) return Found();
            return find_plan(*plans, ATTENTION_BACKWARD, dkdv, q, k);
        };
        Found p = by_plan();
        if (!p) {
            py::gil_scoped_acquire gil;
            Borrow pq(q), pk(k), pv(v), pd(dout), po(out), pl(lse);
            if (plain(q) && plain(k) && plain(v) && plannable({&q, &k, &v})) {
                PyObject *made = PyObject_CallFunctionObjArgs(python.plan_attention_backward, pq.get(), pk.get(), pv.get(), layout->object, py_bool(dkdv), nullptr);
                if (made == nullptr) raise_pending();
                const bool planned = made == Py_True;
                Py_DECREF(made);
                p = planned ? by_plan() : Found();
            }
            if (!p) {
                py::object s = py::float_(scale);
                PyObject *got = PyObject_CallFunctionObjArgs(python.run_attention_backward, pq.get(), pk.get(), pv.get(), pd.get(), po.get(), pl.get(),
                                                             layout->object, s.ptr(), py_bool(causal), py_bool(dkdv), nullptr);
                if (got == nullptr) raise_pending();
                py::tuple t = py::reinterpret_steal<py::tuple>(got);
                variable_list result;
                for (auto x : t) result.push_back(x.is_none() ? Tensor() : THPVariable_Unpack(x.ptr()));
                return result;
            }
        }
        const int *n = p->n.data();          // row wgs, waves, tiles, splits, column wgs, waves, tiles, splits, rows, cols, nnz, batches, head
        Tensor dq = at::empty(q.sizes(), q.options()), delta = at::empty(lse.sizes(), lse.options()), dk, dv;
        if (dkdv) {
            dk = at::empty(k.sizes(), k.options());
            dv = at::empty(v.sizes(), v.options());
        }
        check(lib.attention_gradients(p->bsa_dtype, q.data_ptr(), k.data_ptr(), v.data_ptr(), dout.data_ptr(), out.data_ptr(), lse.data_ptr<float>(),
                                      dq.data_ptr(), dkdv ? dk.data_ptr() : nullptr, dkdv ? dv.data_ptr() : nullptr, delta.data_ptr<float>(),
                                      p->table(0), p->table(1), p->table(2), n[0], n[1], n[2], n[3], p->table(3), p->table(4), p->table(5), n[4],
                                      n[5], n[6], n[7], p.ws(), p->workspace_bytes, n[8], n[9], n[10], n[11], n[12], (float)scale, causal,
                                      current_stream()), *plans, p);
        return {dq, dk, dv};
    }
};

// ---- the calls from Python ------------------------------------------------------------------------------
// The layout's plans, while its tables are those the plans were made from
PlansPtr plans_of(PyObject *layout)
{
    PyObject *capsule = PyObject_GetAttr(layout, python.name_plans);
    if (capsule == nullptr) {
        PyErr_Clear();
        return nullptr;
    }
    PlansPtr plans;
    if (PyCapsule_IsValid(capsule, CAPSULE)) plans = *static_cast<PlansPtr *>(PyCapsule_GetPointer(capsule, CAPSULE));
    Py_DECREF(capsule);
    if (plans == nullptr) return nullptr;
    for (int i = 0; i < 2; ++i) {
        PyObject *table = PyObject_GetAttr(layout, i == 0 ? python.name_row : python.name_col);
        const bool same = table == (i == 0 ? plans->row_layout : plans->col_layout);
        if (table == nullptr) PyErr_Clear();
        Py_XDECREF(table);
        if (!same) return nullptr;
    }
    return plans;
}

bool needs_grad(std::initializer_list<const Tensor *> inputs)
{
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor *t : inputs)
        if (t->requires_grad()) return true;
    return false;
}

PyObject *general(PyObject *apply, PyObject *const *args, Py_ssize_t n) { return PyObject_Vectorcall(apply, args, n, nullptr); }

// truth of an argument, or -1 where Python has to say
int truth(PyObject *x) { return x == Py_True ? 1 : x == Py_False ? 0 : -1; }

PyObject *matmul(PyObject *, PyObject *const *args, Py_ssize_t nargs)
{
    HANDLE_TH_ERRORS
    const int ta = nargs > 4 ? truth(args[4]) : 0, tb = nargs > 5 ? truth(args[5]) : 0;
    if (nargs < 4 || nargs > 6 || ta < 0 || tb < 0 || !THPVariable_CheckExact(args[0]) || !THPVariable_CheckExact(args[1]) || !plain_thread())
        return general(python.matmul, args, nargs);
    const Tensor &a = THPVariable_Unpack(args[0]), &b = THPVariable_Unpack(args[1]);
    int mode = 0;
    while (mode < 3 && args[2] != python.modes[mode]) ++mode;
    if (mode == 3 && PyUnicode_Check(args[2]))
        for (mode = 0; mode < 3 && PyUnicode_Compare(args[2], python.modes[mode]) != 0; ++mode) {}
    if (mode == 3 || !plain(a) || !plain(b) || a.scalar_type() != b.scalar_type() || a.get_device() != b.get_device() || !on_current_device(a) ||
        forward_mode(a) || forward_mode(b))
        return general(python.matmul, args, nargs);
    const PlansPtr plans = plans_of(args[3]);
    if (plans == nullptr) return general(python.matmul, args, nargs);
    const int flags = mode << 2 | ta << 1 | tb;
    Found p = find_plan(*plans, MATMUL, flags, a, b);
    if (!p && plannable({&a, &b})) {
        PyObject *made = PyObject_CallFunctionObjArgs(python.plan_matmul, args[0], args[1], args[2], args[3], py_bool(ta), py_bool(tb), nullptr);
        if (made == nullptr) return nullptr;
        const bool planned = made == Py_True;
        Py_DECREF(made);
        p = planned ? find_plan(*plans, MATMUL, flags, a, b) : Found();
    }
    if (!p || (p->aligned && !(at_16_bytes(a) && at_16_bytes(b)))) return general(python.matmul, args, nargs);
    std::shared_ptr<MatMulNode> node;
    if (needs_grad({&a, &b})) {
        node = std::shared_ptr<MatMulNode>(new MatMulNode(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(a, b));
        node->a_ = SavedVariable(a, false);
        node->b_ = SavedVariable(b, false);
        for (int i = 0; i < 3; ++i) node->mode[i] = i == mode ? 0 : 1;
        node->ta = ta;
        node->tb = tb;
        node->plans = plans;
        node->layout = std::make_unique<PythonRef>(args[3]);
    }
    Tensor c;
    {
        py::gil_scoped_release unlocked;
        c = run_matmul(*plans, p, a, b);
    }
    if (node) torch::autograd::set_history(c, node);
    return THPVariable_Wrap(std::move(c));
    END_HANDLE_TH_ERRORS
}

PyObject *softmax(PyObject *, PyObject *const *args, Py_ssize_t nargs)      // x, layout, scale, causal
{
    HANDLE_TH_ERRORS
    const int causal = nargs == 4 ? truth(args[3]) : -1;
    if (causal < 0 || !(PyFloat_CheckExact(args[2]) || PyLong_CheckExact(args[2])) || !THPVariable_CheckExact(args[0]) || !plain_thread())
        return general(python.softmax, args, nargs);
    const Tensor &x = THPVariable_Unpack(args[0]);
    if (!plain(x) || !on_current_device(x) || forward_mode(x)) return general(python.softmax, args, nargs);
    const PlansPtr plans = plans_of(args[1]);
    if (plans == nullptr) return general(python.softmax, args, nargs);
    const double scale = PyFloat_AsDouble(args[2]);
    if (scale == -1.0 && PyErr_Occurred()) return nullptr;
    Found p = find_plan(*plans, SOFTMAX_FORWARD, 0, x, Tensor());
    if (!p && plannable({&x})) {
        PyObject *made = PyObject_CallFunctionObjArgs(python.plan_softmax, args[0], args[1], nullptr);
        if (made == nullptr) return nullptr;
        const bool planned = made == Py_True;
        Py_DECREF(made);
        p = planned ? find_plan(*plans, SOFTMAX_FORWARD, 0, x, Tensor()) : Found();
    }
    if (!p) return general(python.softmax, args, nargs);
    std::shared_ptr<SoftmaxNode> node;
    if (needs_grad({&x})) {
        node = std::shared_ptr<SoftmaxNode>(new SoftmaxNode(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(x));
        node->scale = scale;
        node->plans = plans;
        node->layout = std::make_unique<PythonRef>(args[1]);
    }
    Tensor y;
    {
        py::gil_scoped_release unlocked;
        const int *n = p->n.data();          // wgs, waves, rows, cols, nnz, batches
        y = at::empty(x.sizes(), x.options());
        check(lib.softmax_forward(p->bsa_dtype, x.data_ptr(), y.data_ptr(), p->table(0), p->table(1), p->table(2), n[0], n[1], n[2], n[3], n[4], n[5],
                                  (float)scale, causal, current_stream()), *plans, p);
    }
    if (node) {
        torch::autograd::set_history(y, node);
        node->y_ = SavedVariable(y, true);
    }
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

PyObject *attention(PyObject *, PyObject *const *args, Py_ssize_t nargs)    // q, k, v, layout, scale, causal
{
    HANDLE_TH_ERRORS
    const int causal = nargs == 6 ? truth(args[5]) : -1;
    if (causal < 0 || !(PyFloat_CheckExact(args[4]) || PyLong_CheckExact(args[4])) || !THPVariable_CheckExact(args[0]) ||
        !THPVariable_CheckExact(args[1]) || !THPVariable_CheckExact(args[2]) || !plain_thread())
        return general(python.attention, args, nargs);
    const Tensor &q = THPVariable_Unpack(args[0]), &k = THPVariable_Unpack(args[1]), &v = THPVariable_Unpack(args[2]);
    for (const Tensor *t : {&q, &k, &v})
        if (!plain(*t) || forward_mode(*t) || t->scalar_type() != q.scalar_type() || t->get_device() != q.get_device() || !at_16_bytes(*t))
            return general(python.attention, args, nargs);
    if (!on_current_device(q) || k.sizes() != v.sizes()) return general(python.attention, args, nargs);
    const PlansPtr plans = plans_of(args[3]);
    if (plans == nullptr) return general(python.attention, args, nargs);
    const double scale = PyFloat_AsDouble(args[4]);
    if (scale == -1.0 && PyErr_Occurred()) return nullptr;
    Found p = find_plan(*plans, ATTENTION_FORWARD, 0, q, k);
    if (!p && plannable({&q, &k, &v})) {
        PyObject *made = PyObject_CallFunctionObjArgs(python.plan_attention, args[0], args[1], args[2], args[3], nullptr);
        if (made == nullptr) return nullptr;
        const bool planned = made == Py_True;
        Py_DECREF(made);
        p = planned ? find_plan(*plans, ATTENTION_FORWARD, 0, q, k) : Found();
    }
    if (!p) return general(python.attention, args, nargs);
    std::shared_ptr<AttentionNode> node;
    if (needs_grad({&q, &k, &v})) {
        node = std::shared_ptr<AttentionNode>(new AttentionNode(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(q, k, v));
        node->q_ = SavedVariable(q, false);
        node->k_ = SavedVariable(k, false);
        node->v_ = SavedVariable(v, false);
        node->scale = scale;
        node->causal = causal;
        node->plans = plans;
        node->layout = std::make_unique<PythonRef>(args[3]);
    }
    Tensor out, lse;
    {
        py::gil_scoped_release unlocked;
        const int *n = p->n.data();          // wgs, waves, tiles, splits, rows, cols, nnz, batches, head
        out = at::empty(q.sizes(), q.options());
        if (node) lse = at::empty(q.sizes().slice(0, q.dim() - 1), q.options().dtype(at::kFloat));
        check(lib.attention_forward(p->bsa_dtype, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), node ? lse.data_ptr<float>() : nullptr,
                                    p->table(0), p->table(1), p->table(2), n[0], n[1], n[2], n[3], p.ws(), p->workspace_bytes, n[4], n[5], n[6],
                                    n[7], n[8], (float)scale, causal, current_stream()), *plans, p);
    }
    if (node) {
        torch::autograd::set_history(out, node);
        node->out_ = SavedVariable(out, true);
        node->lse_ = SavedVariable(lse, false);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// entry points (addresses by name), Python functions (by name), the two modules' dicts
PyObject *setup(PyObject *, PyObject *args)
{
    PyObject *entries, *functions, *first, *second;
    if (!PyArg_ParseTuple(args, "O!O!O!O!", &PyDict_Type, &entries, &PyDict_Type, &functions, &PyDict_Type, &first, &PyDict_Type, &second))
        return nullptr;
    auto address = [&](const char *name, auto &fn) {
        PyObject *x = PyDict_GetItemString(entries, name);
        fn = reinterpret_cast<std::decay_t<decltype(fn)>>(x ? PyLong_AsUnsignedLongLong(x) : 0);
        if (fn == nullptr && !PyErr_Occurred()) PyErr_Format(PyExc_KeyError, "%s", name);
    };
    decltype(&bsa_version) version = nullptr;
    address("bsa_version", version);
    if (version != nullptr && version() != BSA_VERSION)
        PyErr_Format(PyExc_ImportError, "bsa_host_calls.so was built for version %d of the library, which is %d: build both", BSA_VERSION, version());
    if (PyErr_Occurred()) return nullptr;
    address("bsa_matmul", lib.matmul);
    address("bsa_matmul_dsd_runs", lib.runs);
    address("bsa_matmul_dds_panels", lib.panels);
    address("bsa_weight_grad", lib.weight_grad);
    address("bsa_softmax_forward", lib.softmax_forward);
    address("bsa_softmax_backward", lib.softmax_backward);
    address("bsa_attention_forward", lib.attention_forward);
    address("bsa_attention_gradients", lib.attention_gradients);
    auto function = [&](const char *name, PyObject *&f) {
        PyObject *x = PyDict_GetItemString(functions, name);
        if (x == nullptr) PyErr_Format(PyExc_KeyError, "%s", name);
        Py_XINCREF(x);
        f = x;
    };
    function("matmul", python.matmul);
    function("softmax", python.softmax);
    function("attention", python.attention);
    function("plan_matmul", python.plan_matmul);
    function("plan_weight", python.plan_weight);
    function("plan_softmax", python.plan_softmax);
    function("plan_softmax_backward", python.plan_softmax_backward);
    function("plan_attention", python.plan_attention);
    function("plan_attention_backward", python.plan_attention_backward);
    function("run_matmul", python.run_matmul);
    function("run_weight", python.run_weight);
    function("run_softmax_backward", python.run_softmax_backward);
    function("run_attention_backward", python.run_attention_backward);
    function("failed", python.failed);
    Py_INCREF(first);
    Py_INCREF(second);
    python.settings[0] = reinterpret_cast<PyDictObject *>(first);
    python.settings[1] = reinterpret_cast<PyDictObject *>(second);
    python.name_plans = PyUnicode_InternFromString("_plans");
    python.name_row = PyUnicode_InternFromString("row_layout");
    python.name_col = PyUnicode_InternFromString("col_layout");
    const char *modes[3] = {"sdd", "dsd", "dds"};
    for (int i = 0; i < 3; ++i) python.modes[i] = PyUnicode_InternFromString(modes[i]);
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"setup", setup, METH_VARARGS, nullptr},
    {"new_plans", new_plans, METH_VARARGS, nullptr},
    {"add_plan", add_plan, METH_VARARGS, nullptr},
    {"new_space", new_space, METH_O, nullptr},
    {"drop_space", drop_space, METH_O, nullptr},
    {"plan_workspaces", plan_workspaces, METH_O, nullptr},
    {"matmul", (PyCFunction)(void (*)(void))matmul, METH_FASTCALL, "matmul(a, b, mode, layout, trans_a=False, trans_b=False)"},
    {"softmax", (PyCFunction)(void (*)(void))softmax, METH_FASTCALL, "softmax(x, layout, scale, causal)"},
    {"attention", (PyCFunction)(void (*)(void))attention, METH_FASTCALL, "attention(q, k, v, layout, scale, causal)"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "bsa_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_bsa_host_calls()
{
    PyObject *m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", BSA_TORCH_VERSION) != 0) Py_CLEAR(m);
    return m;
}

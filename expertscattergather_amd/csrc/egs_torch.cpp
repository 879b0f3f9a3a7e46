// CPython module `_egs_torch`: the launchers and the two autograd Functions on torch tensors, in C++.
//
// At the default shape a training step needs about 43 us on the GPU, and at an eighth of it half of that, while the same step
// issued through Python - tensor checks, allocations, the routing-table bookkeeping and two torch.autograd.Function nodes
// whose backward has to take the interpreter lock on the engine's thread - needed 100 us of host time.  This module does
// what hip_kernels.py does for the operands that programs normally have (dense, aligned, one element type, on the current
// device) and *declines*, by returning None before it has done anything, for all others: hip_kernels.py then takes its own
// way, which is the definition of what the calls mean.  Nothing here launches a kernel: everything goes through the C ABI of
// include/egs_hip.h.
//
// Reference counterparts: egs/triton_kernels.py:361-578 (launchers), :581-639 (autograd Functions).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <atomic>
#include <tuple>
#include <vector>

#include "egs_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------------------------ what the fast way takes
// Key sets that mean "this is not simply memory on the GPU" (wrappers of transforms and tracers, lazily negated views).
const c10::DispatchKeySet kNotPlain({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                     c10::DispatchKey::Functionalize, c10::DispatchKey::Python, c10::DispatchKey::ZeroTensor,
                                     c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});

bool plain_object(PyObject *o)
{
    return Py_TYPE(o) == (PyTypeObject *)THPVariableClass || Py_TYPE(o) == (PyTypeObject *)ParameterClass;
}
bool plain(const Tensor &t)
{
    return t.defined() && t.is_cuda() && t.layout() == c10::kStrided && !t.key_set().has_any(kNotPlain);
}
// contiguous and on a 16-byte boundary: what the sizes of the workspaces are planned for
bool dense16(const Tensor &t) { return t.is_contiguous() && ((uintptr_t)t.const_data_ptr() & 15) == 0; }
bool no_modes() { return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !torch::jit::tracer::isTracing(); }

int type_id(at::ScalarType t)
{
    return t == at::kFloat ? EGS_F32 : t == at::kHalf ? EGS_F16 : t == at::kBFloat16 ? EGS_BF16 : -1;
}
int ind_type_id(at::ScalarType t)
{
    return t == at::kLong ? EGS_IND_I64 : t == at::kInt ? EGS_IND_I32 : t == at::kShort ? EGS_IND_I16 : t == at::kByte ? EGS_IND_U8 : -1;
}

struct Problem {
    egs_dims d;
    int dt, ind;
    c10::DeviceIndex dev;
    bool ok;
};

// `A` is the activation ([B,T,I] when `rows`, else [B,E,K,J]); W is [E,I,J] when `eij`, else [E,J,I]
Problem problem_of(const Tensor &A, const Tensor &W, const Tensor &Ind, bool rows, bool eij, int64_t T)
{
    Problem p{};
    if (!plain(A) || !plain(W) || !plain(Ind)) return p;
    if (W.dim() != 3 || Ind.dim() != 3 || A.dim() != (rows ? 3 : 4)) return p;
    p.dt = type_id(A.scalar_type());
    p.ind = ind_type_id(Ind.scalar_type());
    if (p.dt < 0 || p.ind < 0 || W.scalar_type() != A.scalar_type()) return p;
    const c10::Device dev = A.device();
    if (W.device() != dev || Ind.device() != dev || dev.index() != c10::hip::current_device()) return p;
    if (!dense16(A) || !dense16(W) || !Ind.is_contiguous()) return p;
    const int64_t E = W.size(0), I = W.size(eij ? 1 : 2), J = W.size(eij ? 2 : 1), B = Ind.size(0), K = Ind.size(2);
    if (Ind.size(1) != E || A.size(0) != B) return p;
    if (rows ? A.size(2) != I : (A.size(1) != E || A.size(2) != K || A.size(3) != J)) return p;
    if (rows) T = A.size(1);
    const int64_t most = INT32_MAX;
    if (B < 1 || T < 1 || E < 1 || K < 1 || I < 1 || J < 1 || B > most || T > most || E > most || K > most || I > most || J > most) return p;
    p.d = {(int32_t)B, (int32_t)T, (int32_t)E, (int32_t)K, (int32_t)I, (int32_t)J};
    p.dev = dev.index();
    p.ok = true;
    return p;
}

// the gradient of an output of these sizes, in the operands' type
bool grad_fits(const Tensor &g, const Tensor &A, at::IntArrayRef sizes)
{
    return plain(g) && g.scalar_type() == A.scalar_type() && g.device() == A.device() && g.sizes().equals(sizes);
}

Tensor empty_gpu(at::IntArrayRef sizes, at::ScalarType type, const Problem &p)
{
    return at::detail::empty_cuda(sizes, type, c10::Device(c10::DeviceType::CUDA, p.dev), std::nullopt);
}

void *stream_of(const Tensor &t) { return (void *)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void raise_status(int rc, const char *what)
{
    if (rc == EGS_OK) return;
    std::string msg = egs_status_string(rc);
    if (rc == EGS_ERR_HIP) msg += std::string(": ") + egs_last_hip_error();
    TORCH_CHECK(false, what, ": ", msg, " (egs_status ", rc, ")");
}

struct Scratch {                // per call, from the caching allocator: stream-ordered and graph-pool aware
    Tensor buf;
    void *ptr = nullptr;
    size_t bytes = 0;
    Scratch(int op, int mode, const Problem &p)
    {
        bytes = egs_workspace_bytes(op, mode, &p.d, p.dt);
        if (bytes == 0) return;
        buf = empty_gpu({(int64_t)bytes}, at::kByte, p);
        ptr = buf.data_ptr();
    }
};

// ------------------------------------------------------------------------------ the four launchers
Tensor gather_forward(const Problem &p, const Tensor &X, const Tensor &W, const Tensor &Ind, const Tensor &build, int act = EGS_ACT_NONE,
                      const Tensor &bias = Tensor())
{
    Tensor Y = empty_gpu({p.d.B, p.d.E, p.d.K, p.d.J}, X.scalar_type(), p);
    const int rc = egs_expert_gather_act_forward(X.const_data_ptr(), W.const_data_ptr(), bias.defined() ? bias.const_data_ptr() : nullptr,
                                                 Ind.const_data_ptr(), Y.data_ptr(),
                                                 build.defined() ? build.data_ptr() : nullptr,
                                                 build.defined() ? (size_t)build.numel() : 0, &p.d, (int64_t)p.d.T * p.d.I, p.d.I, p.dt,
                                                 p.ind, act, stream_of(X));
    raise_status(rc, "expert_gather_forward_call");
    return Y;
}

Tensor scatter_forward(const Problem &p, const Tensor &Y, const Tensor &W, const Tensor &Ind, const Tensor &table, int mode,
                       const Tensor &bias = Tensor())
{
    Tensor out = empty_gpu({p.d.B, p.d.T, p.d.I}, Y.scalar_type(), p);
    Scratch ws(EGS_OP_GEMM_SCATTER, mode, p);
    const int rc = egs_expert_scatter_bias_forward(Y.const_data_ptr(), W.const_data_ptr(), bias.defined() ? bias.const_data_ptr() : nullptr,
                                                    Ind.const_data_ptr(),
                                                    table.defined() ? table.const_data_ptr() : nullptr,
                                                    table.defined() ? (size_t)table.numel() : 0, out.data_ptr(), ws.ptr, ws.bytes, &p.d,
                                                    p.dt, p.ind, mode, stream_of(Y));
    raise_status(rc, "expert_scatter_forward_call");
    return out;
}

struct Grads { Tensor in, W, bias; };

Grads gather_backward(const Problem &p, const Tensor &X, const Tensor &W, const Tensor &Ind, const Tensor &table,
                                          const Tensor &grad_in, int mode, bool with_bias = false)
{
    const Tensor grad = dense16(grad_in) ? grad_in : grad_in.clone(at::MemoryFormat::Contiguous);
    Tensor gX = empty_gpu({p.d.B, p.d.T, p.d.I}, X.scalar_type(), p);
    Tensor gW = empty_gpu({p.d.E, p.d.I, p.d.J}, X.scalar_type(), p);
    Scratch ws(EGS_OP_GATHER_BACKWARD, mode, p);
    const int rc = egs_expert_gather_backward_table(X.const_data_ptr(), W.const_data_ptr(), Ind.const_data_ptr(),
                                                    table.defined() ? table.const_data_ptr() : nullptr,
                                                    table.defined() ? (size_t)table.numel() : 0, grad.const_data_ptr(), gX.data_ptr(),
                                                    gW.data_ptr(), ws.ptr, ws.bytes, &p.d, (int64_t)p.d.T * p.d.I, p.d.I, p.dt, p.ind, mode,
                                                    stream_of(X));
    raise_status(rc, "expert_gather_backward_call");
    Tensor gb;
    if (with_bias) {
        gb = empty_gpu({p.d.E, 1, p.d.J}, X.scalar_type(), p);
        raise_status(egs_gather_bias_grad(grad.const_data_ptr(), gb.data_ptr(), &p.d, p.dt, stream_of(X)), "egs_gather_bias_grad");
    }
    return {gX, gW, gb};
}

Grads scatter_backward(const Problem &p, const Tensor &Y, const Tensor &W, const Tensor &Ind, const Tensor &grad_in, bool with_bias = false)
{
    // rows of the incoming gradient may be strided (unit stride inside a row, everything on the 16-byte grid); what else
    // comes - an expanded scalar, a transposed view - is copied
    Tensor grad = grad_in;
    const int64_t es = grad.element_size();
    int64_t ld_t = grad.stride(1), ld_b = grad.stride(0);
    if (dense16(grad)) {
        ld_t = p.d.I; ld_b = (int64_t)p.d.T * p.d.I;
    } else if ((grad.stride(2) != 1 && p.d.I > 1) || ld_t < p.d.I || ld_b < 0 || (ld_t * es) % 16 || (ld_b * es) % 16 ||
               ((uintptr_t)grad.const_data_ptr() & 15)) {
        grad = grad.clone(at::MemoryFormat::Contiguous);
        ld_t = p.d.I; ld_b = (int64_t)p.d.T * p.d.I;
    }
    Tensor gY = empty_gpu({p.d.B, p.d.E, p.d.K, p.d.J}, Y.scalar_type(), p);
    Tensor gW = empty_gpu({p.d.E, p.d.J, p.d.I}, Y.scalar_type(), p);
    Scratch ws(EGS_OP_SCATTER_BACKWARD, EGS_SCATTER_DETERMINISTIC, p);
    int rc = egs_expert_scatter_backward(Y.const_data_ptr(), W.const_data_ptr(), Ind.const_data_ptr(), grad.const_data_ptr(),
                                         gY.data_ptr(), gW.data_ptr(), ws.ptr, ws.bytes, &p.d, ld_b, ld_t, p.dt, p.ind, stream_of(Y));
    if (rc == EGS_ERR_WORKSPACE && !grad.is_contiguous()) {
        // the workspace is sized for dense operands; strided rows can select kernels that need more
        grad = grad.contiguous();
        rc = egs_expert_scatter_backward(Y.const_data_ptr(), W.const_data_ptr(), Ind.const_data_ptr(), grad.const_data_ptr(), gY.data_ptr(),
                                         gW.data_ptr(), ws.ptr, ws.bytes, &p.d, (int64_t)p.d.T * p.d.I, p.d.I, p.dt, p.ind, stream_of(Y));
    }
    raise_status(rc, "expert_scatter_backward_call");
    Tensor gb;
    if (with_bias) {
        gb = empty_gpu({p.d.E, 1, p.d.I}, Y.scalar_type(), p);
        if (grad.is_contiguous()) { ld_t = p.d.I; ld_b = (int64_t)p.d.T * p.d.I; }
        raise_status(egs_scatter_bias_grad(grad.const_data_ptr(), Ind.const_data_ptr(), gb.data_ptr(), &p.d, ld_b, ld_t, p.dt, p.ind, stream_of(Y)),
                     "egs_scatter_bias_grad");
    }
    return {gY, gW, gb};
}

// ------------------------------------------------------------------------------ routing table kept with Ind
// The same entry that hip_kernels.py keeps in Ind.__dict__ (interpreter lock held in all of this):
// ((data_ptr, version, dtype, (B, T, E, K, I, J), dtype id, stream, capture id), table)
PyObject *g_table_attr = nullptr;       // "_egs_routing_table"

struct TableKey {
    uint64_t ptr, version, stream, capture;
    PyObject *dtype;            // borrowed
    egs_dims d;
    int dt, ind;
};

bool same_int(PyObject *o, uint64_t v)
{
    if (!PyLong_Check(o)) return false;
    const unsigned long long got = PyLong_AsUnsignedLongLong(o);
    if (got == (unsigned long long)-1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return got == v;
}

bool same_key(PyObject *key, const TableKey &k)
{
    if (!PyTuple_Check(key) || PyTuple_GET_SIZE(key) != 7) return false;
    PyObject *dims = PyTuple_GET_ITEM(key, 3);
    const int32_t want[6] = {k.d.B, k.d.T, k.d.E, k.d.K, k.d.I, k.d.J};
    if (!same_int(PyTuple_GET_ITEM(key, 0), k.ptr) || !same_int(PyTuple_GET_ITEM(key, 1), k.version) ||
        PyTuple_GET_ITEM(key, 2) != k.dtype || !PyTuple_Check(dims) || PyTuple_GET_SIZE(dims) != 6 ||
        !same_int(PyTuple_GET_ITEM(key, 4), (uint64_t)k.dt) || !same_int(PyTuple_GET_ITEM(key, 5), k.stream) ||
        !same_int(PyTuple_GET_ITEM(key, 6), k.capture))
        return false;
    for (int i = 0; i < 6; ++i)
        if (!same_int(PyTuple_GET_ITEM(dims, i), (uint64_t)want[i])) return false;
    return true;
}

// `applies`: these sizes have a table and one may be kept with this Ind; `table`: the one it has, if it is valid now
struct TableState {
    bool applies = false;
    size_t bytes = 0;
    Tensor table;
    TableKey key{};
};

TableState table_state(PyObject *ind_obj, const Tensor &Ind, const Problem &p, bool cache)
{
    TableState s;
    // a tensor made under inference mode has no version counter; a subclass may not have this tensor's memory
    if (!cache || Py_TYPE(ind_obj) != (PyTypeObject *)THPVariableClass || Ind.is_inference()) return s;
    s.bytes = egs_routing_table_bytes(&p.d, p.dt);
    if (s.bytes == 0) return s;
    s.key.stream = (uint64_t)(uintptr_t)stream_of(Ind);
    unsigned long long capture = 0;
    if (egs_stream_capture_id((void *)(uintptr_t)s.key.stream, &capture) != EGS_OK) return s;
    s.key.capture = capture;
    s.key.ptr = (uint64_t)(uintptr_t)Ind.const_data_ptr();
    s.key.version = (uint64_t)Ind._version();
    s.key.dtype = (PyObject *)torch::getTHPDtype(Ind.scalar_type());
    s.key.d = p.d; s.key.dt = p.dt; s.key.ind = p.ind;
    s.applies = true;
    PyObject **dict = _PyObject_GetDictPtr(ind_obj);
    if (dict == nullptr || *dict == nullptr) return s;
    PyObject *entry = PyDict_GetItem(*dict, g_table_attr);      // borrowed
    if (entry == nullptr || !PyTuple_Check(entry) || PyTuple_GET_SIZE(entry) != 2) return s;
    PyObject *tab = PyTuple_GET_ITEM(entry, 1);
    if (THPVariable_CheckExact(tab) && same_key(PyTuple_GET_ITEM(entry, 0), s.key)) s.table = THPVariable_Unpack(tab);
    return s;
}

void keep_table(PyObject *ind_obj, const TableKey &k, const Tensor &table)
{
    PyObject *tab = THPVariable_Wrap(table);
    if (tab == nullptr) throw python_error();
    PyObject *entry = Py_BuildValue("((KKO(iiiiii)iKK)N)", (unsigned long long)k.ptr, (unsigned long long)k.version, k.dtype, k.d.B, k.d.T,
                                    k.d.E, k.d.K, k.d.I, k.d.J, k.dt, (unsigned long long)k.stream, (unsigned long long)k.capture, tab);
    if (entry == nullptr) throw python_error();
    const int rc = PyObject_SetAttr(ind_obj, g_table_attr, entry);
    Py_DECREF(entry);
    if (rc != 0) throw python_error();
}

// What a gather's backward needs to know to use the routing table of its forward: everything that the entry above is checked by
// in any other call, and what the entry's owner may do to it meanwhile.  No interpreter lock is taken for it (looking the entry
// up again in the backward was 4 us of an 87 us training step):
//   - the indices: the memory, the version, the sizes and the type, against the ones the node now sees (saved-tensor hooks may hand back
//     another tensor);
//   - the stream and the capture that the backward runs in;
//   - invalidate_routing_table(Ind), which counts up the version of the table tensor, and set_routing_table_cache(False).
// What no longer holds is not used: the indices are sorted.
std::atomic<bool> g_tables_allowed{true};       // set_routing_table_cache's word (a forward is told with the call)

constexpr size_t kTableKey = 13;        // numbers of a table's key, at the end of the node's "numbers"
void save_table(AutogradContext *ctx, std::vector<int64_t> &numbers, const TableKey &k, const Tensor &table)
{
    ctx->saved_data["table"] = table;
    const int64_t key[kTableKey] = {(int64_t)k.ptr, (int64_t)k.version, (int64_t)k.stream, (int64_t)k.capture, k.d.B, k.d.T, k.d.E,
                                    k.d.K, k.d.I, k.d.J, k.dt, k.ind, (int64_t)table._version()};
    numbers.insert(numbers.end(), key, key + kTableKey);
}

Tensor table_of_backward(AutogradContext *ctx, const std::vector<int64_t> &numbers, const Tensor &Ind, const Problem &p)
{
    const auto it = ctx->saved_data.find("table");
    if (it == ctx->saved_data.end() || !g_tables_allowed.load(std::memory_order_acquire) || Ind.is_inference()) return Tensor();
    const Tensor table = it->second.toTensor();
    const uint64_t stream = (uint64_t)(uintptr_t)stream_of(Ind);
    unsigned long long capture = 0;
    if (egs_stream_capture_id((void *)(uintptr_t)stream, &capture) != EGS_OK) return Tensor();
    const int64_t now[kTableKey] = {(int64_t)(uintptr_t)Ind.const_data_ptr(), (int64_t)Ind._version(), (int64_t)stream, (int64_t)capture, p.d.B, p.d.T,
                                    p.d.E, p.d.K, p.d.I, p.d.J, p.dt, p.ind, (int64_t)table._version()};
    return numbers.size() >= kTableKey && std::equal(now, now + kTableKey, numbers.end() - kTableKey) ? table : Tensor();
}

// hip_kernels.py (borrowed; null: not imported under its name)
PyObject *g_owner_name = nullptr;       // "expertscattergather_amd.hip_kernels"
PyObject *owner()
{
    PyObject *modules = PyImport_GetModuleDict();
    return modules == nullptr ? nullptr : PyDict_GetItem(modules, g_owner_name);
}

struct Gil {                    // for the autograd engine's threads, which have a thread state but not the lock
    PyGILState_STATE state;
    Gil() : state(PyGILState_Ensure()) {}
    ~Gil() { PyGILState_Release(state); }
};

// A backward whose operands are not for this way - saved-tensor hooks may hand back another type, layout, alignment or kind of
// tensor than was saved - by the function `name` of hip_kernels.py, with the saved tensors, the gradient, `option` and whether
// there is a bias; returns (gradient of the input, of W, of the bias or None).
Grads backward_in_python(const char *name, const variable_list &saved, const Tensor &grad, int option, bool with_bias)
{
    auto fail = [] {
        python_error err;
        err.persist();
        throw err;
    };
    Gil gil;
    PyObject *module = owner();
    TORCH_CHECK(module != nullptr, name, ": expertscattergather_amd.hip_kernels is not loaded");
    PyObject *args[4] = {THPVariable_Wrap(saved[0]), THPVariable_Wrap(saved[1]), THPVariable_Wrap(saved[2]), THPVariable_Wrap(grad)};
    PyObject *res = nullptr;
    if (args[0] != nullptr && args[1] != nullptr && args[2] != nullptr && args[3] != nullptr)
        res = PyObject_CallMethod(module, name, "OOOOiO", args[0], args[1], args[2], args[3], option, with_bias ? Py_True : Py_False);
    for (PyObject *a : args) Py_XDECREF(a);
    if (res == nullptr) fail();
    Grads g;
    Tensor *out[3] = {&g.in, &g.W, &g.bias};
    if (PyTuple_Check(res) && PyTuple_GET_SIZE(res) == 3)
        for (int i = 0; i < 3; ++i)
            if (THPVariable_Check(PyTuple_GET_ITEM(res, i))) *out[i] = THPVariable_Unpack(PyTuple_GET_ITEM(res, i));
    Py_DECREF(res);
    return g;
}

// ------------------------------------------------------------------------------ autograd
// Same contract as the Python Functions of hip_kernels.py: what is saved is the inputs (and the routing table that was valid in the
// forward, with what it was valid for); the scatter mode is the forward's; both gradients are always computed.
struct ExpertGatherFunctionNative : public torch::autograd::Function<ExpertGatherFunctionNative> {
    static Tensor forward(AutogradContext *ctx, const Tensor &X, const Tensor &W, const Tensor &Ind, const std::optional<Tensor> &bias,
                          const TableState &ts, const std::optional<Tensor> &build, int64_t mode)
    {
        ctx->save_for_backward({X, W, Ind});
        std::vector<int64_t> numbers = {mode, (int64_t)bias.has_value()};
        const Tensor &table = build.has_value() ? *build : ts.table;
        if (table.defined() && !table.is_inference()) save_table(ctx, numbers, ts.key, table);      // (one made there has no version)
        ctx->saved_data["numbers"] = std::move(numbers);
        return gather_forward(problem_of(X, W, Ind, true, true, 0), X, W, Ind, build.value_or(Tensor()), EGS_ACT_NONE, bias.value_or(Tensor()));
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const Tensor &X = saved[0], &W = saved[1], &Ind = saved[2];
        const std::vector<int64_t> numbers = ctx->saved_data.at("numbers").toIntVector();
        const int mode = (int)numbers[0];
        const bool bias = numbers[1] != 0;
        const Problem p = problem_of(X, W, Ind, true, true, 0);
        Grads g;
        if (p.ok && grad_fits(grads[0], X, {p.d.B, p.d.E, p.d.K, p.d.J})) {
            at::AutoDispatchBelowADInplaceOrView below;
            g = gather_backward(p, X, W, Ind, table_of_backward(ctx, numbers, Ind, p), grads[0], mode, bias);
        } else {
            g = backward_in_python("_gather_backward_of_node", saved, grads[0], mode, bias);
        }
        return {g.in, g.W, Tensor(), g.bias, Tensor(), Tensor(), Tensor()};
    }
};

struct ExpertScatterFunctionNative : public torch::autograd::Function<ExpertScatterFunctionNative> {
    static Tensor forward(AutogradContext *ctx, const Tensor &Y, const Tensor &W, const Tensor &Ind, const std::optional<Tensor> &bias,
                          const std::optional<Tensor> &table, int64_t T, int64_t mode)
    {
        ctx->save_for_backward({Y, W, Ind});
        ctx->saved_data["T"] = T;
        ctx->saved_data["bias"] = bias.has_value();
        return scatter_forward(problem_of(Y, W, Ind, false, false, T), Y, W, Ind, table.value_or(Tensor()), (int)mode, bias.value_or(Tensor()));
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads)
    {
        const auto saved = ctx->get_saved_variables();
        const Tensor &Y = saved[0], &W = saved[1], &Ind = saved[2];
        const bool bias = ctx->saved_data["bias"].toBool();
        const Problem p = problem_of(Y, W, Ind, false, false, ctx->saved_data["T"].toInt());
        Grads g;
        if (p.ok && grad_fits(grads[0], Y, {p.d.B, p.d.T, p.d.I})) {
            at::AutoDispatchBelowADInplaceOrView below;
            g = scatter_backward(p, Y, W, Ind, grads[0], bias);
        } else {
            g = backward_in_python("_scatter_backward_of_node", saved, grads[0], 0, bias);
        }
        return {g.in, g.W, Tensor(), g.bias, Tensor(), Tensor(), Tensor()};
    }
};

bool records(const Tensor &a, const Tensor &b, const Tensor &c)
{
    return at::GradMode::is_enabled() && (a.requires_grad() || b.requires_grad() || (c.defined() && c.requires_grad()));
}
// [E,1,N] in the operands' type, dense
bool bias_fits(const Tensor &b, const Tensor &W, int64_t E, int64_t N)
{
    return plain(b) && b.dim() == 3 && b.size(0) == E && b.size(1) == 1 && b.size(2) == N && b.scalar_type() == W.scalar_type() &&
           b.device() == W.device() && b.is_contiguous();
}
std::optional<Tensor> some(const Tensor &t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }
bool has_tangent(const Tensor &t) { return t._fw_grad(0).defined(); }

// ------------------------------------------------------------------------------ Python entry points
struct NoGil {
    PyThreadState *save;
    NoGil() : save(PyEval_SaveThread()) {}
    ~NoGil() { PyEval_RestoreThread(save); }
};

bool want(Py_ssize_t nargs, Py_ssize_t n, const char *name)
{
    if (nargs == n) return true;
    PyErr_Format(PyExc_TypeError, "%s takes %zd arguments, got %zd", name, n, nargs);
    return false;
}

// the compute type of hip_kernels._compute_dtype for operands of one type: that type, if `out_dtype` does not ask for another
bool type_fits(PyObject *out_dtype, const Tensor &t)
{
    if (!THPDtype_Check(out_dtype)) return false;
    const at::ScalarType want_t = ((THPDtype *)out_dtype)->scalar_type;
    return want_t == at::kFloat || want_t == t.scalar_type();
}

bool flag(PyObject *o) { return o == Py_True; }

PyObject *pair(std::pair<Tensor, Tensor> &&t)
{
    PyObject *a = THPVariable_Wrap(std::move(t.first)), *b = THPVariable_Wrap(std::move(t.second));
    if (a == nullptr || b == nullptr) { Py_XDECREF(a); Py_XDECREF(b); return nullptr; }
    return Py_BuildValue("(NN)", a, b);
}

// gather_forward(X, W, Ind, out_dtype, mode, keep_table, record, bias or None) -> Y or None; record: with an autograd node where
// one is due
PyObject *py_gather_forward(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (!want(n, 8, "gather_forward")) return nullptr;
    if (!plain_object(a[0]) || !plain_object(a[1]) || !plain_object(a[2]) || (a[7] != Py_None && !plain_object(a[7]))) Py_RETURN_NONE;
    const Tensor &X = THPVariable_Unpack(a[0]), &W = THPVariable_Unpack(a[1]), &Ind = THPVariable_Unpack(a[2]);
    const Problem p = problem_of(X, W, Ind, true, true, 0);
    if (!p.ok || !type_fits(a[3], X) || !no_modes()) Py_RETURN_NONE;
    const bool record = flag(a[6]);
    Tensor bias;
    if (a[7] != Py_None) {
        bias = THPVariable_Unpack(a[7]);
        if (!bias_fits(bias, W, p.d.E, p.d.J)) Py_RETURN_NONE;
    }
    if (record && (has_tangent(X) || has_tangent(W) || (bias.defined() && has_tangent(bias)))) Py_RETURN_NONE;
    const TableState ts = table_state(a[2], Ind, p, flag(a[5]));
    Tensor table, Y;
    const int64_t mode = PyLong_AsLong(a[4]);
    const bool build = ts.applies && !ts.table.defined();   // first sight of these indices: built in this launch
    {
        NoGil nogil;
        if (build) table = empty_gpu({(int64_t)ts.bytes}, at::kByte, p);
        if (record && records(X, W, bias)) Y = ExpertGatherFunctionNative::apply(X, W, Ind, some(bias), ts, some(table), mode);
        else Y = gather_forward(p, X, W, Ind, table, EGS_ACT_NONE, bias);
    }
    if (build) keep_table(a[2], ts.key, table);
    return THPVariable_Wrap(std::move(Y));
    END_HANDLE_TH_ERRORS
}

// scatter_forward(Y, W, Ind, T, out_dtype, mode, keep_table, record, bias or None) -> out or None
PyObject *py_scatter_forward(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (!want(n, 9, "scatter_forward")) return nullptr;
    if (!plain_object(a[0]) || !plain_object(a[1]) || !plain_object(a[2]) || !PyLong_CheckExact(a[3]) || (a[8] != Py_None && !plain_object(a[8])))
        Py_RETURN_NONE;
    const Tensor &Y = THPVariable_Unpack(a[0]), &W = THPVariable_Unpack(a[1]), &Ind = THPVariable_Unpack(a[2]);
    int overflow = 0;
    const int64_t T = PyLong_AsLongLongAndOverflow(a[3], &overflow);
    if (overflow != 0) Py_RETURN_NONE;
    const Problem p = problem_of(Y, W, Ind, false, false, T);
    if (!p.ok || !type_fits(a[4], Y) || !no_modes()) Py_RETURN_NONE;
    const bool record = flag(a[7]);
    Tensor bias;
    if (a[8] != Py_None) {
        bias = THPVariable_Unpack(a[8]);
        if (!bias_fits(bias, W, p.d.E, p.d.I)) Py_RETURN_NONE;
    }
    if (record && (has_tangent(Y) || has_tangent(W) || (bias.defined() && has_tangent(bias)))) Py_RETURN_NONE;
    const int mode = (int)PyLong_AsLong(a[5]);
    const TableState ts = table_state(a[2], Ind, p, flag(a[6]));
    Tensor out;
    {
        NoGil nogil;
        if (record && records(Y, W, bias)) out = ExpertScatterFunctionNative::apply(Y, W, Ind, some(bias), some(ts.table), T, (int64_t)mode);
        else out = scatter_forward(p, Y, W, Ind, ts.table, mode, bias);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// gather_backward(X, W, Ind, grad_output, out_dtype, mode, keep_table) -> (grad_X, grad_W) or None
PyObject *py_gather_backward(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (!want(n, 7, "gather_backward")) return nullptr;
    for (int i = 0; i < 4; ++i)
        if (!plain_object(a[i])) Py_RETURN_NONE;
    const Tensor &X = THPVariable_Unpack(a[0]), &W = THPVariable_Unpack(a[1]), &Ind = THPVariable_Unpack(a[2]), &G = THPVariable_Unpack(a[3]);
    const Problem p = problem_of(X, W, Ind, true, true, 0);
    if (!p.ok || !type_fits(a[4], X) || !no_modes() || !plain(G) || G.scalar_type() != X.scalar_type() || G.device() != X.device() ||
        !G.sizes().equals({p.d.B, p.d.E, p.d.K, p.d.J}) || !dense16(G))
        Py_RETURN_NONE;
    const int mode = (int)PyLong_AsLong(a[5]);
    const TableState ts = table_state(a[2], Ind, p, flag(a[6]));
    Grads g;
    {
        NoGil nogil;
        g = gather_backward(p, X, W, Ind, ts.table, G, mode);
    }
    return pair({g.in, g.W});
    END_HANDLE_TH_ERRORS
}

// scatter_backward(Y, W, Ind, grad_X, out_dtype) -> (grad_Y, grad_W) or None
PyObject *py_scatter_backward(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (!want(n, 5, "scatter_backward")) return nullptr;
    for (int i = 0; i < 4; ++i)
        if (!plain_object(a[i])) Py_RETURN_NONE;
    const Tensor &Y = THPVariable_Unpack(a[0]), &W = THPVariable_Unpack(a[1]), &Ind = THPVariable_Unpack(a[2]), &G = THPVariable_Unpack(a[3]);
    if (G.dim() != 3) Py_RETURN_NONE;
    const Problem p = problem_of(Y, W, Ind, false, false, G.size(1));
    if (!p.ok || !type_fits(a[4], Y) || !no_modes() || !plain(G) || G.scalar_type() != Y.scalar_type() || G.device() != Y.device() ||
        G.size(0) != p.d.B || G.size(2) != p.d.I || !dense16(G))
        Py_RETURN_NONE;
    Grads g;
    {
        NoGil nogil;
        g = scatter_backward(p, Y, W, Ind, G);
    }
    return pair({g.in, g.W});
    END_HANDLE_TH_ERRORS
}

// router(logits, K, ind_dtype) -> (Ind, scores) or None
PyObject *py_router(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (!want(n, 3, "router")) return nullptr;
    if (!plain_object(a[0]) || !PyLong_CheckExact(a[1]) || !THPDtype_Check(a[2])) Py_RETURN_NONE;
    const Tensor &logits = THPVariable_Unpack(a[0]);
    const at::ScalarType it = ((THPDtype *)a[2])->scalar_type;
    const long long K = PyLong_AsLongLong(a[1]);
    const int dt = plain(logits) ? type_id(logits.scalar_type()) : -1, ind = ind_type_id(it);
    if (dt < 0 || ind < 0 || logits.dim() != 3 || !logits.is_contiguous() || !no_modes() || has_tangent(logits) ||
        logits.device().index() != c10::hip::current_device() || (at::GradMode::is_enabled() && logits.requires_grad()))
        Py_RETURN_NONE;
    const int64_t B = logits.size(0), T = logits.size(1), E = logits.size(2);
    if (B < 1 || T < 1 || E < 1 || K < 1 || K > T || B > INT32_MAX || T > INT32_MAX || E > INT32_MAX) Py_RETURN_NONE;
    Tensor Ind, scores;
    int rc;
    {
        NoGil nogil;
        Problem p{};
        p.dev = logits.device().index();
        Ind = empty_gpu({B, E, K}, it, p);
        scores = empty_gpu({B, E, K}, at::kFloat, p);
        const size_t ws_bytes = egs_expert_choice_router_workspace_bytes((int32_t)B, (int32_t)T, (int32_t)E);
        Tensor ws;
        if (ws_bytes > 0) ws = empty_gpu({(int64_t)ws_bytes}, at::kByte, p);
        rc = egs_expert_choice_router(logits.const_data_ptr(), Ind.data_ptr(), (float *)scores.data_ptr(), ws_bytes > 0 ? ws.data_ptr() : nullptr,
                                      ws_bytes, (int32_t)B, (int32_t)T, (int32_t)E, (int32_t)K, dt, ind, stream_of(logits));
    }
    if (rc == EGS_ERR_UNSUPPORTED) Py_RETURN_NONE;
    raise_status(rc, "expert_choice_router");
    return pair({Ind, scores});
    END_HANDLE_TH_ERRORS
}

// mlp_forward(X, W_gather, W_scatter, Ind, activation, mode, keep_table, block) -> out, or None.  block: by the one-kernel block
// where it takes the operands; else the gather with the activation in its launch, and the scatter
PyObject *py_mlp_forward(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (!want(n, 8, "mlp_forward")) return nullptr;
    for (int i = 0; i < 4; ++i)
        if (!plain_object(a[i])) Py_RETURN_NONE;
    const Tensor &X = THPVariable_Unpack(a[0]), &Wg = THPVariable_Unpack(a[1]), &Ws = THPVariable_Unpack(a[2]), &Ind = THPVariable_Unpack(a[3]);
    const Problem p = problem_of(X, Wg, Ind, true, true, 0);
    if (!p.ok || !no_modes() || !plain(Ws) || Ws.dim() != 3 || Ws.scalar_type() != X.scalar_type() || Ws.device() != X.device() ||
        !dense16(Ws) || Ws.size(0) != p.d.E || Ws.size(1) != p.d.J || Ws.size(2) != p.d.I)
        Py_RETURN_NONE;
    const int act = (int)PyLong_AsLong(a[4]) & ~EGS_ACT_ROUND_FIRST, round = (int)PyLong_AsLong(a[4]) & EGS_ACT_ROUND_FIRST, mode = (int)PyLong_AsLong(a[5]);
    Tensor out;
    if (flag(a[7]) && egs_expert_mlp_supported(&p.d, p.dt)) {
        NoGil nogil;
        out = empty_gpu({p.d.B, p.d.T, p.d.I}, X.scalar_type(), p);
        const int rc = egs_expert_mlp_forward(X.const_data_ptr(), Wg.const_data_ptr(), Ws.const_data_ptr(), Ind.const_data_ptr(), out.data_ptr(),
                                              &p.d, (int64_t)p.d.T * p.d.I, p.d.I, p.dt, p.ind, act, stream_of(X));
        raise_status(rc, "expert_mlp_forward");
    } else {
        if (p.dt == EGS_F32 && act != EGS_ACT_NONE) Py_RETURN_NONE;
        TableState ts = table_state(a[3], Ind, p, flag(a[6]));
        Tensor table = ts.table;
        const bool build = ts.applies && !table.defined();
        {
            NoGil nogil;
            if (build) table = empty_gpu({(int64_t)ts.bytes}, at::kByte, p);
            const Tensor Y = gather_forward(p, X, Wg, Ind, build ? table : Tensor(), act | round);
            out = scatter_forward(p, Y, Ws, Ind, table, mode);
        }
        if (build) keep_table(a[3], ts.key, table);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// set_table_cache(allowed): from now on, also for the backward of calls made before
PyObject *py_set_table_cache(PyObject *, PyObject *on)
{
    g_tables_allowed.store(flag(on), std::memory_order_release);
    Py_RETURN_NONE;
}

PyObject *py_abi_version(PyObject *, PyObject *) { return PyLong_FromLong(egs_abi_version()); }

PyMethodDef methods[] = {
    {"gather_forward", (PyCFunction)(void (*)(void))py_gather_forward, METH_FASTCALL, "Y, or None: not for this way"},
    {"scatter_forward", (PyCFunction)(void (*)(void))py_scatter_forward, METH_FASTCALL, "out, or None: not for this way"},
    {"gather_backward", (PyCFunction)(void (*)(void))py_gather_backward, METH_FASTCALL, "(grad_X, grad_W), or None: not for this way"},
    {"scatter_backward", (PyCFunction)(void (*)(void))py_scatter_backward, METH_FASTCALL, "(grad_Y, grad_W), or None: not for this way"},
    {"router", (PyCFunction)(void (*)(void))py_router, METH_FASTCALL, "(Ind, scores), or None: not for this way"},
    {"mlp_forward", (PyCFunction)(void (*)(void))py_mlp_forward, METH_FASTCALL, "out, or None: not for this way"},
    {"set_table_cache", py_set_table_cache, METH_O, "whether routing tables may be read from now on"},
    {"abi_version", py_abi_version, METH_NOARGS, "ABI version of the library this module is linked to"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_egs_torch", "launchers and autograd Functions of libegs_hip.so on torch tensors", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__egs_torch(void)
{
    g_table_attr = PyUnicode_InternFromString("_egs_routing_table");
    g_owner_name = PyUnicode_InternFromString("expertscattergather_amd.hip_kernels");
    if (g_table_attr == nullptr || g_owner_name == nullptr) return nullptr;
    return PyModule_Create(&module);
}

// The entry points of the Python package as native callables.
//
// A call of a small product is host time: on an MI355X host 8.2 us through the Python function and ctypes (m = n = k = 512, calls in a
// row), of which the launch itself takes 2.5.  The rest was made of Python: attribute look-ups and checks of every tensor, the
// allocation, fifteen converted arguments.  Here a call is parsed, checked and launched without running Python: 5.1 us.
//
// An Entry wraps the package's Python function of the same name and takes the plain calls off it -- plain tensors of the expected
// dimensions on the GPU, integers, defaults.  Everything else (other types, views it does not take, an explicit stream, active
// dispatch or function modes, tracing, wrong arguments) goes to the Python function with the arguments as they came, which
// handles it or raises as ever.
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>
#include <cstring>

#include "../../include/ptoamd.h"

namespace {

constexpr int MAX_PARAMS = 16;
PyObject* g_error = nullptr;  // the package's PtoAmdError

// Thrown where a call is none of the plain ones.
struct NotPlain {};

struct Call {
    PyObject* v[MAX_PARAMS];  // by position; null: not given

    bool given(int i) const { return v[i] != nullptr && v[i] != Py_None; }
    void only_default(int i) const
    {
        if (given(i))
            throw NotPlain{};
    }
    int integer(int i) const
    {
        if (v[i] == nullptr || !PyLong_CheckExact(v[i]))
            throw NotPlain{};
        int overflow = 0;
        const long x = PyLong_AsLongAndOverflow(v[i], &overflow);
        if (overflow != 0 || x > INT_MAX || x < INT_MIN)
            throw NotPlain{};
        return (int)x;
    }
    int integer(int i, int missing) const { return v[i] == nullptr ? missing : integer(i); }
    bool truth(int i, bool missing) const
    {
        if (v[i] == nullptr)
            return missing;
        if (v[i] != Py_True && v[i] != Py_False)
            throw NotPlain{};
        return v[i] == Py_True;
    }
    int flags(int i) const { return v[i] == Py_True ? 1 : v[i] == Py_False ? 0 : integer(i, 0); }
    // a plain device tensor; contiguous, or where the call forwards its row pitch a matrix of contiguous rows
    const at::Tensor& tensor(int i, int dim, bool strided) const
    {
        if (v[i] == nullptr || !THPVariable_CheckExact(v[i]))
            throw NotPlain{};
        const at::Tensor& t = THPVariable_Unpack(v[i]);
        static const c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                                  c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                                  c10::DispatchKey::ZeroTensor});
        if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() || t.key_set().has_any(wrapped) || t.dim() != dim)
            throw NotPlain{};
        if (!t.is_contiguous() && !(strided && dim == 2 && t.stride(1) == 1))
            throw NotPlain{};
        return t;
    }
};

int extent(int64_t x)
{
    if (x > INT_MAX || x < INT_MIN)
        throw NotPlain{};
    return (int)x;
}

at::ScalarType out_type(int type)
{
    switch (type) {
        case PTOAMD_F32: return at::kFloat;
        case PTOAMD_F16: return at::kHalf;
        case PTOAMD_BF16: return at::kBFloat16;
        case PTOAMD_I32: return at::kInt;
        default: throw NotPlain{};
    }
}

at::Tensor empty(at::IntArrayRef shape, at::ScalarType type, const at::Tensor& like)
{
    return at::empty(shape, at::TensorOptions().dtype(type).device(like.device()));
}

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

void* address(const at::Tensor& t) { return t.data_ptr(); }
void* address(const at::Tensor* t) { return t == nullptr ? nullptr : t->data_ptr(); }
template <class T>
T* address_as(const at::Tensor& t)
{
    return static_cast<T*>(t.data_ptr());
}

// What a launch does without the interpreter: threads run meanwhile, as they do behind a ctypes call.
struct Released {
    PyThreadState* state = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(state); }
};

struct Failure {
    const char* what;
    int rc;
};
void check(int rc, const char* what)
{
    if (rc != 0)
        throw Failure{what, rc};
}

PyObject* wrap(at::Tensor&& t) { return THPVariable_Wrap(std::move(t)); }

// ---- the entry points: parameters in the order of the package's functions ------------------------------------------------

// a, b, ab_type, c_type, b_layout, c_in, relu, m, n, k, stream, out, bias, workspace
PyObject* gemm(const Call& c)
{
    for (int i : {5, 7, 8, 9, 10})
        c.only_default(i);
    const at::Tensor &a = c.tensor(0, 2, true), &b = c.tensor(1, 2, true);
    const int ab_type = c.integer(2), c_type = c.integer(3, PTOAMD_F32), b_layout = c.integer(4, PTOAMD_B_DN), relu = c.flags(6);
    const int m = extent(a.size(0)), k = extent(a.size(1)), n = extent(b_layout == PTOAMD_B_DN ? b.size(0) : b.size(1));
    const int lda = extent(a.stride(0)), ldb = extent(b.stride(0));
    const at::Tensor* bias = c.given(12) ? &c.tensor(12, 1, false) : nullptr;
    const at::Tensor* ws = c.given(13) ? &c.tensor(13, 1, false) : nullptr;
    at::Tensor out;
    if (c.given(11))
        out = c.tensor(11, 2, true);
    const at::ScalarType type = out.defined() ? at::kByte : out_type(c_type);
    {
        Released no_gil;
        if (!out.defined())
            out = empty({m, n}, type, a);
        const int ldc = extent(out.stride(0));
        if (ws != nullptr)
            check(ptoamd_gemm_ws(address(out), c_type, address(a), address(b), ab_type, nullptr, address(bias), m, n, k, lda, ldb, ldc, b_layout, relu,
                                 address(ws), ws->nbytes(), stream()), "ptoamd_gemm_ws");
        else if (bias != nullptr)
            check(ptoamd_gemm_bias(address(out), c_type, address(a), address(b), ab_type, nullptr, address(bias), m, n, k, lda, ldb, ldc, b_layout, relu,
                                   stream()), "ptoamd_gemm_bias");
        else
            check(ptoamd_gemm(address(out), c_type, address(a), address(b), ab_type, nullptr, m, n, k, lda, ldb, ldc, b_layout, relu, stream()),
                  "ptoamd_gemm");
    }
    return wrap(std::move(out));
}

// a, b, scale_a, scale_b, b_layout, want_acc, stream, out
PyObject* gemm_w8a8(const Call& c)
{
    c.only_default(6);
    if (c.truth(5, false))
        throw NotPlain{};
    const at::Tensor &a = c.tensor(0, 2, true), &b = c.tensor(1, 2, true), &sa = c.tensor(2, 1, false), &sb = c.tensor(3, 1, false);
    const int b_layout = c.integer(4, PTOAMD_B_DN);
    const int m = extent(a.size(0)), k = extent(a.size(1)), n = extent(b_layout == PTOAMD_B_DN ? b.size(0) : b.size(1));
    const int lda = extent(a.stride(0)), ldb = extent(b.stride(0));
    at::Tensor out;
    if (c.given(7))
        out = c.tensor(7, 2, true);
    {
        Released no_gil;
        if (!out.defined())
            out = empty({m, n}, at::kBFloat16, a);
        check(ptoamd_gemm_w8a8(address(out), nullptr, address_as<const int8_t>(a), address_as<const int8_t>(b), address_as<const float>(sa),
                               address_as<const float>(sb), m, n, k, lda, ldb, extent(out.stride(0)), b_layout, stream()), "ptoamd_gemm_w8a8");
    }
    return wrap(std::move(out));
}

// a, b, sa, sb, m, n, k, a_type, b_type, c_type, sa_layout, sb_layout, b_layout, c_in, stream, out  (workspace, bias: the Python function)
PyObject* gemm_mx(const Call& c)
{
    for (int i : {13, 14, 15})
        c.only_default(i);
    const at::Tensor &a = c.tensor(0, 2, false), &b = c.tensor(1, 2, false), &sa = c.tensor(2, 2, false), &sb = c.tensor(3, 2, false);
    const int m = c.integer(4), n = c.integer(5), k = c.integer(6), a_type = c.integer(7), b_type = c.integer(8), c_type = c.integer(9, PTOAMD_F32);
    const int sa_layout = c.integer(10, PTOAMD_MX_A_ND), sb_layout = c.integer(11, PTOAMD_MX_B_DN), b_layout = c.integer(12, PTOAMD_B_DN);
    if (m < 0 || n < 0)
        throw NotPlain{};
    const at::ScalarType type = out_type(c_type);
    at::Tensor out;
    {
        Released no_gil;
        out = empty({m, n}, type, a);
        check(ptoamd_gemm_mx(address(out), c_type, address(a), address(b), a_type, b_type, address_as<const uint8_t>(sa), address_as<const uint8_t>(sb),
                             sa_layout, sb_layout, nullptr, m, n, k, k, b_layout == PTOAMD_B_DN ? k : n, extent(out.stride(0)), b_layout, stream()),
              "ptoamd_gemm_mx");
    }
    return wrap(std::move(out));
}

// a_bf16, w, sw, n, k, c_type, stream, out
PyObject* gemv_mxfp4(const Call& c)
{
    for (int i : {6, 7})
        c.only_default(i);
    const at::Tensor &a = c.tensor(0, 2, true), &w = c.tensor(1, 2, false), &sw = c.tensor(2, 2, false);
    const int n = c.integer(3), k = c.integer(4), c_type = c.integer(5, PTOAMD_F32), m = extent(a.size(0)), lda = extent(a.stride(0));
    if (n < 0)
        throw NotPlain{};
    const at::ScalarType type = out_type(c_type);
    at::Tensor out;
    {
        Released no_gil;
        out = empty({m, n}, type, w);
        check(ptoamd_gemv_mxfp4(address(out), c_type, address(a), address_as<const uint8_t>(w), address_as<const uint8_t>(sw), m, n, k, lda, k,
                                extent(out.stride(0)), stream()), "ptoamd_gemv_mxfp4");
    }
    return wrap(std::move(out));
}

// a_bf16, packed, n, k, c_type, stream, out
PyObject* gemv_mxfp4_packed(const Call& c)
{
    for (int i : {5, 6})
        c.only_default(i);
    const at::Tensor &a = c.tensor(0, 2, true), &w = c.tensor(1, 1, false);
    const int n = c.integer(2), k = c.integer(3), c_type = c.integer(4, PTOAMD_F32), m = extent(a.size(0)), lda = extent(a.stride(0));
    if (n < 0)
        throw NotPlain{};
    const at::ScalarType type = out_type(c_type);
    at::Tensor out;
    {
        Released no_gil;
        out = empty({m, n}, type, w);
        check(ptoamd_gemv_mxfp4_packed(address(out), c_type, address(a), address_as<const uint8_t>(w), m, n, k, lda, extent(out.stride(0)), stream()),
              "ptoamd_gemv_mxfp4_packed");
    }
    return wrap(std::move(out));
}

// src, scale, offset, stream, out
PyObject* tquant_int8(const Call& c)
{
    for (int i : {3, 4})
        c.only_default(i);
    const at::Tensor &src = c.tensor(0, 2, false), &scale = c.tensor(1, 1, false);
    const at::Tensor* offset = c.given(2) ? &c.tensor(2, 1, false) : nullptr;
    const int rows = extent(src.size(0)), cols = extent(src.size(1));
    at::Tensor out;
    {
        Released no_gil;
        out = empty({rows, cols}, offset == nullptr ? at::kChar : at::kByte, src);
        check(ptoamd_tquant_int8(address(out), address_as<const float>(src), address_as<const float>(scale), static_cast<const float*>(address(offset)),
                                 rows, cols, stream()), "ptoamd_tquant_int8");
    }
    return wrap(std::move(out));
}

// src, alg, axis, want_aux, stream, out
PyObject* tquant_mx(const Call& c)
{
    for (int i : {4, 5})
        c.only_default(i);
    const at::Tensor& src = c.tensor(0, 2, false);
    const int alg = c.integer(1), axis = c.integer(2, 1), rows = extent(src.size(0)), cols = extent(src.size(1));
    const bool aux = c.truth(3, true), fp4 = alg == PTOAMD_OCP_MXFP4 || alg == PTOAMD_NV_MXFP4;
    const at::ScalarType t = src.scalar_type();
    const int src_type = t == at::kFloat ? PTOAMD_F32 : t == at::kHalf ? PTOAMD_F16 : t == at::kBFloat16 ? PTOAMD_BF16 : -1;
    if (src_type < 0)
        throw NotPlain{};
    const int64_t grows = axis == 1 ? rows : rows / 32, gcols = axis == 1 ? cols / 32 : cols;
    at::Tensor codes, exps, maxima, scaling;
    {
        Released no_gil;
        codes = empty({rows, fp4 ? cols / 2 : cols}, at::kByte, src);
        exps = empty({grows, gcols}, at::kByte, src);
        if (aux) {
            maxima = empty({grows, gcols}, at::kFloat, src);
            scaling = empty({grows, gcols}, at::kFloat, src);
        }
        check(ptoamd_tquant_mx(address_as<uint8_t>(codes), address_as<uint8_t>(exps), aux ? address_as<float>(maxima) : nullptr,
                               aux ? address_as<float>(scaling) : nullptr, address(src), src_type, rows, cols, alg, axis, stream()), "ptoamd_tquant_mx");
    }
    PyObject* result = PyTuple_New(aux ? 4 : 2);
    if (result == nullptr)
        return nullptr;
    PyTuple_SET_ITEM(result, 0, wrap(std::move(codes)));
    PyTuple_SET_ITEM(result, 1, wrap(std::move(exps)));
    if (aux) {
        PyTuple_SET_ITEM(result, 2, wrap(std::move(maxima)));
        PyTuple_SET_ITEM(result, 3, wrap(std::move(scaling)));
    }
    return result;
}

// src, scale, offset, stream, out
PyObject* tdequant(const Call& c)
{
    for (int i : {3, 4})
        c.only_default(i);
    const at::Tensor &src = c.tensor(0, 2, false), &scale = c.tensor(1, 1, false), &offset = c.tensor(2, 1, false);
    const at::ScalarType t = src.scalar_type();
    const int src_type = t == at::kChar ? PTOAMD_I8 : t == at::kShort ? PTOAMD_I16 : t == at::kInt ? PTOAMD_I32 : -1;
    if (src_type < 0)
        throw NotPlain{};
    const int rows = extent(src.size(0)), cols = extent(src.size(1));
    at::Tensor out;
    {
        Released no_gil;
        out = empty({rows, cols}, at::kFloat, src);
        check(ptoamd_tdequant(address_as<float>(out), address(src), src_type, address_as<const float>(scale), address_as<const float>(offset), rows,
                              cols, stream()), "ptoamd_tdequant");
    }
    return wrap(std::move(out));
}

struct Native {
    const char* name;
    PyObject* (*run)(const Call&);
    int required;
    const char* params[MAX_PARAMS];
};
const Native natives[] = {
    {"gemm", gemm, 3, {"a", "b", "ab_type", "c_type", "b_layout", "c_in", "relu", "m", "n", "k", "stream", "out", "bias", "workspace"}},
    {"gemm_w8a8", gemm_w8a8, 4, {"a", "b", "scale_a", "scale_b", "b_layout", "want_acc", "stream", "out"}},
    {"gemm_mx", gemm_mx, 9, {"a", "b", "sa", "sb", "m", "n", "k", "a_type", "b_type", "c_type", "sa_layout", "sb_layout", "b_layout", "c_in", "stream", "out"}},
    {"gemv_mxfp4", gemv_mxfp4, 5, {"a_bf16", "w", "sw", "n", "k", "c_type", "stream", "out"}},
    {"gemv_mxfp4_packed", gemv_mxfp4_packed, 4, {"a_bf16", "packed", "n", "k", "c_type", "stream", "out"}},
    {"tquant_int8", tquant_int8, 2, {"src", "scale", "offset", "stream", "out"}},
    {"tquant_mx", tquant_mx, 2, {"src", "alg", "axis", "want_aux", "stream", "out"}},
    {"tdequant", tdequant, 3, {"src", "scale", "offset", "stream", "out"}},
};

// ---- the callable -------------------------------------------------------------------------------------------------------

struct Entry {
    PyObject_HEAD
    vectorcallfunc call;
    PyObject* python;  // the package's function
    PyObject* dict;
    PyObject* weak;
    const Native* native;
    PyObject* params[MAX_PARAMS];  // interned names
    int count;
};

// dispatch or function modes, functorch levels, tracing: anything that sees torch's own calls
bool modes_active()
{
    static const c10::DispatchKeySet keys({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                           c10::DispatchKey::FuncTorchDynamicLayerBackMode, c10::DispatchKey::Functionalize, c10::DispatchKey::Tracer});
    return c10::impl::tls_local_dispatch_key_set().included_.has_any(keys) || at::impl::torch_function_mode_enabled();
}

bool parse(const Entry* e, Call& c, PyObject* const* args, Py_ssize_t n, PyObject* kwnames)
{
    if (n > e->count)
        return false;
    for (int i = 0; i < e->count; ++i)
        c.v[i] = i < n ? args[i] : nullptr;
    const Py_ssize_t keywords = kwnames == nullptr ? 0 : PyTuple_GET_SIZE(kwnames);
    for (Py_ssize_t q = 0; q < keywords; ++q) {
        PyObject* name = PyTuple_GET_ITEM(kwnames, q);
        int i = 0;
        while (i < e->count && e->params[i] != name)
            ++i;
        if (i == e->count || c.v[i] != nullptr)  // (a name that is not interned as well)
            return false;
        c.v[i] = args[n + q];
    }
    for (int i = 0; i < e->native->required; ++i)
        if (c.v[i] == nullptr)
            return false;
    return true;
}

PyObject* entry_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames)
{
    const Entry* e = reinterpret_cast<const Entry*>(self);
    Call c;
    if (parse(e, c, args, PyVectorcall_NARGS(nargsf), kwnames) && !modes_active()) {
        HANDLE_TH_ERRORS
        try {
            return e->native->run(c);
        } catch (const NotPlain&) {
        } catch (const Failure& f) {
            PyErr_Format(g_error, "%s failed (%d): %s", f.what, f.rc, ptoamd_last_error());
            return nullptr;
        }
        END_HANDLE_TH_ERRORS
    }
    return PyObject_Vectorcall(e->python, args, nargsf, kwnames);
}

int entry_traverse(PyObject* self, visitproc visit, void* arg)
{
    Entry* e = reinterpret_cast<Entry*>(self);
    Py_VISIT(e->python);
    Py_VISIT(e->dict);
    return 0;
}
int entry_clear(PyObject* self)
{
    Entry* e = reinterpret_cast<Entry*>(self);
    Py_CLEAR(e->python);
    Py_CLEAR(e->dict);
    return 0;
}
void entry_dealloc(PyObject* self)
{
    PyObject_GC_UnTrack(self);
    if (reinterpret_cast<Entry*>(self)->weak != nullptr)
        PyObject_ClearWeakRefs(self);
    entry_clear(self);
    for (PyObject* p : reinterpret_cast<Entry*>(self)->params)
        Py_XDECREF(p);
    PyObject_GC_Del(self);
}
PyObject* entry_repr(PyObject* self) { return PyObject_Repr(reinterpret_cast<Entry*>(self)->python); }
// what a function has and this does not: its attributes, __code__, __defaults__, __globals__ ...
PyObject* entry_getattro(PyObject* self, PyObject* name)
{
    PyObject* own = PyObject_GenericGetAttr(self, name);
    if (own != nullptr || !PyErr_ExceptionMatches(PyExc_AttributeError))
        return own;
    PyErr_Clear();
    return PyObject_GetAttr(reinterpret_cast<Entry*>(self)->python, name);
}
// as a function: by its qualified name in its module
PyObject* entry_reduce(PyObject* self, PyObject*) { return PyObject_GetAttrString(reinterpret_cast<Entry*>(self)->python, "__qualname__"); }
PyObject* entry_same(PyObject* self, PyObject*)
{
    Py_INCREF(self);
    return self;
}

// (a class attribute binds to its instances)
PyObject* entry_get(PyObject* self, PyObject* instance, PyObject*)
{
    if (instance == nullptr || instance == Py_None)
        return entry_same(self, nullptr);
    return PyMethod_New(self, instance);
}

PyMethodDef entry_methods[] = {{"__reduce__", entry_reduce, METH_NOARGS, nullptr},
                               {"__copy__", entry_same, METH_NOARGS, nullptr},
                               {"__deepcopy__", entry_same, METH_O, nullptr},
                               {nullptr, nullptr, 0, nullptr}};

PyTypeObject entry_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* wrap_function(PyObject*, PyObject* function)
{
    PyObject* name = PyObject_GetAttrString(function, "__name__");
    const char* text = name == nullptr ? nullptr : PyUnicode_AsUTF8(name);
    if (text == nullptr) {
        Py_XDECREF(name);
        return nullptr;
    }
    const Native* native = nullptr;
    for (const Native& n : natives)
        if (strcmp(n.name, text) == 0)
            native = &n;
    Py_DECREF(name);
    if (native == nullptr) {
        PyErr_SetString(PyExc_ValueError, "no native entry point of this name");
        return nullptr;
    }
    Entry* e = PyObject_GC_New(Entry, &entry_type);
    if (e == nullptr)
        return nullptr;
    memset(reinterpret_cast<char*>(e) + sizeof(PyObject), 0, sizeof(Entry) - sizeof(PyObject));
    e->call = entry_call;
    e->native = native;
    Py_INCREF(function);
    e->python = function;
    e->dict = PyDict_New();
    while (e->count < MAX_PARAMS && native->params[e->count] != nullptr) {
        e->params[e->count] = PyUnicode_InternFromString(native->params[e->count]);
        ++e->count;
    }
    PyObject_GC_Track(e);
    for (const char* attr : {"__module__", "__name__", "__qualname__", "__doc__"}) {
        PyObject* value = PyObject_GetAttrString(function, attr);
        if (e->dict == nullptr || value == nullptr || PyDict_SetItemString(e->dict, attr, value) != 0) {
            Py_XDECREF(value);
            Py_DECREF(e);
            return nullptr;
        }
        Py_DECREF(value);
    }
    if (PyDict_SetItemString(e->dict, "__wrapped__", function) != 0) {  // (what inspect.signature follows)
        Py_DECREF(e);
        return nullptr;
    }
    return reinterpret_cast<PyObject*>(e);
}

PyObject* set_error(PyObject*, PyObject* type)
{
    Py_INCREF(type);
    Py_XDECREF(g_error);
    g_error = type;
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"entry_point", wrap_function, METH_O, "The native form of the package's function of that name."},
                         {"set_error", set_error, METH_O, "The exception that a failing call raises."},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "ptoamd_binding", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_ptoamd_binding()
{
    entry_type.tp_name = "ptoamd_binding.EntryPoint";
    entry_type.tp_basicsize = sizeof(Entry);
    entry_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC | Py_TPFLAGS_HAVE_VECTORCALL;
    entry_type.tp_vectorcall_offset = offsetof(Entry, call);
    entry_type.tp_call = PyVectorcall_Call;
    entry_type.tp_dictoffset = offsetof(Entry, dict);
    entry_type.tp_weaklistoffset = offsetof(Entry, weak);
    entry_type.tp_descr_get = entry_get;
    entry_type.tp_traverse = entry_traverse;
    entry_type.tp_clear = entry_clear;
    entry_type.tp_dealloc = entry_dealloc;
    entry_type.tp_repr = entry_repr;
    entry_type.tp_getattro = entry_getattro;
    entry_type.tp_methods = entry_methods;
    if (PyType_Ready(&entry_type) < 0)
        return nullptr;
    PyObject* m = PyModule_Create(&module);
    // (what the package compares before it takes an entry point from here; the Python version is in the file's name)
    if (m != nullptr && PyModule_AddStringConstant(m, "torch_id", PTOAMD_TORCH_ID) != 0)
        Py_CLEAR(m);
    return m;
}

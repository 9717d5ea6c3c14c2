// The host side of a repeated call, in native code: a GEMM entry point that has served a call once (yan_amd/jit_kernels) leaves here what
// its launch takes, under the sizes, strides, types, devices and alignment of its tensors and its plain arguments. A later call that agrees in all of
// them would pass the same checks and make the same launch from other addresses; it is made from here. Everything else, and whatever could
// have changed the plan (the compute-unit cap, the environment switches), goes back to Python; so does a launch with a workspace on a stream
// that has none yet, and under a capture, which has its own. A launch without one is recorded into a capture as it is.
//
// What it is for: one 1 x 2112 x 7168 FP8 call costs the host 8.5 us from Python and 3.5 from here, of which 2.5 are the launch; the kernel takes
// 5. Two streams in turn, with a workspace each: 23.4 us for both calls and the switches of streams by Python, 14.0 from here.
// What it compiles in of torch's objects holds for one torch: `built_for` names it, and host_calls.py uses no module built for another.
// Nothing is kept by address or identity: addresses are read from the tensors of each call, the workspace from split_k.py's own record.
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <cstdint>
#include <cstring>
#include <memory>
#include <string>
#include <unordered_map>
#include <utility>
#include <vector>

namespace {

constexpr int kMaxKey = 96, kMaxArgs = 20, kMaxFloats = 2;
constexpr size_t kMaxCalls = 4096;          // then the table starts anew: a program of ever new sizes does not grow it

enum Kind : int { kTensor = 0, kConstant = 1, kStream = 2, kWorkspace = 3 };

struct Launch {
    std::vector<int64_t> key;
    std::string name;                           // for the error message
    void* function;
    int count;
    bool workspace;
    std::array<int, kMaxArgs> kind;
    std::array<int64_t, kMaxArgs> value;        // a constant, or which tensor
};

std::unordered_multimap<uint64_t, std::shared_ptr<Launch>> g_launches;
PyObject *g_utils, *g_split_k, *g_os, *g_environ, *g_environ_bytes, *g_device, *g_stream, *g_capturing;
PyObject *s_num_sms, *s_last, *s_book, *s_eager, *s_suspect, *s_failed, *s_environ, *b_split_k, *b_tune;

struct Call {
    int64_t key[kMaxKey];
    int used = 0;
    uint64_t address[16];
    int tensors = 0;
    float floats[kMaxFloats] = {0.f, 0.f};
    int num_floats = 0;
    int64_t device = -1;
    bool put(int64_t v) {
        if (used == kMaxKey) return false;
        key[used++] = v;
        return true;
    }
    uint64_t hash() const {
        uint64_t h = 0x9e3779b97f4a7c15ull + used;
        for (int i = 0; i < used; ++i) {
            h ^= uint64_t(key[i]);
            h *= 0xff51afd7ed558ccdull;
            h ^= h >> 32;
        }
        return h;
    }
};

// A C long out of a Python int; false for anything else.
bool plain_int(PyObject* o, int64_t* v) {
    if (!o || !PyLong_CheckExact(o)) return false;
    *v = PyLong_AsLongLong(o);
    if (*v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

bool call_int(PyObject* f, PyObject* arg, int64_t* v) {
    PyObject* r = arg ? PyObject_CallOneArg(f, arg) : PyObject_CallNoArgs(f);
    if (!r) {
        PyErr_Clear();
        return false;
    }
    const bool ok = plain_int(r, v);
    Py_DECREF(r);
    return ok;
}

// What the arguments of a call are apart from their addresses. False: not a call for this file.
bool describe(Call& c, PyObject* const* objs, Py_ssize_t n) {
    int64_t entry, sms;
    if (n < 2 || n > 16 || !plain_int(objs[0], &entry)) return false;
    if (!plain_int(PyDict_GetItemWithError(g_utils, s_num_sms), &sms)) return false;
    if (!call_int(g_device, nullptr, &c.device)) return false;
    if (!c.put(entry) || !c.put(sms) || !c.put(c.device)) return false;
    for (Py_ssize_t i = 1; i < n; ++i) {
        PyObject* o = objs[i];
        if (THPVariable_CheckExact(o)) {
            const at::Tensor& t = THPVariable_Unpack(o);
            if (t.layout() != at::kStrided || !t.is_cuda() || t.device().index() != c.device) return false;
            const auto sizes = t.sizes(), strides = t.strides();
            const uint64_t address = reinterpret_cast<uint64_t>(t.data_ptr());
            // (of an address Python looks at nothing but the alignment, scales_for_kernel)
            if (!c.put((int64_t(t.scalar_type()) * 64 + int64_t(sizes.size())) * 16 + int64_t(address % 16))) return false;
            for (size_t d = 0; d < sizes.size(); ++d)
                if (!c.put(sizes[d]) || !c.put(strides[d])) return false;
            c.address[c.tensors++] = address;
        } else if (PyFloat_CheckExact(o)) {
            if (c.num_floats == kMaxFloats || !c.put(-7)) return false;
            c.floats[c.num_floats++] = float(PyFloat_AS_DOUBLE(o));
        } else {
            int64_t v;
            if (!plain_int(o, &v) || !c.put(-9) || !c.put(v)) return false;
        }
    }
    return true;
}

std::shared_ptr<Launch> find(const Call& c) {
    const auto range = g_launches.equal_range(c.hash());
    for (auto it = range.first; it != range.second; ++it)
        if (int(it->second->key.size()) == c.used && std::memcmp(it->second->key.data(), c.key, size_t(c.used) * 8) == 0) return it->second;
    return nullptr;
}

// The switches as they are when nobody has touched them: K may be split, tiles are not timed.
bool usual_switches() {
    if (PyDict_GetItemWithError(g_os, s_environ) != g_environ) return false;
    auto on = [](PyObject* name, bool otherwise) {
        PyObject* v = PyDict_GetItemWithError(g_environ_bytes, name);
        if (!v) return otherwise;
        if (!PyBytes_CheckExact(v)) return !otherwise;
        return !(PyBytes_GET_SIZE(v) == 0 || (PyBytes_GET_SIZE(v) == 1 && PyBytes_AS_STRING(v)[0] == '0'));
    };
    return on(b_split_k, true) && !on(b_tune, false);
}

#if !defined(__x86_64__) || !defined(__linux__)
#error "launch_with passes arguments as the System V ABI of x86-64 does"
#endif
// Integer arguments go where integers go and floating-point ones where those go, whatever their order among each other (x86-64).
template <size_t... I>
int launch_with(void* f, const uint64_t* a, const float* fl, std::index_sequence<I...>) {
    int rc = 0;
    reinterpret_cast<void (*)(decltype(a[I] + 0)..., int*, float, float)>(f)(a[I]..., &rc, fl[0], fl[1]);
    return rc;
}
template <int N>
int launch_of(int count, void* f, const uint64_t* a, const float* fl) {
    if (count == N) return launch_with(f, a, fl, std::make_index_sequence<N>{});
    if constexpr (N > 1) return launch_of<N - 1>(count, f, a, fl);
    return -1;
}

// The workspace of eager launches on a stream and the token that goes with it, as new references: the latest launch's if it was on this
// stream (split_k._last), else what the book holds for it, unless a launch there failed. False: for Python to make or clear.
bool eager_workspace(int64_t device, int64_t stream, PyObject** token, PyObject** workspace) {
    PyObject* last = PyDict_GetItemWithError(g_split_k, s_last);
    int64_t index, owner;
    if (last && PyTuple_CheckExact(last) && PyTuple_GET_SIZE(last) == 2) {
        PyObject *t = PyTuple_GET_ITEM(last, 0), *w = PyTuple_GET_ITEM(last, 1);
        if (PyTuple_CheckExact(t) && PyTuple_GET_SIZE(t) == 3 && PyTuple_GET_ITEM(t, 2) == Py_None && plain_int(PyTuple_GET_ITEM(t, 0), &index) &&
            index == device && plain_int(PyTuple_GET_ITEM(t, 1), &owner) && owner == stream && THPVariable_CheckExact(w)) {
            Py_INCREF(*token = t);
            Py_INCREF(*workspace = w);
            return true;
        }
    }
    PyObject* book = PyDict_GetItemWithError(g_split_k, s_book);
    PyObject* held = book ? PyObject_GetAttr(book, s_eager) : nullptr;
    PyObject* suspect = held ? PyObject_GetAttr(book, s_suspect) : nullptr;
    PyObject* key = suspect ? Py_BuildValue("(LL)", (long long)device, (long long)stream) : nullptr;
    bool found = false;
    if (key && PyDict_CheckExact(held) && PyAnySet_Check(suspect)) {
        PyObject* w = PyDict_GetItemWithError(held, key);
        if (w && THPVariable_CheckExact(w) && PySet_Contains(suspect, key) == 0) {
            Py_INCREF(w);
            if ((*token = Py_BuildValue("(LLO)", (long long)device, (long long)stream, Py_None))) {
                *workspace = w;
                found = true;
            } else Py_DECREF(w);
        }
    }
    Py_XDECREF(key);
    Py_XDECREF(suspect);
    Py_XDECREF(held);
    return found;
}

// A launch that reported an error, as the Python way reports it. It is not made again: the code can be that of an older error of this
// thread, asked for behind a launch that did run (c = alpha a b + beta c would be applied twice).
PyObject* launch_failed(const std::string& name, PyObject* token, int rc) {
    if (token) {
        PyObject* mark = PyDict_GetItemWithError(g_split_k, s_failed);
        PyObject* done = mark ? PyObject_CallOneArg(mark, token) : nullptr;
        Py_XDECREF(done);
        if (PyErr_Occurred()) return nullptr;
    }
    return PyErr_Format(PyExc_AssertionError, "%s failed with HIP error %d", name.c_str(), rc);
}

// call(entry, *arguments): True if the launch was made, AssertionError if it failed.
PyObject* call(PyObject*, PyObject* const* objs, Py_ssize_t n) {
    if (!g_utils || g_launches.empty()) Py_RETURN_FALSE;
    try {
        Call c;
        if (!usual_switches() || !describe(c, objs, n)) Py_RETURN_FALSE;
        // held, not looked at in the table: what is called below can run other Python code, and other threads, that clear it
        const std::shared_ptr<const Launch> l = find(c);
        if (!l) Py_RETURN_FALSE;
        PyObject* device = PyLong_FromLongLong(c.device);
        int64_t stream;
        const bool have_stream = call_int(g_stream, device, &stream);
        Py_DECREF(device);
        if (!have_stream) Py_RETURN_FALSE;
        PyObject *workspace = nullptr, *token = nullptr;
        uint64_t workspace_address = 0;
        if (l->workspace) {
            // a capture has its own
            PyObject* capturing = PyObject_CallNoArgs(g_capturing);
            const bool eager = capturing == Py_False;
            Py_XDECREF(capturing);
            if (!eager || !eager_workspace(c.device, stream, &token, &workspace)) {
                PyErr_Clear();
                Py_RETURN_FALSE;
            }
            workspace_address = reinterpret_cast<uint64_t>(THPVariable_Unpack(workspace).data_ptr());
        }
        uint64_t args[kMaxArgs];
        for (int i = 0; i < l->count; ++i) {
            switch (l->kind[i]) {
                case kTensor: args[i] = c.address[l->value[i]]; break;
                case kConstant: args[i] = uint64_t(l->value[i]); break;
                case kStream: args[i] = uint64_t(stream); break;
                default: args[i] = workspace_address;
            }
        }
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = launch_of<kMaxArgs>(l->count, l->function, args, c.floats);
        Py_END_ALLOW_THREADS
        Py_XDECREF(workspace);
        PyObject* const failed = rc != 0 ? launch_failed(l->name, token, rc) : nullptr;
        Py_XDECREF(token);
        if (rc != 0) return failed;
        Py_RETURN_TRUE;
    } catch (...) {         // a tensor without storage, say: the checks in Python will say so
        PyErr_Clear();
        Py_RETURN_FALSE;
    }
}

// remember((entry, *arguments), name, address, ((kind, value), ...)): the launch that served these arguments.
PyObject* remember(PyObject*, PyObject* args) {
    PyObject *objs, *spec;
    const char* name;
    unsigned long long address;
    if (!PyArg_ParseTuple(args, "O!sKO!", &PyTuple_Type, &objs, &name, &address, &PyTuple_Type, &spec)) return nullptr;
    try {
        Call c;
        std::vector<PyObject*> items;
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(objs); ++i) items.push_back(PyTuple_GET_ITEM(objs, i));
        const Py_ssize_t count = PyTuple_GET_SIZE(spec);
        if (!g_utils || count < 1 || count > kMaxArgs || !describe(c, items.data(), Py_ssize_t(items.size()))) Py_RETURN_FALSE;
        auto l = std::make_shared<Launch>();
        l->key.assign(c.key, c.key + c.used);
        l->name = name;
        l->function = reinterpret_cast<void*>(address);
        l->count = int(count);
        l->workspace = false;
        for (Py_ssize_t i = 0; i < count; ++i) {
            long long kind, value;
            if (!PyArg_ParseTuple(PyTuple_GET_ITEM(spec, i), "LL", &kind, &value)) return nullptr;
            if (kind < kTensor || kind > kWorkspace || (kind == kTensor && (value < 0 || value >= c.tensors))) Py_RETURN_FALSE;
            l->kind[size_t(i)] = int(kind);
            l->value[size_t(i)] = value;
            l->workspace |= kind == kWorkspace;
        }
        if (g_launches.size() >= kMaxCalls) g_launches.clear();
        const auto range = g_launches.equal_range(c.hash());
        auto at = range.first;
        while (at != range.second && at->second->key != l->key) ++at;
        if (at != range.second) at->second = std::move(l);
        else g_launches.emplace(c.hash(), std::move(l));
        Py_RETURN_TRUE;
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_FALSE;
    }
}

PyObject* forget(PyObject*, PyObject*) {
    g_launches.clear();
    Py_RETURN_NONE;
}

// setup(utils' globals, split_k's globals, os' globals, os.environ, its bytes, current device, raw stream of a device, whether it captures)
PyObject* setup(PyObject*, PyObject* args) {
    if (!PyArg_ParseTuple(args, "O!O!O!OO!OOO", &PyDict_Type, &g_utils, &PyDict_Type, &g_split_k, &PyDict_Type, &g_os, &g_environ, &PyDict_Type,
                          &g_environ_bytes, &g_device, &g_stream, &g_capturing)) {
        g_utils = nullptr;
        return nullptr;
    }
    for (PyObject* o : {g_utils, g_split_k, g_os, g_environ, g_environ_bytes, g_device, g_stream, g_capturing}) Py_INCREF(o);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(call)), METH_FASTCALL, nullptr},
    {"remember", remember, METH_VARARGS, nullptr},
    {"forget", forget, METH_NOARGS, nullptr},
    {"setup", setup, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__host_calls() {
    s_num_sms = PyUnicode_InternFromString("_num_sms");
    s_last = PyUnicode_InternFromString("_last");
    s_book = PyUnicode_InternFromString("_book");
    s_eager = PyUnicode_InternFromString("eager");
    s_suspect = PyUnicode_InternFromString("suspect");
    s_failed = PyUnicode_InternFromString("split_k_launch_failed");
    s_environ = PyUnicode_InternFromString("environ");
    b_split_k = PyBytes_FromString("YAN_SPLIT_K");
    b_tune = PyBytes_FromString("YAN_TUNE_TILES");
    PyObject* m = PyModule_Create(&module_def);
    if (m && PyModule_AddStringConstant(m, "built_for", YAN_BUILT_FOR) != 0) Py_CLEAR(m);
    return m;
}

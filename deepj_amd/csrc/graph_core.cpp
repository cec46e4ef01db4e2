// The recording half of the tensor backend as a CPython extension: buffers, the lazy graph's bookkeeping and command words,
// and the tensors' link to their buffers.  deepj_amd/compute_graph.py, tensor.py and hip_backend.py derive from and call these
// types; what an operation records, the order of a flush and the error texts are theirs.
//
// Why native: recording is host time that no kernel hides (a tensor is read, the graph runs, the program goes on recording).
// In Python an operation took some sixteen calls and objects, 3 to 5 us, and a round trip through ctypes 8 us more.  An attention
// layer that reads its tensors back 20 times: 870 -> 560 us; six training steps of some 70 operations: 3040 -> 2270; a
// feed-forward layer of 15 operations: 202 -> 177.
//
// A tensor's death is what releases its buffer.  Each tensor knows the (graph, id) pairs under which it is tracked and tells
// those graphs when it goes; a graph that goes first takes itself out of its tensors.  Neither holds the other alive.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <initializer_list>
#include <mutex>
#include <new>
#include <string>
#include <unordered_map>
#include <unordered_set>
#include <utility>
#include <vector>

namespace {

struct Graph;
struct Tensor;

PyObject *g_empty, *g_zeros, *g_float32, *g_pack, *g_unpack;       // numpy's and compute_graph.py's (set_helpers)
PyTypeObject *g_tensor_class;                                      // deepj_amd.Tensor
std::unordered_map<int, std::pair<int, std::vector<int>>> g_op_meta;     // opcode -> stride, buffer slots
int g_fill_op;

// Attributes as a class in Python has them: a size is whatever counts (numpy's integers too), a flag whatever is true or not.
template <class T> T &at_offset(PyObject *o, void *offset) { return *reinterpret_cast<T *>(reinterpret_cast<char *>(o) + reinterpret_cast<size_t>(offset)); }
bool deleted(PyObject *v) {
    if (v) return false;
    PyErr_SetString(PyExc_AttributeError, "can't delete attribute");
    return true;
}
PyObject *get_size(PyObject *o, void *offset) { return PyLong_FromSsize_t(at_offset<Py_ssize_t>(o, offset)); }
int set_size(PyObject *o, PyObject *v, void *offset) {
    if (deleted(v)) return -1;
    PyObject *number = PyNumber_Long(v);
    const Py_ssize_t n = number ? PyLong_AsSsize_t(number) : -1;
    Py_XDECREF(number);
    if (n == -1 && PyErr_Occurred()) return -1;
    at_offset<Py_ssize_t>(o, offset) = n;
    return 0;
}
PyObject *get_flag(PyObject *o, void *offset) { return PyBool_FromLong(at_offset<char>(o, offset)); }
int set_flag(PyObject *o, PyObject *v, void *offset) {
    const int is = deleted(v) ? -1 : PyObject_IsTrue(v);
    if (is < 0) return -1;
    at_offset<char>(o, offset) = (char)is;
    return 0;
}
#define ATTRIBUTE(name, kind, type, field) {name, get_##kind, set_##kind, nullptr, reinterpret_cast<void *>(offsetof(type, field))}

// ── GpuBuffer ───────────────────────────────────────────────────────────────
struct Buffer {
    PyObject_HEAD
    int id;
    Py_ssize_t rows, cols;
    char needs_upload, cpu_stale, allocated;
    PyObject *graph;                       // the graph that tracks it: told when a tensor lets go of this buffer
};
extern PyTypeObject BufferType, GraphType, TensorType;
inline bool is_buffer(PyObject *o) { return o && PyObject_TypeCheck(o, &BufferType); }

Buffer *new_buffer(int id, Py_ssize_t rows, Py_ssize_t cols, bool needs_upload, bool allocated, PyObject *graph) {
    Buffer *b = reinterpret_cast<Buffer *>(BufferType.tp_alloc(&BufferType, 0));
    if (!b) return nullptr;
    b->id = id; b->rows = rows; b->cols = cols;
    b->needs_upload = needs_upload; b->cpu_stale = 0; b->allocated = allocated;
    Py_XINCREF(graph);
    b->graph = graph;
    return b;
}
int buffer_init(Buffer *self, PyObject *args, PyObject *kw) {
    static const char *names[] = {"id", "rows", "cols", "needs_upload", "graph", nullptr};
    int id, needs;
    Py_ssize_t rows, cols;
    PyObject *graph = Py_None;
    if (!PyArg_ParseTupleAndKeywords(args, kw, "innp|O", const_cast<char **>(names), &id, &rows, &cols, &needs, &graph)) return -1;
    self->id = id; self->rows = rows; self->cols = cols;
    self->needs_upload = (char)needs; self->cpu_stale = 0; self->allocated = 1;
    Py_INCREF(graph);
    Py_XSETREF(self->graph, graph);
    return 0;
}
int buffer_traverse(Buffer *self, visitproc visit, void *arg) { Py_VISIT(self->graph); return 0; }
int buffer_clear(Buffer *self) { Py_CLEAR(self->graph); return 0; }
void buffer_dealloc(Buffer *self) {
    PyObject_GC_UnTrack(self);
    Py_CLEAR(self->graph);
    Py_TYPE(self)->tp_free(reinterpret_cast<PyObject *>(self));
}
PyObject *buffer_float_count(Buffer *self, PyObject *) { return PyLong_FromSsize_t(self->rows * self->cols); }
PyMemberDef buffer_members[] = {
    {"id", T_INT, offsetof(Buffer, id), 0, nullptr},
    {"graph", T_OBJECT, offsetof(Buffer, graph), 0, nullptr},
    {nullptr, 0, 0, 0, nullptr}};
PyGetSetDef buffer_getset[] = {
    ATTRIBUTE("rows", size, Buffer, rows),
    ATTRIBUTE("cols", size, Buffer, cols),
    ATTRIBUTE("needsUpload", flag, Buffer, needs_upload),
    ATTRIBUTE("cpuStale", flag, Buffer, cpu_stale),
    ATTRIBUTE("allocatedOnGpu", flag, Buffer, allocated),
    {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyMethodDef buffer_methods[] = {{"floatCount", (PyCFunction)buffer_float_count, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};

// ── tensors ─────────────────────────────────────────────────────────────────
struct Track { Graph *graph; int id; };
struct Tensor {
    PyObject_HEAD
    Py_ssize_t rows, cols;
    PyObject *data;                        // the host copy, once there is one (None or null before)
    PyObject *tag;
    std::vector<Track> tracks;
};
inline bool has_data(const Tensor *t) { return t->data && t->data != Py_None; }
inline Buffer *tag_of(const Tensor *t) { return is_buffer(t->tag) ? reinterpret_cast<Buffer *>(t->tag) : nullptr; }

// What a flush sends: values (a copy: the tensor may change before), or how many zeros.
struct Upload {
    int id;
    int64_t count;
    float *values;                         // null: zeros
};

struct Native {                            // the library's calls
    int (*alloc)(const int32_t *, const int32_t *, int32_t);
    int (*upload)(int32_t, const float *, int64_t);
    int (*download)(int32_t, float *, int64_t);
    int (*release)(const int32_t *, int32_t);
    int (*flush)(const int32_t *, int32_t);
    const char *(*error)();
};

struct State {
    std::vector<int32_t> cmd;
    int64_t ops = 0;
    std::vector<Buffer *> allocs;          // strong
    std::vector<Upload> uploads;
    int64_t uploads_taken_out = 0;         // how often some of them were
    std::unordered_map<int, Tensor *> tensors;     // null: it has died
    std::vector<int> maybe_orphans;
    std::vector<int32_t> gone;             // no longer tracked, and still to be released
};
struct Graph {
    PyObject_HEAD
    PyObject *runtime, *zero_buffers, *host_array;
    int next_id;
    Native native;
    PyObject *others;                      // null, None, or what else it tracks: {id: weak reference} (ComputeGraph, compute_graph.py)
    PyTypeObject *native_type;             // a runtime of exactly this class, with nothing set on it, is spoken to directly
    State *s;
};

bool has_other(Graph *g, int id) {
    if (!g->others || !PyDict_Check(g->others)) return false;
    PyObject *key = PyLong_FromLong(id);
    const bool r = key && PyDict_Contains(g->others, key) == 1;
    Py_XDECREF(key);
    PyErr_Clear();
    return r;
}
void drop_other(Graph *g, int id) {
    PyObject *key = PyLong_FromLong(id);
    if (!key || PyDict_DelItem(g->others, key) != 0) PyErr_Clear();
    Py_XDECREF(key);
}
void track(Graph *g, int id, Tensor *t) {
    if (has_other(g, id)) drop_other(g, id);
    Tensor *&slot = g->s->tensors[id];
    if (slot == t) return;
    if (slot)
        for (Track &k : slot->tracks)
            if (k.graph == g && k.id == id) { k = slot->tracks.back(); slot->tracks.pop_back(); break; }
    slot = t;
    t->tracks.push_back({g, id});
}
void forget(Graph *g, int id) {            // the graph no longer tracks this buffer
    auto it = g->s->tensors.find(id);
    if (it == g->s->tensors.end()) return;
    if (Tensor *t = it->second)
        for (Track &k : t->tracks)
            if (k.graph == g && k.id == id) { k = t->tracks.back(); t->tracks.pop_back(); break; }
    g->s->tensors.erase(it);
}

PyObject *tensor_new(PyTypeObject *type, PyObject *, PyObject *) {
    Tensor *t = reinterpret_cast<Tensor *>(type->tp_alloc(type, 0));
    if (t) new (&t->tracks) std::vector<Track>();
    return reinterpret_cast<PyObject *>(t);
}
int tensor_traverse(Tensor *t, visitproc visit, void *arg) { Py_VISIT(t->data); Py_VISIT(t->tag); return 0; }
int tensor_clear(Tensor *t) { Py_CLEAR(t->data); Py_CLEAR(t->tag); return 0; }
void tensor_dealloc(Tensor *t) {
    PyObject_GC_UnTrack(t);
    for (const Track &k : t->tracks) {
        k.graph->s->tensors[k.id] = nullptr;
        k.graph->s->maybe_orphans.push_back(k.id);
    }
    t->tracks.~vector();
    Py_CLEAR(t->data);
    Py_CLEAR(t->tag);
    Py_TYPE(t)->tp_free(reinterpret_cast<PyObject *>(t));
}
// Tensor(rows, cols), or a copy of another tensor (Tensor.java:50-59)
int tensor_init(Tensor *t, PyObject *args, PyObject *kw) {
    static const char *names[] = {"rows", "cols", nullptr};
    PyObject *rows, *cols = Py_None;
    if (!PyArg_ParseTupleAndKeywords(args, kw, "O|O", const_cast<char **>(names), &rows, &cols)) return -1;
    if (PyObject_TypeCheck(rows, &TensorType)) {
        PyObject *r = PyObject_CallMethod(rows, "materialize", nullptr);
        if (!r) return -1;
        Py_DECREF(r);
        Tensor *src = reinterpret_cast<Tensor *>(rows);
        t->rows = src->rows; t->cols = src->cols;
        PyObject *data = PyObject_GetAttrString(rows, "data");
        PyObject *copy = data ? PyObject_CallMethod(data, "copy", nullptr) : nullptr;
        Py_XDECREF(data);
        if (!copy) return -1;
        Py_XSETREF(t->data, copy);
        return 0;
    }
    PyObject *ri = PyNumber_Long(rows), *ci = ri ? PyNumber_Long(cols) : nullptr;
    if (ci) { t->rows = PyLong_AsSsize_t(ri); t->cols = PyLong_AsSsize_t(ci); }
    Py_XDECREF(ri);
    Py_XDECREF(ci);
    if (PyErr_Occurred()) return -1;
    if (t->rows < 0 || t->cols < 0) { PyErr_SetString(PyExc_ValueError, "negative dimensions are not allowed"); return -1; }
    return 0;
}
// The host copy as it is (zeros before anything was put there)
PyObject *tensor_data(Tensor *t, void *) {
    if (!has_data(t)) {
        PyObject *a = PyObject_CallFunction(g_zeros, "(nn)O", t->rows, t->cols, g_float32);
        if (!a) return nullptr;
        Py_XSETREF(t->data, a);
    }
    Py_INCREF(t->data);
    return t->data;
}
int tensor_set_data(Tensor *t, PyObject *v, void *) {
    if (!v) v = Py_None;
    Py_INCREF(v);
    Py_XSETREF(t->data, v);
    return 0;
}
PyObject *tensor_get_tag(Tensor *t, PyObject *) {
    PyObject *o = t->tag ? t->tag : Py_None;
    Py_INCREF(o);
    return o;
}
Graph *plain_graph(PyObject *o);
// tag: borrowed.  The graph that tracks the buffer it had is told; false: it raised something (the tag is in place all the same).
bool set_tag(Tensor *t, PyObject *tag) {
    PyObject *old = t->tag;
    Py_INCREF(tag);
    t->tag = tag;
    bool ok = true;
    if (old && old != tag && is_buffer(old)) {
        PyObject *g = reinterpret_cast<Buffer *>(old)->graph;
        if (Graph *plain = g ? plain_graph(g) : nullptr) {
            plain->s->maybe_orphans.push_back(reinterpret_cast<Buffer *>(old)->id);
        } else if (g && g != Py_None) {
            PyObject *r = PyObject_CallMethod(g, "tensorLetGo", "O", old);
            ok = r != nullptr;
            Py_XDECREF(r);
        }
    }
    Py_XDECREF(old);
    return ok;
}
PyObject *tensor_set_tag(Tensor *t, PyObject *tag) {
    if (!set_tag(t, tag)) return nullptr;
    Py_RETURN_NONE;
}
PyMemberDef tensor_members[] = {
    {"_data", T_OBJECT, offsetof(Tensor, data), 0, nullptr},
    {"_gpu_tag", T_OBJECT, offsetof(Tensor, tag), 0, nullptr},
    {nullptr, 0, 0, 0, nullptr}};
PyGetSetDef tensor_getset[] = {
    ATTRIBUTE("rows", size, Tensor, rows),
    ATTRIBUTE("cols", size, Tensor, cols),
    {"data", (getter)tensor_data, (setter)tensor_set_data, "The host copy as it is (zeros before anything was put there); numpy() brings it up to date first.", nullptr},
    {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyMethodDef tensor_methods[] = {
    {"getGpuTag", (PyCFunction)tensor_get_tag, METH_NOARGS, nullptr},
    {"setGpuTag", (PyCFunction)tensor_set_tag, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

// ── the graph ───────────────────────────────────────────────────────────────
PyObject *graph_new(PyTypeObject *type, PyObject *, PyObject *) {
    Graph *g = reinterpret_cast<Graph *>(type->tp_alloc(type, 0));
    if (g) g->s = new State();
    return reinterpret_cast<PyObject *>(g);
}
void drop_uploads(State *s) {
    for (Upload &u : s->uploads) free(u.values);
    s->uploads.clear();
    s->uploads_taken_out++;
}
void drop_allocs(State *s) {
    std::vector<Buffer *> gone;
    gone.swap(s->allocs);
    for (Buffer *b : gone) Py_DECREF(b);
}
int graph_traverse(Graph *g, visitproc visit, void *arg) {
    Py_VISIT(g->runtime); Py_VISIT(g->zero_buffers); Py_VISIT(g->host_array); Py_VISIT(g->native_type); Py_VISIT(g->others);
    for (Buffer *b : g->s->allocs) Py_VISIT(b);
    return 0;
}
int graph_clear(Graph *g) {
    Py_CLEAR(g->runtime); Py_CLEAR(g->zero_buffers); Py_CLEAR(g->host_array); Py_CLEAR(g->native_type); Py_CLEAR(g->others);
    drop_allocs(g->s);
    return 0;
}
void graph_dealloc(Graph *g) {
    PyObject_GC_UnTrack(g);
    graph_clear(g);
    for (auto &e : g->s->tensors)
        if (e.second) {
            auto &k = e.second->tracks;
            k.erase(std::remove_if(k.begin(), k.end(), [g](const Track &x) { return x.graph == g; }), k.end());
        }
    drop_uploads(g->s);
    delete g->s;
    Py_TYPE(g)->tp_free(reinterpret_cast<PyObject *>(g));
}
// GraphCore(runtime, zero_buffers or None, host_array, native class or None, addresses of its calls)
int graph_init(Graph *g, PyObject *args, PyObject *) {
    PyObject *runtime, *zero, *host, *type, *calls;
    if (!PyArg_ParseTuple(args, "OOOOO", &runtime, &zero, &host, &type, &calls)) return -1;
    if (runtime == Py_None) { PyErr_SetString(PyExc_TypeError, "runtime"); return -1; }          // Objects.requireNonNull
    auto keep = [](PyObject *&slot, PyObject *o) { Py_INCREF(o); Py_XSETREF(slot, o); };
    keep(g->runtime, runtime); keep(g->zero_buffers, zero); keep(g->host_array, host);
    if (type != Py_None) {
        unsigned long long p[6];
        if (!PyArg_ParseTuple(calls, "KKKKKK", p, p + 1, p + 2, p + 3, p + 4, p + 5)) return -1;
        static_assert(sizeof(Native) == sizeof(p), "six addresses");
        memcpy(&g->native, p, sizeof(p));
        PyObject *t = reinterpret_cast<PyObject *>(g->native_type);
        keep(t, type);
        g->native_type = reinterpret_cast<PyTypeObject *>(t);
    }
    return 0;
}
struct Methods {                           // attributes of a class as they were, and whether some class still has them
    std::vector<std::pair<PyObject *, PyObject *>> of;
    PyTypeObject *seen = nullptr;
    unsigned seen_tag = 0;
    bool seen_same = false;
    bool take(PyTypeObject *type, PyObject *names) {
        PyObject *list = PySequence_Tuple(names);
        if (!list) return false;
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(list); i++) {
            PyObject *name = PyTuple_GET_ITEM(list, i), *value = _PyType_Lookup(type, name);
            if (!value) { PyErr_SetObject(PyExc_AttributeError, name); Py_DECREF(list); return false; }
            Py_INCREF(name);
            Py_INCREF(value);
            of.emplace_back(name, value);
        }
        Py_DECREF(list);
        return true;
    }
    bool same(PyTypeObject *type) {        // (a class's version changes with it and with its bases)
        if (type == seen && PyType_HasFeature(type, Py_TPFLAGS_VALID_VERSION_TAG) && type->tp_version_tag == seen_tag) return seen_same;
        bool all = !of.empty();
        for (const auto &m : of) all = all && _PyType_Lookup(type, m.first) == m.second;
        seen = type;
        seen_tag = type->tp_version_tag;
        seen_same = all;
        return all;
    }
};
Methods g_tensor_methods, g_graph_methods, g_runtime_methods, g_native_methods;
PyTypeObject *g_runtime_class, *g_native_class;                    // deepj_amd.HipGpuRuntime, HipNative
PyObject *g_general;                       // compute_graph.py's {name: function of the graph}

// Whether the graph makes the library's calls itself: not where something was put in place of a method that would make them.
bool direct(Graph *g) {
    if (!g->native_type || Py_TYPE(g->runtime) != g->native_type) return false;
    if (g->native_type == g_runtime_class && !(g_runtime_methods.same(g_runtime_class) && g_native_methods.same(g_native_class))) return false;
    PyObject **d = _PyObject_GetDictPtr(g->runtime);
    return !d || !*d || PyDict_GET_SIZE(*d) == 0;
}
// The library's calls run one at a time, as it asks of its callers, and without the interpreter's lock, as through ctypes: an upload
// copies its values and may wait for a full ring, a flush may grow the workspace, a download waits for the device.  Whoever is
// about to make one holds this from before it takes out of a graph what it sends until it has noted what became of that (in the
// same thread again where a finaliser makes another); other threads record on meanwhile.
std::recursive_mutex g_calls;
struct Calls {
    Calls() {
        if (g_calls.try_lock()) return;
        Py_BEGIN_ALLOW_THREADS
        g_calls.lock();
        Py_END_ALLOW_THREADS
    }
    ~Calls() { g_calls.unlock(); }
    Calls(const Calls &) = delete;
    // Runs f, which makes calls and returns the first code that is not 0; false, with the library's text raised, if there is one.
    template <class F> bool operator()(Graph *g, F &&f) const {
        const Native n = g->native;
        std::string text;
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = f(n, text);
        Py_END_ALLOW_THREADS
        if (rc == 0) return true;
        PyObject *message = PyUnicode_DecodeUTF8(text.data(), (Py_ssize_t)text.size(), "replace");
        if (message) { PyErr_SetObject(PyExc_RuntimeError, message); Py_DECREF(message); }
        return false;
    }
};
int noted(int rc, const Native &n, std::string &text) {
    if (rc != 0) text = n.error();
    return rc;
}

// A copy of the tensor's host values as fp32 in row order: straight where they are that already, through pack_f32 otherwise.
bool add_upload(Graph *g, int id, Tensor *t) {
    Upload u{id, 0, nullptr};
    if (!has_data(t)) {
        if (g->zero_buffers != Py_None) {  // cleared on the device, where the runtime can, instead of sending zeros
            u.count = t->rows * t->cols;
            g->s->uploads.push_back(u);
            return true;
        }
        PyObject *d = tensor_data(t, nullptr);
        if (!d) return false;
        Py_DECREF(d);
    }
    Py_buffer v;
    PyObject *packed = nullptr;
    bool plain = PyObject_GetBuffer(t->data, &v, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) == 0;
    if (plain && !(v.itemsize == 4 && v.format && strcmp(v.format, "f") == 0)) { PyBuffer_Release(&v); plain = false; }
    if (!plain) {
        PyErr_Clear();
        packed = PyObject_CallFunctionObjArgs(g_pack, t, nullptr);
        if (!packed) return false;
        if (PyObject_GetBuffer(packed, &v, PyBUF_C_CONTIGUOUS) != 0) { Py_DECREF(packed); return false; }
    }
    u.count = v.len / 4;
    u.values = static_cast<float *>(malloc(v.len ? v.len : 1));
    if (u.values) memcpy(u.values, v.buf, v.len);
    PyBuffer_Release(&v);
    Py_XDECREF(packed);
    if (!u.values) { PyErr_NoMemory(); return false; }
    g->s->uploads.push_back(u);
    return true;
}

// The values of a new buffer from 1 MiB on are sent as they are instead of being copied for the flush (three weights of 11 MB:
// 7.8 ms to their first result with the copies, 1.8 without): nothing recorded refers to the buffer yet, so it does not matter when they arrive.
// false: not of that kind, or it could not be sent: the flush sends it, and says why it cannot.
bool send_now(Graph *g, Buffer *b, Tensor *t) {
    constexpr Py_ssize_t kLarge = 1 << 20;
    if (!has_data(t) || t->rows * t->cols * 4 < kLarge || !direct(g)) return false;
    Py_buffer v;
    if (PyObject_GetBuffer(t->data, &v, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) != 0) { PyErr_Clear(); return false; }
    bool sent = false;
    if (v.itemsize == 4 && v.format && strcmp(v.format, "f") == 0 && v.len == t->rows * t->cols * 4) {
        const int32_t id = b->id, size = (int32_t)(t->rows * t->cols);
        const Calls calls;
        sent = calls(g, [&](const Native &n, std::string &text) {
            int rc = noted(n.alloc(&id, &size, 1), n, text);
            if (rc == 0 && (rc = noted(n.upload(id, static_cast<const float *>(v.buf), size), n, text)) != 0) (void)n.release(&id, 1);
            return rc;
        });
        if (sent) b->allocated = 1;
        else PyErr_Clear();
    }
    PyBuffer_Release(&v);
    return sent;
}

// What is looked into here: a tensor whose class leaves its sizes, values and buffer as Tensor has them.  One that does not is an
// object that stands in for a tensor (ComputeGraph, compute_graph.py).
Tensor *tensor(PyObject *o) { return PyObject_TypeCheck(o, &TensorType) && g_tensor_methods.same(Py_TYPE(o)) ? reinterpret_cast<Tensor *>(o) : nullptr; }
Tensor *as_tensor(PyObject *o) {
    if (PyObject_TypeCheck(o, &TensorType)) return reinterpret_cast<Tensor *>(o);
    PyErr_Format(PyExc_TypeError, "expected a Tensor, not %.100s", Py_TYPE(o)->tp_name);
    return nullptr;
}
// Sizes, rows and columns travel as 32-bit words.
bool fits_words(Py_ssize_t rows, Py_ssize_t cols) {
    if (rows <= INT32_MAX && cols <= INT32_MAX && rows * cols <= INT32_MAX) return true;
    PyErr_Format(PyExc_OverflowError, "a buffer of %zdx%zd: more than 32 bits count", rows, cols);
    return false;
}
// A buffer held through what may run meanwhile: another thread while values are sent, a host array of some other class.
struct Held {
    Buffer *b;
    explicit Held(Buffer *taken) : b(taken) {}             // takes the caller's reference
    ~Held() { Py_XDECREF(b); }
    Held(const Held &) = delete;
    Buffer *operator->() const { return b; }
    explicit operator bool() const { return b != nullptr; }
};
Buffer *ensure(Graph *g, Tensor *t) {      // a reference of the caller's
    if (Buffer *b = tag_of(t)) {
        Py_INCREF(b);
        auto it = g->s->tensors.find(b->id);
        if (it == g->s->tensors.end() || it->second != t) {
            track(g, b->id, t);
            Py_INCREF(g);
            Py_XSETREF(b->graph, reinterpret_cast<PyObject *>(g));
        }
        if (b->needs_upload) {
            PyObject *d = has_data(t) ? nullptr : tensor_data(t, nullptr);
            Py_XDECREF(d);
            if (!has_data(t) || !add_upload(g, b->id, t)) { Py_DECREF(b); return nullptr; }
            b->needs_upload = 0;
            b->cpu_stale = 0;
        }
        return b;
    }
    if (!fits_words(t->rows, t->cols)) return nullptr;
    Buffer *b = new_buffer(g->next_id, t->rows, t->cols, true, false, reinterpret_cast<PyObject *>(g));
    if (!b) return nullptr;
    g->next_id++;
    Py_INCREF(b);                          // (two: the caller's, and the list's of what is to be made)
    const bool sent = send_now(g, b, t);
    if (!sent && !add_upload(g, b->id, t)) { Py_DECREF(b); Py_DECREF(b); return nullptr; }
    if (sent) Py_DECREF(b);
    else g->s->allocs.push_back(b);        // (takes the reference)
    if (!set_tag(t, reinterpret_cast<PyObject *>(b))) { Py_DECREF(b); return nullptr; }
    track(g, b->id, t);
    return b;
}
Buffer *new_output(Graph *g, Py_ssize_t rows, Py_ssize_t cols) {       // a reference of the caller's
    if (!fits_words(rows, cols)) return nullptr;
    Buffer *b = new_buffer(g->next_id, rows, cols, false, false, reinterpret_cast<PyObject *>(g));
    if (!b) return nullptr;
    g->next_id++;
    b->cpu_stale = 1;
    Py_INCREF(b);
    g->s->allocs.push_back(b);
    return b;
}
PyObject *output_tensor(Graph *g, Buffer *b) {
    PyObject *o = tensor_new(g_tensor_class, nullptr, nullptr);
    if (!o) return nullptr;
    Tensor *t = reinterpret_cast<Tensor *>(o);
    t->rows = b->rows; t->cols = b->cols;
    Py_INCREF(b);
    t->tag = reinterpret_cast<PyObject *>(b);
    track(g, b->id, t);
    Py_INCREF(g);
    Py_XSETREF(b->graph, reinterpret_cast<PyObject *>(g));
    return o;
}
bool bind(Graph *g, Tensor *t, Buffer *b) {
    if (!set_tag(t, reinterpret_cast<PyObject *>(b))) return false;
    track(g, b->id, t);
    Py_INCREF(g);
    Py_XSETREF(b->graph, reinterpret_cast<PyObject *>(g));
    return true;
}
// The result of a recorded operation: a new tensor, or `into` on its new buffer.  Takes the caller's reference to out.
PyObject *finish(Graph *g, Buffer *out, Tensor *into) {
    PyObject *r;
    if (!into) r = output_tensor(g, out);
    else if ((r = bind(g, into, out) ? Py_None : nullptr)) Py_INCREF(r);
    Py_DECREF(out);
    return r;
}
inline void emit(Graph *g, std::initializer_list<int64_t> words) {
    for (int64_t w : words) g->s->cmd.push_back((int32_t)w);
    g->s->ops++;
}
bool read_float_bits(PyObject *o, int32_t &bits) {
    const double d = PyFloat_AsDouble(o);
    if (d == -1.0 && PyErr_Occurred()) return false;
    const float f = (float)d;
    memcpy(&bits, &f, 4);
    return true;
}
bool read_int(PyObject *o, int64_t &v) {
    v = PyLong_AsLongLong(o);
    return !(v == -1 && PyErr_Occurred());
}
bool arity(Py_ssize_t n, Py_ssize_t want) {
    if (n == want) return true;
    PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
    return false;
}

// An object that stands in for a tensor is looked after by methods of ComputeGraph.
PyObject *graph_ensure(Graph *g, PyObject *o) {
    if (Tensor *t = tensor(o)) return reinterpret_cast<PyObject *>(ensure(g, t));
    return PyObject_CallMethod(reinterpret_cast<PyObject *>(g), "_ensureOther", "O", o);
}
PyObject *graph_new_output(Graph *g, PyObject *const *a, Py_ssize_t n) {
    int64_t r, c;
    if (!arity(n, 2) || !read_int(a[0], r) || !read_int(a[1], c)) return nullptr;
    return reinterpret_cast<PyObject *>(new_output(g, r, c));
}
Buffer *as_buffer(PyObject *o) {
    if (is_buffer(o)) return reinterpret_cast<Buffer *>(o);
    PyErr_Format(PyExc_TypeError, "expected a GpuBuffer, not %.100s", Py_TYPE(o)->tp_name);
    return nullptr;
}
PyObject *graph_output_tensor(Graph *g, PyObject *o) {
    Buffer *b = as_buffer(o);
    return b ? output_tensor(g, b) : nullptr;
}
PyObject *graph_bind(Graph *g, PyObject *const *a, Py_ssize_t n) {
    if (!arity(n, 2)) return nullptr;
    Buffer *b = as_buffer(a[1]);
    if (!b) return nullptr;
    Tensor *t = tensor(a[0]);
    if (!t) return PyObject_CallMethod(reinterpret_cast<PyObject *>(g), "_bindOther", "OO", a[0], a[1]);
    if (!bind(g, t, b)) return nullptr;
    Py_RETURN_NONE;
}
PyObject *graph_let_go(Graph *g, PyObject *o) {
    Buffer *b = as_buffer(o);
    if (!b) return nullptr;
    g->s->maybe_orphans.push_back(b->id);
    Py_RETURN_NONE;
}
PyObject *graph_emit(Graph *g, PyObject *const *a, Py_ssize_t n) {     // one operation's words
    const size_t at = g->s->cmd.size();
    for (Py_ssize_t i = 0; i < n; i++) {
        int64_t w;
        bool ok = read_int(a[i], w);
        if (ok && (w < INT32_MIN || w > INT32_MAX)) { PyErr_SetString(PyExc_OverflowError, "a command word is 32 bits"); ok = false; }
        if (!ok) { g->s->cmd.resize(at); return nullptr; }
        g->s->cmd.push_back((int32_t)w);
    }
    g->s->ops++;
    Py_RETURN_NONE;
}

// ── operations of the backend: check, inputs, output, words ─────────────────
// They go past the graph's own methods, so only where those are ComputeGraph's and the operands tensors; everything else - a class
// derived from it, a method replaced, an object that stands in for a graph or a tensor - takes the way through the methods
// (compute_graph.py).
Graph *plain_graph(PyObject *o) {
    if (!PyObject_TypeCheck(o, &GraphType) || !g_graph_methods.same(Py_TYPE(o))) return nullptr;
    PyObject **d = _PyObject_GetDictPtr(o);
    if (d && *d && PyDict_GET_SIZE(*d) > 0)
        for (const auto &m : g_graph_methods.of)
            if (PyDict_Contains(*d, m.first) != 0) { PyErr_Clear(); return nullptr; }
    return reinterpret_cast<Graph *>(o);
}
PyObject *general(const char *name, PyObject *const *v, Py_ssize_t n) {
    PyObject *f = g_general ? PyDict_GetItemString(g_general, name) : nullptr;
    if (!f) return PyErr_Format(PyExc_RuntimeError, "no function for %s", name);
    return PyObject_Vectorcall(f, v, (size_t)n, nullptr);
}

// (graph, opcode, name, a, b, in place)
PyObject *record_binary(PyObject *, PyObject *const *v, Py_ssize_t n) {
    int64_t op;
    Graph *g = n == 6 ? plain_graph(v[0]) : nullptr;
    Tensor *a = g ? tensor(v[3]) : nullptr, *b = a ? tensor(v[4]) : nullptr;
    if (!b) return general("binary", v, n);
    if (!read_int(v[1], op)) return nullptr;
    if (a->rows != b->rows || a->cols != b->cols) return PyErr_Format(PyExc_ValueError, "Shape mismatch for %U: %zdx%zd vs %zdx%zd", v[2], a->rows, a->cols, b->rows, b->cols);
    const Held ga(ensure(g, a)), gb(ga ? ensure(g, b) : nullptr);
    Buffer *out = gb ? new_output(g, a->rows, a->cols) : nullptr;
    if (!out) return nullptr;
    emit(g, {op, ga->id, gb->id, out->id, out->rows * out->cols});
    return finish(g, out, v[5] == Py_True ? a : nullptr);
}
// (graph, opcode, a, in place)
PyObject *record_unary(PyObject *, PyObject *const *v, Py_ssize_t n) {
    int64_t op;
    Graph *g = n == 4 ? plain_graph(v[0]) : nullptr;
    Tensor *a = g ? tensor(v[2]) : nullptr;
    if (!a) return general("unary", v, n);
    if (!read_int(v[1], op)) return nullptr;
    const Held ga(ensure(g, a));
    Buffer *out = ga ? new_output(g, a->rows, a->cols) : nullptr;
    if (!out) return nullptr;
    emit(g, {op, ga->id, out->id, out->rows * out->cols});
    return finish(g, out, v[3] == Py_True ? a : nullptr);
}
// (graph, opcode, a, scalar, in place)
PyObject *record_scalar(PyObject *, PyObject *const *v, Py_ssize_t n) {
    int64_t op;
    int32_t bits;
    Graph *g = n == 5 ? plain_graph(v[0]) : nullptr;
    Tensor *a = g ? tensor(v[2]) : nullptr;
    if (!a) return general("scalar", v, n);
    if (!read_int(v[1], op) || !read_float_bits(v[3], bits)) return nullptr;
    const Held ga(ensure(g, a));
    Buffer *out = ga ? new_output(g, a->rows, a->cols) : nullptr;
    if (!out) return nullptr;
    emit(g, {op, ga->id, out->id, bits, out->rows * out->cols});
    return finish(g, out, v[4] == Py_True ? a : nullptr);
}
// (graph, opcode, a, output rows, output columns): an operation whose words end with the input's rows and columns
PyObject *record_shaped(PyObject *, PyObject *const *v, Py_ssize_t n) {
    int64_t op, rows, cols;
    Graph *g = n == 5 ? plain_graph(v[0]) : nullptr;
    Tensor *a = g ? tensor(v[2]) : nullptr;
    if (!a) return general("shaped", v, n);
    if (!read_int(v[1], op) || !read_int(v[3], rows) || !read_int(v[4], cols)) return nullptr;
    const Held ga(ensure(g, a));
    Buffer *out = ga ? new_output(g, rows, cols) : nullptr;
    if (!out) return nullptr;
    emit(g, {op, ga->id, out->id, a->rows, a->cols});
    return finish(g, out, nullptr);
}
PyObject *two_shaped(Graph *g, int64_t op, Tensor *a, Tensor *b) {     // out like a; a's rows and columns
    const Held ga(ensure(g, a)), gb(ga ? ensure(g, b) : nullptr);
    Buffer *out = gb ? new_output(g, a->rows, a->cols) : nullptr;
    if (!out) return nullptr;
    emit(g, {op, ga->id, gb->id, out->id, a->rows, a->cols});
    return finish(g, out, nullptr);
}
// (graph, opcode, a, b): words end with a's rows and columns (shapes checked by the caller)
PyObject *record_pair(PyObject *, PyObject *const *v, Py_ssize_t n) {
    int64_t op;
    Graph *g = n == 4 ? plain_graph(v[0]) : nullptr;
    Tensor *a = g ? tensor(v[2]) : nullptr, *b = a ? tensor(v[3]) : nullptr;
    if (!b) return general("pair", v, n);
    return read_int(v[1], op) ? two_shaped(g, op, a, b) : nullptr;
}
// (graph, opcode, a, row vector)
PyObject *record_rows(PyObject *, PyObject *const *v, Py_ssize_t n) {
    int64_t op;
    Graph *g = n == 4 ? plain_graph(v[0]) : nullptr;
    Tensor *a = g ? tensor(v[2]) : nullptr, *b = a ? tensor(v[3]) : nullptr;
    if (!b) return general("rowBroadcast", v, n);
    if (b->rows != 1 || b->cols != a->cols) return PyErr_Format(PyExc_ValueError, "Expected row vector 1x%zd but got %zdx%zd", a->cols, b->rows, b->cols);
    return read_int(v[1], op) ? two_shaped(g, op, a, b) : nullptr;
}
// (graph, opcode, a, column vector)
PyObject *record_cols(PyObject *, PyObject *const *v, Py_ssize_t n) {
    int64_t op;
    Graph *g = n == 4 ? plain_graph(v[0]) : nullptr;
    Tensor *a = g ? tensor(v[2]) : nullptr, *b = a ? tensor(v[3]) : nullptr;
    if (!b) return general("colBroadcast", v, n);
    if (b->rows != a->rows || b->cols != 1) return PyErr_Format(PyExc_ValueError, "Expected col vector %zdx1 but got %zdx%zd", a->rows, b->rows, b->cols);
    return read_int(v[1], op) ? two_shaped(g, op, a, b) : nullptr;
}
// (graph, opcode, a, b)
PyObject *record_matmul(PyObject *, PyObject *const *v, Py_ssize_t n) {
    int64_t op;
    Graph *g = n == 4 ? plain_graph(v[0]) : nullptr;
    Tensor *a = g ? tensor(v[2]) : nullptr, *b = a ? tensor(v[3]) : nullptr;
    if (!b) return general("matmul", v, n);
    if (!read_int(v[1], op)) return nullptr;
    if (a->cols != b->rows) return PyErr_Format(PyExc_ValueError, "Shape mismatch for matmul: %zdx%zd vs %zdx%zd", a->rows, a->cols, b->rows, b->cols);
    const Held ga(ensure(g, a)), gb(ga ? ensure(g, b) : nullptr);
    Buffer *out = gb ? new_output(g, a->rows, b->cols) : nullptr;
    if (!out) return nullptr;
    emit(g, {op, ga->id, gb->id, out->id, a->rows, b->cols, a->cols});
    return finish(g, out, nullptr);
}
// (graph, opcode, w, g, m, v, lr, beta1, beta2, eps, weight decay, c1, c2): the first, third and fourth are updated where they are
PyObject *record_adamw(PyObject *, PyObject *const *v, Py_ssize_t n) {
    int64_t op;
    int32_t bits[7];
    Graph *g = n == 13 ? plain_graph(v[0]) : nullptr;
    Tensor *t[4] = {};
    for (int i = 0; g && i < 4; i++)
        if (!(t[i] = tensor(v[2 + i]))) g = nullptr;
    if (!g) return general("adamW", v, n);
    if (!read_int(v[1], op)) return nullptr;
    const Held w(ensure(g, t[0])), gw(w ? ensure(g, t[1]) : nullptr), mt(gw ? ensure(g, t[2]) : nullptr), vt(mt ? ensure(g, t[3]) : nullptr);
    if (!vt) return nullptr;
    for (int i = 0; i < 7; i++)
        if (!read_float_bits(v[6 + i], bits[i])) return nullptr;
    emit(g, {op, w->id, gw->id, mt->id, vt->id, bits[0], bits[1], bits[2], bits[3], bits[4], bits[5], bits[6], t[0]->rows * t[0]->cols});
    for (Buffer *b : {w.b, mt.b, vt.b}) { b->cpu_stale = 1; b->needs_upload = 0; }
    Py_RETURN_NONE;
}

// ── flush ───────────────────────────────────────────────────────────────────
// A runtime in Python is handed one thing after the other; the library all of it in one go (flush_native).
PyObject *int_array(const std::vector<int32_t> &v) {       // array.array("i", v): what a runtime in Python is handed
    static PyObject *type = nullptr;
    if (!type) {
        PyObject *m = PyImport_ImportModule("array");
        type = m ? PyObject_GetAttrString(m, "array") : nullptr;
        Py_XDECREF(m);
        if (!type) return nullptr;
    }
    return PyObject_CallFunction(type, "sy#", "i", reinterpret_cast<const char *>(v.data()), (Py_ssize_t)(v.size() * 4));
}
bool call(PyObject *r) {
    Py_XDECREF(r);
    return r != nullptr;
}
// (A call may record and flush itself: what it has handed over then is no longer the first of what waits.)
bool allocate_pending(Graph *g) {
    State *s = g->s;
    while (!s->allocs.empty()) {
        const std::vector<Buffer *> taken = s->allocs;
        std::vector<int32_t> ids, sizes;
        for (Buffer *b : taken) { Py_INCREF(b); ids.push_back(b->id); sizes.push_back((int32_t)(b->rows * b->cols)); }
        PyObject *a = int_array(ids), *b = a ? int_array(sizes) : nullptr;
        const bool ok = b && call(PyObject_CallMethod(g->runtime, "allocBuffers", "OOn", a, b, (Py_ssize_t)taken.size()));
        Py_XDECREF(a);
        Py_XDECREF(b);
        std::vector<Buffer *> done;
        if (ok) {
            const std::unordered_set<Buffer *> made(taken.begin(), taken.end());
            auto at = std::stable_partition(s->allocs.begin(), s->allocs.end(), [&](Buffer *w) { return !made.count(w); });
            done.assign(at, s->allocs.end());
            s->allocs.erase(at, s->allocs.end());
            for (Buffer *w : taken) w->allocated = 1;
        }
        for (Buffer *w : done) Py_DECREF(w);
        for (Buffer *w : taken) Py_DECREF(w);
        if (!ok) return false;
    }
    return true;
}
bool upload_pending(Graph *g) {
    State *s = g->s;
    while (!s->uploads.empty()) {
        const size_t count = s->uploads.size();
        const int64_t taken_out = s->uploads_taken_out;        // (other: an inner flush has sent them)
        PyObject *zeros = nullptr;                             // first: a buffer's zeros come before whatever else is sent to it
        for (size_t i = 0; i < count && s->uploads_taken_out == taken_out; i++) {
            const Upload u = s->uploads[i];
            if (u.values) continue;
            if (!zeros && !(zeros = PyList_New(0))) return false;
            PyObject *pair = Py_BuildValue("(iL)", u.id, (long long)u.count);
            const bool ok = pair && PyList_Append(zeros, pair) == 0;
            Py_XDECREF(pair);
            if (!ok) { Py_DECREF(zeros); return false; }
        }
        if (zeros) {
            const bool ok = call(PyObject_CallFunctionObjArgs(g->zero_buffers, zeros, nullptr));
            Py_DECREF(zeros);
            if (!ok) return false;
        }
        for (size_t i = 0; i < count && s->uploads_taken_out == taken_out; i++) {
            const Upload u = s->uploads[i];
            if (!u.values) continue;
            PyObject *a = PyObject_CallFunction(g_empty, "nO", (Py_ssize_t)u.count, g_float32);
            Py_buffer v;
            if (!a || PyObject_GetBuffer(a, &v, PyBUF_CONTIG) != 0) { Py_XDECREF(a); return false; }
            if (s->uploads_taken_out == taken_out) memcpy(v.buf, u.values, v.len);
            PyBuffer_Release(&v);
            const bool ok = s->uploads_taken_out != taken_out || call(PyObject_CallMethod(g->runtime, "uploadBuffer", "iO", u.id, a));
            Py_DECREF(a);
            if (!ok) return false;
        }
        if (s->uploads_taken_out != taken_out) continue;
        for (size_t i = 0; i < count; i++) free(s->uploads[i].values);
        s->uploads.erase(s->uploads.begin(), s->uploads.begin() + count);
        s->uploads_taken_out++;
    }
    return true;
}
bool execute_pending(Graph *g) {           // fails before its first launch: the ops stay recorded
    State *s = g->s;
    if (s->ops == 0) { s->cmd.clear(); return true; }
    std::vector<int32_t> cmd;
    cmd.swap(s->cmd);
    const int64_t ops = s->ops;
    s->ops = 0;
    PyObject *a = int_array(cmd);
    const bool ok = a && call(PyObject_CallMethod(g->runtime, "flushOps", "On", a, (Py_ssize_t)cmd.size()));
    Py_XDECREF(a);
    if (!ok) {
        cmd.insert(cmd.end(), s->cmd.begin(), s->cmd.end());
        s->cmd.swap(cmd);
        s->ops += ops;
    } else if (s->cmd.empty()) {           // keep the memory
        cmd.clear();
        s->cmd.swap(cmd);
    }
    return ok;
}
bool referenced_by_pending_ops(Graph *g, int id) {
    const auto &c = g->s->cmd;
    for (size_t pos = 0; pos < c.size();) {
        auto m = g_op_meta.find(c[pos]);
        if (m == g_op_meta.end()) return true;             // unknown op: be conservative
        for (int slot : m->second.second)
            if (pos + slot < c.size() && c[pos + slot] == id) return true;
        pos += m->second.first;
    }
    return false;
}
bool release_ids(Graph *g, const std::vector<int32_t> &ids) {
    if (direct(g)) {
        const Calls calls;
        return calls(g, [&](const Native &n, std::string &text) { return noted(n.release(ids.data(), (int32_t)ids.size()), n, text); });
    }
    PyObject *a = int_array(ids);
    const bool ok = a && call(PyObject_CallMethod(g->runtime, "releaseBuffers", "On", a, (Py_ssize_t)ids.size()));
    Py_XDECREF(a);
    return ok;
}
void collect_orphans(Graph *g) {           // into gone
    State *s = g->s;
    if (s->maybe_orphans.empty()) return;
    std::vector<int> candidates;
    candidates.swap(s->maybe_orphans);
    std::vector<int32_t> orphans;
    for (int id : candidates) {
        auto it = s->tensors.find(id);
        const bool other = it == s->tensors.end();
        if (other) {
            if (!has_other(g, id)) continue;               // unknown, or seen before
            PyObject *held = PyObject_CallMethod(reinterpret_cast<PyObject *>(g), "_otherHolds", "i", id);
            const bool stays = held != Py_False;
            if (!held) PyErr_WriteUnraisable(reinterpret_cast<PyObject *>(g));
            Py_XDECREF(held);
            if (stays) continue;
        } else if (Tensor *t = it->second) {
            Buffer *b = tag_of(t);
            if (b && b->id == id) continue;
        }
        if (s->ops > 0 && referenced_by_pending_ops(g, id)) { s->maybe_orphans.push_back(id); continue; }
        orphans.push_back(id);
        if (other) drop_other(g, id);
        else forget(g, id);
    }
    if (orphans.empty()) return;
    if (!s->allocs.empty() || !s->uploads.empty()) {
        auto gone = [&](int id) { return std::find(orphans.begin(), orphans.end(), id) != orphans.end(); };
        std::vector<Buffer *> dropped;
        auto keep = s->allocs.begin();
        for (Buffer *b : s->allocs) if (gone(b->id)) dropped.push_back(b); else *keep++ = b;
        s->allocs.erase(keep, s->allocs.end());
        auto at = s->uploads.begin();
        for (Upload &u : s->uploads) if (gone(u.id)) free(u.values); else *at++ = u;
        s->uploads.erase(at, s->uploads.end());
        s->uploads_taken_out++;
        for (Buffer *b : dropped) Py_DECREF(b);
    }
    s->gone.insert(s->gone.end(), orphans.begin(), orphans.end());
}
bool release_gone(Graph *g) {
    std::vector<int32_t> ids;
    ids.swap(g->s->gone);
    return ids.empty() || release_ids(g, ids);
}
bool release_orphans(Graph *g) {
    collect_orphans(g);
    return release_gone(g);
}
// Taken out of the graph first, so that what other threads record meanwhile is the next flush's; what was not done goes back in front
// of it (all uploads, where one of them failed).
bool flush_native(Graph *g) {
    State *s = g->s;
    std::vector<Buffer *> allocs;
    std::vector<Upload> uploads;
    std::vector<int32_t> cmd, ids, sizes, fills;
    allocs.swap(s->allocs); uploads.swap(s->uploads); cmd.swap(s->cmd);
    const int64_t ops = s->ops;
    s->ops = 0;
    for (Buffer *b : allocs) { ids.push_back(b->id); sizes.push_back((int32_t)(b->rows * b->cols)); }
    for (const Upload &u : uploads)        // (a buffer's zeros come before whatever else is sent to it)
        if (!u.values)
            for (int64_t w : {(int64_t)g_fill_op, (int64_t)u.id, (int64_t)0, u.count}) fills.push_back((int32_t)w);
    bool made = false, sent = false;
    const Calls calls;                     // (held by flush already)
    const bool ok = calls(g, [&](const Native &n, std::string &text) {
        int rc = 0;
        if (!ids.empty() && (rc = noted(n.alloc(ids.data(), sizes.data(), (int32_t)ids.size()), n, text)) != 0) return rc;
        made = true;
        if (!fills.empty() && (rc = noted(n.flush(fills.data(), (int32_t)fills.size()), n, text)) != 0) return rc;
        for (const Upload &u : uploads)
            if (u.values && (rc = noted(n.upload(u.id, u.values, u.count), n, text)) != 0) return rc;
        sent = true;
        return ops > 0 ? noted(n.flush(cmd.data(), (int32_t)cmd.size()), n, text) : 0;
    });
    if (sent) {
        for (Upload &u : uploads) free(u.values);
    } else {
        uploads.insert(uploads.end(), s->uploads.begin(), s->uploads.end());
        s->uploads.swap(uploads);
    }
    if (!ok) {                             // fails before its first launch: the ops stay recorded
        cmd.insert(cmd.end(), s->cmd.begin(), s->cmd.end());
        s->cmd.swap(cmd);
        s->ops += ops;
    } else if (s->cmd.empty()) {           // keep the memory
        cmd.clear();
        s->cmd.swap(cmd);
    }
    if (made) {
        for (Buffer *b : allocs) { b->allocated = 1; Py_DECREF(b); }
    } else {
        allocs.insert(allocs.end(), s->allocs.begin(), s->allocs.end());
        s->allocs.swap(allocs);
    }
    return ok;
}
// A download behind it takes along what is to be released: one time less that the interpreter's lock is given up and taken.
bool flush(Graph *g, bool download_follows = false) {
    if (direct(g)) {
        const Calls calls;
        if ((g->s->ops != 0 || !g->s->allocs.empty()) && !flush_native(g)) return false;
        collect_orphans(g);
        return download_follows || release_gone(g);
    }
    if (g->s->ops == 0 && g->s->allocs.empty()) return release_orphans(g);
    return allocate_pending(g) && upload_pending(g) && execute_pending(g) && release_orphans(g);
}
bool flush_method(Graph *g, bool download_follows = false) { return plain_graph(reinterpret_cast<PyObject *>(g)) ? flush(g, download_follows) : call(PyObject_CallMethod(reinterpret_cast<PyObject *>(g), "flush", nullptr)); }
PyObject *graph_flush(Graph *g, PyObject *) {
    if (!flush(g)) return nullptr;
    Py_RETURN_NONE;
}

// The buffer's values in the tensor's host array: written there directly, and into an array of the runtime's own kind where
// the tensor has none yet.
bool fetch(Graph *g, Buffer *b, PyObject *flat) {          // flat: contiguous fp32 of the buffer's size
    if (!direct(g)) return call(PyObject_CallMethod(g->runtime, "downloadBuffer", "iO", b->id, flat));
    Py_buffer v;
    if (PyObject_GetBuffer(flat, &v, PyBUF_CONTIG) != 0) return false;
    const Calls calls;
    std::vector<int32_t> gone;
    gone.swap(g->s->gone);
    const bool ok = calls(g, [&](const Native &n, std::string &text) {
        const int rc = gone.empty() ? 0 : noted(n.release(gone.data(), (int32_t)gone.size()), n, text);
        return rc ? rc : noted(n.download(b->id, static_cast<float *>(v.buf), v.len / 4), n, text);
    });
    PyBuffer_Release(&v);
    return ok;
}
bool download(Graph *g, Buffer *b, Tensor *t) {
    const Py_ssize_t count = b->rows * b->cols;
    bool plain = false;
    if (has_data(t)) {
        Py_buffer v;
        plain = PyObject_GetBuffer(t->data, &v, PyBUF_CONTIG | PyBUF_FORMAT) == 0;
        if (plain) {
            plain = v.itemsize == 4 && v.format && strcmp(v.format, "f") == 0;
            const Py_ssize_t have = v.len / 4;
            PyBuffer_Release(&v);
            if (plain && have != count) {
                PyErr_Format(PyExc_ValueError, "Size mismatch: src has %zd floats but tensor is %zdx%zd", count, t->rows, t->cols);
                return false;
            }
        } else {
            PyErr_Clear();
        }
    }
    if (plain) {
        if (direct(g)) return fetch(g, b, t->data);
        PyObject *flat = PyObject_CallMethod(t->data, "reshape", "i", -1);
        const bool ok = flat && fetch(g, b, flat);
        Py_XDECREF(flat);
        return ok;
    }
    PyObject *flat = PyObject_CallFunction(g->host_array, "n", count);
    bool ok = flat && fetch(g, b, flat);
    if (ok && !has_data(t) && count == t->rows * t->cols) {
        PyObject *shaped = PyObject_CallMethod(flat, "reshape", "nn", t->rows, t->cols);
        ok = shaped != nullptr;
        if (ok) Py_XSETREF(t->data, shaped);
    } else if (ok) {
        ok = call(PyObject_CallFunctionObjArgs(g_unpack, flat, t, nullptr));
    }
    Py_XDECREF(flat);
    return ok;
}
PyObject *graph_materialize(Graph *g, PyObject *o) {
    Tensor *t = tensor(o);
    if (!t) return PyObject_CallMethod(reinterpret_cast<PyObject *>(g), "_materializeOther", "O", o);
    Buffer *b = tag_of(t);
    if (!b || !b->cpu_stale) Py_RETURN_NONE;
    Py_INCREF(b);
    bool ok = flush_method(g, true) && download(g, b, t);
    if (ok) b->cpu_stale = 0;
    Py_DECREF(b);
    if (!g->s->gone.empty()) {             // (the download was not made)
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        ok = release_gone(g) && ok;
        if (type) { PyErr_Clear(); PyErr_Restore(type, value, trace); }
    }
    if (!ok) return nullptr;
    Py_RETURN_NONE;
}
PyObject *graph_release_all(Graph *g, PyObject *) {
    if (!flush_method(g)) return nullptr;
    State *s = g->s;
    std::vector<int32_t> ids;
    if (g->others && PyDict_Check(g->others)) {
        PyObject *more = PyObject_CallMethod(reinterpret_cast<PyObject *>(g), "_releaseOthers", nullptr), *list = more ? PySequence_Tuple(more) : nullptr;
        Py_XDECREF(more);
        if (!list) return nullptr;
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(list); i++) ids.push_back((int32_t)PyLong_AsLong(PyTuple_GET_ITEM(list, i)));
        Py_DECREF(list);
        if (PyErr_Occurred()) return nullptr;
    }
    for (auto &e : s->tensors) ids.push_back(e.first);
    std::sort(ids.begin(), ids.end());
    for (int id : ids) {
        auto it = s->tensors.find(id);
        Tensor *t = it == s->tensors.end() ? nullptr : it->second;
        Buffer *b = t ? tag_of(t) : nullptr;
        if (!b || !b->cpu_stale) continue;
        Py_INCREF(t);
        Py_INCREF(b);
        const bool ok = download(g, b, t);
        if (ok) b->cpu_stale = b->needs_upload = 0;
        Py_DECREF(b);
        Py_DECREF(t);
        if (!ok) return nullptr;
    }
    for (int id : ids) {
        auto it = s->tensors.find(id);
        Tensor *t = it == s->tensors.end() ? nullptr : it->second;
        if (!t) continue;
        Py_INCREF(t);
        const bool ok = set_tag(t, Py_None);
        Py_DECREF(t);
        if (!ok) return nullptr;
    }
    if (!ids.empty() && !release_ids(g, ids)) return nullptr;
    while (!s->tensors.empty()) forget(g, s->tensors.begin()->first);
    Py_CLEAR(g->others);
    s->maybe_orphans.clear();
    drop_allocs(s);
    drop_uploads(s);
    s->cmd.clear();
    s->ops = 0;
    g->next_id = 0;
    Py_RETURN_NONE;
}
// (id, tensor): its host values are sent there; (buffer, tensor): the buffer's values come into its host array; (id): no tensor of
// its own has it; (id): whatever had it is gone
PyObject *graph_upload(Graph *g, PyObject *const *a, Py_ssize_t n) {
    int64_t id;
    if (!arity(n, 2) || !read_int(a[0], id)) return nullptr;
    Tensor *t = as_tensor(a[1]);
    if (!t || !add_upload(g, (int)id, t)) return nullptr;
    Py_RETURN_NONE;
}
PyObject *graph_download(Graph *g, PyObject *const *a, Py_ssize_t n) {
    if (!arity(n, 2)) return nullptr;
    Buffer *b = as_buffer(a[0]);
    Tensor *t = b ? as_tensor(a[1]) : nullptr;
    if (!t || !download(g, b, t)) return nullptr;
    Py_RETURN_NONE;
}
PyObject *graph_forget(Graph *g, PyObject *o) {
    int64_t id;
    if (!read_int(o, id)) return nullptr;
    forget(g, (int)id);
    Py_RETURN_NONE;
}
PyObject *graph_lost(Graph *g, PyObject *o) {
    int64_t id;
    if (!read_int(o, id)) return nullptr;
    g->s->maybe_orphans.push_back((int)id);
    Py_RETURN_NONE;
}
PyObject *graph_is_empty(Graph *g, PyObject *) { return PyBool_FromLong(g->s->ops == 0); }

#define FAST(name, f) {name, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef graph_methods[] = {
    {"ensureGpuBuffer", (PyCFunction)graph_ensure, METH_O, nullptr},
    FAST("newOutputBuffer", graph_new_output),
    {"createOutputTensor", (PyCFunction)graph_output_tensor, METH_O, nullptr},
    FAST("bindTensorToBuffer", graph_bind),
    {"tensorLetGo", (PyCFunction)graph_let_go, METH_O, "Tensor.setGpuTag: the buffer is no longer the tag of a tensor that had it."},
    FAST("_emit", graph_emit),
    FAST("_upload", graph_upload),
    FAST("_download", graph_download),
    {"_forget", (PyCFunction)graph_forget, METH_O, nullptr},
    {"_lost", (PyCFunction)graph_lost, METH_O, nullptr},
    {"isEmpty", (PyCFunction)graph_is_empty, METH_NOARGS, nullptr},
    {"flush", (PyCFunction)graph_flush, METH_NOARGS, nullptr},
    {"materialize", (PyCFunction)graph_materialize, METH_O, nullptr},
    {"releaseAll", (PyCFunction)graph_release_all, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyMemberDef graph_members[] = {
    {"runtime", T_OBJECT_EX, offsetof(Graph, runtime), 0, nullptr},
    {"_others", T_OBJECT, offsetof(Graph, others), 0, nullptr},
    {nullptr, 0, 0, 0, nullptr}};

PyTypeObject BufferType = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyTypeObject GraphType = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyTypeObject TensorType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// set_helpers(numpy.empty, numpy.zeros, numpy.float32, pack_f32, unpack_f32_into, op meta {opcode: (stride, slots)}, fill opcode)
PyObject *set_helpers(PyObject *, PyObject *args) {
    PyObject *p[5], *meta;
    if (!PyArg_ParseTuple(args, "OOOOOO!i", p, p + 1, p + 2, p + 3, p + 4, &PyDict_Type, &meta, &g_fill_op)) return nullptr;
    PyObject **slot[5] = {&g_empty, &g_zeros, &g_float32, &g_pack, &g_unpack};
    for (int i = 0; i < 5; i++) { Py_INCREF(p[i]); Py_XSETREF(*slot[i], p[i]); }
    PyObject *key, *value;
    for (Py_ssize_t pos = 0; PyDict_Next(meta, &pos, &key, &value);) {
        int stride;
        PyObject *slots;
        if (!PyArg_ParseTuple(value, "iO!", &stride, &PyTuple_Type, &slots)) return nullptr;
        std::vector<int> s;
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(slots); i++) s.push_back((int)PyLong_AsLong(PyTuple_GET_ITEM(slots, i)));
        if (PyErr_Occurred()) return nullptr;
        g_op_meta[(int)PyLong_AsLong(key)] = {stride, s};
    }
    Py_RETURN_NONE;
}
PyObject *set_tensor_class(PyObject *, PyObject *o) {
    if (!PyType_Check(o) || !PyType_IsSubtype(reinterpret_cast<PyTypeObject *>(o), &TensorType)) {
        PyErr_SetString(PyExc_TypeError, "a class derived from TensorCore");
        return nullptr;
    }
    PyObject *names = Py_BuildValue("(sssssss)", "rows", "cols", "data", "_data", "_gpu_tag", "getGpuTag", "setGpuTag");
    const bool ok = names && g_tensor_methods.take(reinterpret_cast<PyTypeObject *>(o), names);
    Py_XDECREF(names);
    if (!ok) return nullptr;
    Py_INCREF(o);
    g_tensor_class = reinterpret_cast<PyTypeObject *>(o);
    Py_RETURN_NONE;
}
// set_methods({name: function}, ComputeGraph, names): the way through a graph's methods, and which those are
PyObject *set_methods(PyObject *, PyObject *args) {
    PyObject *functions, *graph, *names;
    if (!PyArg_ParseTuple(args, "O!O!O", &PyDict_Type, &functions, &PyType_Type, &graph, &names)) return nullptr;
    if (!g_graph_methods.take(reinterpret_cast<PyTypeObject *>(graph), names)) return nullptr;
    Py_INCREF(functions);
    Py_XSETREF(g_general, functions);
    Py_RETURN_NONE;
}
// set_native(HipGpuRuntime, names, HipNative, names): the methods that calls by address stand for
PyObject *set_native(PyObject *, PyObject *args) {
    PyObject *runtime, *names, *native, *native_names;
    if (!PyArg_ParseTuple(args, "O!OO!O", &PyType_Type, &runtime, &names, &PyType_Type, &native, &native_names)) return nullptr;
    if (!g_runtime_methods.take(reinterpret_cast<PyTypeObject *>(runtime), names)) return nullptr;
    if (!g_native_methods.take(reinterpret_cast<PyTypeObject *>(native), native_names)) return nullptr;
    Py_INCREF(runtime);
    Py_INCREF(native);
    g_runtime_class = reinterpret_cast<PyTypeObject *>(runtime);
    g_native_class = reinterpret_cast<PyTypeObject *>(native);
    Py_RETURN_NONE;
}
PyMethodDef module_methods[] = {
    FAST("binary", record_binary),
    FAST("unary", record_unary),
    FAST("scalar", record_scalar),
    FAST("shaped", record_shaped),
    FAST("pair", record_pair),
    FAST("rowBroadcast", record_rows),
    FAST("colBroadcast", record_cols),
    FAST("matmul", record_matmul),
    FAST("adamW", record_adamw),
    {"set_methods", set_methods, METH_VARARGS, nullptr},
    {"set_native", set_native, METH_VARARGS, nullptr},
    {"set_helpers", set_helpers, METH_VARARGS, nullptr},
    {"set_tensor_class", set_tensor_class, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_graph_core", nullptr, -1, module_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__graph_core() {
    BufferType.tp_name = "deepj_amd.GpuBuffer";
    BufferType.tp_doc = "GpuBuffer.java:9-32.";
    BufferType.tp_basicsize = sizeof(Buffer);
    BufferType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
    BufferType.tp_new = PyType_GenericNew;
    BufferType.tp_init = (initproc)buffer_init;
    BufferType.tp_traverse = (traverseproc)buffer_traverse;
    BufferType.tp_clear = (inquiry)buffer_clear;
    BufferType.tp_dealloc = (destructor)buffer_dealloc;
    BufferType.tp_members = buffer_members;
    BufferType.tp_getset = buffer_getset;
    BufferType.tp_methods = buffer_methods;

    TensorType.tp_name = "deepj_amd._graph_core.TensorCore";
    TensorType.tp_basicsize = sizeof(Tensor);
    TensorType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
    TensorType.tp_new = tensor_new;
    TensorType.tp_init = (initproc)tensor_init;
    TensorType.tp_traverse = (traverseproc)tensor_traverse;
    TensorType.tp_clear = (inquiry)tensor_clear;
    TensorType.tp_dealloc = (destructor)tensor_dealloc;
    TensorType.tp_members = tensor_members;
    TensorType.tp_getset = tensor_getset;
    TensorType.tp_methods = tensor_methods;

    GraphType.tp_name = "deepj_amd._graph_core.GraphCore";
    GraphType.tp_basicsize = sizeof(Graph);
    GraphType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC;
    GraphType.tp_new = graph_new;
    GraphType.tp_init = (initproc)graph_init;
    GraphType.tp_traverse = (traverseproc)graph_traverse;
    GraphType.tp_clear = (inquiry)graph_clear;
    GraphType.tp_dealloc = (destructor)graph_dealloc;
    GraphType.tp_members = graph_members;
    GraphType.tp_methods = graph_methods;

    if (PyType_Ready(&BufferType) < 0 || PyType_Ready(&TensorType) < 0 || PyType_Ready(&GraphType) < 0) return nullptr;
    PyObject *m = PyModule_Create(&module_def);
    if (!m) return nullptr;
    Py_INCREF(&BufferType);
    Py_INCREF(&TensorType);
    Py_INCREF(&GraphType);
    if (PyModule_AddObject(m, "GpuBuffer", reinterpret_cast<PyObject *>(&BufferType)) < 0 ||
        PyModule_AddObject(m, "TensorCore", reinterpret_cast<PyObject *>(&TensorType)) < 0 ||
        PyModule_AddObject(m, "GraphCore", reinterpret_cast<PyObject *>(&GraphType)) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}

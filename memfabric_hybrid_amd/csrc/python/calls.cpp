// The Python face's way into the C API: address and length sequences become 64-bit words here, not in
// the interpreter.
//
// What it replaces: a ctypes array filled element by element costs 40 to 60 ns an element (a 122-segment batch
// 15 us of interpreter before a 4.4 us copy, 4096 pages in numpy arrays 700 us before a 50 us copy).  Here an int
// of a list is read where it lies (about 1 ns), and an array of 64-bit integers, which may be read-only, is handed to the
// library as it is: the library only reads it.  The interpreter lock is released for the call itself, as ctypes does; while it is, an array that was handed over must
// not be written to by another thread (the rule of the C API's own arrays).
//
// The words of the sequences of one call live in a workspace that the thread keeps between calls, up to kKeptWords, until it ends.
// A call takes it out of the thread's hands: an element's __int__ may make a batch call of its own.  The module is linked against libmf_hip_dataplane.so.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>
#if PY_VERSION_HEX < 0x030C0000
#include <longintrepr.h>
#endif

#include <cstddef>
#include <cstdint>
#include <cstring>
#include <memory>
#include <new>
#include <utility>

#include "../../../include/mf_hip_dataplane.h"
#include "../../../include/mf_xcopy_api.h"

namespace {

constexpr size_t kKeptWords = 1u << 17;   // 1 MiB a thread: three sequences of 43 000 elements
constexpr int kNoHandle = -1;             // what the transfer methods answer before initialize()

struct Workspace {
    std::unique_ptr<uint64_t[]> words;
    size_t capacity = 0;

    uint64_t *Room(size_t n)
    {
        if (n > capacity) {
            words.reset();
            words.reset(new (std::nothrow) uint64_t[n]);
            capacity = words ? n : 0;
        }
        return words.get();
    }
};
thread_local Workspace t_workspace;   // what the thread's last call has left; empty while a call uses it

inline uint64_t WordOfInt(PyObject *o)   // an int, modulo 2^64
{
#if PY_VERSION_HEX < 0x030C0000
    const auto *v = reinterpret_cast<const PyLongObject *>(o);
    switch (Py_SIZE(o)) {   // digits of PyLong_SHIFT bits, least significant first; addresses have two
        case 0:
            return 0;
        case 1:
            return v->ob_digit[0];
        case 2:
            return v->ob_digit[0] | static_cast<uint64_t>(v->ob_digit[1]) << PyLong_SHIFT;
        default:
            break;
    }
#endif
    return PyLong_AsUnsignedLongLongMask(o);
}

// int(o) modulo 2^64.  Returns false with an exception set.
bool WordOf(PyObject *o, uint64_t &out)
{
    if (PyLong_Check(o)) {
        out = WordOfInt(o);
        return true;
    }
    PyObject *as = PyNumber_Long(o);
    if (as == nullptr) {
        return false;
    }
    out = WordOfInt(as);
    Py_DECREF(as);
    return true;
}

// A handle, stream or address argument: None, an int, or a ctypes pointer value.
bool PointerOf(PyObject *o, void *&out)
{
    uint64_t word = 0;
    if (o == Py_None) {
        out = nullptr;
        return true;
    }
    if (!PyLong_Check(o)) {
        PyObject *value = PyObject_GetAttrString(o, "value");
        if (value == nullptr) {
            return false;
        }
        const bool ok = value == Py_None || WordOf(value, word);
        Py_DECREF(value);
        out = reinterpret_cast<void *>(word);
        return ok;
    }
    out = reinterpret_cast<void *>(WordOfInt(o));
    return true;
}

bool FlagsOf(PyObject *o, uint32_t &out)
{
    uint64_t word = 0;
    if (!WordOf(o, word)) {
        return false;
    }
    out = static_cast<uint32_t>(word);
    return true;
}

// One sequence argument: a list, a tuple, an array of 64-bit integers or anything else that can be iterated.
class Words {
public:
    ~Words()
    {
        if (viewed_) {
            PyBuffer_Release(&view_);
        }
        Py_XDECREF(items_);
    }

    bool Open(PyObject *o)
    {
        if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o) && PyObject_CheckBuffer(o)) {
            if (PyObject_GetBuffer(o, &view_, PyBUF_FORMAT | PyBUF_C_CONTIGUOUS) == 0) {
                viewed_ = true;
                if (view_.ndim == 1 && view_.itemsize == 8 && Integer64(view_.format) &&
                    reinterpret_cast<uintptr_t>(view_.buf) % 8 == 0) {
                    count_ = static_cast<size_t>(view_.shape[0]);
                    return true;
                }
                viewed_ = false;
                PyBuffer_Release(&view_);
            } else {
                PyErr_Clear();   // not contiguous, or no format: element by element
            }
        }
        items_ = PySequence_Fast(o, "expected a sequence of integers");
        if (items_ == nullptr) {
            return false;
        }
        count_ = static_cast<size_t>(PySequence_Fast_GET_SIZE(items_));
        return true;
    }

    size_t Count() const
    {
        return count_;
    }
    bool NeedsRoom() const
    {
        return !viewed_;
    }

    // The first n elements as words: the array itself, or `room` filled.  nullptr with an exception set on failure.
    const uint64_t *Read(size_t n, uint64_t *room)
    {
        if (viewed_) {
            return static_cast<const uint64_t *>(view_.buf);
        }
        for (size_t i = 0; i < n; ++i) {
            if (static_cast<size_t>(PySequence_Fast_GET_SIZE(items_)) < n) {   // an element's __int__ may have changed the list
                PyErr_SetString(PyExc_RuntimeError, "sequence changed while it was read");
                return nullptr;
            }
            i += PlainInts(PySequence_Fast_ITEMS(items_) + i, n - i, room + i);
            if (i == n) {
                break;
            }
            PyObject *item = PySequence_Fast_GET_ITEM(items_, static_cast<Py_ssize_t>(i));
            Py_INCREF(item);
            const bool ok = WordOf(item, room[i]);
            Py_DECREF(item);
            if (!ok) {
                return nullptr;
            }
        }
        return room;
    }

private:
    // The ints in front of the first element that is none.  No Python code runs meanwhile, so the sequence stays as it is.
    static size_t PlainInts(PyObject *const *__restrict items, size_t n, uint64_t *__restrict room)
    {
        constexpr size_t kAhead = 24;
        size_t i = 0;
        for (; i < n && PyLong_CheckExact(items[i]); ++i) {
            if (i + kAhead < n) {
                __builtin_prefetch(items[i + kAhead]);
            }
            room[i] = WordOfInt(items[i]);
        }
        return i;
    }

    static bool Integer64(const char *format)
    {
        if (format == nullptr) {
            return false;
        }
        if (*format == '@' || *format == '=' || *format == '<') {
            ++format;
        }
        return (*format == 'Q' || *format == 'q' || *format == 'L' || *format == 'l') && format[1] == '\0';
    }

    Py_buffer view_{};
    bool viewed_ = false;
    PyObject *items_ = nullptr;
    size_t count_ = 0;
};

// The three sequences of a batch.
class Batch {
public:
    Batch() : workspace_(std::exchange(t_workspace, Workspace{})) {}
    ~Batch()
    {
        if (workspace_.capacity <= kKeptWords && workspace_.capacity > t_workspace.capacity) {
            t_workspace = std::move(workspace_);
        }
    }
    Batch(const Batch &) = delete;
    Batch &operator=(const Batch &) = delete;
    bool Open(PyObject *a, PyObject *b, PyObject *c)
    {
        return words_[0].Open(a) && words_[1].Open(b) && words_[2].Open(c);
    }
    size_t Count(int i) const
    {
        return words_[i].Count();
    }
    bool Read(size_t n)
    {
        size_t needed = 1;   // never a null array, whatever n
        for (const Words &w : words_) {
            needed += w.NeedsRoom() ? n : 0;
        }
        uint64_t *room = workspace_.Room(needed);
        if (room == nullptr) {
            PyErr_NoMemory();
            return false;
        }
        for (int i = 0; i < 3; ++i) {
            at_[i] = words_[i].Read(n, room);
            if (at_[i] == nullptr) {
                if (!PyErr_Occurred()) {
                    at_[i] = room;   // an empty array may have no address
                } else {
                    return false;
                }
            }
            room += words_[i].NeedsRoom() ? n : 0;
        }
        return true;
    }
    void **Pointers(int i) const
    {
        return reinterpret_cast<void **>(const_cast<uint64_t *>(at_[i]));
    }
    uint64_t *Sizes() const
    {
        return const_cast<uint64_t *>(at_[2]);
    }

private:
    Workspace workspace_;
    Words words_[3];
    const uint64_t *at_[3] = {};
};

bool Arguments(Py_ssize_t given, Py_ssize_t wanted)
{
    if (given != wanted) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", wanted, given);
        return false;
    }
    return true;
}

// copy(handle, source, destination, size, type, flags)
PyObject *Copy(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    void *handle = nullptr;
    uint64_t size = 0;
    uint32_t type = 0;
    uint32_t flags = 0;
    void *source = nullptr;
    void *target = nullptr;
    if (!Arguments(count, 6) || !PointerOf(args[0], handle) || !PointerOf(args[1], source) || !PointerOf(args[2], target) ||
        !WordOf(args[3], size) || !FlagsOf(args[4], type) || !FlagsOf(args[5], flags)) {
        return nullptr;
    }
    smem_copy_params params{source, target, size};
    int32_t ret = 0;
    Py_BEGIN_ALLOW_THREADS;
    ret = smem_bm_copy(handle, &params, static_cast<smem_bm_copy_type>(type), flags);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(ret);
}

// copy_batch(handle, sources, destinations, sizes, count, type, flags)
PyObject *CopyBatch(PyObject *, PyObject *const *args, Py_ssize_t given)
{
    void *handle = nullptr;
    uint32_t type = 0;
    uint32_t flags = 0;
    if (!Arguments(given, 7) || !PointerOf(args[0], handle) || !FlagsOf(args[5], type) || !FlagsOf(args[6], flags)) {
        return nullptr;
    }
    const Py_ssize_t n = PyNumber_AsSsize_t(args[4], PyExc_OverflowError);
    if (n == -1 && PyErr_Occurred()) {
        return nullptr;
    }
    Batch batch;
    if (!batch.Open(args[1], args[2], args[3])) {
        return nullptr;
    }
    for (int i = 0; i < 3; ++i) {
        if (n < 0 || static_cast<uint64_t>(n) > UINT32_MAX || static_cast<size_t>(n) > batch.Count(i)) {
            return PyLong_FromLong(SM_INVALID_PARAM);   // fewer elements than the batch is said to have
        }
    }
    if (!batch.Read(static_cast<size_t>(n))) {
        return nullptr;
    }
    smem_batch_copy_params params{batch.Pointers(0), batch.Pointers(1), batch.Sizes(), static_cast<uint32_t>(n)};
    int32_t ret = 0;
    Py_BEGIN_ALLOW_THREADS;
    ret = smem_bm_copy_batch(handle, &params, static_cast<smem_bm_copy_type>(type), flags);
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(ret);
}

// transfer_batch(handle, write, peer, buffers, peer buffers, lengths, submit, stream, flags)
PyObject *TransferBatch(PyObject *, PyObject *const *args, Py_ssize_t given)
{
    if (!Arguments(given, 9)) {
        return nullptr;
    }
    void *handle = nullptr;
    void *stream = nullptr;
    uint32_t flags = 0;
    if (!PointerOf(args[0], handle)) {
        return nullptr;
    }
    if (handle == nullptr) {
        return PyLong_FromLong(kNoHandle);
    }
    Batch batch;
    if (!batch.Open(args[3], args[4], args[5])) {
        return nullptr;
    }
    const size_t n = batch.Count(0);
    if (n != batch.Count(1) || n != batch.Count(2) || n > UINT32_MAX) {
        return PyLong_FromLong(kNoHandle);
    }
    const char *peer = PyUnicode_AsUTF8(args[2]);
    if (peer == nullptr || !PointerOf(args[7], stream) || !FlagsOf(args[8], flags) || !batch.Read(n)) {
        return nullptr;
    }
    const bool write = args[1] == Py_True;
    const bool submit = args[6] == Py_True;
    const auto size = static_cast<uint32_t>(n);
    void **local = batch.Pointers(0);
    void **remote = batch.Pointers(1);
    static_assert(sizeof(size_t) == sizeof(uint64_t), "64-bit sizes expected");
    auto *lengths = reinterpret_cast<size_t *>(batch.Sizes());
    int32_t ret = 0;
    Py_BEGIN_ALLOW_THREADS;
    if (write) {
        auto *from = const_cast<const void **>(local);
        ret = submit ? smem_trans_batch_write_submit(handle, from, peer, remote, lengths, size, stream, flags)
                     : smem_trans_batch_write(handle, from, peer, remote, lengths, size, flags);
    } else {
        auto *from = const_cast<const void **>(remote);
        ret = submit ? smem_trans_batch_read_submit(handle, local, peer, from, lengths, size, stream, flags)
                     : smem_trans_batch_read(handle, local, peer, from, lengths, size, flags);
    }
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(ret);
}

// fill(array, values): a writable array of 64-bit words from as many integers
PyObject *Fill(PyObject *, PyObject *const *args, Py_ssize_t given)
{
    if (!Arguments(given, 2)) {
        return nullptr;
    }
    Words values;
    if (!values.Open(args[1])) {
        return nullptr;
    }
    Py_buffer target;
    if (PyObject_GetBuffer(args[0], &target, PyBUF_WRITABLE | PyBUF_C_CONTIGUOUS) != 0) {
        return nullptr;
    }
    const size_t n = values.Count();
    const uint64_t *at = nullptr;
    if (static_cast<size_t>(target.len) < 8 * n) {
        PyErr_SetString(PyExc_ValueError, "array is too short");
    } else {
        at = values.Read(n, static_cast<uint64_t *>(target.buf));
        if (at != nullptr && at != target.buf) {
            std::memmove(target.buf, at, 8 * n);
        }
    }
    PyBuffer_Release(&target);
    if (PyErr_Occurred()) {
        return nullptr;
    }
    Py_RETURN_NONE;
}

template <class F>
PyCFunction AsMethod(F f)
{
    return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

// A function of the C API that takes addresses and numbers only, in the place of its ctypes object: plain ints, and None for an address, go to it as
// they are; a call with anything else, and every attribute, is the ctypes object's.  ctypes looks a converter up and calls it for every argument: a dispatch
// and a combine of the decode path, 22 arguments, take the host 2.1 us less so (2 tokens, both calls, 8.9 -> 7.6 us), a table's four 0.35.
struct Direct {
    PyObject_HEAD
    vectorcallfunc call;
    PyObject *function;     // the ctypes object
    PyObject *(*direct)(const uint64_t *args);      // null once something has been set on that: its types may be others
    const char *kinds;      // an argument each: 'p' address, 'i' number
};

bool Plain(PyObject *const *args, const char *kinds, uint64_t *words)
{
    for (; *kinds != '\0'; ++kinds, ++args, ++words) {
        if (PyLong_CheckExact(*args)) {
            *words = WordOfInt(*args);
        } else if (*args == Py_None && *kinds == 'p') {
            *words = 0;
        } else {
            return false;
        }
    }
    return true;
}

PyObject *CallDirect(PyObject *self, PyObject *const *args, size_t nargsf, PyObject *names)
{
    const auto *d = reinterpret_cast<const Direct *>(self);
    constexpr size_t kMost = 16;
    uint64_t words[kMost];
    if (names == nullptr && d->direct != nullptr && static_cast<size_t>(PyVectorcall_NARGS(nargsf)) == std::strlen(d->kinds) &&
        Plain(args, d->kinds, words)) {
        return d->direct(words);
    }
    return PyObject_Vectorcall(d->function, args, nargsf, names);
}

template <class T>
T *Address(uint64_t word)
{
    return reinterpret_cast<T *>(word);
}

uint32_t Number(uint64_t word)
{
    return static_cast<uint32_t>(word);
}

PyObject *MoeDispatch(const uint64_t *a)
{
    int32_t ret = 0;
    Py_BEGIN_ALLOW_THREADS;
    ret = mf_moe_dispatch(Address<const void>(a[0]), Address<const int32_t>(a[1]), Number(a[2]), Number(a[3]), Number(a[4]), Number(a[5]),
                          Address<void>(a[6]), Address<int32_t>(a[7]), Address<int32_t>(a[8]), Address<int32_t>(a[9]), Address<int32_t>(a[10]),
                          Address<void>(a[11]), a[12], Address<void>(a[13]));
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(ret);
}

PyObject *MoeCombine(const uint64_t *a)
{
    int32_t ret = 0;
    Py_BEGIN_ALLOW_THREADS;
    ret = mf_moe_combine(Address<const void>(a[0]), Address<const int32_t>(a[1]), Address<const float>(a[2]), Number(a[3]), Number(a[4]), Number(a[5]),
                         Address<void>(a[6]), Address<void>(a[7]));
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(ret);
}

PyObject *DeviceTable(const uint64_t *a)
{
    int32_t ret = 0;
    Py_BEGIN_ALLOW_THREADS;
    ret = mf_xcopy_device_table(Address<const void>(a[0]), Number(a[1]), static_cast<int32_t>(Number(a[2])), Address<void>(a[3]));
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(ret);
}

struct DirectKind {
    const char *name;
    const char *kinds;
    PyObject *(*direct)(const uint64_t *args);
};
constexpr DirectKind kDirects[] = {
    {"mf_moe_dispatch", "ppiiiippppppip", MoeDispatch},
    {"mf_moe_combine", "pppiiipp", MoeCombine},
    {"mf_xcopy_device_table", "piip", DeviceTable},
};

void DirectDealloc(PyObject *self)
{
    PyTypeObject *type = Py_TYPE(self);
    Py_XDECREF(reinterpret_cast<Direct *>(self)->function);
    type->tp_free(self);
    Py_DECREF(type);
}

PyObject *DirectGet(PyObject *self, PyObject *name)
{
    PyObject *function = reinterpret_cast<Direct *>(self)->function;
    if (PyUnicode_CompareWithASCIIString(name, "_as_parameter_") == 0) {    // where ctypes is given a function
        Py_INCREF(function);
        return function;
    }
    return PyObject_GetAttr(function, name);
}

int DirectSet(PyObject *self, PyObject *name, PyObject *value)
{
    auto *d = reinterpret_cast<Direct *>(self);
    d->direct = nullptr;
    return PyObject_SetAttr(d->function, name, value);
}

PyMemberDef g_directMembers[] = {
    {"__vectorcalloffset__", T_PYSSIZET, offsetof(Direct, call), READONLY, nullptr},
    {nullptr, 0, 0, 0, nullptr},
};
PyType_Slot g_directSlots[] = {
    {Py_tp_dealloc, reinterpret_cast<void *>(DirectDealloc)},
    {Py_tp_getattro, reinterpret_cast<void *>(DirectGet)},
    {Py_tp_setattro, reinterpret_cast<void *>(DirectSet)},
    {Py_tp_call, reinterpret_cast<void *>(PyVectorcall_Call)},
    {Py_tp_members, g_directMembers},
    {0, nullptr},
};
PyType_Spec g_directSpec = {"_calls.Direct", sizeof(Direct), 0,
                            Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL | Py_TPFLAGS_DISALLOW_INSTANTIATION, g_directSlots};
PyTypeObject *g_directType = nullptr;

// direct(name, function): what stands for the ctypes object of that function, or the object itself where there is nothing
PyObject *MakeDirect(PyObject *, PyObject *const *args, Py_ssize_t given)
{
    if (!Arguments(given, 2)) {
        return nullptr;
    }
    const char *name = PyUnicode_AsUTF8(args[0]);
    if (name == nullptr) {
        return nullptr;
    }
    for (const DirectKind &kind : kDirects) {
        if (std::strcmp(kind.name, name) == 0) {
            auto *d = PyObject_New(Direct, g_directType);
            if (d == nullptr) {
                return nullptr;
            }
            d->call = CallDirect;
            Py_INCREF(args[1]);
            d->function = args[1];
            d->direct = kind.direct;
            d->kinds = kind.kinds;
            return reinterpret_cast<PyObject *>(d);
        }
    }
    Py_INCREF(args[1]);
    return args[1];
}

PyMethodDef g_methods[] = {
    {"copy", AsMethod(Copy), METH_FASTCALL, "copy(handle, source, destination, size, type, flags) -> code"},
    {"copy_batch", AsMethod(CopyBatch), METH_FASTCALL,
     "copy_batch(handle, sources, destinations, sizes, count, type, flags) -> code"},
    {"transfer_batch", AsMethod(TransferBatch), METH_FASTCALL,
     "transfer_batch(handle, write, peer, buffers, peer_buffers, lengths, submit, stream, flags) -> code"},
    {"direct", AsMethod(MakeDirect), METH_FASTCALL, "direct(name, function): a function that is called without ctypes where that is possible"},
    {"fill", AsMethod(Fill), METH_FASTCALL, "fill(array, values): the values as 64-bit words in the array"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_calls", "Native calls of the Python face.", -1, g_methods,
                        nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls(void)
{
    g_directType = reinterpret_cast<PyTypeObject *>(PyType_FromSpec(&g_directSpec));
    return g_directType == nullptr ? nullptr : PyModule_Create(&g_module);
}

// CPython module tensorrt_amd._plugin_call: the two calls of a plugin's runtime that a Python host makes per layer and
// pass, with the tensor descriptions read from the Python objects here.  Filling ctypes structures from Python costs 6
// to 8 us per enqueue, twice what the launch itself takes (SkipLayerNorm of 1024 x 768 FP32, whose kernel takes 3.9 us:
// 10.4 us per call with the structures filled in Python, 4.1 us with this module).
//
// Nothing is linked: the C functions of include/trtamd_plugin_c.h come in as addresses, so the module does not depend on
// where the plugin library lies.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "trtamd_plugin_c.h"

#include <memory>
#include <new>

namespace
{

PyObject *gDims, *gType, *gFormat, *gScale; // interned attribute names

constexpr Py_ssize_t kInline = 8; // tensors per side that need no heap allocation

bool asInt64(PyObject* o, int64_t& out)
{
    if (PyLong_Check(o))
    {
        out = PyLong_AsLongLong(o);
    }
    else
    {
        PyObject* n = PyNumber_Long(o); // numpy integers and the like
        if (!n)
        {
            return false;
        }
        out = PyLong_AsLongLong(n);
        Py_DECREF(n);
    }
    return out != -1 || !PyErr_Occurred();
}

bool asPointer(PyObject* o, void*& out)
{
    PyObject* n = PyNumber_Long(o);
    if (!n)
    {
        return false;
    }
    unsigned long long const v = PyLong_AsUnsignedLongLongMask(n);
    Py_DECREF(n);
    out = reinterpret_cast<void*>(v);
    return !PyErr_Occurred();
}

bool intAttribute(PyObject* o, PyObject* name, int32_t& out)
{
    PyObject* a = PyObject_GetAttr(o, name);
    int64_t v = 0;
    bool const ok = a && asInt64(a, v);
    Py_XDECREF(a);
    out = static_cast<int32_t>(v);
    return ok;
}

// The fields that the runtime calls read: dims, type, format, scale.
bool readDesc(PyObject* t, trtamd_tensor_desc& d)
{
    PyObject* dims = PyObject_GetAttr(t, gDims);
    PyObject* seq = dims ? PySequence_Fast(dims, "dims must be a sequence") : nullptr;
    Py_XDECREF(dims);
    if (!seq)
    {
        return false;
    }
    Py_ssize_t const n = PySequence_Fast_GET_SIZE(seq);
    bool ok = n <= TRTAMD_MAX_DIMS;
    if (!ok)
    {
        PyErr_SetString(PyExc_IndexError, "invalid index");
    }
    for (Py_ssize_t i = 0; ok && i < n; ++i)
    {
        ok = asInt64(PySequence_Fast_GET_ITEM(seq, i), d.dims[i]);
    }
    Py_DECREF(seq);
    d.nb_dims = static_cast<int32_t>(n);
    if (!ok || !intAttribute(t, gType, d.type) || !intAttribute(t, gFormat, d.format))
    {
        return false;
    }
    PyObject* s = PyObject_GetAttr(t, gScale);
    PyObject* f = s ? PyNumber_Float(s) : nullptr;
    Py_XDECREF(s);
    if (!f)
    {
        return false;
    }
    d.scale = static_cast<float>(PyFloat_AS_DOUBLE(f));
    Py_DECREF(f);
    return true;
}

// A Python sequence of n items turned into C values, in place for the usual few and on the heap beyond.
template <typename T>
class Values
{
public:
    template <typename Read>
    bool fill(PyObject* sequence, Read read)
    {
        PyObject* seq = PySequence_Fast(sequence, "a sequence is required");
        if (!seq)
        {
            return false;
        }
        mCount = PySequence_Fast_GET_SIZE(seq);
        if (mCount > kInline)
        {
            mHeap.reset(new (std::nothrow) T[static_cast<size_t>(mCount)]{}); // no exception may leave for the interpreter
            if (!mHeap)
            {
                Py_DECREF(seq);
                PyErr_NoMemory();
                return false;
            }
        }
        bool ok = true;
        for (Py_ssize_t i = 0; ok && i < mCount; ++i)
        {
            ok = read(PySequence_Fast_GET_ITEM(seq, i), data()[i]);
        }
        Py_DECREF(seq);
        return ok;
    }
    T* data()
    {
        return mCount > kInline ? mHeap.get() : mInline;
    }
    int32_t count() const
    {
        return static_cast<int32_t>(mCount);
    }

private:
    T mInline[kInline]{};
    std::unique_ptr<T[]> mHeap;
    Py_ssize_t mCount{0};
};

using OnShapeChange = int32_t (*)(void*, trtamd_tensor_desc const*, int32_t, trtamd_tensor_desc const*, int32_t);
using Enqueue = int32_t (*)(void*, trtamd_tensor_desc const*, int32_t, trtamd_tensor_desc const*, int32_t,
    void const* const*, void* const*, void*, void*);

// on_shape_change(function address, plugin handle, inputs, outputs) -> status
PyObject* onShapeChange(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    void *fn, *plugin;
    Values<trtamd_tensor_desc> in, out;
    if (n != 4)
    {
        PyErr_SetString(PyExc_TypeError, "on_shape_change takes 4 arguments");
        return nullptr;
    }
    if (!asPointer(args[0], fn) || !asPointer(args[1], plugin) || !in.fill(args[2], readDesc) || !out.fill(args[3], readDesc))
    {
        return nullptr;
    }
    int32_t status;
    Py_BEGIN_ALLOW_THREADS
    status = reinterpret_cast<OnShapeChange>(fn)(plugin, in.data(), in.count(), out.data(), out.count());
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
}

// enqueue(function address, plugin handle, input descriptions, output descriptions, input addresses, output addresses,
// workspace, stream) -> status
PyObject* enqueue(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    void *fn, *plugin, *workspace, *stream;
    Values<trtamd_tensor_desc> in, out;
    Values<void*> inputs, outputs;
    if (n != 8)
    {
        PyErr_SetString(PyExc_TypeError, "enqueue takes 8 arguments");
        return nullptr;
    }
    if (!asPointer(args[0], fn) || !asPointer(args[1], plugin) || !in.fill(args[2], readDesc) || !out.fill(args[3], readDesc)
        || !inputs.fill(args[4], asPointer) || !outputs.fill(args[5], asPointer) || !asPointer(args[6], workspace)
        || !asPointer(args[7], stream))
    {
        return nullptr;
    }
    int32_t status;
    Py_BEGIN_ALLOW_THREADS
    status = reinterpret_cast<Enqueue>(fn)(
        plugin, in.data(), in.count(), out.data(), out.count(), inputs.data(), outputs.data(), workspace, stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
}

PyMethodDef gMethods[] = {
    {"on_shape_change", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(onShapeChange)), METH_FASTCALL,
        "IPluginV3OneRuntime::onShapeChange"},
    {"enqueue", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(enqueue)), METH_FASTCALL,
        "IPluginV3OneRuntime::enqueue / IPluginV2DynamicExt::enqueue"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef gModule = {PyModuleDef_HEAD_INIT, "_plugin_call", "Runtime calls of the plugins", -1, gMethods, nullptr,
    nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__plugin_call(void)
{
    gDims = PyUnicode_InternFromString("dims");
    gType = PyUnicode_InternFromString("type");
    gFormat = PyUnicode_InternFromString("format");
    gScale = PyUnicode_InternFromString("scale");
    return gDims && gType && gFormat && gScale ? PyModule_Create(&gModule) : nullptr;
}

// The part of the Python interface that runs for every call: operators submitted on the default stream without a wait, the
// planes of a list of torch tensors and batches of them, tensors of the library's own memory, the results that are handed out
// again and torch's views of them. In Python one call of an operator was 5.3 to 6.2 us of the interpreter beside 2 to 3 us of the
// library, a result tensor 2.0 us, a batch of 61 images another 43 us.
//
// What is here does what its Python counterpart does or leaves the call to it (pyapi._submit), before anything has happened:
// other streams, waits, threads at the containers' marks, arguments of other types.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <cvcuda/OpConvertTo.h>
#include <cvcuda/OpCropFlipNormalizeReformat.h>
#include <cvcuda/OpCvtColor.h>
#include <cvcuda/OpNormalize.h>
#include <cvcuda/OpReformat.h>
#include <cvcuda/OpResize.h>
#include <cvcuda/OpResizeCropConvertReformat.h>
#include <cvcuda/OpWarpAffine.h>
#include <cvcuda/OpWarpPerspective.h>
#include <nvcv/Tensor.h>
#include <structmember.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>
#include <cstring>
#include <memory>

namespace {

// names of pyapi and of the containers
PyObject *s_submit, *s_Tensor, *s_ImageBatchVarShape, *s_lock, *s_followed, *s_tls, *s_stack, *s_check, *s_t, *s_handle, *s_wrote, *s_read,
    *s_kind, *s_acquire, *s_release, *s_torch, *s_C, *s_getDevice, *s_getStream, *s_value, *s_key, *s_meta, *s_nbytes, *s_np, *s_dtype, *s_made,
    *s_sizeOf;

// A new reference that goes with the scope.
struct Ref
{
    PyObject *o;
    explicit Ref(PyObject *obj = nullptr)
        : o(obj)
    {
    }
    ~Ref()
    {
        Py_XDECREF(o);
    }
    Ref(const Ref &)            = delete;
    Ref &operator=(const Ref &) = delete;
    explicit operator bool() const
    {
        return o != nullptr;
    }
};

// `api`: pyapi's dictionary, which bind() makes the `self` of the functions that use it (each copy of the package in a process
// has its own). Its names are looked up in each call: they can be replaced. Borrowed.
PyObject *Name(PyObject *api, PyObject *name)
{
    return PyDict_GetItem(api, name);
}

// The key of the current device's default stream (0, -1, -2 ...) where that is the current stream: false elsewhere, and where
// a Python error is set.
bool DefaultStreamKey(PyObject *api, long &key)
{
    PyObject *tls = Name(api, s_tls);
    if (tls == nullptr)
    {
        return false;
    }
    Ref stack(PyObject_GetAttr(tls, s_stack));
    if (!stack && PyErr_ExceptionMatches(PyExc_AttributeError))
    {
        // a thread's first call: the list that `with stream:` would make, so that the next call finds it
        PyErr_Clear();
        stack.o = PyList_New(0);
        if (stack && PyObject_SetAttr(tls, s_stack, stack.o) < 0)
        {
            return false;
        }
    }
    if (!stack || PyObject_IsTrue(stack.o) != 0)
    {
        return false;
    }
    PyObject *torch = Name(api, s_torch);
    Ref       c(torch != nullptr ? PyObject_GetAttr(torch, s_C) : nullptr);
    if (!c)
    {
        return false;
    }
    Ref device(PyObject_CallMethodNoArgs(c.o, s_getDevice));
    Ref stream(device ? PyObject_CallMethodOneArg(c.o, s_getStream, device.o) : nullptr);
    if (!stream || PyObject_IsTrue(stream.o) != 0)
    {
        return false;
    }
    key = -PyLong_AsLong(device.o);
    return !PyErr_Occurred();
}

enum Kind
{
    kNone,
    kTensor,
    kBatch
};

// The pointer that an object's `handle` (a ctypes.c_void_p) holds.
bool Pointer(PyObject *obj, void *&p)
{
    Ref h(PyObject_GetAttr(obj, s_handle)), value(h ? PyObject_GetAttr(h.o, s_value) : nullptr);
    if (!value || !PyLong_CheckExact(value.o))
    {
        PyErr_Clear();
        return false;
    }
    p = PyLong_AsVoidPtr(value.o);
    if (PyErr_Occurred())
    {
        PyErr_Clear();
        return false;
    }
    return true;
}

// The library's handle of a container of pyapi.
Kind HandleOf(PyObject *api, PyObject *obj, void *&handle)
{
    const bool tensor = Py_TYPE(obj) == reinterpret_cast<PyTypeObject *>(Name(api, s_Tensor));
    if (!tensor && Py_TYPE(obj) != reinterpret_cast<PyTypeObject *>(Name(api, s_ImageBatchVarShape)))
    {
        return kNone;
    }
    Ref inner(tensor ? PyObject_GetAttr(obj, s_t) : nullptr);
    if (tensor && !inner)
    {
        PyErr_Clear();
        return kNone;
    }
    return Pointer(tensor ? inner.o : obj, handle) && handle != nullptr ? (tensor ? kTensor : kBatch) : kNone;
}

bool Int(PyObject *o, int &v)
{
    const long l = PyLong_Check(o) ? PyLong_AsLong(o) : LONG_MAX;
    v            = (int)l;
    if (l == -1 && PyErr_Occurred())
    {
        PyErr_Clear();
        return false;
    }
    return l >= INT_MIN && l <= INT_MAX;
}

bool Real(PyObject *o, double &v)
{
    v = PyFloat_CheckExact(o) ? PyFloat_AS_DOUBLE(o) : 0;
    return PyFloat_CheckExact(o);
}

// `n` floats of a list or tuple.
bool Reals(PyObject *o, float *v, Py_ssize_t n)
{
    if (!(PyList_CheckExact(o) || PyTuple_CheckExact(o)) || PySequence_Fast_GET_SIZE(o) != n)
    {
        return false;
    }
    for (Py_ssize_t i = 0; i < n; ++i)
    {
        double d;
        if (!Real(PySequence_Fast_GET_ITEM(o, i), d))
        {
            return false;
        }
        v[i] = (float)d;
    }
    return true;
}

bool Pair(PyObject *o, int &x, int &y)
{
    return PyTuple_CheckExact(o) && PyTuple_GET_SIZE(o) == 2 && Int(PyTuple_GET_ITEM(o, 0), x) && Int(PyTuple_GET_ITEM(o, 1), y);
}

// One call of an operator: its C function and its arguments, in the order of the package's operator classes.
struct Call
{
    int                kind;
    NVCVOperatorHandle op;
    void              *h[5];
    bool               batch, flag;
    int                i[6];
    double             d[4];
    float              m[9], bv[4];

    bool Parse(PyObject *api, PyObject *const *a, Py_ssize_t n)
    {
        auto handles = [&](std::initializer_list<int> at)
        {
            int k = 0;
            for (int index : at)
            {
                const Kind got = HandleOf(api, a[index], h[k]);
                if (k == 0)
                {
                    batch = got == kBatch;
                }
                if (got == kNone)
                {
                    return false;
                }
                ++k;
            }
            return true;
        };
        switch (kind)
        {
        case 1: // Resize
        case 2: // CvtColor
            return n == 3 && handles({0, 1}) && Int(a[2], i[0]);
        case 3: // Reformat
            return n == 2 && handles({0, 1}) && !batch;
        case 4: // ConvertTo
            return n == 4 && handles({0, 1}) && !batch && Real(a[2], d[0]) && Real(a[3], d[1]);
        case 5: // Normalize
            return n == 8 && handles({0, 1, 2, 3}) && Real(a[4], d[0]) && Real(a[5], d[1]) && Real(a[6], d[2]) && Int(a[7], i[0]) && i[0] >= 0;
        case 6: // ResizeCropConvertReformat
            flag = n == 9 && a[8] == Py_True;
            return n == 9 && handles({0, 1}) && Pair(a[2], i[0], i[1]) && Int(a[3], i[2]) && Pair(a[4], i[3], i[4]) && Int(a[5], i[5])
                && Real(a[6], d[0]) && Real(a[7], d[1]) && PyBool_Check(a[8]);
        case 7: // CropFlipNormalizeReformat
            return n == 12 && handles({0, 1, 2, 5, 6}) && HandleOf(api, a[7], h4) != kNone && batch && Int(a[3], i[0]) && Real(a[4], d[0])
                && Real(a[8], d[1]) && Real(a[9], d[2]) && Real(a[10], d[3]) && Int(a[11], i[1]) && i[1] >= 0;
        case 8: // WarpAffine
        case 9: // WarpPerspective
            return n == 6 && handles({0, 1}) && (batch ? HandleOf(api, a[2], h[2]) != kNone : Reals(a[2], m, kind == 8 ? 6 : 9)) && Int(a[3], i[0])
                && Int(a[4], i[1]) && Reals(a[5], bv, 4);
        default:
            return false;
        }
    }

    void *h4 = nullptr; // CropFlipNormalizeReformat's scale

    template<class H>
    H As(int k) const
    {
        return reinterpret_cast<H>(h[k]);
    }

    NVCVStatus Submit() const
    {
        using T = NVCVTensorHandle;
        using B = NVCVImageBatchHandle;
        const auto interp = (NVCVInterpolationType)i[0];
        switch (kind)
        {
        case 1:
            return batch ? cvcudaResizeVarShapeSubmit(op, nullptr, As<B>(0), As<B>(1), interp)
                         : cvcudaResizeSubmit(op, nullptr, As<T>(0), As<T>(1), interp);
        case 2:
            return batch ? cvcudaCvtColorVarShapeSubmit(op, nullptr, As<B>(0), As<B>(1), (NVCVColorConversionCode)i[0])
                         : cvcudaCvtColorSubmit(op, nullptr, As<T>(0), As<T>(1), (NVCVColorConversionCode)i[0]);
        case 3:
            return cvcudaReformatSubmit(op, nullptr, As<T>(0), As<T>(1));
        case 4:
            return cvcudaConvertToSubmit(op, nullptr, As<T>(0), As<T>(1), d[0], d[1]);
        case 5:
            return batch ? cvcudaNormalizeVarShapeSubmit(op, nullptr, As<B>(0), As<T>(1), As<T>(2), As<B>(3), (float)d[0], (float)d[1],
                                                         (float)d[2], (uint32_t)i[0])
                         : cvcudaNormalizeSubmit(op, nullptr, As<T>(0), As<T>(1), As<T>(2), As<T>(3), (float)d[0], (float)d[1], (float)d[2],
                                                 (uint32_t)i[0]);
        case 6:
        {
            const NVCVSize2D size = {i[0], i[1]};
            const int2       at   = {i[3], i[4]};
            return batch ? cvcudaResizeCropConvertReformatVarShapeSubmit(op, nullptr, As<B>(0), As<T>(1), size, (NVCVInterpolationType)i[2], at,
                                                                         (NVCVChannelManip)i[5], (float)d[0], (float)d[1], flag)
                         : cvcudaResizeCropConvertReformatSubmit(op, nullptr, As<T>(0), As<T>(1), size, (NVCVInterpolationType)i[2], at,
                                                                 (NVCVChannelManip)i[5], (float)d[0], (float)d[1], flag);
        }
        case 7:
            return cvcudaCropFlipNormalizeReformatSubmit(op, nullptr, As<B>(0), As<T>(1), As<T>(2), (NVCVBorderType)i[0], (float)d[0],
                                                         As<T>(3), As<T>(4), reinterpret_cast<T>(h4), (float)d[1], (float)d[2], (float)d[3],
                                                         (uint32_t)i[1]);
        default:
        {
            const float4 c = {bv[0], bv[1], bv[2], bv[3]};
            const auto   border = (NVCVBorderType)i[1];
            if (kind == 8)
            {
                return batch ? cvcudaWarpAffineVarShapeSubmit(op, nullptr, As<B>(0), As<B>(1), As<T>(2), i[0], border, c)
                             : cvcudaWarpAffineSubmit(op, nullptr, As<T>(0), As<T>(1), m, i[0], border, c);
            }
            return batch ? cvcudaWarpPerspectiveVarShapeSubmit(op, nullptr, As<B>(0), As<B>(1), As<T>(2), i[0], border, c)
                         : cvcudaWarpPerspectiveSubmit(op, nullptr, As<T>(0), As<T>(1), m, i[0], border, c);
        }
        }
    }
};

// The container's attributes (a new reference), null where it has none.
PyObject *AttributesOf(PyObject *obj)
{
    PyObject *dict = PyObject_GenericGetDict(obj, nullptr);
    if (dict == nullptr)
    {
        PyErr_Clear();
    }
    return dict;
}

bool SameKey(PyObject *o, long key)
{
    return PyLong_CheckExact(o) && PyLong_AsLong(o) == key;
}

// Whether a mark (stream, event) is absent or of stream `key`.
bool WroteBy(PyObject *attributes, long key)
{
    PyObject *wrote = PyDict_GetItem(attributes, s_wrote);
    return wrote == nullptr || (PyTuple_CheckExact(wrote) && PyTuple_GET_SIZE(wrote) == 2 && SameKey(PyTuple_GET_ITEM(wrote, 0), key));
}

bool ReadBy(PyObject *attributes, long key)
{
    PyObject *read = PyDict_GetItem(attributes, s_read);
    if (read == nullptr)
    {
        return true;
    }
    PyObject  *other;
    Py_ssize_t at = 0;
    if (!PyDict_CheckExact(read))
    {
        return false;
    }
    while (PyDict_Next(read, &at, &other, nullptr))
    {
        if (!SameKey(other, key))
        {
            return false;
        }
    }
    return true;
}

// Whether no container of the call has a mark of another stream.
bool NothingToWaitFor(PyObject *reads, PyObject *writes, long key)
{
    for (Py_ssize_t k = 0; k < PyList_GET_SIZE(reads); ++k)
    {
        Ref attributes(AttributesOf(PyList_GET_ITEM(reads, k)));
        if (!attributes || !WroteBy(attributes.o, key))
        {
            return false;
        }
    }
    for (Py_ssize_t k = 0; k < PyList_GET_SIZE(writes); ++k)
    {
        Ref attributes(AttributesOf(PyList_GET_ITEM(writes, k)));
        if (!attributes || !WroteBy(attributes.o, key) || !ReadBy(attributes.o, key))
        {
            return false;
        }
    }
    return true;
}

// The marks of a call on default stream `key`: as pyapi._submit leaves them, without an event.
bool Mark(PyObject *reads, PyObject *writes, PyObject *key)
{
    for (Py_ssize_t k = 0; k < PyList_GET_SIZE(reads); ++k)
    {
        Ref       attributes(AttributesOf(PyList_GET_ITEM(reads, k)));
        PyObject *read = attributes ? PyDict_GetItem(attributes.o, s_read) : nullptr;
        if (read != nullptr)
        {
            if (PyDict_GetItem(read, key) != Py_None && PyDict_SetItem(read, key, Py_None) < 0)
            {
                return false;
            }
            continue;
        }
        Ref fresh(PyDict_New());
        if (!fresh || PyDict_SetItem(fresh.o, key, Py_None) < 0 || PyObject_SetAttr(PyList_GET_ITEM(reads, k), s_read, fresh.o) < 0)
        {
            return false;
        }
    }
    for (Py_ssize_t k = 0; k < PyList_GET_SIZE(writes); ++k)
    {
        PyObject *obj = PyList_GET_ITEM(writes, k);
        Ref       attributes(AttributesOf(obj));
        PyObject *was = attributes ? PyDict_GetItem(attributes.o, s_wrote) : nullptr, *read = attributes ? PyDict_GetItem(attributes.o, s_read) : nullptr;
        // (marks that stand already stay; another thread may have set others meanwhile)
        const bool stands = was != nullptr && PyTuple_CheckExact(was) && PyTuple_GET_SIZE(was) == 2 && PyTuple_GET_ITEM(was, 1) == Py_None
                         && PyObject_RichCompareBool(PyTuple_GET_ITEM(was, 0), key, Py_EQ) == 1;
        if (!stands)
        {
            Ref wrote(PyTuple_Pack(2, key, Py_None));
            if (!wrote || PyObject_SetAttr(obj, s_wrote, wrote.o) < 0)
            {
                return false;
            }
        }
        if (read == nullptr || !PyDict_CheckExact(read) || PyDict_GET_SIZE(read) != 0)
        {
            Ref none(PyDict_New());
            if (!none || PyObject_SetAttr(obj, s_read, none.o) < 0)
            {
                return false;
            }
        }
    }
    return true;
}

// submit(stream, reads, writes, op, *args): pyapi._submit for calls on the current device's default stream, given as None, that
// wait for nothing; others are handed on to it.
PyObject *Submit(PyObject *api, PyObject *const *a, Py_ssize_t n)
{
    auto handOn = [&]() -> PyObject *
    {
        PyObject *submit = Name(api, s_submit);
        return submit != nullptr ? PyObject_Vectorcall(submit, a, (size_t)n, nullptr)
                                 : (PyErr_SetString(PyExc_RuntimeError, "pyapi is gone"), nullptr);
    };
    Call call;
    long key;
    if (n < 4 || a[0] != Py_None || !PyList_CheckExact(a[1]) || !PyList_CheckExact(a[2]) || !DefaultStreamKey(api, key))
    {
        PyErr_Clear();
        return handOn();
    }
    Ref   kind(PyObject_GetAttr(a[3], s_kind));
    void *op = nullptr;
    if (!kind || !Int(kind.o, call.kind) || !Pointer(a[3], op) || !call.Parse(api, a + 4, n - 4))
    {
        PyErr_Clear();
        return handOn();
    }
    call.op = reinterpret_cast<NVCVOperatorHandle>(op);
    Ref       keyObject(PyLong_FromLong(key));
    PyObject *lock = Name(api, s_lock), *followed = Name(api, s_followed);
    // the marks are read under their lock; where another thread holds it, Python waits for it
    Ref got(lock != nullptr && followed != nullptr && keyObject ? PyObject_CallMethodOneArg(lock, s_acquire, Py_False) : nullptr);
    if (!got || got.o != Py_True)
    {
        PyErr_Clear();
        return handOn();
    }
    PyObject  *calls = PyDict_GetItem(followed, keyObject.o);
    const bool plain = (calls == nullptr || PyObject_IsTrue(calls) == 0) && NothingToWaitFor(a[1], a[2], key);
    Ref        released(PyObject_CallMethodNoArgs(lock, s_release));
    if (!plain)
    {
        PyErr_Clear();
        return handOn();
    }
    NVCVStatus status;
    Py_BEGIN_ALLOW_THREADS
    status = call.Submit();
    Py_END_ALLOW_THREADS
    if (status != NVCV_SUCCESS)
    {
        PyObject *check = Name(api, s_check);
        Ref       value(PyLong_FromLong((long)status));
        Ref       raised(check != nullptr && value ? PyObject_CallOneArg(check, value.o) : nullptr);
        if (!PyErr_Occurred())
        {
            PyErr_SetString(PyExc_RuntimeError, "the operator failed");
        }
        return nullptr;
    }
    Ref        held(PyObject_CallMethodNoArgs(lock, s_acquire));
    const bool ok = held && Mark(a[1], a[2], keyObject.o);
    if (held)
    {
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        Ref freed(PyObject_CallMethodNoArgs(lock, s_release));
        PyErr_Restore(type, value, trace);
    }
    if (!ok)
    {
        return nullptr;
    }
    Py_RETURN_NONE;
}

// default_stream_key(): pyapi._default_stream_key(None) outside `with stream:`; None inside, where Python looks at the stream.
PyObject *DefaultKey(PyObject *api, PyObject *)
{
    long key;
    if (DefaultStreamKey(api, key))
    {
        return PyLong_FromLong(key);
    }
    if (PyErr_Occurred())
    {
        return nullptr;
    }
    Py_RETURN_NONE;
}

// planes(buffers): (channels, packed NVCVImagePlaneStrided array) of torch tensors on the GPU of one element type and channel
// count, each (H, W) or (H, W, C); None where a buffer is anything else.
PyObject *Planes(PyObject *, PyObject *buffers)
{
    Ref list(PySequence_Fast(buffers, "buffers: a sequence"));
    if (!list)
    {
        return nullptr;
    }
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(list.o);
    Ref              out(PyBytes_FromStringAndSize(nullptr, n * (Py_ssize_t)sizeof(NVCVImagePlaneStrided)));
    if (!out)
    {
        return nullptr;
    }
    auto          *plane    = reinterpret_cast<NVCVImagePlaneStrided *>(PyBytes_AS_STRING(out.o));
    int64_t        channels = 0;
    at::ScalarType type     = at::kByte;
    try
    {
        for (Py_ssize_t k = 0; k < n; ++k)
        {
            PyObject *obj = PySequence_Fast_GET_ITEM(list.o, k);
            if (!THPVariable_CheckExact(obj))
            {
                Py_RETURN_NONE;
            }
            const at::Tensor &t = THPVariable_Unpack(obj);
            if (!t.is_cuda() || t.requires_grad() || t.layout() != at::kStrided || t.dim() < 2 || t.dim() > 3 || t.numel() == 0)
            {
                Py_RETURN_NONE;
            }
            const int64_t c = t.dim() == 3 ? t.size(2) : 1;
            if (k > 0 && (c != channels || t.scalar_type() != type))
            {
                Py_RETURN_NONE;
            }
            channels = c;
            type     = t.scalar_type();
            const int64_t row = (t.is_contiguous() ? t.size(1) * c : t.stride(0)) * (int64_t)t.element_size();
            if (t.size(0) > INT32_MAX || t.size(1) > INT32_MAX || row > INT32_MAX || row < INT32_MIN)
            {
                PyErr_SetString(PyExc_OverflowError, "image sizes and row pitches are 32-bit numbers");
                return nullptr;
            }
            std::memset(&plane[k], 0, sizeof(plane[k]));
            plane[k].width     = (int32_t)t.size(1);
            plane[k].height    = (int32_t)t.size(0);
            plane[k].rowStride = (int32_t)row;
            plane[k].basePtr   = static_cast<decltype(plane[k].basePtr)>(t.data_ptr());
        }
    }
    catch (const std::exception &)
    {
        Py_RETURN_NONE; // (a tensor without memory of its own ...: as_image says what is wrong with it)
    }
    return Py_BuildValue("LO", (long long)channels, out.o);
}

// tensor_alloc(shape, dtype, layout, base_align, row_align): (status, handle) of a tensor with memory of its own.
PyObject *TensorAlloc(PyObject *, PyObject *args)
{
    PyObject          *shape;
    unsigned long long dtype;
    const char        *layout;
    int                base, row;
    if (!PyArg_ParseTuple(args, "OKsii", &shape, &dtype, &layout, &base, &row))
    {
        return nullptr;
    }
    Ref list(PySequence_Fast(shape, "shape: a sequence"));
    if (!list)
    {
        return nullptr;
    }
    const Py_ssize_t rank = PySequence_Fast_GET_SIZE(list.o), letters = (Py_ssize_t)std::strlen(layout);
    if (rank > NVCV_TENSOR_MAX_RANK || letters > NVCV_TENSOR_MAX_RANK)
    {
        PyErr_SetString(PyExc_ValueError, "too many dimensions");
        return nullptr;
    }
    int64_t extents[NVCV_TENSOR_MAX_RANK];
    for (Py_ssize_t k = 0; k < rank; ++k)
    {
        extents[k] = PyLong_AsLongLong(PySequence_Fast_GET_ITEM(list.o, k));
        if (extents[k] == -1 && PyErr_Occurred())
        {
            return nullptr;
        }
    }
    NVCVTensorLayout order = {};
    std::memcpy(order.data, layout, (size_t)letters);
    order.rank = (int32_t)letters;
    NVCVTensorRequirements needs;
    NVCVTensorHandle       handle = nullptr;
    NVCVStatus             status;
    Py_BEGIN_ALLOW_THREADS
    status = nvcvTensorCalcRequirements((int32_t)rank, extents, (NVCVDataType)dtype, order, base, row, &needs);
    if (status == NVCV_SUCCESS)
    {
        status = nvcvTensorConstruct(&needs, nullptr, &handle);
    }
    Py_END_ALLOW_THREADS
    return Py_BuildValue("iK", (int)status, (unsigned long long)reinterpret_cast<uintptr_t>(handle));
}

// torch_view(handle, float32, device, owner): a torch tensor over a library tensor's memory, which keeps `owner`; None where it
// has no elements, strides that are no multiples of them, or lies on another device than `device`.
PyObject *TorchView(PyObject *, PyObject *args)
{
    unsigned long long handle;
    int                isFloat, device;
    PyObject          *owner;
    if (!PyArg_ParseTuple(args, "KiiO", &handle, &isFloat, &device, &owner))
    {
        return nullptr;
    }
    NVCVTensorData data;
    if (nvcvTensorExportData(reinterpret_cast<NVCVTensorHandle>((uintptr_t)handle), &data) != NVCV_SUCCESS)
    {
        Py_RETURN_NONE; // (Python's way reports it)
    }
    const int64_t size = isFloat ? 4 : 1;
    int64_t       strides[NVCV_TENSOR_MAX_RANK];
    for (int32_t k = 0; k < data.rank; ++k)
    {
        if (data.shape[k] == 0 || data.buffer.strided.strides[k] % size != 0)
        {
            Py_RETURN_NONE;
        }
        strides[k] = data.buffer.strided.strides[k] / size;
    }
    try
    {
        // torch keeps the owner for as long as it keeps the deleter, which it drops where the tensor cannot be made, uncalled
        Py_INCREF(owner);
        std::shared_ptr<PyObject> kept(owner,
                                       [](PyObject *o)
                                       {
                                           if (Py_IsInitialized())
                                           {
                                               const PyGILState_STATE state = PyGILState_Ensure();
                                               Py_DECREF(o);
                                               PyGILState_Release(state);
                                           }
                                       });
        const auto options = at::TensorOptions().dtype(isFloat ? at::kFloat : at::kByte).device(at::kCUDA);
        at::Tensor t = at::from_blob(data.buffer.strided.basePtr, at::IntArrayRef(data.shape, data.rank), at::IntArrayRef(strides, data.rank),
                                     [kept = std::move(kept)](void *) {}, options);
        if (t.device().index() != device)
        {
            Py_RETURN_NONE;
        }
        return THPVariable_Wrap(std::move(t));
    }
    catch (const std::exception &e)
    {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

// batch_alloc(capacity): (status, handle) of an image batch.
PyObject *BatchAlloc(PyObject *, PyObject *capacity)
{
    int n;
    if (!Int(capacity, n))
    {
        PyErr_SetString(PyExc_TypeError, "capacity: a 32-bit number");
        return nullptr;
    }
    NVCVImageBatchVarShapeRequirements needs;
    NVCVImageBatchHandle               handle = nullptr;
    NVCVStatus                         status;
    Py_BEGIN_ALLOW_THREADS
    status = nvcvImageBatchVarShapeCalcRequirements(n, &needs);
    if (status == NVCV_SUCCESS)
    {
        status = nvcvImageBatchVarShapeConstruct(&needs, nullptr, &handle);
    }
    Py_END_ALLOW_THREADS
    return Py_BuildValue("iK", (int)status, (unsigned long long)reinterpret_cast<uintptr_t>(handle));
}

// push_planes(batch's handle, format, planes' array as planes() gives it): status.
PyObject *PushPlanes(PyObject *, PyObject *args)
{
    unsigned long long handle, format;
    const char        *planes;
    Py_ssize_t         bytes;
    if (!PyArg_ParseTuple(args, "KKy#", &handle, &format, &planes, &bytes))
    {
        return nullptr;
    }
    NVCVStatus status;
    Py_BEGIN_ALLOW_THREADS
    status = nvcvxImageBatchVarShapePushBuffers(reinterpret_cast<NVCVImageBatchHandle>((uintptr_t)handle), format,
                                                reinterpret_cast<const NVCVImagePlaneStrided *>(planes),
                                                (int32_t)(bytes / (Py_ssize_t)sizeof(NVCVImagePlaneStrided)));
    Py_END_ALLOW_THREADS
    return PyLong_FromLong((long)status);
}

// batch_state(batch's handle): (status, number of images, the format that all of them have, 0 without one).
PyObject *BatchState(PyObject *, PyObject *handle)
{
    auto *h = reinterpret_cast<NVCVImageBatchHandle>(PyLong_AsVoidPtr(handle));
    if (PyErr_Occurred())
    {
        return nullptr;
    }
    int32_t         n      = 0;
    NVCVImageFormat format = NVCV_IMAGE_FORMAT_NONE;
    NVCVStatus      status = nvcvImageBatchGetNumImages(h, &n);
    if (status == NVCV_SUCCESS)
    {
        status = nvcvImageBatchVarShapeGetUniqueFormat(h, &format);
    }
    return Py_BuildValue("iiK", (int)status, (int)n, (unsigned long long)format);
}

// tensor_release(handle), batch_release(handle): gives a reference back.
template<class Handle, NVCVStatus (*DecRef)(Handle, int *)>
PyObject *Release(PyObject *, PyObject *handle)
{
    auto *h = reinterpret_cast<Handle>(PyLong_AsVoidPtr(handle));
    if (PyErr_Occurred())
    {
        return nullptr;
    }
    Py_BEGIN_ALLOW_THREADS
    (void)DecRef(h, nullptr);
    Py_END_ALLOW_THREADS
    Py_RETURN_NONE;
}

// ---- operators' results that are handed out again: see pyapi._Outputs, which is this type by another name. Its tables are
// touched under the interpreter's lock alone, and no object is given up between a table and the numbers that go with it.
struct Outputs
{
    PyObject_HEAD
    PyObject *api;  // pyapi's dictionary
    PyObject *free; // (shape, element type, layout, device) -> list of the library's tensors
    long long bytes, count, mostBytes, mostTensors;
};

int OutputsInit(PyObject *self, PyObject *args, PyObject *)
{
    auto     *o = reinterpret_cast<Outputs *>(self);
    PyObject *api;
    if (!PyArg_ParseTuple(args, "O!", &PyDict_Type, &api))
    {
        return -1;
    }
    Py_INCREF(api);
    Py_XSETREF(o->api, api);
    Py_XSETREF(o->free, PyDict_New());
    o->bytes = o->count = 0;
    o->mostBytes        = 256 << 20;
    o->mostTensors      = 64;
    return o->free != nullptr ? 0 : -1;
}

// (pyapi's dictionary holds the object that holds it: a copy of the package that nobody has any more goes by the collector)
int OutputsTraverse(PyObject *self, visitproc visit, void *arg)
{
    auto *o = reinterpret_cast<Outputs *>(self);
    Py_VISIT(Py_TYPE(self));
    Py_VISIT(o->api);
    Py_VISIT(o->free);
    return 0;
}

int OutputsCollect(PyObject *self)
{
    auto *o  = reinterpret_cast<Outputs *>(self);
    o->bytes = o->count = 0;
    Py_CLEAR(o->free);
    Py_CLEAR(o->api);
    return 0;
}

void OutputsDealloc(PyObject *self)
{
    PyTypeObject *type = Py_TYPE(self);
    PyObject_GC_UnTrack(self);
    (void)OutputsCollect(self);
    type->tp_free(self);
    Py_DECREF(type);
}

// Whether it has its tables: not before __init__, nor once the collector has taken them (an error is set).
bool OutputsLive(const Outputs *o)
{
    if (o->api != nullptr && o->free != nullptr)
    {
        return true;
    }
    PyErr_SetString(PyExc_RuntimeError, "no tables of results");
    return false;
}

// The tables as they were, with empty ones in their place (a new reference).
PyObject *OutputsTakeAll(Outputs *o)
{
    PyObject *empty = PyDict_New();
    if (empty == nullptr)
    {
        return nullptr;
    }
    PyObject *all = o->free;
    o->free       = empty;
    o->bytes = o->count = 0;
    return all;
}

// clear(): gives everything held back to the allocator; False if there was nothing.
PyObject *OutputsClear(PyObject *self, PyObject *)
{
    auto *o = reinterpret_cast<Outputs *>(self);
    if (!OutputsLive(o))
    {
        return nullptr;
    }
    const bool held = o->count != 0;
    Ref        all(OutputsTakeAll(o));
    return all ? PyBool_FromLong(held) : nullptr;
}

// get(shape, dtype, layout): a tensor for a result.
PyObject *OutputsGet(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    auto *o = reinterpret_cast<Outputs *>(self);
    if (n != 3)
    {
        PyErr_SetString(PyExc_TypeError, "get(shape, dtype, layout)");
        return nullptr;
    }
    if (!OutputsLive(o))
    {
        return nullptr;
    }
    Ref       shape(PySequence_Tuple(a[0])); // (a tuple itself)
    PyObject *np = Name(o->api, s_np), *torch = Name(o->api, s_torch);
    Ref       dtypes(shape && np != nullptr ? PyObject_GetAttr(np, s_dtype) : nullptr);
    if (!dtypes || !PyType_Check(dtypes.o))
    {
        return nullptr;
    }
    Ref dtype(nullptr);
    if (PyObject_TypeCheck(a[1], reinterpret_cast<PyTypeObject *>(dtypes.o)))
    {
        Py_INCREF(a[1]);
        dtype.o = a[1];
    }
    else
    {
        dtype.o = PyObject_CallOneArg(dtypes.o, a[1]);
    }
    Ref c(dtype && torch != nullptr ? PyObject_GetAttr(torch, s_C) : nullptr);
    Ref device(c ? PyObject_CallMethodNoArgs(c.o, s_getDevice) : nullptr);
    Ref key(device ? PyTuple_Pack(4, shape.o, dtype.o, a[2], device.o) : nullptr);
    if (!key)
    {
        return nullptr;
    }
    Ref       raw(nullptr);
    PyObject *kept = PyDict_GetItemWithError(o->free, key.o);
    if (kept == nullptr && PyErr_Occurred())
    {
        return nullptr;
    }
    const bool again = kept != nullptr && PyList_GET_SIZE(kept) > 0;
    if (again)
    {
        const Py_ssize_t last = PyList_GET_SIZE(kept) - 1;
        raw.o                 = PyList_GET_ITEM(kept, last);
        Py_INCREF(raw.o);
        if (PyList_SetSlice(kept, last, last + 1, nullptr) < 0)
        {
            return nullptr;
        }
        --o->count;
        Ref size(PyObject_GetAttr(raw.o, s_nbytes));
        o->bytes -= size ? PyLong_AsLongLong(size.o) : 0;
        if (PyErr_Occurred())
        {
            return nullptr;
        }
    }
    else
    {
        PyObject *make = Name(o->api, s_made);
        raw.o = make != nullptr ? PyObject_CallFunctionObjArgs(make, shape.o, dtype.o, a[2], nullptr) : nullptr;
        if (!raw)
        {
            return nullptr;
        }
    }
    PyObject *type = Name(o->api, s_Tensor);
    if (type == nullptr || !PyType_Check(type))
    {
        PyErr_SetString(PyExc_TypeError, "Tensor is no type");
        return nullptr;
    }
    Ref none(PyTuple_New(0));
    Ref out(none ? reinterpret_cast<PyTypeObject *>(type)->tp_new(reinterpret_cast<PyTypeObject *>(type), none.o, nullptr) : nullptr);
    Ref attributes(out ? PyObject_GenericGetDict(out.o, nullptr) : nullptr);
    Ref meta(attributes ? PyTuple_Pack(3, shape.o, dtype.o, PyObject_IsTrue(a[2]) == 1 ? a[2] : Py_None) : nullptr);
    if (!meta || PyDict_SetItem(attributes.o, s_t, raw.o) < 0 || PyDict_SetItem(attributes.o, s_meta, meta.o) < 0)
    {
        return nullptr;
    }
    if (again) // another stream's first use of it waits for the default stream's last
    {
        Ref by(PyNumber_Negative(device.o)), wrote(by ? PyTuple_Pack(2, by.o, Py_None) : nullptr);
        if (!wrote || PyDict_SetItem(attributes.o, s_wrote, wrote.o) < 0)
        {
            return nullptr;
        }
    }
    if (PyDict_SetItem(attributes.o, s_key, key.o) < 0) // (the last: from here on it comes back)
    {
        return nullptr;
    }
    Py_INCREF(out.o);
    return out.o;
}

// put(tensor): keeps the library's tensor of one whose owner is gone, if every use of it was on its device's default stream.
PyObject *OutputsPut(PyObject *self, PyObject *tensor)
{
    auto *o = reinterpret_cast<Outputs *>(self);
    Ref   attributes(AttributesOf(tensor));
    // (where the interpreter is ending, names and attributes may be gone: then it is not kept)
    PyObject *key = attributes ? PyDict_GetItem(attributes.o, s_key) : nullptr, *raw = attributes ? PyDict_GetItem(attributes.o, s_t) : nullptr;
    if (key == nullptr || raw == nullptr || !PyTuple_CheckExact(key) || PyTuple_GET_SIZE(key) != 4 || o->free == nullptr)
    {
        Py_RETURN_NONE;
    }
    const long by = -PyLong_AsLong(PyTuple_GET_ITEM(key, 3));
    if (PyErr_Occurred() || !WroteBy(attributes.o, by) || !ReadBy(attributes.o, by))
    {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    Ref held(raw);
    Py_INCREF(raw);
    Ref size(PyObject_GetAttr(raw, s_nbytes));
    if (!size)
    {
        PyErr_Clear();
        PyObject *sizeOf = Name(o->api, s_sizeOf);
        size.o           = sizeOf != nullptr && sizeOf != Py_None ? PyObject_CallOneArg(sizeOf, raw) : nullptr;
        if (!size || PyObject_SetAttr(raw, s_nbytes, size.o) < 0)
        {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
    }
    const long long bytes = PyLong_AsLongLong(size.o);
    if (PyErr_Occurred())
    {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    Ref drop(nullptr);
    if (o->count >= o->mostTensors || o->bytes + bytes > o->mostBytes)
    {
        drop.o = OutputsTakeAll(o);
    }
    if (bytes <= o->mostBytes / 4)
    {
        Ref       fresh(PyDict_GetItem(o->free, key) == nullptr ? PyList_New(0) : nullptr);
        PyObject *kept = fresh ? PyDict_SetDefault(o->free, key, fresh.o) : PyDict_GetItem(o->free, key);
        if (kept != nullptr && PyList_Append(kept, raw) == 0)
        {
            o->bytes += bytes;
            ++o->count;
        }
        PyErr_Clear();
    }
    Py_RETURN_NONE;
}

PyMethodDef kOutputsMethods[] = {
    {"get", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(OutputsGet)), METH_FASTCALL, nullptr},
    {"put", OutputsPut, METH_O, nullptr},
    {"clear", OutputsClear, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyMemberDef kOutputsMembers[] = {
    {"most_bytes", T_LONGLONG, offsetof(Outputs, mostBytes), 0, nullptr},
    {"most_tensors", T_LONGLONG, offsetof(Outputs, mostTensors), 0, nullptr},
    {"_bytes", T_LONGLONG, offsetof(Outputs, bytes), READONLY, nullptr},
    {"_count", T_LONGLONG, offsetof(Outputs, count), READONLY, nullptr},
    {nullptr, 0, 0, 0, nullptr},
};

PyType_Slot kOutputsSlots[] = {
    {Py_tp_init, reinterpret_cast<void *>(OutputsInit)}, {Py_tp_dealloc, reinterpret_cast<void *>(OutputsDealloc)},
    {Py_tp_traverse, reinterpret_cast<void *>(OutputsTraverse)}, {Py_tp_clear, reinterpret_cast<void *>(OutputsCollect)},
    {Py_tp_new, reinterpret_cast<void *>(PyType_GenericNew)}, {Py_tp_methods, kOutputsMethods},
    {Py_tp_members, kOutputsMembers}, {0, nullptr},
};

PyType_Spec kOutputsSpec = {"_cvcuda_native.Outputs", sizeof(Outputs), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC,
                                  kOutputsSlots};

PyMethodDef kBound[] = {
    {"submit", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(Submit)), METH_FASTCALL, nullptr},
    {"default_stream_key", DefaultKey, METH_NOARGS, nullptr},
};

// bind(pyapi's dictionary): (submit, default_stream_key) for it.
PyObject *Bind(PyObject *, PyObject *names)
{
    if (!PyDict_Check(names))
    {
        PyErr_SetString(PyExc_TypeError, "bind(dict)");
        return nullptr;
    }
    Ref submit(PyCFunction_New(&kBound[0], names)), key(PyCFunction_New(&kBound[1], names));
    return submit && key ? PyTuple_Pack(2, submit.o, key.o) : nullptr;
}

PyMethodDef kMethods[] = {
    {"bind", Bind, METH_O, nullptr},
    {"planes", Planes, METH_O, nullptr},
    {"tensor_alloc", TensorAlloc, METH_VARARGS, nullptr},
    {"torch_view", TorchView, METH_VARARGS, nullptr},
    {"tensor_release", Release<NVCVTensorHandle, nvcvTensorDecRef>, METH_O, nullptr},
    {"batch_alloc", BatchAlloc, METH_O, nullptr},
    {"push_planes", PushPlanes, METH_VARARGS, nullptr},
    {"batch_state", BatchState, METH_O, nullptr},
    {"batch_release", Release<NVCVImageBatchHandle, nvcvImageBatchDecRef>, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_cvcuda_native", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__cvcuda_native(void)
{
    const struct
    {
        PyObject  **name;
        const char *text;
    } names[] = {
        {&s_submit, "_submit"},   {&s_Tensor, "Tensor"},   {&s_ImageBatchVarShape, "ImageBatchVarShape"},
        {&s_lock, "_events_lock"}, {&s_followed, "_followed"}, {&s_tls, "_stream_tls"},
        {&s_stack, "stack"},      {&s_check, "check"},     {&s_t, "_t"},
        {&s_handle, "handle"},    {&s_wrote, "_wrote"},    {&s_read, "_read"},
        {&s_kind, "_native"},     {&s_acquire, "acquire"}, {&s_release, "release"},
        {&s_torch, "torch"},      {&s_C, "_C"},            {&s_getDevice, "_cuda_getDevice"},
        {&s_getStream, "_cuda_getCurrentRawStream"},
        {&s_value, "value"},      {&s_key, "_key"},        {&s_meta, "_meta"},
        {&s_nbytes, "_nbytes"},   {&s_np, "np"},           {&s_dtype, "dtype"},
        {&s_made, "_new_result"}, {&s_sizeOf, "_bytes_of"},
    };
    for (const auto &n : names)
    {
        if ((*n.name = PyUnicode_InternFromString(n.text)) == nullptr)
        {
            return nullptr;
        }
    }
    Ref module(PyModule_Create(&kModule)), outputs(PyType_FromSpec(&kOutputsSpec));
    if (!module || !outputs || PyModule_AddObjectRef(module.o, "Outputs", outputs.o) < 0)
    {
        return nullptr;
    }
    Py_INCREF(module.o);
    return module.o;
}

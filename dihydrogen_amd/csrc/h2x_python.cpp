// CPython entry to the C ABI for the calls that the layers make once per step.
//
// A call through ctypes wraps every pointer in an object and looks its argument
// types up; a layer call that launches one or two kernels of a few microseconds
// spent more time on that than the GPU on the work.  Here each entry point is
// one METH_FASTCALL function whose argument conversions are generated from its
// C signature: integers and floats as they are, and for a pointer None, an
// address, a torch tensor (what its data_ptr() returns, or raises; where that is torch's own method and no mode
// listens, it is not called, see data_ptr_of), any other object with a get_base_ptr() method (a local tensor: the
// method is asked, also where there is a data_ptr() too, or, where it is the one given to pointer_types(), what it does
// is done here, 0.1 us less than in Python), or one with a data_ptr() method alone. Every function returns what the C
// function returns (a status or a size). The GIL is released during the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <exception>
#include <tuple>
#include <type_traits>
#include <utility>

#include "h2x.h"

namespace
{

PyObject *s_data_ptr = nullptr, *s_get_base_ptr = nullptr, *s_data = nullptr, *s_base_bytes = nullptr; // interned names
PyTypeObject *s_torch_tensor = nullptr, *s_local_tensor = nullptr;
PyObject *s_base_ptr_method = nullptr, *s_base_bytes_property = nullptr; // of s_local_tensor
bool s_torch_is_known = false; // torch tensors lie in memory as this file was compiled for
unsigned int s_known_torch_version = 0; // tag of the class of torch tensors, when its data_ptr() was looked at
unsigned int s_known_version = 0;

bool as_address(PyObject* address, void** out)
{
    *out = PyLong_AsVoidPtr(address);
    return *out != nullptr || !PyErr_Occurred();
}

// What o's method returns, an address; false: an exception is set.
bool address_by(PyObject* method, PyObject* o, void** out)
{
    PyObject* const address = PyObject_CallMethodNoArgs(o, method);
    const bool ok = address && as_address(address, out);
    Py_XDECREF(address);
    return ok;
}

// What holds for all pointers of a call, until Python code runs.
struct Look
{
    bool is_new = true, plain = false;
};

// Whether the data_ptr() of torch tensors is the method that torch has in C++ (a class that nobody has changed since
// has its version tag still), and no mode for torch's functions is on, which would be told of the call.
bool calls_are_plain()
{
    PyTypeObject* const t = s_torch_tensor;
    const bool valid = PyType_HasFeature(t, Py_TPFLAGS_VALID_VERSION_TAG);
    if (!valid || t->tp_version_tag != s_known_torch_version)
    {
        PyObject* const method = _PyType_Lookup(t, s_data_ptr);
        if (t->tp_getattro != PyObject_GenericGetAttr || !method || Py_TYPE(method) != &PyMethodDescr_Type)
            return false;
        if (PyType_HasFeature(t, Py_TPFLAGS_VALID_VERSION_TAG)) // (the look-up may have given it one)
            s_known_torch_version = t->tp_version_tag;
    }
    return !at::impl::torch_function_mode_enabled();
}

// Whether what o.data_ptr() does is known: o is a torch tensor of that very class, and has no data_ptr() of its own.
bool has_plain_data_ptr(PyObject* o, Look* look)
{
    if (!s_torch_is_known || Py_TYPE(o) != s_torch_tensor)
        return false;
    if (look->is_new)
        *look = {false, calls_are_plain()};
    if (!look->plain)
        return false;
    PyObject** const own = _PyObject_GetDictPtr(o);
    return !own || !*own || !PyDict_GetItemWithError(*own, s_data_ptr);
}

// What o.data_ptr() returns. A torch tensor is asked as a C++ object where it can be: through its Python method, with
// an object made of the address and taken apart again, a pointer took 40 ns, of which a batch-norm backward pass has 14
// and a shuffle between 16 ranks 32.
// (One that has no memory to point to raises what the method raises.)
bool data_ptr_of(PyObject* o, void** out, Look* look)
{
    if (has_plain_data_ptr(o, look))
    {
        try
        {
            *out = THPVariable_Unpack(o).data_ptr();
            return true;
        }
        catch (const std::exception&)
        {
        }
    }
    look->is_new = true;
    return address_by(s_data_ptr, o, out);
}

// Whether the class of local tensors still reads `data` and `base_bytes` as it did and has the get_base_ptr() that is known.
// A class that nobody has changed since it was looked at has its version tag still.
bool class_is_known()
{
    PyTypeObject* const t = s_local_tensor;
    const bool valid = PyType_HasFeature(t, Py_TPFLAGS_VALID_VERSION_TAG);
    if (valid && t->tp_version_tag == s_known_version)
        return true;
    if (t->tp_getattro != PyObject_GenericGetAttr
        || PyDict_GetItemWithError(t->tp_dict, s_get_base_ptr) != s_base_ptr_method
        || PyDict_GetItemWithError(t->tp_dict, s_base_bytes) != s_base_bytes_property
        || PyDict_GetItemWithError(t->tp_dict, s_data))
        return false;
    if (valid)
        s_known_version = t->tp_version_tag;
    return true;
}

// What the get_base_ptr() of a local tensor of that very class returns: data.data_ptr() + base_bytes, read from the object's
// dictionary (three look-ups; by way of attributes 40 ns more).  0: not such a tensor, or not yet; -1: an exception is set.
int base_of(PyObject* o, void** out, Look* look)
{
    if (Py_TYPE(o) != s_local_tensor || !class_is_known())
        return 0;
    PyObject** const own = _PyObject_GetDictPtr(o);
    if (!own || !*own || PyDict_GetItemWithError(*own, s_get_base_ptr)) // (replaced on the object)
        return 0;
    PyObject *const data = PyDict_GetItemWithError(*own, s_data), *const bytes = PyDict_GetItemWithError(*own, s_base_bytes);
    if (!data || !bytes)
        return 0;
    const Py_ssize_t offset = PyLong_AsSsize_t(bytes);
    if (offset == -1 && PyErr_Occurred())
        return -1;
    Py_INCREF(data);
    const bool ok = data_ptr_of(data, out, look);
    Py_DECREF(data);
    if (!ok)
        return -1;
    *out = reinterpret_cast<void*>(reinterpret_cast<uintptr_t>(*out) + offset);
    return 1;
}

bool address_of(PyObject* o, void** out, Look* look)
{
    if (const int known = base_of(o, out, look))
        return known > 0;
    if (s_torch_tensor && PyObject_TypeCheck(o, s_torch_tensor))
        return data_ptr_of(o, out, look);
    look->is_new = true;
    PyObject* const method = PyObject_GetAttr(o, s_get_base_ptr);
    if (!method)
    {
        if (!PyErr_ExceptionMatches(PyExc_AttributeError))
            return false;
        PyErr_Clear();
        return address_by(s_data_ptr, o, out);
    }
    PyObject* const address = PyObject_CallNoArgs(method);
    Py_DECREF(method);
    const bool ok = address && as_address(address, out);
    Py_XDECREF(address);
    return ok;
}

template <typename P>
bool convert(PyObject* o, P* out, Look* look)
{
    if constexpr (std::is_pointer<P>::value)
    {
        if (o == Py_None)
        {
            *out = nullptr;
            return true;
        }
        if (PyLong_Check(o))
        {
            void* const p = PyLong_AsVoidPtr(o);
            *out = reinterpret_cast<P>(p);
            return p != nullptr || !PyErr_Occurred();
        }
        void* p;
        if (!address_of(o, &p, look))
            return false;
        *out = reinterpret_cast<P>(p);
        return true;
    }
    else if constexpr (std::is_floating_point<P>::value)
    {
        const double v = PyFloat_AsDouble(o);
        *out = static_cast<P>(v);
        return v != -1.0 || !PyErr_Occurred();
    }
    else
    {
        const long long v = PyLong_AsLongLong(o);
        *out = static_cast<P>(v);
        return v != -1 || !PyErr_Occurred();
    }
}

template <auto F>
struct Entry;

template <typename R, typename... P, R (*F)(P...)>
struct Entry<F>
{
    template <size_t... I>
    static PyObject* call(PyObject* const* args, std::index_sequence<I...>)
    {
        std::tuple<P...> v;
        Look look;
        if (!(convert(args[I], &std::get<I>(v), &look) && ...))
            return nullptr;
        R result;
        Py_BEGIN_ALLOW_THREADS
        result = F(std::get<I>(v)...);
        Py_END_ALLOW_THREADS
        if constexpr (std::is_signed<R>::value)
            return PyLong_FromLong(result);
        else
            return PyLong_FromSize_t(result);
    }

    static PyObject* fastcall(PyObject*, PyObject* const* args, Py_ssize_t nargs)
    {
        if (nargs != static_cast<Py_ssize_t>(sizeof...(P)))
            return PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd",
                                static_cast<Py_ssize_t>(sizeof...(P)), nargs);
        return call(args, std::index_sequence_for<P...>{});
    }
};

// Whether torch is the one whose headers this file was compiled with, and has a torch tensor's address where they say.
// (Another one's tensors are asked by their method.)
bool is_known_torch(PyObject* type, PyObject* version, PyObject* tensor)
{
    if (PyUnicode_CompareWithASCIIString(version, H2X_TORCH_VERSION) != 0 || reinterpret_cast<PyObject*>(Py_TYPE(tensor)) != type)
        return false;
    void* by_method;
    if (!address_by(s_data_ptr, tensor, &by_method))
    {
        PyErr_Clear();
        return false;
    }
    return THPVariable_Unpack(tensor).data_ptr() == by_method;
}

// pointer_types(torch.Tensor, the class of local tensors, its get_base_ptr, its base_bytes, torch.__version__, a torch
// tensor with memory): whether torch tensors are asked for their addresses as C++ objects.
PyObject* pointer_types(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    if (nargs != 6 || !PyType_Check(args[0]) || !PyType_Check(args[1]) || !PyUnicode_Check(args[4]))
        return PyErr_Format(PyExc_TypeError, "two types, a function, a property, a version and a tensor");
    const bool known = is_known_torch(args[0], args[4], args[5]);
    nargs = 4; // what is kept
    PyObject* const before[] = {reinterpret_cast<PyObject*>(s_torch_tensor), reinterpret_cast<PyObject*>(s_local_tensor),
                                s_base_ptr_method, s_base_bytes_property};
    for (Py_ssize_t i = 0; i < nargs; ++i)
        Py_INCREF(args[i]);
    s_torch_tensor = reinterpret_cast<PyTypeObject*>(args[0]);
    s_local_tensor = reinterpret_cast<PyTypeObject*>(args[1]);
    s_base_ptr_method = args[2];
    s_base_bytes_property = args[3];
    s_known_version = s_known_torch_version = 0;
    s_torch_is_known = known;
    for (PyObject* const o : before)
        Py_XDECREF(o);
    return PyBool_FromLong(known);
}

// same_buffers(addresses, *lists): whether the buffers of the lists of local tensors, one list after the other, lie at
// the addresses of the tuple (0: a tensor without a buffer), and are as many.
PyObject* same_buffers(PyObject*, PyObject* const* args, Py_ssize_t nargs)
{
    if (nargs < 1 || !PyTuple_Check(args[0]))
        return PyErr_Format(PyExc_TypeError, "a tuple of addresses");
    const Py_ssize_t n = PyTuple_GET_SIZE(args[0]);
    Py_ssize_t k = 0;
    Look look;
    for (Py_ssize_t a = 1; a < nargs; ++a)
    {
        if (!PyList_Check(args[a]))
            return PyErr_Format(PyExc_TypeError, "a list of tensors");
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(args[a]); ++i, ++k)
        {
            if (k == n)
                Py_RETURN_FALSE;
            PyObject* const tensor = PyList_GET_ITEM(args[a], i);
            Py_INCREF(tensor); // code that runs for `data` may drop it from the list
            PyObject* const data = PyObject_GetAttr(tensor, s_data);
            look.is_new |= Py_TYPE(tensor) != s_local_tensor || !class_is_known(); // of that class `data` runs no code
            Py_DECREF(tensor);
            void* p = nullptr;
            const bool ok = data && (data == Py_None || data_ptr_of(data, &p, &look));
            Py_XDECREF(data);
            if (!ok)
                return nullptr;
            if (PyLong_AsVoidPtr(PyTuple_GET_ITEM(args[0], k)) != p)
                return PyErr_Occurred() ? nullptr : PyBool_FromLong(0);
        }
    }
    if (PyErr_Occurred())
        return nullptr;
    return PyBool_FromLong(k == n);
}

#define H2X_ENTRY(NAME)                                                                            \
    {                                                                                              \
        #NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Entry<NAME>::fastcall)), \
            METH_FASTCALL, nullptr                                                                 \
    }

PyMethodDef s_methods[] = {H2X_ENTRY(h2x_bn_channel_sums_and_sqsums),
                           H2X_ENTRY(h2x_bn_channel_sums_and_sqsums_strided),
                           H2X_ENTRY(h2x_bn_sums_to_statistics),
                           H2X_ENTRY(h2x_bn_batch_normalization),
                           H2X_ENTRY(h2x_bn_batch_normalization_strided),
                           H2X_ENTRY(h2x_bn_batch_normalization_clearing),
                           H2X_ENTRY(h2x_bn_backprop1),
                           H2X_ENTRY(h2x_bn_backprop1_strided),
                           H2X_ENTRY(h2x_bn_backprop2),
                           H2X_ENTRY(h2x_bn_backprop2_strided),
                           H2X_ENTRY(h2x_bn_backprop2_clearing),
                           H2X_ENTRY(h2x_bn_forward_local),
                           H2X_ENTRY(h2x_bn_backward_local),
                           H2X_ENTRY(h2x_bn_team_state_needed),
                           H2X_ENTRY(h2x_bn_ordered_state_needed),
                           H2X_ENTRY(h2x_bn_team_state_needed_clearing),
                           H2X_ENTRY(h2x_bn_forward_once),
                           H2X_ENTRY(h2x_bn_forward_clearing),
                           H2X_ENTRY(h2x_bn_backward_clearing),
                           H2X_ENTRY(h2x_bn_backward_once),
                           H2X_ENTRY(h2x_tensor_transform),
                           H2X_ENTRY(h2x_tensor_reduce_sum),
                           H2X_ENTRY(h2x_softmax_channel_forward),
                           H2X_ENTRY(h2x_softmax_channel_backward),
                           H2X_ENTRY(h2x_softmax_instance_max),
                           H2X_ENTRY(h2x_softmax_instance_exp),
                           H2X_ENTRY(h2x_softmax_instance_normalize),
                           H2X_ENTRY(h2x_softmax_instance_forward_local),
                           H2X_ENTRY(h2x_softmax_instance_backward_local),
                           H2X_ENTRY(h2x_softmax_instance_workspace_bytes),
                           H2X_ENTRY(h2x_softmax_instance_state_needed),
                           H2X_ENTRY(h2x_softmax_instance_forward_once),
                           H2X_ENTRY(h2x_softmax_instance_backward_once),
                           H2X_ENTRY(h2x_softmax_instance_dot),
                           H2X_ENTRY(h2x_softmax_instance_gradient),
                           H2X_ENTRY(h2x_halo_pack_or_unpack_batched),
                           H2X_ENTRY(h2x_halo_clear),
                           H2X_ENTRY(h2x_halo_clear_batched),
                           H2X_ENTRY(h2x_halo_exchange_fused),
                           H2X_ENTRY(h2x_halo_grid_exchange),
                           H2X_ENTRY(h2x_halo_grid_fold),
                           H2X_ENTRY(h2x_halo_grid_clear),
                           H2X_ENTRY(h2x_shuffle_direct),
                           H2X_ENTRY(h2x_shuffle_pack_batched),
                           H2X_ENTRY(h2x_shuffle_unpack_batched),
                           {"pointer_types",
                            reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&pointer_types)), METH_FASTCALL, nullptr},
                           {"same_buffers",
                            reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&same_buffers)), METH_FASTCALL, nullptr},
                           {nullptr, nullptr, 0, nullptr}};

PyModuleDef s_module = {PyModuleDef_HEAD_INIT, "_h2xcall", "Native calls into libh2x.so.", -1,
                        s_methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__h2xcall(void)
{
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    s_data = PyUnicode_InternFromString("data");
    s_base_bytes = PyUnicode_InternFromString("base_bytes");
    s_get_base_ptr = PyUnicode_InternFromString("get_base_ptr");
    if (!s_data_ptr || !s_data || !s_base_bytes || !s_get_base_ptr)
        return nullptr;
    return PyModule_Create(&s_module);
}

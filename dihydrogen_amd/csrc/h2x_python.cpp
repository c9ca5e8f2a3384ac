// CPython entry to the C ABI for the calls that the layers make once per step.
//
// A call through ctypes wraps every pointer in an object and looks its argument
// types up; a layer call that launches one or two kernels of a few microseconds
// spent more time on that than the GPU on the work.  Here each entry point is
// one METH_FASTCALL function whose argument conversions are generated from its
// C signature: integers and floats as they are, and for a pointer None, an
// address, or any object with a data_ptr() method (a torch tensor).  Every
// function returns what the C function returns (a status or a size).  The GIL
// is released during the call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "h2x.h"

namespace
{

PyObject* s_data_ptr = nullptr; // interned "data_ptr"

template <typename P>
bool convert(PyObject* o, P* out)
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
        PyObject* const address = PyObject_CallMethodNoArgs(o, s_data_ptr);
        if (!address)
            return false;
        void* const p = PyLong_AsVoidPtr(address);
        Py_DECREF(address);
        *out = reinterpret_cast<P>(p);
        return p != nullptr || !PyErr_Occurred();
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
        if (!(convert(args[I], &std::get<I>(v)) && ...))
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
                           {nullptr, nullptr, 0, nullptr}};

PyModuleDef s_module = {PyModuleDef_HEAD_INIT, "_h2xcall", "Native calls into libh2x.so.", -1,
                        s_methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__h2xcall(void)
{
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    if (!s_data_ptr)
        return nullptr;
    return PyModule_Create(&s_module);
}

// Tensor-level calls onto the C ABI for Python, one C call each.
//
// mccl_amd/hip_ops.py checks its tensors in Python and calls the C ABI through ctypes: 5 us of host
// time around a launch of 2.5, more than a small fold takes on the GPU, and 150 us for the 240
// tensors of a ring step's fold list.  The functions here take the well-formed calls: they check the
// same conditions, launch and return the library's status, which hip_ops raises from.  Everything
// else (wrong device, layout, type or size) gives None, with nothing done, and hip_ops then goes
// through it by itself and reports.  A call that has reached the library is never made again: its
// status may be an error although the kernels were launched (one that an earlier call left on the
// thread, or the second of two launches), and folds and compress update their operands in place.
#include <torch/extension.h>
#include <torch/csrc/autograd/python_variable.h>

#include <c10/hip/HIPStream.h>

#include <vector>

#include "../../../include/mccl_hip.h"
#include "FastCalls.hpp"

namespace mccl {

namespace {

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

// The tensor behind `o` when it is a contiguous GPU tensor, else null.
const at::Tensor* gpu_tensor(PyObject* o) {
    if (!THPVariable_Check(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.is_cuda() && t.is_contiguous() ? &t : nullptr;
}
const at::Tensor* gpu_tensor(PyObject* o, at::ScalarType dtype, uint64_t min_numel) {
    const at::Tensor* t = gpu_tensor(o);
    return t && t->scalar_type() == dtype && static_cast<uint64_t>(t->numel()) >= min_numel ? t : nullptr;
}

// ... a byte tensor that holds `rows` rows of `stride` > 0 bytes (whatever their product).
const at::Tensor* gpu_rows(PyObject* o, uint64_t rows, int64_t stride) {
    const at::Tensor* t = gpu_tensor(o, at::kByte, 1);
    return t && static_cast<uint64_t>(t->numel() / stride) >= rows ? t : nullptr;
}

bool kernel_dtype(at::ScalarType t) {
    switch (t) {
        case at::kByte: case at::kInt: case at::kLong: case at::kHalf: case at::kFloat: case at::kBool: case at::kBFloat16:
            return true;
        default:
            return false;
    }
}

bool same(const at::Tensor* a, const at::Tensor* b) {
    return a && b && a->scalar_type() == b->scalar_type() && a->sizes() == b->sizes();
}

bool get_int(PyObject* o, int64_t* v) {
    if (!PyLong_CheckExact(o)) return false;
    *v = PyLong_AsLongLong(o);
    if (*v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}
bool get_float(PyObject* o, float* v) {
    if (!PyFloat_CheckExact(o)) return false;
    *v = static_cast<float>(PyFloat_AS_DOUBLE(o));
    return true;
}
// None or a float: *given says which.
bool get_scale(PyObject* o, int* given, float* v) {
    *given = o != Py_None;
    *v = 0.0f;
    return !*given || get_float(o, v);
}

// Calls the library without the interpreter lock, as ctypes does.
template <class F>
PyObject* launch(F&& f) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(rc);
}

// A list or tuple as an array of its items.
bool items(PyObject* seq, PyObject*** v, Py_ssize_t* n) {
    if (!PyList_CheckExact(seq) && !PyTuple_CheckExact(seq)) return false;
    *v = PySequence_Fast_ITEMS(seq);
    *n = PySequence_Fast_GET_SIZE(seq);
    return true;
}

// (dst, src, op)
PyObject* fold2(PyObject*, PyObject* const* a, Py_ssize_t n) {
    int64_t op;
    if (n != 3 || !get_int(a[2], &op)) Py_RETURN_NONE;
    const at::Tensor *d = gpu_tensor(a[0]), *s = gpu_tensor(a[1]);
    if (!same(d, s) || !kernel_dtype(d->scalar_type())) Py_RETURN_NONE;
    return launch([&] {
        return mccl_hip_fold2(d->data_ptr(), s->data_ptr(), d->numel(), static_cast<int>(d->scalar_type()), static_cast<int>(op), stream());
    });
}

// (dst, src, scale)
PyObject* fold2_scale(PyObject*, PyObject* const* a, Py_ssize_t n) {
    float f;
    if (n != 3 || !get_float(a[2], &f)) Py_RETURN_NONE;
    const at::Tensor *d = gpu_tensor(a[0]), *s = gpu_tensor(a[1]);
    if (!same(d, s) || !kernel_dtype(d->scalar_type())) Py_RETURN_NONE;
    return launch([&] {
        return mccl_hip_fold2_scale(d->data_ptr(), s->data_ptr(), d->numel(), static_cast<int>(d->scalar_type()), f, stream());
    });
}

// (dsts, srcs, op)
PyObject* fold2_batch(PyObject*, PyObject* const* a, Py_ssize_t n) {
    int64_t op;
    PyObject **dv, **sv;
    Py_ssize_t nd, ns;
    if (n != 3 || !get_int(a[2], &op) || !items(a[0], &dv, &nd) || !items(a[1], &sv, &ns) || nd != ns || nd == 0) Py_RETURN_NONE;
    std::vector<void*> dp(nd);
    std::vector<const void*> sp(nd);
    std::vector<uint64_t> cnt(nd);
    at::ScalarType dtype = at::kFloat;
    for (Py_ssize_t i = 0; i < nd; i++) {
        const at::Tensor *d = gpu_tensor(dv[i]), *s = gpu_tensor(sv[i]);
        if (i == 0 && d) dtype = d->scalar_type();
        if (!same(d, s) || d->scalar_type() != dtype) Py_RETURN_NONE;
        dp[i] = d->data_ptr();
        sp[i] = s->data_ptr();
        cnt[i] = static_cast<uint64_t>(d->numel());
    }
    if (!kernel_dtype(dtype)) Py_RETURN_NONE;
    return launch([&] {
        return mccl_hip_fold2_batch(dp.data(), sp.data(), cnt.data(), static_cast<uint32_t>(nd), static_cast<int>(dtype), static_cast<int>(op), stream());
    });
}

// (out, ins, op, schedule, bucket_elems, scale or None, stepwise)
PyObject* ring_fold(PyObject*, PyObject* const* a, Py_ssize_t n) {
    int64_t op, schedule, bucket, stepwise;
    int scaled;
    float f;
    PyObject** iv;
    Py_ssize_t ni;
    if (n != 7 || !items(a[1], &iv, &ni) || ni < 1 || ni > MCCL_HIP_MAX_WORLD || !get_int(a[2], &op) || !get_int(a[3], &schedule) ||
        !get_int(a[4], &bucket) || bucket < 1 || !get_scale(a[5], &scaled, &f) || !get_int(a[6], &stepwise))
        Py_RETURN_NONE;
    const at::Tensor* out = gpu_tensor(a[0]);
    if (!out || !kernel_dtype(out->scalar_type())) Py_RETURN_NONE;
    const void* in[MCCL_HIP_MAX_WORLD];
    for (Py_ssize_t i = 0; i < ni; i++) {
        const at::Tensor* t = gpu_tensor(iv[i]);
        if (!t || t->scalar_type() != out->scalar_type() || t->numel() != out->numel()) Py_RETURN_NONE;
        in[i] = t->data_ptr();
    }
    return launch([&] {
        return mccl_hip_ring_fold(out->data_ptr(), in, static_cast<int>(ni), out->numel(), bucket, static_cast<int>(schedule),
                                  static_cast<int>(out->scalar_type()), static_cast<int>(op), scaled, f, static_cast<int>(stepwise), stream());
    });
}

// (grad, residual, ratio, bucket_elems, wire, workspace, wire_stride, status or None)
PyObject* topk_compress(PyObject*, PyObject* const* a, Py_ssize_t n) {
    int64_t bucket, stride;
    if (n != 8 || !PyFloat_CheckExact(a[2]) || !get_int(a[3], &bucket) || !get_int(a[6], &stride) || bucket < 1 || stride < 4) Py_RETURN_NONE;
    const double ratio = PyFloat_AS_DOUBLE(a[2]);
    const at::Tensor* g = gpu_tensor(a[0], at::kFloat, 1);
    if (!g) Py_RETURN_NONE;
    const uint64_t count = static_cast<uint64_t>(g->numel());
    const uint64_t be = std::min<uint64_t>(bucket, count), nb = (count + be - 1) / be;
    const at::Tensor* r = gpu_tensor(a[1], at::kFloat, count);
    const at::Tensor* w = gpu_rows(a[4], nb, stride);
    const at::Tensor* ws = gpu_tensor(a[5], at::kByte, 1);
    const at::Tensor* st = a[7] == Py_None ? nullptr : gpu_tensor(a[7], at::kInt, 1);
    if (!r || static_cast<uint64_t>(r->numel()) != count || !w || !ws || (a[7] != Py_None && !st)) Py_RETURN_NONE;
    return launch([&] {
        return mccl_hip_topk_compress(g->data_ptr<float>(), r->data_ptr<float>(), count, be, ratio, w->data_ptr(), stride,
                                      ws->data_ptr(), ws->numel(), st ? st->data_ptr<int>() : nullptr, stream());
    });
}

// (acc, wires, wire_stride, bucket_elems, scale or None, status or None, workspace)
PyObject* sparse_accumulate(PyObject*, PyObject* const* a, Py_ssize_t n) {
    int64_t stride, bucket;
    int scaled;
    float f;
    PyObject** wv;
    Py_ssize_t nw;
    if (n != 7 || !items(a[1], &wv, &nw) || nw < 1 || nw > MCCL_HIP_MAX_WORLD || !get_int(a[2], &stride) || stride < 4 ||
        !get_int(a[3], &bucket) || bucket < 1 || !get_scale(a[4], &scaled, &f))
        Py_RETURN_NONE;
    const at::Tensor* acc = gpu_tensor(a[0], at::kFloat, 1);
    const at::Tensor* st = a[5] == Py_None ? nullptr : gpu_tensor(a[5], at::kInt, 1);
    const at::Tensor* ws = gpu_tensor(a[6], at::kByte, 1);
    if (!acc || !ws || (a[5] != Py_None && !st)) Py_RETURN_NONE;
    const uint64_t count = static_cast<uint64_t>(acc->numel());
    const uint64_t be = std::min<uint64_t>(bucket, count), nb = (count + be - 1) / be;
    const void* wires[MCCL_HIP_MAX_WORLD];
    for (Py_ssize_t i = 0; i < nw; i++) {
        const at::Tensor* w = gpu_rows(wv[i], nb, stride);
        if (!w) Py_RETURN_NONE;
        wires[i] = w->data_ptr();
    }
    return launch([&] {
        return mccl_hip_sparse_accumulate(acc->data_ptr<float>(), count, bucket, wires, static_cast<int>(nw), stride, scaled, f,
                                          st ? st->data_ptr<int>() : nullptr, ws->data_ptr(), ws->numel(), stream());
    });
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    return F(self, args, n);
    END_HANDLE_TH_ERRORS
}

#define MCCL_FAST(NAME) \
    { "_fast_" #NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&guarded<NAME>)), METH_FASTCALL, nullptr }

PyMethodDef kMethods[] = {
    MCCL_FAST(fold2), MCCL_FAST(fold2_scale), MCCL_FAST(fold2_batch), MCCL_FAST(ring_fold),
    MCCL_FAST(topk_compress), MCCL_FAST(sparse_accumulate), {nullptr, nullptr, 0, nullptr},
};

}  // namespace

void add_fast_calls(PyObject* module) {
    if (PyModule_AddFunctions(module, kMethods) != 0) throw py::error_already_set();
}

}  // namespace mccl

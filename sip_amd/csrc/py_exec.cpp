// CPython module _asdfft_py: one call from Plan.execute / Istft.execute to the C ABI.
//
// Through ctypes an exec took two or three tensor descriptors (argument arrays, create, destroy), the
// stream and the entry point itself, about 10.9 us of host time a call, which bounded every transform
// whose kernels take less.  The same calls from here are below 1 us besides the launch.  Anything but
// plain HIP tensors of exact type torch.Tensor returns NotImplemented, and the caller goes the ctypes way.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>

#include <c10/hip/HIPStream.h>

#include "acl_meta.h"
#include "fft_api.h"

namespace {

using namespace AsdSip;

// Dense descriptor of a tensor's shape and address, as N.AclTensor makes it: float32 or, for every
// other type, complex64.
class View {
public:
    explicit View(const at::Tensor& t)
    {
        const auto sizes = t.sizes();
        const size_t n = sizes.size();
        if (n > kMaxRank) return;
        int64_t strides[kMaxRank];
        int64_t step = 1;
        for (size_t i = n; i-- > 0;) {
            strides[i] = step;
            step *= sizes[i];
        }
        ptr_ = aclCreateTensor(sizes.data(), n, t.scalar_type() == at::kFloat ? ACL_FLOAT : ACL_COMPLEX64, strides, 0,
                               ACL_FORMAT_ND, sizes.data(), n, t.data_ptr());
    }
    ~View()
    {
        if (ptr_ != nullptr) aclDestroyTensor(ptr_);
    }
    View(const View&) = delete;
    View& operator=(const View&) = delete;
    aclTensor* get() const { return ptr_; }

private:
    static constexpr size_t kMaxRank = 16;  // aclCreateTensor's own limit
    aclTensor* ptr_ = nullptr;
};

bool plain(PyObject* o) { return THPVariable_CheckExact(o) && THPVariable_Unpack(o).is_cuda(); }

// torch's default stream is the null stream, refused by asdFftSetStream; hipStreamLegacy is its name.
hipStream_t stream_of(const at::Tensor& t)
{
    const hipStream_t s = c10::hip::getCurrentHIPStream(t.device().index()).stream();
    return s != nullptr ? s : hipStreamLegacy;
}

PyObject* not_here()
{
    Py_INCREF(Py_NotImplemented);
    return Py_NotImplemented;
}

// None, or (entry point, status) of the first call that failed.
template <typename Exec>
PyObject* run(PyObject* handle, PyObject* workspace, const at::Tensor& x, const char* name, Exec exec)
{
    const asdFftHandle h = PyLong_AsVoidPtr(handle);
    if (h == nullptr && PyErr_Occurred()) return nullptr;
    void* ws = workspace == Py_None ? nullptr : THPVariable_Unpack(workspace).data_ptr();
    const hipStream_t stream = stream_of(x);
    const char* fn = "asdFftSetWorkspace";
    AspbStatus st = ACL_SUCCESS;
    Py_BEGIN_ALLOW_THREADS
    if (ws != nullptr) st = asdFftSetWorkspace(h, ws);
    if (st == ACL_SUCCESS) {
        fn = "asdFftSetStream";
        st = asdFftSetStream(h, stream);
    }
    if (st == ACL_SUCCESS) {
        fn = name;
        st = exec(h);
    }
    Py_END_ALLOW_THREADS
    if (st == ACL_SUCCESS) Py_RETURN_NONE;
    return Py_BuildValue("(si)", fn, (int)st);
}

// execute(handle, kind, workspace or None, input, output)
PyObject* execute(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (n != 5) {
        PyErr_SetString(PyExc_TypeError, "execute takes 5 arguments");
        return nullptr;
    }
    if (!plain(args[3]) || !plain(args[4]) || !(args[2] == Py_None || plain(args[2]))) return not_here();
    const at::Tensor &x = THPVariable_Unpack(args[3]), &y = THPVariable_Unpack(args[4]);
    View vx(x), vy(y);
    if (vx.get() == nullptr || vy.get() == nullptr) return not_here();
    const long kind = PyLong_AsLong(args[1]);
    if (kind == -1 && PyErr_Occurred()) return nullptr;
    switch (kind) {
        case ASCEND_FFT_C2C:
            return run(args[0], args[2], x, "asdFftExecC2C",
                       [&](asdFftHandle h) { return asdFftExecC2C(h, vx.get(), vy.get()); });
        case ASCEND_FFT_R2C:
            return run(args[0], args[2], x, "asdFftExecR2C",
                       [&](asdFftHandle h) { return asdFftExecR2C(h, vx.get(), vy.get()); });
        case ASCEND_FFT_C2R:
            return run(args[0], args[2], x, "asdFftExecC2R",
                       [&](asdFftHandle h) { return asdFftExecC2R(h, vx.get(), vy.get()); });
        default: return not_here();
    }
    END_HANDLE_TH_ERRORS
}

// execute_istft(handle, workspace or None, spectrum, window, output)
PyObject* execute_istft(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    if (n != 5) {
        PyErr_SetString(PyExc_TypeError, "execute_istft takes 5 arguments");
        return nullptr;
    }
    for (int i = 2; i < 5; i++) {
        if (!plain(args[i])) return not_here();
    }
    if (!(args[1] == Py_None || plain(args[1]))) return not_here();
    const at::Tensor &x = THPVariable_Unpack(args[2]), &w = THPVariable_Unpack(args[3]), &y = THPVariable_Unpack(args[4]);
    View vx(x), vw(w), vy(y);
    if (vx.get() == nullptr || vw.get() == nullptr || vy.get() == nullptr) return not_here();
    return run(args[0], args[1], x, "asdFftExecIstft",
               [&](asdFftHandle h) { return asdFftExecIstft(h, vx.get(), vw.get(), vy.get()); });
    END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"execute", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&execute)), METH_FASTCALL, nullptr},
    {"execute_istft", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&execute_istft)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_asdfft_py", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__asdfft_py() { return PyModule_Create(&kModule); }

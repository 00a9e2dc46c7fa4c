// The Python wrappers' plain calls in native code: checks, output allocation,
// kargs and launch of one GEMM or activation quantizer.
//
// A decode GEMM or a small quantizer runs 2-10 us on the GPU, and its Python
// wrapper took 14.5 us of host time: two 1.7 us allocations, 1.8 us for the
// stream object, 1.3 us for the device guard, 4-4.6 us in the launch itself,
// the rest checks, ctypes conversions and record_stream calls.  Here the same
// steps take 5.0-5.5 us, most of it the launch: one token through a 7168 ->
// 2112 block-scale layer (quantizer and GEMM) 26 -> 12.1 us per pass.
//
// Every function returns None for a call that is not plain -- another
// tensor type than torch.Tensor, a shape, stride, type or device the entry
// does not take, a tensor off the current device, a split-K workspace that
// is not there yet, a launch that fails -- and the Python wrapper then goes
// through its own checks, which raise, allocate or launch as they always
// did.  Nothing is kept from one call to the next.
#include <climits>
#include <cstring>

#include <Python.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/VirtualGuardImpl.h>

#include "qgemm.h"

namespace {

// libqgemm.so's functions, as Python's loaded library has them
struct Lib {
    decltype(&qgemm_quant_fp8_blockscale_act) quant_bs;
    decltype(&qgemm_quant_fp8_e8m0_act) quant_e8m0;
    decltype(&qgemm_quant_mxfp8) quant_mx8;
    decltype(&qgemm_quant_mxfp4) quant_mx4;
    decltype(&qgemm_e8m0_shuffle_bytes) shuffle_bytes;
    decltype(&gemm_a8w8_blockscale_bpreshuffle) bs;
    decltype(&gemm_a8w8_blockscale_bpreshuffle_workspace_bytes) bs_ws;
    decltype(&gemm_a8w8_blockscale_ldsbypass) bypass;
    decltype(&gemm_a8w8_blockscale_ldsbypass_workspace_bytes) bypass_ws;
    decltype(&qgemm_ldsbypass_b_bytes) bypass_bytes;
    decltype(&gemm_a8w8_mxfp8) mx8;
    decltype(&gemm_a8w8_mxfp8_workspace_bytes) mx8_ws;
    decltype(&gemm_a4w4_mxfp4) mx4;
    decltype(&gemm_a4w4_mxfp4_workspace_bytes) mx4_ws;
    decltype(&gemm_a4w4_mxfp4_bpreshuffle_kid) a4w4;
    decltype(&gemm_a4w4_mxfp4_bpreshuffle_kid_workspace_bytes) a4w4_ws;
    decltype(&launch_blockscale_bpreshuffle) e8m0;
};
Lib lib;
bool bound = false;

// A call the Python wrapper has to make.
struct NotPlain {};
void need(bool ok) {
    if (!ok) throw NotPlain{};
}

const at::Tensor& tensor(PyObject* o) {
    need(THPVariable_CheckExact(o));
    const at::Tensor& t = THPVariable_Unpack(o);
    // strided memory of its own on the GPU: no functorch, fake or nested tensor
    need(t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() &&
         !t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                                   c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                                   c10::DispatchKey::Conjugate, c10::DispatchKey::Negative})));
    return t;
}

int dim(const at::Tensor& t, int i) {
    const int64_t n = t.size(i);
    need(n > 0 && n <= INT_MAX);
    return (int)n;
}

bool shape(const at::Tensor& t, int64_t r, int64_t c) { return t.dim() == 2 && t.size(0) == r && t.size(1) == c; }
bool bytes1(const at::Tensor& t) { return t.element_size() == 1; }
int64_t up(int64_t a, int64_t b) { return (a + b - 1) / b; }
// a batch stride or byte count as the kargs hold it
int i32(int64_t v) {
    need(v >= 0 && v <= INT_MAX);
    return (int)v;
}

// The current stream of the tensors' device, which has to be current.
struct Launch {
    c10::impl::VirtualGuardImpl guard{c10::DeviceType::CUDA};
    c10::Device device;
    c10::Stream stream;
    hipStream_t raw;
    explicit Launch(const at::Tensor& t)
        : device(t.device()), stream(guard.getStream(t.device())),
          raw(c10::hip::HIPStreamMasqueradingAsCUDA(stream).stream()) {
        need(guard.getDevice() == device);
    }
    // the caching allocator keeps the memory until this stream is past the call
    void record(const at::Tensor& t) const { guard.recordDataPtrOnStream(t.storage().data_ptr(), stream); }
    at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type) const {
        return at::empty(sizes, at::TensorOptions().dtype(type).device(device));
    }
};

struct Unlocked {    // without the GIL
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// The cached split-K workspace of this device and stream, of at least `want`
// bytes; the Python wrapper makes one that is missing or too small.
at::Tensor workspace(PyObject* dict, const Launch& l, size_t want) {
    need(PyDict_Check(dict));
    PyObject* key = Py_BuildValue("(in)", (int)l.device.index(), (Py_ssize_t)(intptr_t)l.raw);
    need(key != nullptr);
    PyObject* o = PyDict_GetItem(dict, key);
    Py_DECREF(key);
    need(o != nullptr);
    const at::Tensor t = tensor(o);
    need((size_t)t.nbytes() >= want);
    return t;
}

template <class Query, class Run>
void launch(const Launch& l, PyObject* ws_dict, Query query, Run run) {
    size_t want = 0;
    {
        Unlocked u;
        want = query();
    }
    at::Tensor ws;
    if (want) ws = workspace(ws_dict, l, want);
    hipError_t st;
    {
        Unlocked u;
        st = want ? run(ws.data_ptr(), (size_t)ws.nbytes()) : run((void*)nullptr, (size_t)0);
    }
    need(st == hipSuccess);
}

PyObject* none() { Py_RETURN_NONE; }

template <class F>
PyObject* guarded(F f) {
    try {
        need(bound);
        return f();
    } catch (...) {
        PyErr_Clear();
        return none();
    }
}

// gemm(kind, A, B, A_scale, B_scale, dtype, n, workspaces): kind 0 K-panel
// block scales, 1 B'' block scales (n columns), 2 MXFP8, 3 MXFP4, 4 MXFP4 in
// aiter's formats, 5 E8M0 block scales
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject* {
        need(nargs == 8 && PyLong_Check(args[0]) && THPDtype_Check(args[5]) && PyLong_Check(args[6]));
        const long kind = PyLong_AsLong(args[0]), n_arg = PyLong_AsLong(args[6]);
        const at::ScalarType out_type = reinterpret_cast<THPDtype*>(args[5])->scalar_type;
        need(out_type == at::kBFloat16 || out_type == at::kFloat);
        const int out = out_type == at::kBFloat16 ? QGEMM_OUT_BF16 : QGEMM_OUT_FP32;
        const at::Tensor &A = tensor(args[1]), &B = tensor(args[2]), &SA = tensor(args[3]), &SB = tensor(args[4]);
        need(A.dim() == 2 && bytes1(A) && bytes1(B) && A.is_contiguous() && B.is_contiguous());
        need(B.device() == A.device() && SA.device() == A.device() && SB.device() == A.device());
        const int m = dim(A, 0), kb = dim(A, 1);
        const Launch l(A);
        const auto done = [&](const at::Tensor& y) {
            for (const at::Tensor* t : {&A, &B, &SA, &SB, &y}) l.record(*t);
            return THPVariable_Wrap(y);
        };
        if (kind == 0 || kind == 1) {
            need(kb % 128 == 0);
            const int kg = kb / 128;
            int64_t n = n_arg;
            if (kind == 0) {
                need(B.dim() == 3 && B.size(0) == kg && B.size(2) == 128);
                n = B.size(1);
            }
            need(n > 0 && n <= INT_MAX && (kind == 0 || (size_t)B.nbytes() == lib.bypass_bytes((int)n, kb)));
            need(SA.scalar_type() == at::kFloat && SB.scalar_type() == at::kFloat && shape(SA, m, kg) &&
                 shape(SB, up(n, 128), kg) && SB.is_contiguous());
            int sfa = m;
            if (SA.is_contiguous()) sfa = m > 1 ? 1 : m;
            else need(SA.stride(0) == 1 && SA.stride(1) == m);
            const at::Tensor y = l.empty({m, n}, out_type);
            if (kind == 0) {
                const opus_gemm_kargs a{A.data_ptr(), B.data_ptr(), y.data_ptr(), m, (int)n, kb, 1, kb, 128, (int)n,
                                        i32((int64_t)m * kb), i32(n * kb), i32(m * n), SA.data_ptr(), SB.data_ptr(), sfa,
                                        kg, i32((int64_t)m * kg), i32(SB.size(0) * kg)};
                launch(l, args[7], [&] { return lib.bs_ws(&a); },
                       [&](void* w, size_t b) { return lib.bs(&a, out, w, b, l.raw); });
            } else {
                const opus_gemm_ldsbypass_kargs a{A.data_ptr(), nullptr, B.data_ptr(), y.data_ptr(), m, (int)n, kb, 1, kb,
                                                  128, (int)n, i32((int64_t)m * kb), i32(n * kb), i32(m * n),
                                                  SA.data_ptr(), SB.data_ptr(), sfa, kg, i32((int64_t)m * kg),
                                                  i32(SB.size(0) * kg), i32((int64_t)B.nbytes())};
                launch(l, args[7], [&] { return lib.bypass_ws(&a); },
                       [&](void* w, size_t b) { return lib.bypass(&a, out, w, b, l.raw); });
            }
            return done(y);
        }
        const bool fp4 = kind == 3 || kind == 4;
        const int64_t k = fp4 ? 2 * (int64_t)kb : kb;
        need(k <= INT_MAX && k % (fp4 ? 256 : 128) == 0 && B.dim() == 2 && B.size(1) == kb && bytes1(SA) && bytes1(SB));
        const int n = dim(B, 0);
        const int kg = (int)(k / 32);
        if (kind == 2 || kind == 3) {
            need(shape(SA, m, kg) && shape(SB, n, kg) && SA.is_contiguous() && SB.is_contiguous());
            const at::Tensor y = l.empty({m, n}, out_type);
            const opus_gemm_scale_kargs a{A.data_ptr(), B.data_ptr(), y.data_ptr(), m, n, (int)k, 1, kb, kb, n,
                                          i32((int64_t)m * kb), i32((int64_t)n * kb), i32((int64_t)m * n), SA.data_ptr(),
                                          SB.data_ptr(), kg, kg, i32((int64_t)m * kg), i32((int64_t)n * kg)};
            launch(l, args[7], [&] { return fp4 ? lib.mx4_ws(&a) : lib.mx8_ws(&a); },
                   [&](void* w, size_t b) { return (fp4 ? lib.mx4 : lib.mx8)(&a, out, w, b, l.raw); });
            return done(y);
        }
        if (kind == 4) {
            const int64_t blk = 32 * up(kg, 8) * 8;    // bytes of a 32-row block of shuffled scales
            need(n % 16 == 0 && SA.is_contiguous() && SB.is_contiguous() && SA.numel() >= up(m, 32) * blk &&
                 SB.numel() >= up(n, 32) * blk);
            const at::Tensor y = l.empty({m, n}, out_type);
            const opus_gemm_mxfp4_scale_kargs a{A.data_ptr(), B.data_ptr(), y.data_ptr(), m, n, (int)k, 1, kb, kb, n,
                                                i32((int64_t)m * kb), i32((int64_t)n * kb), i32((int64_t)m * n),
                                                SA.data_ptr(), SB.data_ptr(), i32(blk), i32(blk), i32(SA.numel()),
                                                i32(SB.numel()), 0};
            launch(l, args[7], [&] { return lib.a4w4_ws(&a, QGEMM_KID_AUTO); },
                   [&](void* w, size_t b) { return lib.a4w4(&a, out, QGEMM_KID_AUTO, w, b, l.raw); });
            return done(y);
        }
        need(kind == 5);
        const auto e8m0 = [](const at::Tensor& t) {
            return t.scalar_type() == at::kByte || t.scalar_type() == at::kFloat8_e8m0fnu;
        };
        const int kt = kb / 128;
        need(A.scalar_type() == at::kFloat8_e4m3fn && (B.scalar_type() == at::kFloat8_e4m3fn || B.scalar_type() == at::kByte) &&
             e8m0(SA) && e8m0(SB) && m % 256 == 0 && n % 256 == 0 && shape(SA, m, kt) && shape(SB, n / 128, kt) &&
             SB.is_contiguous() && (SA.is_contiguous() || (SA.stride(0) == 1 && SA.stride(1) == m)));
        i32((int64_t)m * n * (out == QGEMM_OUT_BF16 ? 2 : 4));
        const at::Tensor y = l.empty({m, n}, out_type);
        const opus_gemm_scale_kargs a{A.data_ptr(), B.data_ptr(), y.data_ptr(), m, n, kb, 1, kb, kb, n,
                                      i32((int64_t)m * kb), i32((int64_t)n * kb), i32((int64_t)m * n), SA.data_ptr(),
                                      SB.data_ptr(), m, kt, i32((int64_t)m * kt), i32((int64_t)(n / 128) * kt)};
        launch(l, args[7], [] { return (size_t)0; }, [&](void*, size_t) { return lib.e8m0(&a, out, 0, l.raw); });
        return done(y);
    });
}

// quant(kind, x): kind 0 fp32 scales per 1x128 row-major, 1 column-major, 2
// E8M0 per 1x128 column-major, 3 / 4 MXFP8 with row-major / shuffled scales,
// 5 / 6 MXFP4; returns (codes, scales)
PyObject* quant(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject* {
        need(nargs == 2 && PyLong_Check(args[0]));
        const long kind = PyLong_AsLong(args[0]);
        need(kind >= 0 && kind <= 6);
        const at::Tensor& x = tensor(args[1]);
        need(x.dim() == 2 && (x.scalar_type() == at::kFloat || x.scalar_type() == at::kBFloat16));
        const int in = x.scalar_type() == at::kFloat ? QGEMM_IN_FP32 : QGEMM_IN_BF16;
        const int rows = dim(x, 0), k = dim(x, 1);
        need(k % (kind < 3 ? 128 : 32) == 0 && x.stride(1) == 1 && x.stride(0) % 4 == 0);
        const int ld = i32(x.stride(0));
        const Launch l(x);
        const bool fp4 = kind >= 5, shuffle = kind == 4 || kind == 6;
        const int kg = k / (kind < 3 ? 128 : 32), qcols = fp4 ? k / 2 : k;
        const at::Tensor q = l.empty({rows, qcols}, fp4 ? at::kByte : at::kFloat8_e4m3fn);
        const at::ScalarType st = kind < 2 ? at::kFloat : at::kByte;
        at::Tensor s;
        if (shuffle) s = l.empty({(int64_t)lib.shuffle_bytes(rows, kg)}, st);
        else if (kind == 1 || kind == 2) s = l.empty({kg, rows}, st);
        else s = l.empty({rows, kg}, st);
        auto* qp = static_cast<uint8_t*>(q.data_ptr());
        hipError_t status;
        {
            Unlocked u;
            if (kind < 2)
                status = lib.quant_bs(x.data_ptr(), in, rows, k, ld, qp, k, static_cast<float*>(s.data_ptr()),
                                      kind ? 1 : kg, kind ? rows : 1, l.raw);
            else if (kind == 2)
                status = lib.quant_e8m0(x.data_ptr(), in, rows, k, ld, qp, k, static_cast<uint8_t*>(s.data_ptr()), 1, rows,
                                        l.raw);
            else
                status = (fp4 ? lib.quant_mx4 : lib.quant_mx8)(x.data_ptr(), in, rows, k, ld, qp, qcols,
                                                               static_cast<uint8_t*>(s.data_ptr()), kg, shuffle, l.raw);
        }
        need(status == hipSuccess);
        for (const at::Tensor& t : {x, q, s}) l.record(t);
        if (kind == 1 || kind == 2) s = s.t();
        PyObject *a = THPVariable_Wrap(q), *b = THPVariable_Wrap(s), *r = PyTuple_Pack(2, a, b);
        Py_XDECREF(a);
        Py_XDECREF(b);
        return r;
    });
}

// bind(addresses): the library's functions in Lib's order
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    constexpr Py_ssize_t count = sizeof(Lib) / sizeof(void*);
    if (nargs != count) {
        PyErr_SetString(PyExc_TypeError, "bind takes one address per library function");
        return nullptr;
    }
    void* p[count];
    for (Py_ssize_t i = 0; i < count; ++i) {
        p[i] = PyLong_AsVoidPtr(args[i]);
        if (!p[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address");
            return nullptr;
        }
    }
    static_assert(sizeof(p) == sizeof(Lib), "Lib holds function pointers only");
    std::memcpy(&lib, p, sizeof(lib));
    bound = true;
    return none();
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(bind)), METH_FASTCALL, nullptr},
    {"gemm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(gemm)), METH_FASTCALL, nullptr},
    {"quant", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(quant)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast() { return PyModule_Create(&module); }

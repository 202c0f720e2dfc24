// The launchers' plain case in native code: cuvit_amd/_native.so.
//
// A call of the Python binding checks its operands (device, type, contiguity,
// size), finds the stream and crosses ctypes. In Python that is 7 to 10 us,
// more than most of the library's kernels at the sizes of one image take; here
// it is well under one, so a caller's launches follow one another as fast as
// the kernels run.
//
// Every function does the whole of a launcher for the plain case: plain torch
// tensors and whole numbers that pass every check of the Python code. It then
// returns the C ABI's status. For anything else (an address instead of a
// tensor, a tensor subclass, a wrong type, an empty extent, too few elements)
// it touches nothing and returns -1, and the Python code, which names what is
// wrong, takes the call from the start. Nothing is kept between calls.
#include "cuvit/capi.h"

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <climits>
#include <cstddef>
#include <cstdint>
#include <initializer_list>

namespace {

constexpr long kNotPlain = -1;

/// The C ABI as the Python module loaded it (bind()), and its structs' types.
struct Library {
    decltype(&cuvit_layer_norm_f32) layer_norm_f32;
    decltype(&cuvit_layer_norm_bf16) layer_norm_bf16;
    decltype(&cuvit_softmax_f32) softmax_f32;
    decltype(&cuvit_softmax_bf16) softmax_bf16;
    decltype(&cuvit_extract_patches_f32) extract_patches_f32;
    decltype(&cuvit_extract_patches_bf16) extract_patches_bf16;
    decltype(&cuvit_gemm_f32) gemm_f32;
    decltype(&cuvit_gemm_bf16) gemm_bf16;
    decltype(&cuvit_attention_f32) attention_f32;
    decltype(&cuvit_attention_bf16) attention_bf16;
    decltype(&cuvit_preprocess_u8) preprocess_u8;
    decltype(&cuvit_vit_forward) vit_forward;
};
Library library{};
PyObject* gemm_problem_type = nullptr;
PyObject* preprocessing_type = nullptr;

/// A plain torch tensor's fields, or false.
const at::Tensor* plain_tensor(PyObject* object) {
    return THPVariable_CheckExact(object) ? &THPVariable_Unpack(object) : nullptr;
}

/// The address of a contiguous GPU tensor of @p type with at least @p elements
/// (a positive number), or null.
void* operand(PyObject* object, at::ScalarType type, std::int64_t elements) {
    const at::Tensor* const tensor = plain_tensor(object);
    if (tensor == nullptr || !tensor->is_cuda() || tensor->scalar_type() != type || !tensor->has_storage() ||
        !tensor->is_contiguous() || tensor->numel() < elements) {
        return nullptr;
    }
    return tensor->data_ptr();
}

/// A positive C int from a Python int.
bool positive(PyObject* object, int* out) {
    if (!PyLong_CheckExact(object)) {
        return false;
    }
    int overflow = 0;
    const long value = PyLong_AsLongAndOverflow(object, &overflow);
    if (overflow != 0 || value <= 0 || value > INT_MAX) {
        return false;
    }
    *out = static_cast<int>(value);
    return true;
}

/// The product of positive numbers, or false past 2^62.
bool product(std::int64_t* out, std::initializer_list<std::int64_t> factors) {
    std::int64_t total = 1;
    for (const std::int64_t f : factors) {
        if (f > (std::int64_t{1} << 62) / total) {
            return false;
        }
        total *= f;
    }
    *out = total;
    return true;
}

/// torch's current stream for None, else a stream object's handle.
bool stream_of(PyObject* object, cuvit_stream_t* out) {
    if (object == Py_None) {
        *out = reinterpret_cast<cuvit_stream_t>(c10::hip::getCurrentHIPStream().stream());
        return true;
    }
    PyObject* const handle = PyObject_GetAttrString(object, "cuda_stream");
    if (handle == nullptr) {
        PyErr_Clear();
        return false;
    }
    const bool whole = PyLong_CheckExact(handle);
    void* const address = whole ? PyLong_AsVoidPtr(handle) : nullptr;
    Py_DECREF(handle);
    if (PyErr_Occurred() != nullptr) {
        PyErr_Clear();
        return false;
    }
    *out = reinterpret_cast<cuvit_stream_t>(address);
    return whole;
}

/// fp32 or bf16 as the launcher picks it: the argument @p choice, or with None
/// the type of @p object.
bool storage(PyObject* choice, PyObject* object, at::ScalarType* out) {
    if (choice == Py_True || choice == Py_False) {
        *out = choice == Py_True ? at::kBFloat16 : at::kFloat;
        return true;
    }
    const at::Tensor* const tensor = choice == Py_None ? plain_tensor(object) : nullptr;
    if (tensor == nullptr) {
        return false;
    }
    *out = tensor->scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat;
    return true;
}

/// A view of a ctypes struct of exactly @p type.
class Struct {
  public:
    Struct(PyObject* object, PyObject* type, std::size_t bytes) {
        if (reinterpret_cast<PyObject*>(Py_TYPE(object)) != type) {
            return;
        }
        if (PyObject_GetBuffer(object, &view_, PyBUF_SIMPLE) != 0) {
            PyErr_Clear();
            return;
        }
        held_ = true;
        valid_ = static_cast<std::size_t>(view_.len) >= bytes;
    }
    ~Struct() {
        if (held_) {
            PyBuffer_Release(&view_);
        }
    }
    Struct(const Struct&) = delete;
    Struct& operator=(const Struct&) = delete;
    const void* get() const { return valid_ ? view_.buf : nullptr; }

  private:
    Py_buffer view_{};
    bool held_ = false;
    bool valid_ = false;
};

/// Runs a launch without the interpreter lock, as ctypes does.
template <typename Launch> long unlocked(Launch&& launch) {
    long status = 0;
    Py_BEGIN_ALLOW_THREADS
    status = launch();
    Py_END_ALLOW_THREADS
    return status;
}

/// A function's body, with every C++ exception turned into "not plain".
template <typename Body> PyObject* answer(Body&& body) {
    long status = kNotPlain;
    try {
        status = body();
    } catch (...) {
        status = kNotPlain;
    }
    return PyLong_FromLong(status);
}

// (x, gamma, beta, out, rows, columns, epsilon, stream, bf16)
PyObject* layer_norm(PyObject*, PyObject* const* a, Py_ssize_t count) {
    return answer([&]() -> long {
        at::ScalarType type;
        int rows, columns;
        std::int64_t elements;
        cuvit_stream_t stream;
        if (count != 9 || !storage(a[8], a[0], &type) || !positive(a[4], &rows) || !positive(a[5], &columns) ||
            !product(&elements, {rows, columns}) || !PyFloat_CheckExact(a[6])) {
            return kNotPlain;
        }
        const void* const x = operand(a[0], type, elements);
        const auto* const gamma = static_cast<const float*>(operand(a[1], at::kFloat, columns));
        const auto* const beta = static_cast<const float*>(operand(a[2], at::kFloat, columns));
        void* const out = operand(a[3], type, elements);
        const float epsilon = static_cast<float>(PyFloat_AS_DOUBLE(a[6]));
        if (x == nullptr || gamma == nullptr || beta == nullptr || out == nullptr || !stream_of(a[7], &stream)) {
            return kNotPlain;
        }
        return unlocked([&]() -> long {
            return type == at::kFloat
                       ? library.layer_norm_f32(static_cast<const float*>(x), gamma, beta, static_cast<float*>(out),
                                                rows, columns, epsilon, stream)
                       : library.layer_norm_bf16(static_cast<const std::uint16_t*>(x), gamma, beta,
                                                 static_cast<std::uint16_t*>(out), rows, columns, epsilon, stream);
        });
    });
}

// (x, out, rows, columns, stream, bf16)
PyObject* softmax(PyObject*, PyObject* const* a, Py_ssize_t count) {
    return answer([&]() -> long {
        at::ScalarType type;
        int rows, columns;
        std::int64_t elements;
        cuvit_stream_t stream;
        if (count != 6 || !storage(a[5], a[0], &type) || !positive(a[2], &rows) || !positive(a[3], &columns) ||
            !product(&elements, {rows, columns})) {
            return kNotPlain;
        }
        const void* const x = operand(a[0], type, elements);
        void* const out = operand(a[1], type, elements);
        if (x == nullptr || out == nullptr || !stream_of(a[4], &stream)) {
            return kNotPlain;
        }
        return unlocked([&]() -> long {
            return type == at::kFloat
                       ? library.softmax_f32(static_cast<const float*>(x), static_cast<float*>(out), rows, columns,
                                             stream)
                       : library.softmax_bf16(static_cast<const std::uint16_t*>(x), static_cast<std::uint16_t*>(out),
                                              rows, columns, stream);
        });
    });
}

// (images, patches, batch, channels, height, width, patch, stream, bf16)
PyObject* extract_patches(PyObject*, PyObject* const* a, Py_ssize_t count) {
    return answer([&]() -> long {
        at::ScalarType type;
        int batch, channels, height, width, patch;
        std::int64_t elements;
        cuvit_stream_t stream;
        if (count != 9 || !storage(a[8], a[0], &type) || !positive(a[2], &batch) || !positive(a[3], &channels) ||
            !positive(a[4], &height) || !positive(a[5], &width) || !positive(a[6], &patch) ||
            !product(&elements, {batch, channels, height, width})) {
            return kNotPlain;
        }
        const void* const images = operand(a[0], type, elements);
        void* const patches = operand(a[1], type, elements);
        if (images == nullptr || patches == nullptr || !stream_of(a[7], &stream)) {
            return kNotPlain;
        }
        return unlocked([&]() -> long {
            return type == at::kFloat
                       ? library.extract_patches_f32(static_cast<const float*>(images), static_cast<float*>(patches),
                                                     batch, channels, height, width, patch, stream)
                       : library.extract_patches_bf16(static_cast<const std::uint16_t*>(images),
                                                      static_cast<std::uint16_t*>(patches), batch, channels, height,
                                                      width, patch, stream);
        });
    });
}

/// The elements an operand of @p rows rows reaches over the batch, or false
/// where an entry starts before it (or the numbers are past any tensor's).
bool reach(const cuvit_gemm_batch& batch, int rows, int ld, int columns, std::int64_t stride,
           std::int64_t outer_stride, std::int64_t* out) {
    constexpr std::int64_t kLimit = std::int64_t{1} << 31;
    if (stride < 0 || outer_stride < 0 || stride > kLimit || outer_stride > kLimit) {
        return false;
    }
    std::int64_t high;
    if (batch.inner > 0 && batch.inner < batch.count) {
        high = static_cast<std::int64_t>(batch.count / batch.inner - 1) * outer_stride +
               static_cast<std::int64_t>(batch.inner - 1) * stride;
    } else {
        high = static_cast<std::int64_t>(batch.count - 1) * stride;
    }
    if (high > (std::int64_t{1} << 61)) {
        return false;
    }
    *out = high + static_cast<std::int64_t>(rows - 1) * ld + columns;
    return true;
}

// (a, b, bias, c, problem, stream, bf16)
PyObject* gemm(PyObject*, PyObject* const* args, Py_ssize_t count) {
    return answer([&]() -> long {
        at::ScalarType type;
        cuvit_stream_t stream;
        if (count != 7 || !storage(args[6], args[0], &type)) {
            return kNotPlain;
        }
        const Struct view(args[4], gemm_problem_type, sizeof(cuvit_gemm_problem));
        const auto* const p = static_cast<const cuvit_gemm_problem*>(view.get());
        if (p == nullptr || p->m <= 0 || p->n <= 0 || p->k <= 0 || p->batch.count <= 0 ||
            (p->layout != CUVIT_GEMM_NO_TRANSPOSE && p->layout != CUVIT_GEMM_TRANSPOSED)) {
            return kNotPlain;
        }
        const bool transposed = p->layout == CUVIT_GEMM_TRANSPOSED;
        const int b_rows = transposed ? p->n : p->k;
        const int b_columns = transposed ? p->k : p->n;
        const int lda = p->lda != 0 ? p->lda : p->k;
        const int ldb = p->ldb != 0 ? p->ldb : b_columns;
        const int ldc = p->ldc != 0 ? p->ldc : p->n;
        std::int64_t a_reach, b_reach, c_reach;
        if (lda < p->k || ldb < b_columns || ldc < p->n ||
            !reach(p->batch, p->m, lda, p->k, p->batch.stride_a, p->batch.outer_stride_a, &a_reach) ||
            !reach(p->batch, b_rows, ldb, b_columns, p->batch.stride_b, p->batch.outer_stride_b, &b_reach) ||
            !reach(p->batch, p->m, ldc, p->n, p->batch.stride_c, p->batch.outer_stride_c, &c_reach)) {
            return kNotPlain;
        }
        const void* const a = operand(args[0], type, a_reach);
        const void* const b = operand(args[1], type, b_reach);
        const bool with_bias = args[2] != Py_None;
        const auto* const bias =
            with_bias ? static_cast<const float*>(operand(args[2], at::kFloat, p->n)) : nullptr;
        void* const c = operand(args[3], type, c_reach);
        if (a == nullptr || b == nullptr || c == nullptr || (with_bias && bias == nullptr) ||
            !stream_of(args[5], &stream)) {
            return kNotPlain;
        }
        return unlocked([&]() -> long {
            return type == at::kFloat
                       ? library.gemm_f32(static_cast<const float*>(a), static_cast<const float*>(b), bias,
                                          static_cast<float*>(c), p, stream)
                       : library.gemm_bf16(static_cast<const std::uint16_t*>(a), static_cast<const std::uint16_t*>(b),
                                           bias, static_cast<std::uint16_t*>(c), p, stream);
        });
    });
}

// (qkv, context, images, heads, tokens, head_dim, stream)
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t count) {
    return answer([&]() -> long {
        at::ScalarType type;
        int images, heads, tokens, head_dim;
        std::int64_t elements;
        cuvit_stream_t stream;
        if (count != 7 || !storage(Py_None, a[0], &type) || !positive(a[2], &images) || !positive(a[3], &heads) ||
            !positive(a[4], &tokens) || !positive(a[5], &head_dim) ||
            !product(&elements, {3, images, tokens, heads, head_dim})) {
            return kNotPlain;
        }
        const void* const qkv = operand(a[0], type, elements);
        void* const context = operand(a[1], type, elements / 3);
        if (qkv == nullptr || context == nullptr || !stream_of(a[6], &stream)) {
            return kNotPlain;
        }
        return unlocked([&]() -> long {
            return type == at::kFloat
                       ? library.attention_f32(static_cast<const float*>(qkv), static_cast<float*>(context), images,
                                               heads, tokens, head_dim, stream)
                       : library.attention_bf16(static_cast<const std::uint16_t*>(qkv),
                                                static_cast<std::uint16_t*>(context), images, heads, tokens, head_dim,
                                                stream);
        });
    });
}

// (pixels, tensor, batch, width, height, settings, stream)
PyObject* preprocess(PyObject*, PyObject* const* a, Py_ssize_t count) {
    return answer([&]() -> long {
        int batch, width, height;
        std::int64_t in, out;
        cuvit_stream_t stream;
        if (count != 7 || !positive(a[2], &batch) || !positive(a[3], &width) || !positive(a[4], &height)) {
            return kNotPlain;
        }
        const Struct view(a[5], preprocessing_type, sizeof(cuvit_preprocessing));
        const auto* const settings = static_cast<const cuvit_preprocessing*>(view.get());
        if (settings == nullptr || settings->size <= 0 || !product(&in, {batch, height, width, 3}) ||
            !product(&out, {batch, 3, settings->size, settings->size})) {
            return kNotPlain;
        }
        const auto* const pixels = static_cast<const std::uint8_t*>(operand(a[0], at::kByte, in));
        auto* const tensor = static_cast<float*>(operand(a[1], at::kFloat, out));
        if (pixels == nullptr || tensor == nullptr || !stream_of(a[6], &stream)) {
            return kNotPlain;
        }
        return unlocked(
            [&]() -> long { return library.preprocess_u8(pixels, batch, width, height, settings, tensor, stream); });
    });
}

// (handle address, images, logits, batch, image elements, classes, stream)
PyObject* vit_forward(PyObject*, PyObject* const* a, Py_ssize_t count) {
    return answer([&]() -> long {
        int batch, image_elements, classes;
        std::int64_t in, out;
        cuvit_stream_t stream;
        if (count != 7 || !PyLong_CheckExact(a[0]) || !positive(a[3], &batch) || !positive(a[4], &image_elements) ||
            !positive(a[5], &classes) || !product(&in, {batch, image_elements}) || !product(&out, {batch, classes})) {
            return kNotPlain;
        }
        auto* const handle = static_cast<cuvit_vit*>(PyLong_AsVoidPtr(a[0]));
        const auto* const images = static_cast<const float*>(operand(a[1], at::kFloat, in));
        auto* const logits = static_cast<float*>(operand(a[2], at::kFloat, out));
        if (PyErr_Occurred() != nullptr) {
            PyErr_Clear();
            return kNotPlain;
        }
        if (handle == nullptr || images == nullptr || logits == nullptr || !stream_of(a[6], &stream)) {
            return kNotPlain;
        }
        return unlocked([&]() -> long { return library.vit_forward(handle, images, logits, batch, stream); });
    });
}

// (GemmProblem, Preprocessing, address of each of Library's functions in order)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t count) {
    constexpr Py_ssize_t kFunctions = sizeof(Library) / sizeof(void*);
    if (count != 2 + kFunctions) {
        PyErr_SetString(PyExc_TypeError, "bind takes the two struct types and every function's address");
        return nullptr;
    }
    void* addresses[kFunctions];
    for (Py_ssize_t i = 0; i < kFunctions; ++i) {
        addresses[i] = PyLong_AsVoidPtr(a[2 + i]);
        if (addresses[i] == nullptr) {
            if (PyErr_Occurred() == nullptr) {
                PyErr_SetString(PyExc_ValueError, "a function's address is null");
            }
            return nullptr;
        }
    }
    __builtin_memcpy(&library, addresses, sizeof(library));
    Py_INCREF(a[0]);
    Py_INCREF(a[1]);
    Py_XSETREF(gemm_problem_type, a[0]);
    Py_XSETREF(preprocessing_type, a[1]);
    Py_RETURN_NONE;
}

#define CUVIT_FAST(name) \
    {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {CUVIT_FAST(bind),           CUVIT_FAST(layer_norm), CUVIT_FAST(softmax),
                         CUVIT_FAST(extract_patches), CUVIT_FAST(gemm),       CUVIT_FAST(attention),
                         CUVIT_FAST(preprocess),     CUVIT_FAST(vit_forward), {nullptr, nullptr, 0, nullptr}};
#undef CUVIT_FAST

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "The launchers' plain case.", -1, methods,
                      nullptr,               nullptr,   nullptr,                      nullptr};

} // namespace

/// The module, with the PyTorch and Python that it was compiled for: the Python
/// side uses it with these only.
PyMODINIT_FUNC PyInit__native() {
    PyObject* const created = PyModule_Create(&module);
    if (created == nullptr) {
        return nullptr;
    }
    PyObject* const built_for = Py_BuildValue("(sii)", TORCH_VERSION, PY_MAJOR_VERSION, PY_MINOR_VERSION);
    if (built_for == nullptr || PyModule_AddObject(created, "built_for", built_for) != 0) {
        Py_XDECREF(built_for);
        Py_DECREF(created);
        return nullptr;
    }
    return created;
}

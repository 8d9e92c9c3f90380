// Host side of the hot calls in native code: argument checks, output and scratch allocation, stream lookup and the launches
// of libquest_hip.so, as a CPython module over torch's C++ tensors.
//
// Why: a layer at a handful of tokens is 5 to 7 us of GPU work, and its Python host path (asserts, ctypes conversions, device
// context, one allocation per output) took 36 us per call, so every small call ran at the speed of the interpreter.  From here a call of two
// launches takes 8.4 to 11.7 us to issue, module call included (30 calls in a row; boxes and processes differ so much), and one of a single launch
// (quest_linear_few_tokens) 5.1 to 7.2: a launch is about 3.5 us of it, an allocation 0.7.  That, and not the GPU, still bounds the smallest calls.
//
// Contract of every function: either the call is the plain case -- exact torch tensors on one GPU, contiguous, right types, sizes
// and alignment, accepted by the library -- and everything is launched, or None comes back with nothing launched and the
// caller's Python statement of the same call runs, which raises what there is to raise.  (Should a launch itself fail, `block`
// raises, for its stream has changed; the others come back with None, and the Python statement starts over and reports it.)
// Nothing is cached between calls.
#include <Python.h>

#include <ATen/Context.h>
#include <ATen/autocast_mode.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/scaled_dot_product_attention.h>
#include <ATen/ops/silu.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>

#include "../../include/quest_hip.h"

namespace {

constexpr float kHadamardEntry = 181.f / 2048.f;      // bf16(2^-3.5) == fp16(2^-3.5)

// ---- arguments ------------------------------------------------------------------------------------------------------
// Collects what the arguments of one call have in common and whether every one of them is as expected.
struct Args {
    bool ok = true;
    c10::Device dev{c10::DeviceType::CPU};
    at::Tensor none;                  // stands for an argument that is no tensor
    const at::Tensor *tensor(PyObject *o) {
        if (!THPVariable_CheckExact(o)) {
            ok = false;
            return &none;
        }
        const at::Tensor &t = THPVariable_Unpack(o);
        if (!t.is_cuda() || !t.is_contiguous() || t.numel() == 0) {
            ok = false;
        } else if (dev.is_cpu()) {
            dev = t.device();
        } else if (t.device() != dev) {
            ok = false;
        }
        return &t;
    }
    const at::Tensor *tensor(PyObject *o, at::ScalarType type, int64_t numel) {
        const at::Tensor *t = tensor(o);
        if (ok && (t->scalar_type() != type || t->numel() != numel)) ok = false;
        return t;
    }
    const at::Tensor *matrix(PyObject *o, at::ScalarType type, int64_t rows, int64_t cols) {
        const at::Tensor *t = tensor(o);
        if (ok && (t->scalar_type() != type || t->dim() != 2 || t->size(0) != rows || t->size(1) != cols)) ok = false;
        return t;
    }
};

bool is_half(at::ScalarType t) { return t == at::kBFloat16 || t == at::kHalf; }
int dtype_code(at::ScalarType t) { return t == at::kBFloat16 ? QUEST_DTYPE_BF16 : QUEST_DTYPE_FP16; }
bool fits_int(int64_t v) { return v > 0 && v <= 0x7fffffff; }
void *stream_of(c10::Device dev) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream(); }
at::Tensor make(at::IntArrayRef sizes, at::ScalarType type, c10::Device dev) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(dev));
}
PyObject *wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }
PyObject *declined() { Py_RETURN_NONE; }
PyObject *ref(PyObject *o) {
    Py_INCREF(o);
    return o;
}
// Allocations and launches run without the interpreter lock, as calls through ctypes do: a launch can wait for room in its queue.
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    Unlocked() = default;
    Unlocked(const Unlocked &) = delete;
    ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename F>
int on(c10::Device dev, F &&launch) {
    const Unlocked unlocked;
    const c10::DeviceGuard guard(dev);
    return launch(stream_of(dev));
}
int64_t up(int64_t bytes) { return (bytes + 255) & ~(int64_t)255; }
bool at(const at::Tensor *t, unsigned bytes) { return t == nullptr || (reinterpret_cast<uintptr_t>(t->data_ptr()) & (bytes - 1)) == 0; }

// Counts a write into a tensor of the caller's, as torch's own in-place calls do: `unchanged` below goes by that count, and the tensor may
// be a layer's buffer.
void wrote(const at::Tensor &t) {
    if (!t.is_inference()) t.unsafeGetTensorImpl()->bump_version();
}

// Whether `t` is the tensor that something was derived from and still holds what it held: its address and version then are given.
bool unchanged(PyObject *t, PyObject *source, PyObject *address, PyObject *version) {
    if (t != source || !THPVariable_CheckExact(t)) return false;
    const at::Tensor &v = THPVariable_Unpack(t);
    return !v.is_inference() && PyLong_Check(address) && PyLong_AsVoidPtr(address) == v.data_ptr() && PyLong_Check(version) &&
           PyLong_AsLongLong(version) == (long long)v._version();
}

// E2M3 tiles of the packed weight `packed`: a tensor of them, or (tiles, of which tensor, its address, its version) as Linear4bit keeps
// them.  None if there are none, or if the tensor has changed since.
PyObject *tiles_of(PyObject *kept, PyObject *packed) {
    if (!PyTuple_Check(kept)) return kept;
    if (PyTuple_GET_SIZE(kept) != 4 || !unchanged(packed, PyTuple_GET_ITEM(kept, 1), PyTuple_GET_ITEM(kept, 2), PyTuple_GET_ITEM(kept, 3))) return Py_None;
    return PyTuple_GET_ITEM(kept, 0);
}

// What the GEMMs ask of sizes (gemm_check in gemm.hip, e2m3_gemm_check in gemm_e2m3.hip), for calls that launch something before them.
bool gemm_takes(int64_t m, int64_t k, int64_t n, bool tiles) {
    if (tiles)
        return k % 128 == 0 && k <= 65536 && quest_e2m3_tiles_bytes((int)std::min<int64_t>(m + 256, 0x7fffffff), (int)k) < (1ull << 31) &&
               quest_e2m3_tiles_bytes((int)std::min<int64_t>(n + 256, 0x7fffffff), (int)k) < (1ull << 31);
    return k % 32 == 0 && k < 131072 && m * (k / 2) < (1ll << 31) && n * (k / 2) < (1ll << 31);
}

// One activation's codes in scratch memory: packed nibbles, row sums and scales, or E2M3 tiles and scales.
struct Codes {
    uint8_t *codes = nullptr;         // packed nibbles or tiles
    int32_t *row_sum = nullptr;
    void *scale = nullptr;
    bool tiles = false;
    static int64_t body(int64_t m, int64_t k, bool as_tiles) { return up(as_tiles ? (int64_t)quest_e2m3_tiles_bytes((int)m, (int)k) : m * (k / 2)); }
    static int64_t bytes(int64_t m, int64_t k, bool as_tiles) { return body(m, k, as_tiles) + (as_tiles ? 0 : up(4 * m)) + up(2 * m); }
    Codes(void *at, int64_t m, int64_t k, bool as_tiles) : codes((uint8_t *)at), tiles(as_tiles) {
        const int64_t behind = body(m, k, as_tiles);
        row_sum = as_tiles ? nullptr : (int32_t *)(codes + behind);
        scale = codes + behind + (as_tiles ? 0 : up(4 * m));
    }
};

// One projection's weights.
struct Linear {
    const at::Tensor *packed, *scale, *add, *tiles;
    int n, k;
    bool take(Args &args, PyObject *t, at::ScalarType type, bool want_tiles) {
        if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) != 4) return args.ok = false;
        packed = args.tensor(PyTuple_GET_ITEM(t, 0));
        if (!args.ok || packed->scalar_type() != at::kByte || packed->dim() != 2 || !fits_int(packed->size(0)) ||
            !fits_int(packed->size(1) * 2))
            return args.ok = false;
        n = (int)packed->size(0);
        k = (int)packed->size(1) * 2;
        scale = args.tensor(PyTuple_GET_ITEM(t, 1), type, n);
        add = args.tensor(PyTuple_GET_ITEM(t, 2), at::kInt, n);
        PyObject *const form = want_tiles ? tiles_of(PyTuple_GET_ITEM(t, 3), PyTuple_GET_ITEM(t, 0)) : Py_None;
        tiles = form != Py_None ? args.tensor(form, at::kByte, (int64_t)quest_e2m3_tiles_bytes(n, k)) : nullptr;
        return args.ok;
    }
};

// The activation kernel for a GEMM on w: codes of x, of its norm (x + branch first where there is one, in place), or of silu(gate) * up.  It
// reads ahead for the GEMM.
struct Producer {
    int kind = QUEST_PRODUCER_NONE;
    const void *branch = nullptr, *norm_weight = nullptr;
    double eps = 0.;
};
// How much of the weights: what memory gives while the kernel runs (1600M model at 2 x 500 tokens 2953 us without, 2822 to 2828 with 4 to 40 MB).
// Many tokens: nothing of weights that are more than that, for their GEMM is long and the memory busy (layers of 3065 to 11837 tokens x 10000 x 13000
// read 30 to 100 MB ahead and were 1.5 to 3.7 % slower).  A layer on its own gains from 64 to 512 tokens ((91, 1664, 20608) 14.0 -> 13.3 us); fewer
// are bound by the host, more by their products.
// Packed weights of up to 64 tokens: nothing, for that GEMM streams them at once with all its workgroups (1600M model at 1 x 8 tokens 1062 us with, 1032
// without, at 1 x 1 971 and 955, at 1 x 30 1201 and 1174).
size_t read_ahead_bytes(int64_t m, size_t weights) {
    const size_t most = 8000000 + 8000 * (size_t)std::min<int64_t>(m, 2048);
    return m > 2048 && weights > most ? 0 : std::min(weights, most);
}
int quantise_for(const Linear &w, const Codes &q, const void *x, const Producer &p, int m, int k, float had_scale, int dt, void *st) {
    quest_activation a = {};
    a.producer = p.kind, a.x = x, a.branch = p.branch, a.norm_weight = p.norm_weight, a.eps = (float)p.eps;
    a.scale = q.scale, a.x_int_packed = q.tiles ? nullptr : q.codes, a.x_int_row_sum = q.row_sum, a.tiles = q.tiles ? q.codes : nullptr;
    a.size_k = k, a.size_m = m, a.had_scale = had_scale, a.dtype = dt;
    // row blocks of 32 channels: so much of the start of each that the kernel is not kept waiting by it
    a.next_blocks = q.tiles ? (w.n + 31) / 32 : w.n / 32;
    a.next = q.tiles ? w.tiles->data_ptr() : w.packed->data_ptr();
    a.next_pitch = q.tiles ? quest_e2m3_tiles_bytes(32, (k + 127) / 128 * 128) : (size_t)k * 16;
    a.next_bytes = a.next_blocks > 0 && (q.tiles || m > 64) ? read_ahead_bytes(m, a.next_pitch * a.next_blocks) / a.next_blocks : 0;
    return quest_activation_before_gemm(&a, st);
}

// a layer on tiles in one launch, for sizes where the library has that
quest_fused_linear fused(void *out, const void *x, const void *w_tiles, const void *w_scale, int64_t m, int64_t k, int64_t n, float had_scale, int dt) {
    quest_fused_linear l = {};
    l.out = out, l.x = x, l.w_tiles = w_tiles, l.w_scale = w_scale;
    l.size_m = (int)m, l.size_k = (int)k, l.size_n = (int)n, l.had_scale = had_scale, l.dtype = dt;
    return l;
}

// ---- which matrix instructions a layer on its own runs on ------------------------------------------------------------
// sizes that the FP6 kernels address
bool tiles_addressable(int64_t m, int64_t k, int64_t n) { return k <= 65536 && m * n <= (1ll << 30) && m * k <= (5ll << 29); }

// Whether the FP6 layer is one launch (gemm_e2m3_fused.hip) at sizes where the INT8 kernels, one launch themselves up to 16 tokens, are the slower ones
// on the GPU too: 1.0 to 1.6 times from 9 to 128 tokens, (8, 1024, 3072) the same.  That file has the exact rule; what is let through here and not there
// takes two launches, which are no slower than INT8's at these sizes.
bool one_launch_on_tiles(int64_t m, int64_t k, int64_t n) { return 512 < k && k <= 2048 && m * n <= (k <= 1024 ? 820000 : 131072); }

// what harness.py holds under these names: from its E2M3_SHORT_ROWS_TOKENS + 1 tokens on, a layer takes the FP6 kernels with rows of E2M3_MIN_K elements and
// more, or of E2M3_MIN_K_NARROW where it has fewer than E2M3_NARROW channels
struct Lines {
    int64_t min_k, min_k_narrow, narrow, short_rows_tokens;
    bool take(PyObject *const *a) {
        int64_t *const to[4] = {&min_k, &min_k_narrow, &narrow, &short_rows_tokens};
        for (int i = 0; i < 4; i++)
            if (!PyLong_Check(a[i]) || ((*to[i] = PyLong_AsLongLong(a[i])) == -1 && PyErr_Occurred())) return false;
        return true;
    }
};

// Whether the FP6 kernels are the faster ones for an (m, k) x (n, k) layer on its own, quantiser included, with weights that come from HBM (copies of more
// than 300 MB in turn).  The lines were drawn over 2096 sizes, K 128 to 11008, N 136 to 22016, M 33 to 4096, with the FP6 kernels before
// gemm_e2m3_resident.hip, and have not been drawn again.  With today's kernels the path taken is 2.9 % behind the faster one on average over 220
// sizes of these ranges (always FP6: 1.2 %), and 10 % over 260 sizes with rows of 640 to 1664 elements and 512 tokens and more (0.5 %), most at more
// than 4096 tokens with K < 1536 ((6618, 1280, 9712) 1.69).
bool prefers_e2m3(int64_t m, int64_t k, int64_t n, const Lines &lines) {
    if (m < 49 && (m < 9 || k > 2048)) return false;                 // (a few tokens first: their calls are host-bound)
    if (k % 128 != 0 || !tiles_addressable(m, k, n)) return false;
    if (m <= 128 && one_launch_on_tiles(m, k, n)) return true;
    if (m < 49) return false;
    // With short rows and many tokens the GEMM is mostly epilogue either way and the tile-writing activation kernels are a little slower than the
    // row-writing ones: see _enough_per_row in harness.py, the same line
    if (m > lines.short_rows_tokens) return k >= (n >= lines.narrow ? lines.min_k : lines.min_k_narrow);
    // K < 640: as often slower as faster (K = 128: 0.86 at (2000, 22016), 1.49 at (700, 11008); K = 512: 0.88 to 1.42)
    if (k < 640) return false;
    // Some tens of tokens: the weights are the cost, and the tiles are 1.5 x the codes' bytes.  (INT8 / FP6 time: (33, 11008, 11008) 0.72, (64, 4096,
    // 11008) 0.88, (40, 1024, 4096) 0.96; (64, 2048, 2048) 1.06, (64, 11008, 1024) 1.27.)  More than 16384 channels are a second round of the INT8
    // kernel's tiles: (56, 3072, 22016) 1.06.
    if (m <= 64) return (n <= 4096 && k >= 1536) || (n > 16384 && 2048 <= k && k <= 6912);
    // The INT8 kernels' 64 x 64 tiles: half a round of the 256 CUs or less 0.95 to 1.31 (1.08 on average), one nearly full round 0.82 to 1.16 (0.92; (256,
    // 6912, 3072) 0.87, (128, 4096, 8192) 0.87), two rounds 0.82 to 1.10 (0.96) with K >= 4096 and 0.91 to 1.12 (1.01) below, more 0.90 to 1.57 (1.10).
    const int64_t tiles = ((m + 63) >> 6) * ((n + 63) >> 6);
    if (tiles <= 512) return tiles <= 128 || (tiles > 256 && k < 4096);
    return !(m > 3000 && k < 1536 && 512 <= n && n <= 2048);          // (4096, 1280, 512) 0.96; (4096, 1024, 2048) 1.11 by now
}

// What is different for rows that are not whole 128s (`padded` long with the zeros behind them): the quantiser takes no longer ones, and the INT8 side has
// another quantiser, the row kernel, which is the faster one for few rows.  49 to 56 tokens of up to 4096 elements in two launches, INT8 / FP6 GPU time: (50,
// 3104, 4096) 0.89, (50, 4064, 1024) 0.91, (52, 4064, 4096) 0.92, (50, 2272, 2048) 1.00 and 0.94 as a call; with longer rows, more tokens or more channels (50, 6048,
// 1024) 1.09, (50, 4960, 4096) 1.01, (64, 2272, 4096) 1.05, (50, 4064, 18000) 1.18.
// Channels that are not whole 8s: the FP6 epilogue stores them one by one, which short rows do not outweigh where there are few tiles, 256 tokens up (400
// sizes, rows of 672 to 6816): (300, 672, 3319) 0.95, (300, 1376, 17003) 0.94, (500, 672, 2052) 0.83, (500, 2016, 2052) 0.90, (1000, 1376, 1031) 0.97, (2000, 672,
// 1031) 0.94; with more of them (500, 1376, 5569) 1.04, (1000, 1376, 3319) 1.06, (2000, 1376, 2052) 1.01, or fewer tokens (200, 1376, 1031) 1.13.
bool ragged_takes_tiles(int64_t m, int64_t padded, int64_t n) {
    if (n % 8 != 0 && padded <= 2048 && m > 256 && (m <= 384 ? n > 2048 : m * n <= 2200000)) return false;
    return padded <= 32768 && (m > 56 || padded > 4096 || n > 4096 || one_launch_on_tiles(m, padded, n));
}

// the same for Python: three sizes, and for prefers_e2m3 the four lines behind them
template <typename Rule>
PyObject *ask(PyObject *const *a, Py_ssize_t n_args, Py_ssize_t wanted, Rule rule) {
    if (n_args != wanted) return PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", wanted, n_args);
    const long long m = PyLong_AsLongLong(a[0]), k = PyLong_AsLongLong(a[1]), n = PyLong_AsLongLong(a[2]);
    if (PyErr_Occurred()) return nullptr;
    return PyBool_FromLong(rule(m, k, n));
}
PyObject *py_tiles_addressable(PyObject *, PyObject *const *a, Py_ssize_t n_args) { return ask(a, n_args, 3, tiles_addressable); }
PyObject *py_one_launch_on_tiles(PyObject *, PyObject *const *a, Py_ssize_t n_args) { return ask(a, n_args, 3, one_launch_on_tiles); }
PyObject *py_prefers_e2m3(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    Lines lines;
    if (n_args == 7 && !lines.take(a + 3)) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_TypeError, "whole numbers expected");
    return ask(a, n_args, 7, [&](int64_t m, int64_t k, int64_t n) { return prefers_e2m3(m, k, n, lines); });
}

// ---- linear(x, w_packed, w_scale, w_add, w_tiles, bias, had_scale, out[, lines]) -------------------------------------
// The W4A4 linear layer: activation kernel, GEMM, bias.  x (..., K); w_tiles: None, or the weight's E2M3 tiles (see tiles_of) when the
// FP6 kernel is wanted -- with the four lines behind `out`, where prefers_e2m3 and ragged_takes_tiles say so; out: None or the (M, N) result to fill.
PyObject *linear(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    Lines lines;
    if (n_args != 8 && (n_args != 12 || !lines.take(a + 8))) return PyErr_Occurred() ? nullptr : declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *x = args.tensor(a[0]);
    if (!args.ok || !is_half(x->scalar_type()) || x->dim() < 1) return declined();
    const at::ScalarType type = x->scalar_type();
    const int64_t k = x->size(-1), m = x->numel() / k;
    const at::Tensor *w = args.tensor(a[1]);
    if (!args.ok || w->scalar_type() != at::kByte || w->dim() != 2 || w->size(1) * 2 != k) return declined();
    const int64_t n = w->size(0);
    if (!fits_int(m) || !fits_int(k) || !fits_int(n)) return declined();
    const at::Tensor *w_scale = args.tensor(a[2], type, n);
    const at::Tensor *w_add = args.tensor(a[3], at::kInt, n);
    const double had_scale = PyFloat_AsDouble(a[6]);
    // (rows of whole 32s that are not whole 128s come as tiles with zeros behind them, without the transform)
    const int64_t padded = had_scale != 0. || k % 32 != 0 ? k : (k + 127) / 128 * 128;
    PyObject *const tiles_arg = n_args == 8 || (prefers_e2m3(m, padded, n, lines) && (padded == k || ragged_takes_tiles(m, padded, n))) ? tiles_of(a[4], a[1]) : Py_None;
    const bool tiles = tiles_arg != Py_None && args.ok && at(w_scale, 4);      // (the FP6 kernels read scales two at a time)
    const int64_t kt = tiles ? padded : k;
    const at::Tensor *w_tiles = tiles ? args.tensor(tiles_arg, at::kByte, (int64_t)quest_e2m3_tiles_bytes((int)n, (int)kt)) : nullptr;
    const at::Tensor *bias = a[5] == Py_None ? nullptr : args.tensor(a[5], type, n);
    const at::Tensor *given = a[7] == Py_None ? nullptr : args.matrix(a[7], type, m, n);
    if (!args.ok || !gemm_takes(m, kt, n, tiles) || !at(x, 16) || !at(w, 16) || !at(w_tiles, 16) || !at(given, 16)) return declined();
    // (a bias whose derivative is wanted is added by torch)
    if (bias != nullptr && ((at::GradMode::is_enabled() && bias->requires_grad()) || bias->_fw_grad(0).defined())) return declined();

    // (a single launch writes outputs while rows of x are still being read)
    const auto begins = [](const at::Tensor &t) { return reinterpret_cast<uintptr_t>(t.data_ptr()); };
    const bool apart = given == nullptr || begins(*given) + given->nbytes() <= begins(*x) || begins(*x) + x->nbytes() <= begins(*given);
    at::Tensor out;
    const auto result = [&]() {
        if (given != nullptr) return *given;
        c10::SmallVector<int64_t, 5> shape(x->sizes().begin(), x->sizes().end());
        shape.back() = n;
        return make(shape, type, args.dev);
    };
    const int rc = on(args.dev, [&](void *st) {
        const int dt = dtype_code(type);
        if (apart && !tiles && quest_linear_few_tokens_available((int)m, (int)k)) {
            out = result();
            const int rc = quest_linear_few_tokens(out.data_ptr(), x->data_ptr(), (const uint8_t *)w->data_ptr(), (const int32_t *)w_add->data_ptr(), w_scale->data_ptr(),
                                                   bias ? bias->data_ptr() : nullptr, (int)m, (int)k, (int)n, (float)had_scale, dt, st);
            if (rc == QUEST_OK) return rc;
        }
        if (apart && tiles) {
            out = result();
            quest_fused_linear l = fused(out.data_ptr(), x->data_ptr(), w_tiles->data_ptr(), w_scale->data_ptr(), m, k, n, (float)had_scale, dt);
            if (bias != nullptr) l.epilogue = QUEST_EPILOGUE_BIAS, l.bias = bias->data_ptr();
            const int rc = at(bias, 16) ? quest_linear_e2m3_fused(&l, st) : QUEST_ERR_UNSUPPORTED;
            if (rc == QUEST_OK) return rc;
        }
        const at::Tensor hold = make({Codes::bytes(m, kt, tiles)}, at::kByte, args.dev);
        const Codes q(hold.data_ptr(), m, kt, tiles);
        int rc = kt != k && had_scale == 0. ? quest_quantize_e2m3_padded(x->data_ptr(), q.scale, q.codes, (int)k, (int)m, dt, st)
                 : tiles && m >= 64 && m <= 512 ? quantise_for({w, w_scale, w_add, w_tiles, (int)n, (int)k}, q, x->data_ptr(), {}, (int)m, (int)k, (float)had_scale, dt, st)
                 : tiles ? quest_hadamard_quantize_e2m3(x->data_ptr(), q.scale, q.codes, nullptr, nullptr, nullptr, (int)k, (int)m, (float)had_scale, dt, st)
                         : quest_hadamard_quantize_int4(x->data_ptr(), q.scale, q.codes, q.row_sum, nullptr, (int)k, (int)m, (float)had_scale, dt, st);
        if (rc != QUEST_OK) return rc;
        if (!out.defined()) out = result();
        bool add_bias = bias != nullptr;
        if (add_bias) {                                      // in the GEMM's epilogue where the kernel can
            rc = tiles ? quest_fused_matmul_dequantize_bias_e2m3(out.data_ptr(), q.codes, w_tiles->data_ptr(), q.scale, w_scale->data_ptr(), bias->data_ptr(), (int)m, (int)kt, (int)n, dt, st)
                       : quest_fused_matmul_dequantize_bias_int4_int4t(out.data_ptr(), q.codes, (const uint8_t *)w->data_ptr(), q.row_sum, (const int32_t *)w_add->data_ptr(),
                                                                       q.scale, w_scale->data_ptr(), bias->data_ptr(), (int)m, (int)k, (int)n, dt, st);
            add_bias = rc != QUEST_OK;
        }
        if (add_bias || bias == nullptr) {
            rc = tiles ? quest_fused_matmul_dequantize_e2m3(out.data_ptr(), q.codes, w_tiles->data_ptr(), q.scale, w_scale->data_ptr(), (int)m, (int)kt, (int)n, dt, st)
                       : quest_fused_matmul_dequantize_int4_int4t(out.data_ptr(), q.codes, (const uint8_t *)w->data_ptr(), q.row_sum,
                                                                  (const int32_t *)w_add->data_ptr(), q.scale, w_scale->data_ptr(), (int)m, (int)k, (int)n, dt, st);
            if (rc == QUEST_OK && add_bias) out.add_(*bias);
        }
        return rc;
    });
    if (rc != QUEST_OK) return declined();
    return given != nullptr ? ref(a[7]) : wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- gemm(mat_a, mat_b, a_add, b_add, a_mul, b_mul, out) ------------------------------------------------------------
PyObject *gemm(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    if (n_args != 7) return declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *x = args.tensor(a[0]), *w = args.tensor(a[1]);
    if (!args.ok || x->scalar_type() != at::kByte || w->scalar_type() != at::kByte || x->dim() != 2 || w->dim() != 2 ||
        x->size(1) != w->size(1))
        return declined();
    const int64_t m = x->size(0), n = w->size(0), k = w->size(1) * 2;
    if (!fits_int(m) || !fits_int(k) || !fits_int(n)) return declined();
    const at::Tensor *a_add = args.tensor(a[2], at::kInt, m), *b_add = args.tensor(a[3], at::kInt, n);
    const at::Tensor *a_mul = args.tensor(a[4]);
    if (!args.ok || !is_half(a_mul->scalar_type()) || a_mul->numel() != m) return declined();
    const at::ScalarType type = a_mul->scalar_type();
    const at::Tensor *b_mul = args.tensor(a[5], type, n);
    const at::Tensor *given = a[6] == Py_None ? nullptr : args.matrix(a[6], type, m, n);
    if (!args.ok) return declined();
    at::Tensor out;
    const int rc = on(args.dev, [&](void *st) {
        out = given != nullptr ? *given : make({m, n}, type, args.dev);
        return quest_fused_matmul_dequantize_int4_int4t(out.data_ptr(), (const uint8_t *)x->data_ptr(), (const uint8_t *)w->data_ptr(),
                                                        (const int32_t *)a_add->data_ptr(), (const int32_t *)b_add->data_ptr(), a_mul->data_ptr(),
                                                        b_mul->data_ptr(), (int)m, (int)k, (int)n, dtype_code(type), st);
    });
    if (rc != QUEST_OK) return declined();
    return given != nullptr ? ref(a[6]) : wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- matmul_int32(mat_a, mat_b, out) --------------------------------------------------------------------------------
PyObject *matmul_int32(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    if (n_args != 3) return declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *x = args.tensor(a[0]), *w = args.tensor(a[1]);
    if (!args.ok || x->scalar_type() != at::kByte || w->scalar_type() != at::kByte || x->dim() != 2 || w->dim() != 2 ||
        x->size(1) != w->size(1))
        return declined();
    const int64_t m = x->size(0), n = w->size(0), k = w->size(1) * 2;
    if (!fits_int(m) || !fits_int(k) || !fits_int(n)) return declined();
    const at::Tensor *given = a[2] == Py_None ? nullptr : args.matrix(a[2], at::kInt, m, n);
    if (!args.ok) return declined();
    at::Tensor out;
    const int rc = on(args.dev, [&](void *st) {
        out = given != nullptr ? *given : make({m, n}, at::kInt, args.dev);
        return quest_matmul_int4_int4t_int32((int32_t *)out.data_ptr(), (const uint8_t *)x->data_ptr(), (const uint8_t *)w->data_ptr(), (int)m,
                                             (int)k, (int)n, st);
    });
    if (rc != QUEST_OK) return declined();
    return given != nullptr ? ref(a[2]) : wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- hadamard_quantize(x, scale, packed, row_sum, had_scale, rule) -> (scale, packed, row_sum) ------------------------
// scale, packed and row_sum: None or the tensor to fill.
PyObject *hadamard_quantize(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    if (n_args != 6) return declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *x = args.tensor(a[0]);
    if (!args.ok || !is_half(x->scalar_type()) || x->dim() != 2) return declined();
    const at::ScalarType type = x->scalar_type();
    const int64_t m = x->size(0), k = x->size(1);
    if (!fits_int(m) || !fits_int(k)) return declined();
    at::Tensor scale, packed, row_sum;
    if (a[1] != Py_None) scale = *args.tensor(a[1], type, m);
    if (a[2] != Py_None) packed = *args.matrix(a[2], at::kByte, m, k / 2);
    if (a[3] != Py_None) row_sum = *args.tensor(a[3], at::kInt, m);
    const double had_scale = PyFloat_AsDouble(a[4]);
    const long rule = PyLong_AsLong(a[5]);
    if (!args.ok) return declined();
    const int rc = on(args.dev, [&](void *st) {
        if (!scale.defined()) scale = make({m, 1}, type, args.dev);
        if (!packed.defined()) packed = make({m, k / 2}, at::kByte, args.dev);
        if (!row_sum.defined()) row_sum = make({m, 1}, at::kInt, args.dev);
        return quest_hadamard_quantize_int4_rule(x->data_ptr(), scale.data_ptr(), (uint8_t *)packed.data_ptr(), (int32_t *)row_sum.data_ptr(),
                                                 nullptr, (int)k, (int)m, (float)had_scale, (int)rule, dtype_code(type), st);
    });
    if (rc != QUEST_OK) return declined();
    wrote(scale), wrote(packed), wrote(row_sum);
    PyObject *t = PyTuple_New(3);
    if (t == nullptr) return nullptr;
    PyTuple_SET_ITEM(t, 0, a[1] != Py_None ? ref(a[1]) : wrap(std::move(scale)));
    PyTuple_SET_ITEM(t, 1, a[2] != Py_None ? ref(a[2]) : wrap(std::move(packed)));
    PyTuple_SET_ITEM(t, 2, a[3] != Py_None ? ref(a[3]) : wrap(std::move(row_sum)));
    return t;
    END_HANDLE_TH_ERRORS
}

// ---- pack_weight(weight, had_scale, rule) -> (packed, scale, add) ------------------------------------------------------
PyObject *pack_weight(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    if (n_args != 3) return declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *w = args.tensor(a[0]);
    if (!args.ok || !is_half(w->scalar_type()) || w->dim() != 2) return declined();
    const at::ScalarType type = w->scalar_type();
    const int64_t n = w->size(0), k = w->size(1);
    if (!fits_int(n) || !fits_int(k)) return declined();
    const float had_scale = (float)PyFloat_AsDouble(a[1]);
    const int rule = (int)PyLong_AsLong(a[2]);
    at::Tensor packed, scale, add;
    const int rc = on(args.dev, [&](void *st) {
        packed = make({n, k / 2}, at::kByte, args.dev), scale = make({n, 1}, type, args.dev), add = make({n, 1}, at::kInt, args.dev);
        return quest_pack_weight_int4(w->data_ptr(), scale.data_ptr(), (uint8_t *)packed.data_ptr(), (int32_t *)add.data_ptr(), (int)k, (int)n,
                                      had_scale, rule, dtype_code(type), st);
    });
    if (rc != QUEST_OK) return declined();
    PyObject *t = PyTuple_New(3);
    if (t == nullptr) return nullptr;
    PyTuple_SET_ITEM(t, 0, wrap(std::move(packed)));
    PyTuple_SET_ITEM(t, 1, wrap(std::move(scale)));
    PyTuple_SET_ITEM(t, 2, wrap(std::move(add)));
    return t;
    END_HANDLE_TH_ERRORS
}

// ---- hadamard128(x, out, had_scale) ----------------------------------------------------------------------------------
PyObject *hadamard128(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    if (n_args != 3) return declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *x = args.tensor(a[0]);
    if (!args.ok || !is_half(x->scalar_type()) || x->dim() < 1) return declined();
    const int64_t k = x->size(-1), rows = x->numel() / k;
    at::Tensor out;
    if (a[1] != Py_None) out = *args.tensor(a[1], x->scalar_type(), x->numel());
    if (!args.ok || (out.defined() && out.sizes() != x->sizes()) || !fits_int(k) || !fits_int(rows)) return declined();
    const float had_scale = (float)PyFloat_AsDouble(a[2]);
    const int rc = on(args.dev, [&](void *st) {
        if (!out.defined()) out = make(x->sizes(), x->scalar_type(), args.dev);
        return quest_hadamard128(out.data_ptr(), x->data_ptr(), (int)k, (int)rows, had_scale, dtype_code(x->scalar_type()), st);
    });
    if (rc != QUEST_OK) return declined();
    return a[1] != Py_None ? ref(a[1]) : wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- find_scale(x, scale) --------------------------------------------------------------------------------------------
PyObject *find_scale(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    if (n_args != 2) return declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *x = args.tensor(a[0]);
    if (!args.ok || !is_half(x->scalar_type()) || x->dim() != 2) return declined();
    const int64_t m = x->size(0), k = x->size(1);
    at::Tensor scale;
    if (a[1] != Py_None) scale = *args.tensor(a[1], x->scalar_type(), m);
    if (!args.ok || !fits_int(m) || !fits_int(k)) return declined();
    const int rc = on(args.dev, [&](void *st) {
        if (!scale.defined()) scale = make({m, 1}, x->scalar_type(), args.dev);
        return quest_find_scale_int4(scale.data_ptr(), x->data_ptr(), (int)k, (int)m, dtype_code(x->scalar_type()), st);
    });
    if (rc != QUEST_OK) return declined();
    wrote(scale);
    return a[1] != Py_None ? ref(a[1]) : wrap(std::move(scale));
    END_HANDLE_TH_ERRORS
}

// ---- quantize(x, scale, x_int, packed, row_sum, do_dequantize) -> True -----------------------------------------------
PyObject *quantize(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    if (n_args != 6) return declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *x = args.tensor(a[0]);
    if (!args.ok || !is_half(x->scalar_type()) || x->dim() != 2) return declined();
    const int64_t m = x->size(0), k = x->size(1);
    const at::Tensor *scale = args.tensor(a[1], x->scalar_type(), m);
    const at::Tensor *x_int = a[2] == Py_None ? nullptr : args.matrix(a[2], at::kChar, m, k);
    const at::Tensor *packed = a[3] == Py_None ? nullptr : args.matrix(a[3], at::kByte, m, k / 2);
    const at::Tensor *row_sum = a[4] == Py_None ? nullptr : args.tensor(a[4], at::kInt, m);
    if (!args.ok || !fits_int(m) || !fits_int(k)) return declined();
    const int dequantize = PyObject_IsTrue(a[5]);
    if (dequantize < 0) return nullptr;
    const int rc = on(args.dev, [&](void *st) {
        return quest_quantize_int4(x->data_ptr(), scale->data_ptr(), x_int ? (int8_t *)x_int->data_ptr() : nullptr,
                                   packed ? (uint8_t *)packed->data_ptr() : nullptr, row_sum ? (int32_t *)row_sum->data_ptr() : nullptr, (int)k,
                                   (int)m, dequantize, dtype_code(x->scalar_type()), st);
    });
    if (rc != QUEST_OK) return declined();
    for (const at::Tensor *t : {packed, row_sum})
        if (t != nullptr) wrote(*t);
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// ---- add_mul_vv(a_add, a_mul, b_add, b_mul, mat_c, mat_d) -------------------------------------------------------------
PyObject *add_mul_vv(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    if (n_args != 6) return declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *c = args.tensor(a[4]);
    if (!args.ok || c->scalar_type() != at::kInt || c->dim() != 2) return declined();
    const int64_t m = c->size(0), n = c->size(1);
    const at::Tensor *a_mul = args.tensor(a[1]);
    if (!args.ok || !is_half(a_mul->scalar_type()) || a_mul->numel() != m) return declined();
    const at::ScalarType type = a_mul->scalar_type();
    const at::Tensor *a_add = args.tensor(a[0], at::kInt, m), *b_add = args.tensor(a[2], at::kInt, n), *b_mul = args.tensor(a[3], type, n);
    const at::Tensor *given = a[5] == Py_None ? nullptr : args.matrix(a[5], type, m, n);
    if (!args.ok || !fits_int(m) || !fits_int(n)) return declined();
    at::Tensor out;
    const int rc = on(args.dev, [&](void *st) {
        out = given != nullptr ? *given : make({m, n}, type, args.dev);
        return quest_add_mul_vv(out.data_ptr(), (const int32_t *)a_add->data_ptr(), a_mul->data_ptr(), (const int32_t *)b_add->data_ptr(),
                                b_mul->data_ptr(), (const int32_t *)c->data_ptr(), (int)m, (int)n, dtype_code(type), st);
    });
    if (rc != QUEST_OK) return declined();
    return given != nullptr ? ref(a[5]) : wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ---- block(x, branch, freqs, n_head, norm1, eps1, norm2, eps2, qkv, o, gate_up, glu, down, tiles, glu_of) -------------
// One producer-fused decoder block (LlamaBlock.forward_fused with every option at its default): x (B, T, C) is the residual
// stream, updated in place; branch: None, or the previous block's MLP output still to be added.  qkv, o, gate_up, glu, down:
// (packed, scale, add, tiles or None) of the projections, glu the row-interleaved gate / up weights; tiles: which of the
// four GEMMs (bit 0 qkv, 1 o, 2 gate_up, 3 down) run on E2M3 tiles where there are any; glu_of: gate_up's three tensors, their
// addresses and their versions when glu was made from them.  Returns True, or the block's MLP output when it is still to be added.
void launched(int rc, const char *what) {
    TORCH_CHECK(rc == QUEST_OK, what, " failed with status ", rc, ": ", quest_status_string(rc));
}

// the GEMM of a projection on quantised activations: dst = product, or dst += product with the two roundings of x + y
void project(const Linear &w, const Codes &q, void *dst, int m, int dt, void *st, bool add_to_dst = false) {
    if (q.tiles) {
        auto *f = add_to_dst ? quest_fused_matmul_dequantize_add_e2m3 : quest_fused_matmul_dequantize_e2m3;
        launched(f(dst, q.codes, w.tiles->data_ptr(), q.scale, w.scale->data_ptr(), m, w.k, w.n, dt, st), "projection");
    } else {
        auto *f = add_to_dst ? quest_fused_matmul_dequantize_add_int4_int4t : quest_fused_matmul_dequantize_int4_int4t;
        launched(f(dst, q.codes, (const uint8_t *)w.packed->data_ptr(), q.row_sum, (const int32_t *)w.add->data_ptr(),
                   q.scale, w.scale->data_ptr(), m, w.k, w.n, dt, st), "projection");
    }
}

void quantise_into(const Linear &w, const Codes &q, const void *x, int m, int k, int dt, void *st) {
    int rc = quantise_for(w, q, x, {}, m, k, kHadamardEntry, dt, st);
    launched(rc, "activation kernel");
}

// a projection of x without tiles on so few tokens that quantiser and GEMM are one launch; false: nothing was launched
bool project_few(const Linear &w, const void *x, void *dst, int m, int dt, void *st) {
    if (w.tiles != nullptr || !quest_linear_few_tokens_available(m, w.k)) return false;
    const int rc = quest_linear_few_tokens(dst, x, (const uint8_t *)w.packed->data_ptr(), (const int32_t *)w.add->data_ptr(), w.scale->data_ptr(), nullptr, m, w.k, w.n,
                                           kHadamardEntry, dt, st);
    if (rc == QUEST_ERR_UNSUPPORTED) return false;
    launched(rc, "projection");
    return true;
}

// a projection of x, through the norm if there is one, on tiles in one launch; false: nothing was launched
bool project_fused(const Linear &w, const void *x, void *dst, int m, int dt, void *st, int epilogue, const at::Tensor *norm = nullptr, double eps = 0.,
                   const quest_fused_linear &rope = {}) {
    if (w.tiles == nullptr) return false;
    quest_fused_linear l = fused(dst, x, w.tiles->data_ptr(), w.scale->data_ptr(), m, w.k, w.n, kHadamardEntry, dt);
    l.epilogue = epilogue, l.eps = (float)eps, l.norm_weight = norm ? norm->data_ptr() : nullptr;
    l.freqs_cis = rope.freqs_cis, l.seq_len = rope.seq_len, l.rot_cols = rope.rot_cols, l.head_dim = rope.head_dim;
    const int rc = quest_linear_e2m3_fused(&l, st);
    if (rc == QUEST_ERR_UNSUPPORTED || rc == QUEST_ERR_BAD_SHAPE) return false;
    launched(rc, "projection");
    return true;
}

void norm_into(const Linear &w, const Codes &q, at::Tensor &x, const void *branch, const at::Tensor &weight, double eps, int m, int k, int dt, void *st) {
    launched(quantise_for(w, q, x.data_ptr(), {QUEST_PRODUCER_RMSNORM, branch, weight.data_ptr(), eps}, m, k, kHadamardEntry, dt, st), "norm kernel");
}

// whether scaled_dot_product_attention would run the flash kernel whose bits ours gives: not switched off, no backend put before it
// (sdpa_kernel's set_priority), no other flash library preferred
bool default_flash_attention() {
    at::Context &ctx = at::globalContext();
    return ctx.userEnabledFlashSDP() && ctx.sDPPriorityOrder()[0] == at::SDPBackend::flash_attention && ctx.getROCmFAPreferredBackend() != at::ROCmFABackend::Ck;
}

PyObject *block(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    if (n_args != 15) return declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *xp = args.tensor(a[0]);
    if (!args.ok || !is_half(xp->scalar_type()) || xp->dim() != 3) return declined();
    const at::ScalarType type = xp->scalar_type();
    // (the attention below would hand back another type than the kernels after it are told)
    if (at::autocast::is_autocast_enabled(at::kCUDA) && at::autocast::get_autocast_dtype(at::kCUDA) != type) return declined();
    const int64_t b = xp->size(0), t = xp->size(1), c64 = xp->size(2);
    if (!fits_int(b * t) || !fits_int(3 * c64)) return declined();
    const int m = (int)(b * t), c = (int)c64;
    const at::Tensor *branch = a[1] == Py_None ? nullptr : args.tensor(a[1], type, xp->numel());
    const long n_head = PyLong_AsLong(a[3]);
    if (n_head == -1 && PyErr_Occurred()) return nullptr;
    if (n_head <= 0 || c % n_head != 0) return declined();
    const int head_dim = (int)(c / n_head);
    const at::Tensor *freqs = args.tensor(a[2], at::kFloat, t * (head_dim / 2) * 2);
    const at::Tensor *norm1 = args.tensor(a[4], type, c), *norm2 = args.tensor(a[6], type, c);
    const double eps1 = PyFloat_AsDouble(a[5]), eps2 = PyFloat_AsDouble(a[7]);
    const long tiles = PyLong_AsLong(a[13]);
    Linear qkv, o, gate_up, glu, down;
    if (!args.ok || PyErr_Occurred() || !qkv.take(args, a[8], type, tiles & 1) || !o.take(args, a[9], type, tiles & 2) ||
        !gate_up.take(args, a[10], type, false) || !glu.take(args, a[11], type, tiles & 4) || !down.take(args, a[12], type, tiles & 8))
        return declined();
    if (!PyTuple_Check(a[14]) || PyTuple_GET_SIZE(a[14]) != 9) return declined();
    for (int i = 0; i < 3; i++)
        if (!unchanged(PyTuple_GET_ITEM(a[10], i), PyTuple_GET_ITEM(a[14], i), PyTuple_GET_ITEM(a[14], 3 + i), PyTuple_GET_ITEM(a[14], 6 + i)))
            return declined();
    const int hidden = down.k;
    if (qkv.k != c || qkv.n != 3 * c || o.k != c || o.n != c || gate_up.k != c || gate_up.n != 2 * hidden || glu.k != c || glu.n != 2 * hidden ||
        down.n != c || (c & 127) != 0 || (hidden & 127) != 0 || c > 32768 || hidden > 32768 || (head_dim & 7) != 0)
        return declined();
    // the residual stream is updated on the way, so what the kernels ask is asked here
    if (branch == xp || !at(xp, 16) || !at(branch, 16) || !at(freqs, 16) || !at(norm1, 16) || !at(norm2, 16)) return declined();
    for (const Linear *w : {&qkv, &o, &gate_up, &glu, &down})
        if (!gemm_takes(m, w->k, w->n, false) || (w->tiles != nullptr && !gemm_takes(m, w->k, w->n, true)) || !at(w->packed, 16) ||
            !at(w->tiles, 16) || !at(w->scale, 4))
            return declined();

    at::Tensor x = *xp, mlp;                                     // mlp: what is left to be added to x, if anything
    on(args.dev, [&](void *st) {
        const int dt = dtype_code(type);

        // One scratch allocation for the block: the codes that the GEMMs read one after the other; the heads, and where they were the gated
        // unit's outputs; the attention's outputs and, where no GEMM adds them, the output projection's; the down projection's codes.
        // Up to 64 tokens fp16 keeps torch's silu: the kernels' fast exponential gives torch's bits for every bf16 gate, but for two
        // fp16 ones it does not.
        const bool torch_silu = m <= 64 && type == at::kHalf, glu_tiles = glu.tiles != nullptr && !torch_silu, down_tiles = down.tiles != nullptr;
        const int64_t codes_b = std::max({Codes::bytes(m, c, qkv.tiles != nullptr), Codes::bytes(m, c, o.tiles != nullptr), Codes::bytes(m, c, glu_tiles)});
        const int64_t wide_b = up(2 * m * std::max<int64_t>(3 * c64, !glu_tiles && m <= 64 ? 2 * (int64_t)hidden : hidden)), core_b = up(2 * m * c64);
        const at::Tensor scratch = make({codes_b + wide_b + 2 * core_b + Codes::bytes(m, hidden, down_tiles)}, at::kByte, args.dev);
        uint8_t *const codes = (uint8_t *)scratch.data_ptr(), *const wide = codes + codes_b, *const core = wide + wide_b, *const att = core + core_b;
        const Codes act(att + core_b, m, hidden, down_tiles);

        // norm -> q, k, v with q and k rotated
        quest_fused_linear rope = {};
        rope.freqs_cis = (const float *)freqs->data_ptr(), rope.seq_len = (int)t, rope.rot_cols = 2 * c, rope.head_dim = head_dim;
        if (branch != nullptr || !project_fused(qkv, x.data_ptr(), wide, m, dt, st, QUEST_EPILOGUE_ROPE, norm1, eps1, rope)) {
            const Codes q(codes, m, c, qkv.tiles != nullptr);
            norm_into(qkv, q, x, branch ? branch->data_ptr() : nullptr, *norm1, eps1, m, c, dt, st);
            const float *f = (const float *)freqs->data_ptr();
            int rc = q.tiles ? (t >= 32 && head_dim % 32 == 0
                                    ? quest_fused_matmul_dequantize_rope_e2m3(wide, q.codes, qkv.tiles->data_ptr(), q.scale, qkv.scale->data_ptr(), m, c, 3 * c, dt, f, (int)t, 2 * c, head_dim, st)
                                    : QUEST_ERR_UNSUPPORTED)
                             : quest_fused_matmul_dequantize_rope_int4_int4t(wide, q.codes, (const uint8_t *)qkv.packed->data_ptr(), q.row_sum, (const int32_t *)qkv.add->data_ptr(), q.scale, qkv.scale->data_ptr(), m, c, 3 * c, dt, f, (int)t, 2 * c, head_dim, st);
            if (rc == QUEST_ERR_UNSUPPORTED || rc == QUEST_ERR_BAD_SHAPE) {        // nothing was launched: the two calls
                project(qkv, q, wide, m, dt, st);
                rc = quest_rope_interleaved(wide, f, m, (int)t, 3 * c, 2 * c, head_dim, dt, st);
            }
            launched(rc, "QKV projection");
        }
        // causal attention: the library's where ours does not take the heads, gives other bits (a 4-bit quantiser follows) or is not in the
        // place of the library kernel that the caller's choice of backends names
        const void *attended = core;
        at::Tensor theirs;
        int rc = QUEST_ERR_UNSUPPORTED;
        if (t <= QUEST_ATTENTION_SAME_BITS(head_dim) && default_flash_attention())
            rc = quest_causal_attention(core, wide, (int)b, (int)t, (int)n_head, head_dim, dt, st);
        if (rc == QUEST_ERR_UNSUPPORTED) {
            const int64_t row = 3 * c64;
            const at::Tensor heads = scratch.narrow(0, codes_b, 2 * m * row).view(type);
            const auto part = [&](int64_t i) { return heads.as_strided({b, n_head, t, head_dim}, {t * row, head_dim, row, 1}, heads.storage_offset() + i * c64); };
            theirs = at::scaled_dot_product_attention(part(0), part(1), part(2), {}, 0.0, true).transpose(1, 2).contiguous();
            attended = theirs.data_ptr();
        } else {
            launched(rc, "attention");
        }
        // output projection: into the residual stream where its GEMM can add
        bool has_att = project_few(o, attended, att, m, dt, st);
        if (!has_att && !project_fused(o, attended, x.data_ptr(), m, dt, st, QUEST_EPILOGUE_ADD)) {
            const Codes q(codes, m, c, o.tiles != nullptr);
            quantise_into(o, q, attended, m, c, dt, st);
            has_att = !q.tiles && !quest_fused_matmul_dequantize_add_available(m, c, c, st);
            project(o, q, has_att ? (void *)att : x.data_ptr(), m, dt, st, !has_att);
        }
        // norm -> gated unit -> its codes, or, few tokens, its outputs in `gated`
        const void *gated = nullptr;
        at::Tensor torchs;
        if (glu_tiles && !has_att && project_fused(glu, x.data_ptr(), wide, m, dt, st, QUEST_EPILOGUE_SWIGLU, norm2, eps2)) {
            gated = wide;
        } else {
            const Codes q(codes, m, c, glu_tiles);
            norm_into(q.tiles || m > 64 ? glu : gate_up, q, x, has_att ? att : nullptr, *norm2, eps2, m, c, dt, st);
            if (!q.tiles && m <= 64) {
                // the weight-streaming GEMM has no gated epilogue: gate and up side by side, the product inside the quantiser
                project(gate_up, q, wide, m, dt, st);
                if (torch_silu) {
                    const at::Tensor both = scratch.narrow(0, codes_b, 4 * (int64_t)m * hidden).view(type).view({m, 2 * hidden});
                    torchs = at::silu(both.narrow(1, 0, hidden)).mul_(both.narrow(1, hidden, hidden)).contiguous();
                    gated = torchs.data_ptr();
                } else {
                    launched(quantise_for(down, act, wide, {QUEST_PRODUCER_SILU_MUL}, m, hidden, kHadamardEntry, dt, st), "gated unit");
                }
            } else {
                launched(q.tiles ? quest_fused_matmul_dequantize_swiglu_e2m3(wide, q.codes, glu.tiles->data_ptr(), q.scale, glu.scale->data_ptr(), m, c, 2 * hidden, dt, st)
                                 : quest_fused_matmul_dequantize_swiglu_int4_int4t(wide, q.codes, (const uint8_t *)glu.packed->data_ptr(), q.row_sum, (const int32_t *)glu.add->data_ptr(), q.scale, glu.scale->data_ptr(), m, c, 2 * hidden, dt, st),
                         "gated projection");
                gated = wide;
            }
        }
        if (gated != nullptr && project_fused(down, gated, x.data_ptr(), m, dt, st, QUEST_EPILOGUE_ADD)) {
        } else if (down_tiles || quest_fused_matmul_dequantize_add_available(m, hidden, c, st)) {
            if (gated != nullptr) quantise_into(down, act, gated, m, hidden, dt, st);
            project(down, act, x.data_ptr(), m, dt, st, true);
        } else {
            mlp = make({b, t, c64}, type, args.dev);
            if (gated == nullptr || !project_few(down, gated, mlp.data_ptr(), m, dt, st)) {
                if (gated != nullptr) quantise_into(down, act, gated, m, hidden, dt, st);
                project(down, act, mlp.data_ptr(), m, dt, st);
            }
        }
        return 0;
    });
    if (!mlp.defined()) Py_RETURN_TRUE;
    return wrap(std::move(mlp));
    END_HANDLE_TH_ERRORS
}

// ---- last_logits(x, branch, norm_w, eps, head_w) -> (B, 1, V) ----------------------------------------------------------
// Final norm and language-model head for the last position of every sequence of x (B, T, C); branch: None, or what is still to be
// added to x.
PyObject *last_logits(PyObject *, PyObject *const *a, Py_ssize_t n_args) {
    if (n_args != 5) return declined();
    HANDLE_TH_ERRORS
    Args args;
    const at::Tensor *x = args.tensor(a[0]);
    if (!args.ok || !is_half(x->scalar_type()) || x->dim() != 3) return declined();
    const at::ScalarType type = x->scalar_type();
    const int64_t b = x->size(0), t = x->size(1), c = x->size(2);
    const at::Tensor *branch = a[1] == Py_None ? nullptr : args.tensor(a[1], type, x->numel());
    const at::Tensor *norm_w = args.tensor(a[2], type, c), *head = args.tensor(a[4]);
    const double eps = PyFloat_AsDouble(a[3]);
    if (!args.ok || head->scalar_type() != type || head->dim() != 2 || head->size(1) != c || b > 64 || (c & 63) != 0 || !fits_int(c) ||
        !fits_int(head->size(0)) || !at(x, 4) || !at(branch, 4) || !at(norm_w, 4) || !at(head, 16))
        return declined();
    const int64_t v = head->size(0), last = (t - 1) * c * 2;
    at::Tensor logits;
    const int rc = on(args.dev, [&](void *st) {
        const at::Tensor normed = make({b, c}, type, args.dev);
        logits = make({b, 1, v}, type, args.dev);
        const int rc = quest_rmsnorm_rows(normed.data_ptr(), (const uint8_t *)x->data_ptr() + last, branch ? (const uint8_t *)branch->data_ptr() + last : nullptr,
                                          norm_w->data_ptr(), (float)eps, (int)b, (long)(t * c), (int)c, dtype_code(type), st);
        if (rc != QUEST_OK) return rc;
        return quest_dense_rows(logits.data_ptr(), normed.data_ptr(), head->data_ptr(), (int)b, (int)c, (int)v, dtype_code(type), st);
    });
    if (rc != QUEST_OK) return declined();
    return wrap(std::move(logits));
    END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
#define QUEST_FN_AS(name, function) {#name, (PyCFunction)(void (*)(void))function, METH_FASTCALL, nullptr}
#define QUEST_FN(name) QUEST_FN_AS(name, name)
    QUEST_FN_AS(prefers_e2m3, py_prefers_e2m3), QUEST_FN_AS(one_launch_on_tiles, py_one_launch_on_tiles), QUEST_FN_AS(tiles_addressable, py_tiles_addressable),
    QUEST_FN(linear), QUEST_FN(gemm), QUEST_FN(matmul_int32), QUEST_FN(hadamard_quantize), QUEST_FN(pack_weight), QUEST_FN(hadamard128), QUEST_FN(find_scale), QUEST_FN(quantize), QUEST_FN(add_mul_vv), QUEST_FN(block), QUEST_FN(last_logits),
#undef QUEST_FN
#undef QUEST_FN_AS
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "Native host path of quest_amd's hot calls.", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&kModule); }

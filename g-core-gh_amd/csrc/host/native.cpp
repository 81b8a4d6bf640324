// The calls a decode or conversion loop makes thousands of times, from Python's arguments to the C ABI in one step.
//
// Every function takes what its wrapper in gcore_lowp/ has in hand and answers None unless the call is the plain one: exact
// torch tensors, contiguous, on the current GPU, of the types and shapes the kernels take as they are, and accepted by the C
// ABI.  The wrapper then goes through its own checks, conversions and errors as if this file did not exist.  What it saves is
// the interpreter's work per call (attribute look-ups, four or five tensor methods that do nothing, a device guard, ctypes
// conversions).  Where it allocates, launches or waits the interpreter's lock is free, as it is in torch's allocations and in a
// ctypes call: an allocation may wait for the device and a launch for room in a full queue.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <vector>

#include <ATen/ATen.h>
#include <ATen/EmptyTensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPException.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/lowp.h"

namespace {

// addresses in the library that ctypes has loaded (bind)
decltype(&lp_quant_fp8_block) p_quant_fp8;
decltype(&lp_dequant_fp8_block) p_dequant_fp8;
decltype(&lp_dequant_fp4_block) p_dequant_fp4;
decltype(&lp_fp4_to_fp8_amax) p_fp4_amax;
decltype(&lp_fp4_to_fp8_rebase) p_fp4_rebase;
decltype(&lp_gemm_fp8_block) p_gemm;
decltype(&lp_gemm_block_workspace_bytes) p_gemm_ws;
decltype(&lp_host_flag) p_flag;
decltype(&lp_host_table) p_table;
decltype(&lp_quant_fp8_row_colwise_t) p_quant_both;
decltype(&lp_gemm_fp8_grouped) p_grouped;
decltype(&lp_gemm_fp8_grouped_nn) p_grouped_nn;
decltype(&lp_gemm_fp8_rowscale_grouped) p_rowscale;
decltype(&lp_zero_slots) p_zero;
decltype(&lp_gemm_fp8_grouped_rows) p_grouped_rows;

PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    constexpr int count = 15;
    void *a[count];
    if (n != count) { PyErr_SetString(PyExc_TypeError, "bind: fifteen addresses"); return nullptr; }
    for (int i = 0; i < count; ++i) {
        a[i] = PyLong_AsVoidPtr(args[i]);
        if (!a[i]) { if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address"); return nullptr; }
    }
    p_quant_fp8 = (decltype(p_quant_fp8))a[0];
    p_dequant_fp8 = (decltype(p_dequant_fp8))a[1];
    p_dequant_fp4 = (decltype(p_dequant_fp4))a[2];
    p_fp4_amax = (decltype(p_fp4_amax))a[3];
    p_fp4_rebase = (decltype(p_fp4_rebase))a[4];
    p_gemm = (decltype(p_gemm))a[5];
    p_gemm_ws = (decltype(p_gemm_ws))a[6];
    p_flag = (decltype(p_flag))a[7];
    p_table = (decltype(p_table))a[8];
    p_quant_both = (decltype(p_quant_both))a[9];
    p_grouped = (decltype(p_grouped))a[10];
    p_grouped_nn = (decltype(p_grouped_nn))a[11];
    p_rowscale = (decltype(p_rowscale))a[12];
    p_zero = (decltype(p_zero))a[13];
    p_grouped_rows = (decltype(p_grouped_rows))a[14];
    Py_RETURN_NONE;
}

// A tensor the kernels can take as it is; nullptr otherwise.
const at::Tensor *plain(PyObject *o)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.is_cuda() || !t.is_contiguous() || t.numel() == 0 || t.is_conj() || t.is_neg()) return nullptr;
    return &t;
}

// All of them on the device that is current (the kernels are launched there).
template <class... T>
bool here(c10::DeviceIndex dev, const T *...t) { return dev == c10::hip::current_device() && ((t->get_device() == dev) && ...); }

at::Tensor make(at::IntArrayRef sizes, at::ScalarType type, c10::DeviceIndex dev)
{
    return at::detail::empty_cuda(sizes, type, c10::Device(c10::kCUDA, dev), std::nullopt);
}

void *stream(c10::DeviceIndex dev) { return (void *)c10::hip::getCurrentHIPStream(dev).stream(); }

int scale_code(at::ScalarType t)
{
    switch (t) {
    case at::kFloat: return LP_F32;
    case at::kBFloat16: return LP_BF16;
    case at::kFloat8_e8m0fnu: return LP_E8M0;
    default: return -1;
    }
}

at::ScalarType scale_type(int code) { return code == LP_F32 ? at::kFloat : code == LP_BF16 ? at::kBFloat16 : at::kFloat8_e8m0fnu; }

PyObject *pair(const at::Tensor &a, const at::Tensor &b)
{
    PyObject *x = THPVariable_Wrap(a), *y = x ? THPVariable_Wrap(b) : nullptr;
    PyObject *r = y ? PyTuple_Pack(2, x, y) : nullptr;
    Py_XDECREF(x);
    Py_XDECREF(y);
    return r;
}

bool ints(PyObject *const *args, int n, long *out)
{
    for (int i = 0; i < n; ++i) {
        out[i] = PyLong_AsLong(args[i]);
        if (out[i] == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    }
    return true;
}

// What torch throws reaches Python as the exception a call through torch's own bindings raises (torch.OutOfMemoryError of an
// allocation among them).
#define GUARDED(...) HANDLE_TH_ERRORS __VA_ARGS__ END_HANDLE_TH_ERRORS

// Other Python threads run while one of these lives.
struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// Waits until the flag lp_host_flag raises is up.  Watching it for the length of a kernel beats the runtime's own wait (12 us
// against 14 - 20 for a quantisation of 256 x 256 with the check); behind a long queue the runtime waits.
hipError_t wait_flag(const int32_t *flag, hipStream_t st)
{
    const auto begin = std::chrono::steady_clock::now();
    for (int i = 0; !__atomic_load_n(flag, __ATOMIC_ACQUIRE); ++i) {
        if ((i & 63) == 63 && std::chrono::steady_clock::now() - begin > std::chrono::microseconds(200)) return hipStreamSynchronize(st);
        __builtin_ia32_pause();
    }
    return hipSuccess;
}

// (x, bm, bn, scale_mode, scale code, zero_rule, amax_floor, check) -> (codes, scales), with `check` (codes, scales, whether a
// block holds a NaN), which waits for the result
PyObject *quant_fp8(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    long v[5];
    if (n != 8 || !ints(args + 1, 5, v)) Py_RETURN_NONE;
    const double floor = PyFloat_AsDouble(args[6]);
    if (PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
    const bool check = args[7] == Py_True;
    GUARDED(
        const at::Tensor *x = plain(args[0]);
        if (!x) Py_RETURN_NONE;
        const c10::DeviceIndex dev = x->get_device();
        if (!here(dev, x) || x->dim() < 2 || (x->scalar_type() != at::kBFloat16 && x->scalar_type() != at::kFloat)) Py_RETURN_NONE;
        const int64_t rows = x->size(-2), cols = x->size(-1), bm = v[0], bn = v[1];
        if (bm <= 0 || bn <= 0 || rows % bm || cols % bn || v[3] < 0 || v[3] > LP_E8M0) Py_RETURN_NONE;
        const hipStream_t st = c10::hip::getCurrentHIPStream(dev).stream();
        at::Tensor q, s, words;                          // words: NaN count, flag
        int32_t *host = nullptr;
        bool declined = false;
        {
            Unlocked u;
            hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
            if (check) declined = hipStreamIsCapturing(st, &capturing) != hipSuccess || capturing != hipStreamCaptureStatusNone;
            if (check && !declined) {
                words = at::detail::empty_cpu({2}, at::kInt, true);
                host = words.data_ptr<int32_t>();
                host[0] = host[1] = 0;
            }
            if (!declined) {
                at::DimVector grid(x->sizes().begin(), x->sizes().end());
                grid[grid.size() - 2] = rows / bm;
                grid[grid.size() - 1] = cols / bn;
                q = make(x->sizes(), at::kFloat8_e4m3fn, dev), s = make(grid, scale_type((int)v[3]), dev);
                const int rc = p_quant_fp8(x->const_data_ptr(), x->scalar_type() == at::kFloat ? LP_F32 : LP_BF16, x->numel() / cols, cols, (int)bm,
                                       (int)bn, (int)v[2], (float)floor, (int)v[4], q.data_ptr(), s.data_ptr(), (int)v[3], host, st);
                declined = rc != LP_OK;
                // an error of the runtime may be an earlier call's: the kernel may be running
                if (check && rc == LP_ERR_HIP) (void)hipStreamSynchronize(st);
            }
            // the counter and the flag stay allocated until the GPU is through with them (above too)
            if (check && !declined) C10_HIP_CHECK(p_flag(host + 1, st) ? hipStreamSynchronize(st) : wait_flag(host + 1, st));
        }
        if (declined) Py_RETURN_NONE;
        if (!check) return pair(q, s);
        PyObject *two = pair(q, s);
        PyObject *r = two ? PyTuple_Pack(3, PyTuple_GET_ITEM(two, 0), PyTuple_GET_ITEM(two, 1), host[0] ? Py_True : Py_False) : nullptr;
        Py_XDECREF(two);
        return r;
    )
}

// (codes, scales, fp4, FP4 zero rule, out code) -> values; the block is the ratio of the two shapes
PyObject *dequant(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    long v[3];
    if (n != 5 || !ints(args + 2, 3, v)) Py_RETURN_NONE;
    GUARDED(
        const at::Tensor *c = plain(args[0]), *s = plain(args[1]);
        if (!c || !s) Py_RETURN_NONE;
        const c10::DeviceIndex dev = c->get_device();
        if (!here(dev, c, s) || c->dim() < 2 || s->dim() != c->dim() || c->element_size() != 1) Py_RETURN_NONE;
        const int sc = scale_code(s->scalar_type());
        const int64_t rows = c->size(-2), cols = c->size(-1) * (v[0] ? 2 : 1), sr = s->size(-2), scol = s->size(-1);
        if (sc < 0 || rows % sr || cols % scol || (v[2] != LP_F32 && v[2] != LP_BF16)) Py_RETURN_NONE;
        for (int64_t d = 0; d + 2 < c->dim(); ++d)
            if (c->size(d) != s->size(d)) Py_RETURN_NONE;
        at::DimVector shape(c->sizes().begin(), c->sizes().end());
        shape[shape.size() - 1] = cols;
        const int64_t all_rows = c->numel() / c->size(-1);
        const int bm = (int)(rows / sr), bn = (int)(cols / scol);
        at::Tensor out;
        int rc;
        {
            Unlocked u;
            out = make(shape, v[2] == LP_F32 ? at::kFloat : at::kBFloat16, dev);
            rc = v[0] ? p_dequant_fp4(c->const_data_ptr(), s->const_data_ptr(), sc, all_rows, cols, bm, bn, (int)v[1], out.data_ptr(), (int)v[2], stream(dev))
                      : p_dequant_fp8(c->const_data_ptr(), s->const_data_ptr(), sc, all_rows, cols, bm, bn, out.data_ptr(), (int)v[2], stream(dev));
        }
        if (rc) Py_RETURN_NONE;
        return THPVariable_Wrap(out);
    )
}

// (packed, e8m0 scales, kind, scale_mode, zero_rule, scale code of the result, amax_floor) -> (codes, scales); kind 0: re-based,
// kind 1: requantised by amax
PyObject *fp4_to_fp8(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    long v[4];
    if (n != 7 || !ints(args + 2, 4, v)) Py_RETURN_NONE;
    const double floor = PyFloat_AsDouble(args[6]);
    if (PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
    GUARDED(
        const at::Tensor *x = plain(args[0]), *s = plain(args[1]);
        if (!x || !s) Py_RETURN_NONE;
        const c10::DeviceIndex dev = x->get_device();
        if (!here(dev, x, s) || x->dim() != 2 || s->dim() != 2 || x->scalar_type() != at::kChar || s->scalar_type() != at::kFloat8_e8m0fnu)
            Py_RETURN_NONE;
        const int64_t rows = x->size(0), cols = x->size(1) * 2;
        if (rows % 128 || cols % 128 || s->size(0) != rows || s->size(1) != cols / 32 || v[3] < 0 || v[3] > LP_E8M0) Py_RETURN_NONE;
        at::Tensor q, so;
        int rc;
        {
            Unlocked u;
            q = make({rows, cols}, at::kFloat8_e4m3fn, dev), so = make({rows / 128, cols / 128}, scale_type((int)v[3]), dev);
            rc = v[0] ? p_fp4_amax(x->const_data_ptr(), s->const_data_ptr(), rows, cols, (int)v[1], (float)floor, (int)v[2], q.data_ptr(),
                                   so.data_ptr(), (int)v[3], nullptr, stream(dev))
                      : p_fp4_rebase(x->const_data_ptr(), s->const_data_ptr(), rows, cols, q.data_ptr(), so.data_ptr(), (int)v[3], stream(dev));
        }
        if (rc) Py_RETURN_NONE;
        return pair(q, so);
    )
}

// (Aq, As, Bq, Bs, out code) -> C
PyObject *gemm(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    long out_code;
    if (n != 5 || !ints(args + 4, 1, &out_code)) Py_RETURN_NONE;
    GUARDED(
        const at::Tensor *a = plain(args[0]), *sa = plain(args[1]), *b = plain(args[2]), *sb = plain(args[3]);
        if (!a || !sa || !b || !sb) Py_RETURN_NONE;
        const c10::DeviceIndex dev = a->get_device();
        if (!here(dev, a, sa, b, sb) || a->dim() != 2 || sa->dim() != 2 || b->dim() != 2 || sb->dim() != 2) Py_RETURN_NONE;
        if (a->scalar_type() != at::kFloat8_e4m3fn || b->scalar_type() != at::kFloat8_e4m3fn || sa->scalar_type() != sb->scalar_type() ||
            (sa->scalar_type() != at::kFloat && sa->scalar_type() != at::kFloat8_e8m0fnu) || (out_code != LP_BF16 && out_code != LP_F32))
            Py_RETURN_NONE;
        const int64_t M = a->size(0), K = a->size(1), N = b->size(0);
        if (b->size(1) != K || K % 128 || N % 128 || sa->size(0) != M || sa->size(1) != K / 128 || sb->size(0) != N / 128 || sb->size(1) != K / 128)
            Py_RETURN_NONE;
        at::Tensor c;
        int rc;
        {
            Unlocked u;
            at::Tensor ws;
            c = make({M, N}, out_code == LP_BF16 ? at::kBFloat16 : at::kFloat, dev);
            const int scales = scale_code(sa->scalar_type());
            int64_t need = p_gemm_ws(scales, M, N, K);
            if (need > 0) {
                try {
                    ws = make({need}, at::kByte, dev);
                } catch (const c10::OutOfMemoryError &) {
                    need = 0;                                // the kernels that need none are slower, not fewer
                }
            }
            rc = p_gemm(a->const_data_ptr(), sa->const_data_ptr(), b->const_data_ptr(), sb->const_data_ptr(), scales, M, N, K,
                        c.data_ptr(), (int)out_code, need > 0 ? ws.data_ptr() : nullptr, need, stream(dev));
        }
        if (rc) Py_RETURN_NONE;
        return THPVariable_Wrap(c);
    )
}

// The grouped linear: what gcore_lowp/grouped_gemm_fp8.py does with the row counts of the experts, a Python list of ints.  A layer is
// three or four launches forward and up to seven backward; through the interpreter and ctypes they and their tensors took longer
// than the GPU does for an expert-parallel shard (9 experts, 1754 rows, 2048 x 1536, forward and backward: 250 -> 145 us, of which
// autograd's own engine 50; 12 experts, 444 rows, 2048 x 2048, forward alone: 41 -> 29).
struct Experts {
    std::vector<int32_t> offsets;                                   // E + 1
    std::vector<std::array<int32_t, 4>> looped, one, two;           // problems of the weight gradient: {expert, K blocks, K blocks before, 0}
    std::vector<int32_t> empty;
    int64_t blocks = 0;                                             // K blocks of all, an expert padded to whole ones

    bool read(PyObject *list, bool train)
    {
        if (!PyList_CheckExact(list)) return false;
        const Py_ssize_t n = PyList_GET_SIZE(list);
        offsets.reserve(n + 1);
        offsets.push_back(0);
        for (Py_ssize_t e = 0; e < n; ++e) {
            PyObject *o = PyList_GET_ITEM(list, e);
            int over = 0;
            const long m = PyLong_CheckExact(o) ? PyLong_AsLongAndOverflow(o, &over) : -1;
            if (over || m < 0 || m > INT32_MAX - offsets.back()) return false;
            offsets.push_back(offsets.back() + (int32_t)m);
            if (!train) continue;
            const int32_t kb = (int32_t)((m + 127) / 128);
            if (kb == 0) empty.push_back((int32_t)e);
            else (kb == 1 ? one : kb == 2 ? two : looped).push_back({(int32_t)e, kb, (int32_t)blocks, 0});
            blocks += kb;
        }
        // longest first
        std::stable_sort(looped.begin(), looped.end(), [](const auto &a, const auto &b) { return a[1] > b[1]; });
        return true;
    }
    std::vector<int32_t> groups() const
    {
        std::vector<int32_t> w;
        for (const auto *kind : {&looped, &one, &two})
            for (const auto &g : *kind) w.insert(w.end(), g.begin(), g.end());
        w.insert(w.end(), empty.begin(), empty.end());
        return w;
    }
};

PyObject *tuple_of(std::initializer_list<at::Tensor> ts)
{
    PyObject *r = PyTuple_New((Py_ssize_t)ts.size());
    Py_ssize_t i = 0;
    for (const at::Tensor &t : ts) {
        PyObject *o = nullptr;
        if (!t.defined()) { o = Py_None; Py_INCREF(o); }
        else if (r) o = THPVariable_Wrap(t);
        if (!r || !o) { Py_XDECREF(r); Py_XDECREF(o); return nullptr; }
        PyTuple_SET_ITEM(r, i++, o);
    }
    return r;
}

// The experts' weights and rows as the kernels take them
bool grouped_operands(const at::Tensor *x, const at::Tensor *wq, const at::Tensor *ws, at::ScalarType qt, at::ScalarType st, int64_t width)
{
    return x && wq && ws && here(x->get_device(), x, wq, ws) && x->dim() == 2 && wq->dim() == 3 && ws->dim() == 3 && wq->scalar_type() == qt &&
           ws->scalar_type() == st && (x->scalar_type() == at::kBFloat16 || x->scalar_type() == at::kFloat) && wq->size(1) % 128 == 0 &&
           wq->size(2) % 128 == 0 && ws->size(0) == wq->size(0) && ws->size(1) == wq->size(1) / 128 && ws->size(2) == wq->size(2) / 128 &&
           x->size(1) == width;
}

// (x, Wq, Ws, rows per expert, out code, train, backward) -> (out, offsets, problems of the weight gradient, codes and scales of x by
// column); without `train` the last three are None, with no backward to come the offsets are too
PyObject *grouped_forward(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    long out_code;
    if (n != 7 || !ints(args + 4, 1, &out_code) || (out_code != LP_BF16 && out_code != LP_F32)) Py_RETURN_NONE;
    const bool train = args[5] == Py_True, backward = args[6] == Py_True;
    GUARDED(
        const at::Tensor *x = plain(args[0]), *wq = plain(args[1]), *ws = plain(args[2]);
        if (!wq || wq->dim() != 3 || !grouped_operands(x, wq, ws, at::kFloat8_e4m3fn, at::kFloat8_e8m0fnu, wq->size(2))) Py_RETURN_NONE;
        const int64_t rows = x->size(0), K = x->size(1), E = wq->size(0), N = wq->size(1);
        Experts ex;
        if (!ex.read(args[3], train) || (int64_t)ex.offsets.size() != E + 1 || ex.offsets.back() != rows) Py_RETURN_NONE;
        if (train && (uintptr_t)x->const_data_ptr() % 16) Py_RETURN_NONE;
        const c10::DeviceIndex dev = x->get_device();
        const int in_code = x->scalar_type() == at::kFloat ? LP_F32 : LP_BF16;
        at::Tensor out, offs, groups, qt, st;
        int rc;
        {
            Unlocked u;
            void *s_ = stream(dev);
            const at::Tensor q = make({rows, K}, at::kFloat8_e4m3fn, dev), s = make({rows, K / 128}, at::kFloat8_e8m0fnu, dev);
            const auto quantise = [&] {
                return p_quant_fp8(x->const_data_ptr(), in_code, rows, K, 1, 128, LP_SCALE_POW2, 0.0f, LP_ZERO_NONE, q.data_ptr(), s.data_ptr(), LP_E8M0,
                                   nullptr, s_);
            };
            const auto result = [&] { return make({rows, N}, out_code == LP_BF16 ? at::kBFloat16 : at::kFloat, dev); };
            // The row counts go with the GEMM's arguments, by which it also chooses its tiles, unless it refuses (more than 512 experts, 4 GiB)
            const auto multiply = [&] {
                out = result();
                return p_grouped_rows(q.data_ptr(), s.data_ptr(), wq->const_data_ptr(), ws->const_data_ptr(), LP_E8M0, ex.offsets.data(), (int)E, rows, N, K,
                                      out.data_ptr(), (int)out_code, s_);
            };
            rc = LP_ERR_UNSUPPORTED;
            bool quantised = false;
            if (!train && !backward) {
                // nobody else wants the offsets
                rc = quantise();
                quantised = !rc;
                if (!rc) rc = multiply();
            }
            if (rc == LP_ERR_UNSUPPORTED) {
                std::vector<int32_t> words = ex.offsets;
                const int64_t first = (E + 1 + 3) / 4 * 4;                // the problems, 16 bytes each
                if (train) {
                    const std::vector<int32_t> g = ex.groups();
                    words.resize(first, 0);
                    words.insert(words.end(), g.begin(), g.end());
                }
                const at::Tensor table = make({(int64_t)words.size()}, at::kInt, dev);
                offs = table.narrow(0, 0, E + 1);
                rc = p_table(words.data(), (int64_t)words.size(), table.data_ptr<int32_t>(), s_);
                if (!rc && train) {
                    groups = table.narrow(0, first, (int64_t)words.size() - first);
                    qt = make({K * ex.blocks * 128}, at::kByte, dev), st = make({K * ex.blocks}, at::kByte, dev);
                    rc = p_quant_both(x->const_data_ptr(), in_code, rows, K, offs.data_ptr<int32_t>(), (int)E, ex.blocks, 128, q.data_ptr(), s.data_ptr(),
                                      qt.data_ptr(), st.data_ptr(), LP_E8M0, s_);
                } else if (!rc && !quantised) {
                    rc = quantise();
                }
                if (!rc) {
                    rc = out.defined() ? LP_ERR_UNSUPPORTED : multiply();          // defined: refused above
                    if (rc == LP_ERR_UNSUPPORTED)
                        rc = p_grouped(q.data_ptr(), s.data_ptr(), wq->const_data_ptr(), ws->const_data_ptr(), LP_E8M0, offs.data_ptr<int32_t>(), (int)E, rows,
                                       N, K, out.data_ptr(), (int)out_code, s_);
                }
            }
        }
        if (rc) Py_RETURN_NONE;
        return tuple_of({out, offs, groups, qt, st});
    )
}

// (dY, Wq as bytes, Ws as bytes, offsets, problems, codes and scales of x by column, rows per expert, dX wanted, dW wanted, out code)
// -> (dX, dW), None where not wanted
PyObject *grouped_backward(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    long out_code;
    if (n != 11 || !ints(args + 10, 1, &out_code) || (out_code != LP_BF16 && out_code != LP_F32)) Py_RETURN_NONE;
    const bool want_w = args[9] == Py_True;
    if (args[8] != Py_True) Py_RETURN_NONE;
    GUARDED(
        const at::Tensor *dy = plain(args[0]), *wq = plain(args[1]), *ws = plain(args[2]), *offs = plain(args[3]);
        if (!wq || wq->dim() != 3 || !offs || !grouped_operands(dy, wq, ws, at::kByte, at::kByte, wq->size(1))) Py_RETURN_NONE;
        const int64_t rows = dy->size(0), E = wq->size(0), N = wq->size(1), K = wq->size(2);
        const c10::DeviceIndex dev = dy->get_device();
        Experts ex;
        if (!ex.read(args[7], want_w) || (int64_t)ex.offsets.size() != E + 1 || ex.offsets.back() != rows || offs->scalar_type() != at::kInt ||
            offs->numel() != E + 1 || !here(dev, offs) || (uintptr_t)dy->const_data_ptr() % 16)
            Py_RETURN_NONE;
        const at::Tensor *groups = nullptr, *xq = nullptr, *xs = nullptr;
        const int64_t problems = (int64_t)(ex.looped.size() + ex.one.size() + ex.two.size());
        if (want_w) {
            groups = plain(args[4]), xq = plain(args[5]), xs = plain(args[6]);
            if (!groups || !xq || !xs || !here(dev, groups, xq, xs) || groups->scalar_type() != at::kInt || xq->element_size() != 1 || xs->element_size() != 1 ||
                groups->numel() != 4 * problems + (int64_t)ex.empty.size() || xq->numel() != K * ex.blocks * 128 || xs->numel() != K * ex.blocks)
                Py_RETURN_NONE;
        }
        const at::ScalarType type = out_code == LP_BF16 ? at::kBFloat16 : at::kFloat;
        const int in_code = dy->scalar_type() == at::kFloat ? LP_F32 : LP_BF16;
        at::Tensor dx, dw;
        int rc;
        {
            Unlocked u;
            void *s_ = stream(dev);
            const at::Tensor q = make({rows, N}, at::kByte, dev), s = make({rows, N / 128}, at::kByte, dev);
            at::Tensor qt, st;
            if (want_w) {
                qt = make({N * ex.blocks * 128}, at::kByte, dev), st = make({N * ex.blocks}, at::kByte, dev);
                rc = p_quant_both(dy->const_data_ptr(), in_code, rows, N, offs->const_data_ptr<int32_t>(), (int)E, ex.blocks, 128, q.data_ptr(), s.data_ptr(),
                                  qt.data_ptr(), st.data_ptr(), LP_E8M0, s_);
            } else {
                rc = p_quant_fp8(dy->const_data_ptr(), in_code, rows, N, 1, 128, LP_SCALE_POW2, 0.0f, LP_ZERO_NONE, q.data_ptr(), s.data_ptr(), LP_E8M0,
                                 nullptr, s_);
            }
            if (!rc) {
                dx = make({rows, K}, type, dev);
                rc = p_grouped_nn(q.data_ptr(), s.data_ptr(), wq->const_data_ptr(), ws->const_data_ptr(), LP_E8M0, offs->const_data_ptr<int32_t>(), (int)E,
                                  rows, K, N, dx.data_ptr(), (int)out_code, s_);
            }
            if (!rc && want_w) {
                dw = make({E, N, K}, type, dev);
                const int32_t *at = groups->const_data_ptr<int32_t>();
                const bool whole = std::all_of(ex.looped.begin(), ex.looped.end(), [](const auto &g) { return g[1] % 4 == 0; });
                const auto launch = [&](const std::vector<std::array<int32_t, 4>> &kind, int most, int multiple) {
                    if (rc || kind.empty()) return;
                    rc = p_rowscale(qt.data_ptr(), st.data_ptr(), xq->const_data_ptr(), xs->const_data_ptr(), LP_E8M0, at, (int)kind.size(), most, multiple,
                                    N, K, dw.data_ptr(), (int)out_code, s_);
                    at += 4 * kind.size();
                };
                launch(ex.looped, ex.looped.empty() ? 0 : ex.looped[0][1], whole ? 4 : 1);
                launch(ex.one, 1, 1);
                launch(ex.two, 2, 2);
                if (!rc) rc = p_zero(dw.data_ptr(), N * K * (int64_t)dw.element_size(), E, at, (int)ex.empty.size(), s_);
            }
        }
        if (rc) Py_RETURN_NONE;
        return tuple_of({dx, dw});
    )
}

#define ENTRY(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {ENTRY(bind), ENTRY(quant_fp8), ENTRY(dequant), ENTRY(fp4_to_fp8), ENTRY(gemm), ENTRY(grouped_forward), ENTRY(grouped_backward),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_lowp_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject *PyInit__lowp_native()
{
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "built_for", LOWP_BUILT_FOR)) Py_CLEAR(m);
    return m;
}

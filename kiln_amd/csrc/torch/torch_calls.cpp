// The entry points of libkiln_marlin_gemm called from Python without Python: operand checks, output allocation,
// workspace lookup and the C call in one extension function each (CPython fast calls).
//
// What bounds a decode step driven from Python is the host: through ctypes one call cost 9.6 us (argument
// checks, a device context, the stream handle, an allocation and fifteen converted arguments), more than the 4
// to 8 us its kernel runs, so the GPU waited.
//
// Every function handles the plain case -- contiguous tensors of the right types on one device, a workspace that
// is already there -- and answers None to anything else, which tells the caller to take its checked route
// (whose error texts are the reference's).  The library's functions come as addresses (bind), so that the
// callers' choice between the shipped library and the tuning build holds here too.
#include <Python.h>

#include <algorithm>
#include <array>
#include <cstdint>
#include <vector>

#include <ATen/ATen.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "kiln_w4a16.h"

namespace {

struct Library {
    decltype(&kiln_marlin_w4a16_gemm) gemm = nullptr;
    decltype(&kiln_w4a16_gemm_lora) gemm_lora = nullptr;
    decltype(&kiln_w4a16_gemm_swiglu) swiglu = nullptr;
    decltype(&kiln_w4a16_gemm_swiglu_lora) swiglu_lora = nullptr;
    decltype(&kiln_w4a16_mlp) mlp = nullptr;
    decltype(&kiln_w4a16_workspace_bytes) workspace_bytes = nullptr;
    decltype(&kiln_w4a16_mlp_workspace_bytes) mlp_workspace_bytes = nullptr;
    decltype(&kiln_w4a16_stack_adapters) stack_adapters = nullptr;
    decltype(&kiln_w4a16_quantize_and_pack_many_device) quantize = nullptr;
    decltype(&kiln_w4a16_takes_adapter_sides) takes_sides = nullptr;
    decltype(&kiln_w4a16_takes_rank) takes_rank = nullptr;
    decltype(&kiln_w4a16_gemm_adapter_sides) gemm_sides = nullptr;
    decltype(&kiln_w4a16_repack_gptq_device) repack = nullptr;
};
Library g_lib;  // written by bind() under the interpreter lock, like everything below

PyTypeObject *g_stacked_type = nullptr, *g_single_type = nullptr;  // lora.StackedLora, lora.LoraProjectionWeights
PyObject *g_names[6] = {};                                         // interned: a_cat b_cat ranks scales a b
enum { kACat, kBCat, kRanks, kScales, kA, kB };

// marlin_gemm's workspaces, {(device index, stream handle): uint8 tensor}: looked up on every call, so that the
// dictionary is their only owner and what happens to its entries holds here at once.
PyObject *g_workspaces = nullptr;

const at::Tensor *tensor_of(PyObject *o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

bool plain(const at::Tensor &t, at::ScalarType type, int64_t dims, c10::Device device) {
    return t.dim() == dims && t.scalar_type() == type && t.device() == device && t.layout() == at::kStrided && t.is_contiguous();
}

// One GEMM's operands, checked: everything marlin_gemm._check_gemm_args asks for, and contiguity.
struct Problem {
    const at::Tensor *x = nullptr, *b = nullptr, *s = nullptr;
    int m = 0, n = 0, k = 0, groupsize = 0;
    c10::Device device{c10::DeviceType::CPU};
};

bool packed_ok(const at::Tensor &b, const at::Tensor &s, int64_t k, int groupsize, c10::Device device, int64_t *n) {
    if (!plain(b, at::kInt, 2, device) || !plain(s, at::kHalf, 2, device)) return false;
    *n = s.size(1);
    return k > 0 && k % 128 == 0 && *n > 0 && *n % 256 == 0 && b.size(0) == k / 16 && b.size(1) == 2 * *n &&
           s.size(0) == (groupsize == -1 ? 1 : k / 128) && k <= INT32_MAX && *n <= INT32_MAX / 2;
}

// 128 or -1 (per column), compared before it is narrowed; anything else, integers beyond 64 bits included, is the
// checked route's to refuse
bool groupsize_of(PyObject *o, int *groupsize) {
    const long g = PyLong_AsLong(o);
    if (g == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    if (g != 128 && g != -1) return false;
    *groupsize = (int)g;
    return true;
}

// max_rank: 2 for the GEMM entry points, 3 where a [batch, seq, k] activation is taken as well
bool problem_of(PyObject *const *args, int max_rank, Problem *p) {
    p->x = tensor_of(args[0]);
    p->b = tensor_of(args[1]);
    p->s = tensor_of(args[2]);
    if (!p->x || !p->b || !p->s || !g_lib.gemm || !groupsize_of(args[3], &p->groupsize)) return false;
    const at::Tensor &x = *p->x;
    const int64_t rank = x.dim();
    if (rank < 2 || rank > max_rank || !x.is_cuda()) return false;
    p->device = x.device();
    if (!plain(x, at::kBFloat16, rank, p->device)) return false;
    const int64_t k = x.size(rank - 1);
    int64_t n = 0;
    if (!packed_ok(*p->b, *p->s, k, p->groupsize, p->device, &n)) return false;
    const int64_t m = x.numel() / k;
    if (m < 1 || m > INT32_MAX) return false;
    p->m = (int)m;
    p->n = (int)n;
    p->k = (int)k;
    return true;
}

at::Tensor empty_bf16(at::IntArrayRef sizes, c10::Device device) {
    return at::Tensor(at::detail::empty_cuda(sizes, at::kBFloat16, device, std::nullopt));
}

// the result: `given` if the caller passed one of the right form (false: it is of another), else a new tensor
bool output_of(PyObject *given, const at::Tensor &x, int64_t columns, c10::Device device, at::Tensor *out) {
    if (given && given != Py_None) {
        const at::Tensor *t = tensor_of(given);
        if (!t || !plain(*t, at::kBFloat16, 2, device) || t->size(1) != columns || t->size(0) != x.numel() / x.size(x.dim() - 1)) return false;
        *out = *t;
        return true;
    }
    const int64_t rank = x.dim();
    std::array<int64_t, 3> sizes{x.size(0), rank == 3 ? x.size(1) : columns, columns};
    *out = empty_bf16(at::IntArrayRef(sizes.data(), (size_t)rank), device);
    return true;
}

// The device made current for the call, its stream, and that stream's workspace if it holds `bytes`.
struct Launch {
    c10::hip::HIPGuardMasqueradingAsCUDA guard;
    void *stream;
    at::Tensor workspace;
    explicit Launch(c10::Device device)
        : guard(device), stream((void *)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream()) {}
    bool find_workspace(c10::Device device, size_t bytes) {
        PyObject *key = PyTuple_New(2), *index = PyLong_FromLong(device.index()), *handle = PyLong_FromVoidPtr(stream);
        if (key && index && handle && g_workspaces) {
            PyTuple_SET_ITEM(key, 0, index);
            PyTuple_SET_ITEM(key, 1, handle);
            index = handle = nullptr;  // the tuple's now
            const PyObject *found = PyDict_GetItemWithError(g_workspaces, key);
            const at::Tensor *t = found ? tensor_of(const_cast<PyObject *>(found)) : nullptr;
            if (t && plain(*t, at::kByte, 1, device) && (size_t)t->numel() >= bytes) workspace = *t;
        }
        Py_XDECREF(key);
        Py_XDECREF(index);
        Py_XDECREF(handle);
        PyErr_Clear();
        return workspace.defined();
    }
};

bool ints_of(PyObject *o, std::vector<int> *v) {
    if (!PyTuple_CheckExact(o) && !PyList_CheckExact(o)) return false;
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(o);
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject *e = PySequence_Fast_GET_ITEM(o, i);
        if (!PyLong_CheckExact(e)) return false;
        const long value = PyLong_AsLong(e);
        if (value < 1 || value > INT32_MAX) {
            PyErr_Clear();
            return false;
        }
        v->push_back((int)value);
    }
    return true;
}
bool floats_of(PyObject *o, std::vector<float> *v) {
    if (!PyTuple_CheckExact(o) && !PyList_CheckExact(o)) return false;
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(o);
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject *e = PySequence_Fast_GET_ITEM(o, i);
        if (!PyFloat_CheckExact(e)) return false;
        v->push_back((float)PyFloat_AS_DOUBLE(e));
    }
    return true;
}

// Adapters as the library takes them.
struct Adapters {
    at::Tensor a, b;
    std::vector<int> ranks;
    std::vector<float> scales;
    int r_total = 0;
};

bool adapters_ok(const Adapters &l, const Problem &p) {
    return l.r_total >= 1 && l.r_total <= 64 && !l.ranks.empty() && l.ranks.size() <= 8 && l.ranks.size() == l.scales.size() &&
           plain(l.a, at::kBFloat16, 2, p.device) && plain(l.b, at::kBFloat16, 2, p.device) && l.a.size(0) == l.r_total &&
           l.a.size(1) == p.k && l.b.size(0) == p.n && l.b.size(1) == l.r_total;
}

// The launch itself, without the interpreter lock: a full queue makes it wait for the GPU.
int call(const Problem &p, const at::Tensor &out, bool swiglu, const Adapters *l, const Launch &at_) {
    const void *x = p.x->data_ptr(), *b = p.b->data_ptr();
    void *s = p.s->data_ptr(), *c = out.data_ptr(), *ws = at_.workspace.data_ptr();
    const int dev = p.device.index();
    int st;
    Py_BEGIN_ALLOW_THREADS
    if (l) {
        const void *a = l->a.data_ptr(), *lb = l->b.data_ptr();
        const int count = (int)l->ranks.size();
        st = swiglu ? g_lib.swiglu_lora(x, b, c, s, p.m, p.n / 2, p.k, ws, p.groupsize, dev, at_.stream, a, lb, l->r_total, count,
                                        l->ranks.data(), l->scales.data())
                    : g_lib.gemm_lora(x, b, c, s, p.m, p.n, p.k, ws, p.groupsize, dev, at_.stream, a, lb, l->r_total, count,
                                      l->ranks.data(), l->scales.data());
    } else {
        st = swiglu ? g_lib.swiglu(x, b, c, s, p.m, p.n / 2, p.k, ws, p.groupsize, dev, at_.stream)
                    : g_lib.gemm(x, b, c, s, p.m, p.n, p.k, ws, p.groupsize, dev, at_.stream, -1, -1, -1, 16);
    }
    Py_END_ALLOW_THREADS
    return st;
}

// linear(x, b_packed, scales, groupsize, out, swiglu, max_rank)
PyObject *py_linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Problem p;
    if (nargs != 7 || !problem_of(args, (int)PyLong_AsLong(args[6]), &p)) Py_RETURN_NONE;
    const bool swiglu = args[5] == Py_True;
    Launch at_(p.device);
    if (!at_.find_workspace(p.device, g_lib.workspace_bytes(p.m, p.n, p.k))) Py_RETURN_NONE;
    at::Tensor out;
    if (!output_of(args[4], *p.x, swiglu ? p.n / 2 : p.n, p.device, &out)) Py_RETURN_NONE;
    if (call(p, out, swiglu, nullptr, at_) != KILN_W4A16_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// linear_lora(x, b_packed, scales, groupsize, out, swiglu, lora_a, lora_b, ranks, lora_scales)
PyObject *py_linear_lora(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Problem p;
    if (nargs != 10 || !problem_of(args, 2, &p)) Py_RETURN_NONE;
    const bool swiglu = args[5] == Py_True;
    const at::Tensor *a = tensor_of(args[6]), *b = tensor_of(args[7]);
    Adapters l;
    if (!a || !b || !ints_of(args[8], &l.ranks) || !floats_of(args[9], &l.scales)) Py_RETURN_NONE;
    l.a = *a;
    l.b = *b;
    for (int r : l.ranks) l.r_total += r <= 64 ? r : 65;
    if (!adapters_ok(l, p)) Py_RETURN_NONE;
    Launch at_(p.device);
    if (!at_.find_workspace(p.device, g_lib.workspace_bytes(p.m, p.n, p.k))) Py_RETURN_NONE;
    at::Tensor out;
    if (!output_of(args[4], *p.x, swiglu ? p.n / 2 : p.n, p.device, &out)) Py_RETURN_NONE;
    if (call(p, out, swiglu, &l, at_) != KILN_W4A16_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// One projection's adapters among those of a fused call.
struct Side {
    at::Tensor a, b;
    int rank = 0, first = 0, rows = 0;
};

// The adapters of one side (a StackedLora, or a LoraProjectionWeights scaled by `scale`), appended to `l`.
bool add_side(PyObject *o, double scale, const Problem &p, int first, int rows, std::vector<Side> *sides, Adapters *l) {
    const bool stacked = Py_TYPE(o) == g_stacked_type;
    if (!stacked && Py_TYPE(o) != g_single_type) return false;
    PyObject *pa = PyObject_GetAttr(o, g_names[stacked ? kACat : kA]), *pb = PyObject_GetAttr(o, g_names[stacked ? kBCat : kB]);
    PyObject *pr = stacked ? PyObject_GetAttr(o, g_names[kRanks]) : nullptr, *ps = stacked ? PyObject_GetAttr(o, g_names[kScales]) : nullptr;
    Side side;
    bool ok = pa && pb && (!stacked || (pr && ps));
    if (!ok) PyErr_Clear();
    if (ok) {
        const at::Tensor *a = tensor_of(pa), *b = tensor_of(pb);
        ok = a && b && plain(*a, at::kBFloat16, 2, p.device) && plain(*b, at::kBFloat16, 2, p.device) && a->size(1) == p.k &&
             b->size(0) == rows && a->size(0) == b->size(1) && a->size(0) >= 1 && a->size(0) <= 64;
        if (ok) {
            side.a = *a;
            side.b = *b;
            side.rank = (int)a->size(0);
            side.first = first;
            side.rows = rows;
        }
    }
    if (ok && stacked) {
        const size_t before = l->ranks.size();
        ok = ints_of(pr, &l->ranks) && floats_of(ps, &l->scales) && l->ranks.size() == l->scales.size();
        int sum = 0;
        for (size_t i = before; i < l->ranks.size(); ++i) sum += l->ranks[i] <= 64 ? l->ranks[i] : 65;
        ok = ok && sum == side.rank;
    } else if (ok) {
        l->ranks.push_back(side.rank);
        l->scales.push_back((float)scale);
    }
    Py_XDECREF(pa);
    Py_XDECREF(pb);
    Py_XDECREF(pr);
    Py_XDECREF(ps);
    if (!ok) return false;
    l->r_total += side.rank;
    sides->push_back(std::move(side));
    return l->r_total <= 64 && l->ranks.size() <= 8 && sides->size() <= 8;
}

// linear_sides(x, b_packed, scales, groupsize, swiglu, sides, widths, lora_scale, split): a GEMM whose columns belong
// to several projections -- side by side, `widths` columns each, or with `swiglu` gate and up interleaved
// (widths = n_out twice) -- each with its adapters or None.  One projection over all columns with a stacked rank that
// kiln_w4a16_takes_rank names is what the entry points with adapters take as it is.  Else the launch reads every projection's own where
// they lie -- one to three of them, where kiln_w4a16_takes_adapter_sides says so -- and all others become one stacked set in a launch of their own in front.
// `split`: the result comes as one view per projection.
PyObject *py_linear_sides(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Problem p;
    if (nargs != 9 || !problem_of(args, 3, &p)) Py_RETURN_NONE;
    const bool swiglu = args[4] == Py_True, split = args[8] == Py_True;
    std::vector<int> widths;
    if (!PyTuple_CheckExact(args[5]) || !ints_of(args[6], &widths) || PyTuple_GET_SIZE(args[5]) != (Py_ssize_t)widths.size()) Py_RETURN_NONE;
    const double scale = PyFloat_AsDouble(args[7]);
    if (scale == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    Adapters l;
    std::vector<Side> sides;
    int64_t first = 0;
    for (size_t i = 0; i < widths.size(); ++i) {
        PyObject *o = PyTuple_GET_ITEM(args[5], (Py_ssize_t)i);
        if (o != Py_None && !add_side(o, scale, p, swiglu ? (int)(8 * i) : (int)first, widths[i], &sides, &l)) Py_RETURN_NONE;
        first += widths[i];
    }
    if (first != p.n || (swiglu && (widths.size() != 2 || widths[0] != widths[1]))) Py_RETURN_NONE;
    Launch at_(p.device);
    if (!at_.find_workspace(p.device, g_lib.workspace_bytes(p.m, p.n, p.k))) Py_RETURN_NONE;
    kiln_w4a16_adapter_side own[8];
    for (size_t i = 0; i < sides.size(); ++i)
        own[i] = {sides[i].a.data_ptr(), sides[i].b.data_ptr(), sides[i].rank, sides[i].first, sides[i].rows};
    const int n_sides = (int)sides.size(), n_adapters = (int)l.ranks.size();
    const bool as_it_is = n_sides == 1 && sides[0].rows == p.n && g_lib.takes_rank(p.m, p.n, p.k, sides[0].rank, p.device.index());
    const bool in_place = !as_it_is && n_sides > 0 &&
                          g_lib.takes_sides(p.m, p.n, p.k, own, n_sides, swiglu ? 1 : 0, n_adapters, p.device.index());
    if (!sides.empty() && !in_place) {
        const int padded = (l.r_total + 7) / 8 * 8;
        if (as_it_is) {
            l.a = sides[0].a;
            l.b = sides[0].b;
        } else {
            const int64_t a_elems = (int64_t)padded * p.k;  // a multiple of 1024 elements: both parts keep their alignment
            at::Tensor both = empty_bf16({a_elems + (int64_t)p.n * padded}, p.device);
            l.a = both.narrow(0, 0, a_elems).view({padded, p.k});
            l.b = both.narrow(0, a_elems, (int64_t)p.n * padded).view({p.n, padded});
            const void *pa[8], *pb[8];
            int ranks[8], firsts[8], rows[8];
            for (size_t i = 0; i < sides.size(); ++i) {
                pa[i] = own[i].lora_a;
                pb[i] = own[i].lora_b;
                ranks[i] = own[i].rank;
                firsts[i] = own[i].first_row;
                rows[i] = own[i].rows;
            }
            l.ranks.back() += padded - l.r_total;  // the last adapter gets the zero columns
            l.r_total = padded;
            const int st = g_lib.stack_adapters(pa, pb, ranks, firsts, rows, (int)sides.size(), p.k, p.n, padded, swiglu ? 1 : 0,
                                                l.a.data_ptr(), l.b.data_ptr(), at_.stream);
            if (st != KILN_W4A16_OK) Py_RETURN_NONE;
        }
        if (!adapters_ok(l, p)) Py_RETURN_NONE;
    }
    at::Tensor out;
    if (!output_of(nullptr, *p.x, swiglu ? p.n / 2 : p.n, p.device, &out)) Py_RETURN_NONE;
    int st = KILN_W4A16_OK;
    if (in_place) {
        const void *x = p.x->data_ptr(), *b = p.b->data_ptr();
        void *s = p.s->data_ptr(), *c = out.data_ptr(), *ws = at_.workspace.data_ptr();
        const int dev = p.device.index();
        Py_BEGIN_ALLOW_THREADS
        st = g_lib.gemm_sides(x, b, c, s, p.m, p.n, p.k, ws, p.groupsize, dev, at_.stream, own, n_sides, swiglu ? 1 : 0, n_adapters,
                              l.ranks.data(), l.scales.data());
        Py_END_ALLOW_THREADS
    } else {
        st = call(p, out, swiglu, sides.empty() ? nullptr : &l, at_);
    }
    if (st != KILN_W4A16_OK) Py_RETURN_NONE;
    if (!split) return THPVariable_Wrap(std::move(out));
    std::vector<int64_t> w(widths.begin(), widths.end());
    std::vector<at::Tensor> parts = out.split_with_sizes(w, -1);
    PyObject *tuple = PyTuple_New((Py_ssize_t)parts.size());
    if (!tuple) return nullptr;
    for (size_t i = 0; i < parts.size(); ++i) {
        PyObject *t = THPVariable_Wrap(std::move(parts[i]));
        if (!t) {
            Py_DECREF(tuple);
            return nullptr;
        }
        PyTuple_SET_ITEM(tuple, (Py_ssize_t)i, t);
    }
    return tuple;
    END_HANDLE_TH_ERRORS
}

// mlp(x, b_gate_up, s_gate_up, groupsize, b_down, s_down, out)
PyObject *py_mlp(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Problem p;
    if (nargs != 7 || !problem_of(args, 2, &p)) Py_RETURN_NONE;
    const at::Tensor *bd = tensor_of(args[4]), *sd = tensor_of(args[5]);
    int64_t n_down = 0;
    const int n_out = p.n / 2;
    if (!bd || !sd || !packed_ok(*bd, *sd, n_out, p.groupsize, p.device, &n_down)) Py_RETURN_NONE;
    Launch at_(p.device);
    if (!at_.find_workspace(p.device, g_lib.mlp_workspace_bytes(p.m, p.k, n_out, (int)n_down))) Py_RETURN_NONE;
    at::Tensor out;
    if (!output_of(args[6], *p.x, n_down, p.device, &out)) Py_RETURN_NONE;
    const void *x = p.x->data_ptr(), *bgu = p.b->data_ptr(), *sgu = p.s->data_ptr(), *b2 = bd->data_ptr(), *s2 = sd->data_ptr();
    void *y = out.data_ptr(), *ws = at_.workspace.data_ptr();
    int st;
    Py_BEGIN_ALLOW_THREADS
    st = g_lib.mlp(x, bgu, sgu, b2, s2, y, p.m, p.k, n_out, (int)n_down, ws, p.groupsize, p.device.index(), at_.stream);
    Py_END_ALLOW_THREADS
    if (st != KILN_W4A16_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// quantize(inputs, side_by_side, gate_up): every (contiguous bf16 [k, n] weight, groupsize) of the tuple `inputs`, all on one
// device, quantised and packed on the current stream -> a list of (words, scales), None where the shape is not
// supported, and behind them the interleaved pack of each pair of `gate_up`.  The inputs each tuple of `side_by_side` names by
// position (one k, one groupsize) get packed tensors that lie one after the other in memory; a pair of `gate_up` names a
// gate and an up of one shape and groupsize, each in one pair at most.
PyObject *py_quantize(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 3 || !g_lib.quantize || !PyTuple_CheckExact(args[0]) || !PyTuple_CheckExact(args[1]) || !PyTuple_CheckExact(args[2]) ||
        PyTuple_GET_SIZE(args[0]) == 0)
        Py_RETURN_NONE;
    struct Item {
        at::Tensor w, b, s;
        int64_t k = 0, n = 0, groups = 0;
        int g = 0;
        bool supported = false;
        int pair = -1, side = 0;  // the pair it is gate (0) or up (1) of
    };
    std::vector<Item> items((size_t)PyTuple_GET_SIZE(args[0]));
    for (size_t i = 0; i < items.size(); ++i) {
        Item &it = items[i];
        PyObject *pair = PyTuple_GET_ITEM(args[0], (Py_ssize_t)i);
        if (!PyTuple_CheckExact(pair) || PyTuple_GET_SIZE(pair) != 2 || !PyLong_CheckExact(PyTuple_GET_ITEM(pair, 1))) Py_RETURN_NONE;
        const at::Tensor *w = tensor_of(PyTuple_GET_ITEM(pair, 0));
        if (!w || !w->is_cuda() || !plain(*w, at::kBFloat16, 2, i ? items[0].w.device() : w->device()) ||
            !groupsize_of(PyTuple_GET_ITEM(pair, 1), &it.g))
            Py_RETURN_NONE;
        it.w = *w;
        it.k = w->size(0);
        it.n = w->size(1);
        if (it.k > INT32_MAX || it.n > INT32_MAX) Py_RETURN_NONE;
        it.supported = it.k > 0 && it.n > 0 && it.k % 128 == 0 && it.n % 256 == 0;
        it.groups = it.g == -1 ? 1 : it.k / 128;
    }
    const c10::Device device = items[0].w.device();
    c10::hip::HIPGuardMasqueradingAsCUDA guard(device);
    void *stream = (void *)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream();
    auto empty = [&](int64_t elems, at::ScalarType type) { return at::Tensor(at::detail::empty_cuda({elems}, type, device, std::nullopt)); };
    // piece [first, first + n) of the columns of a packed pair of `total` columns
    auto place = [](Item &it, const at::Tensor &b, const at::Tensor &s, int64_t first) {
        it.b = b.as_strided({it.k / 16, 2 * it.n}, {2 * it.n, 1}, first * (it.k / 8));
        it.s = s.as_strided({it.groups, it.n}, {it.n, 1}, first * it.groups);
    };
    std::vector<std::vector<int>> runs((size_t)PyTuple_GET_SIZE(args[1]));
    std::vector<bool> in_run(items.size(), false);
    for (Py_ssize_t r = 0; r < PyTuple_GET_SIZE(args[1]); ++r) {
        std::vector<int> &run = runs[(size_t)r];
        PyObject *o = PyTuple_GET_ITEM(args[1], r);
        if (!PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) == 0) Py_RETURN_NONE;
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(o); ++i) {
            const long at_ = PyLong_AsLong(PyTuple_GET_ITEM(o, i));
            if (at_ < 0 || at_ >= (long)items.size() || !items[(size_t)at_].supported || in_run[(size_t)at_]) {
                PyErr_Clear();
                Py_RETURN_NONE;
            }
            in_run[(size_t)at_] = true;
            run.push_back((int)at_);
            const Item &it = items[(size_t)at_], &head = items[(size_t)run[0]];
            if (it.k != head.k || it.g != head.g) Py_RETURN_NONE;
        }
    }
    struct Pair {
        at::Tensor b, s;
    };
    std::vector<Pair> pairs((size_t)PyTuple_GET_SIZE(args[2]));
    for (size_t p = 0; p < pairs.size(); ++p) {
        PyObject *o = PyTuple_GET_ITEM(args[2], (Py_ssize_t)p);
        if (!PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) != 2) Py_RETURN_NONE;
        Item *sides[2];
        for (int i = 0; i < 2; ++i) {
            const long at_ = PyLong_AsLong(PyTuple_GET_ITEM(o, i));
            if (at_ < 0 || at_ >= (long)items.size() || !items[(size_t)at_].supported || items[(size_t)at_].pair >= 0) {
                PyErr_Clear();
                Py_RETURN_NONE;
            }
            sides[i] = &items[(size_t)at_];
            sides[i]->pair = (int)p;
            sides[i]->side = i;
        }
        const Item &gate = *sides[0], &up = *sides[1];
        if (gate.k != up.k || gate.n != up.n || gate.g != up.g || gate.n > INT32_MAX / 2) Py_RETURN_NONE;
    }
    std::vector<kiln_w4a16_quantize_item> calls;
    calls.reserve(items.size());
    auto queue = [&](const Item &it) {
        calls.push_back({it.w.data_ptr(), (int)it.k, (int)it.n, it.g, it.side, it.b.data_ptr(), it.s.data_ptr(),
                         it.pair < 0 ? nullptr : pairs[(size_t)it.pair].b.data_ptr(),
                         it.pair < 0 ? nullptr : pairs[(size_t)it.pair].s.data_ptr()});
    };
    std::vector<bool> launched(items.size(), false);
    for (size_t r = 0; r < runs.size(); ++r) {
        const Item &head = items[(size_t)runs[r][0]];
        int64_t columns = 0, first = 0;
        bool paired = false;
        for (int i : runs[r]) {
            columns += items[(size_t)i].n;
            paired |= items[(size_t)i].pair >= 0;
        }
        at::Tensor b = empty(head.k / 8 * columns, at::kInt), s = empty(head.groups * columns, at::kHalf);
        for (int i : runs[r]) {
            place(items[(size_t)i], b, s, first);
            first += items[(size_t)i].n;
        }
        // The first run's weights go ahead, as soon as their memory is there, so that the GPU works on them while the host
        // makes the rest ready (a dozen tensors and a launch, 10 to 15 us): one launch of weights with scales per group (per
        // column they would be three) that takes it 6 us and more.  A layer of 2560 / 9216, seven weights: 100.9 -> 97.6 us; the call
        // on layers of other widths, full and linear attention: 4096 / 12288 171 -> 168 and 177 -> 172, 2048 / 5632 (16.8 M and 18.9 M weights in the
        // run) 67.4 -> 65.6 and 66.4 -> 63.9, 1792 / 4864 (13.8 and 15.1) 63.1 -> 63.1 and 61.2 -> 60.5, but 1536 / 5120 (10.2 and 10.6) 62.4 ->
        // 63.9 and 58.1 -> 59.2: the launch more costs what the GPU gains on them.
        if (r == 0 && !paired && head.g == 128 && head.k * columns >= (int64_t)14 << 20 && runs[r].size() < items.size()) {
            for (int i : runs[r]) {
                queue(items[(size_t)i]);
                launched[(size_t)i] = true;
            }
            if (g_lib.quantize(calls.data(), (int)calls.size(), device.index(), stream) != KILN_W4A16_OK) Py_RETURN_NONE;
            calls.clear();
        }
    }
    for (size_t p = 0; p < pairs.size(); ++p) {
        const Item &gate = *std::find_if(items.begin(), items.end(), [&](const Item &it) { return it.pair == (int)p && it.side == 0; });
        pairs[p].b = empty(gate.k / 8 * 2 * gate.n, at::kInt).view({gate.k / 16, 4 * gate.n});
        pairs[p].s = empty(gate.groups * 2 * gate.n, at::kHalf).view({gate.groups, 2 * gate.n});
    }
    for (size_t i = 0; i < items.size(); ++i) {
        Item &it = items[i];
        if (!it.supported || launched[i]) continue;
        if (!it.b.defined()) place(it, empty(it.k / 8 * it.n, at::kInt), empty(it.groups * it.n, at::kHalf), 0);
        queue(it);
    }
    if (g_lib.quantize(calls.data(), (int)calls.size(), device.index(), stream) != KILN_W4A16_OK) Py_RETURN_NONE;
    PyObject *list = PyList_New((Py_ssize_t)(items.size() + pairs.size()));
    if (!list) return nullptr;
    for (size_t i = 0; i < items.size() + pairs.size(); ++i) {
        PyObject *entry = Py_None;
        if (i >= items.size() || items[i].supported) {
            at::Tensor &tb = i < items.size() ? items[i].b : pairs[i - items.size()].b;
            at::Tensor &ts = i < items.size() ? items[i].s : pairs[i - items.size()].s;
            PyObject *b = THPVariable_Wrap(std::move(tb)), *s = THPVariable_Wrap(std::move(ts));
            entry = b && s ? PyTuple_Pack(2, b, s) : nullptr;
            Py_XDECREF(b);
            Py_XDECREF(s);
            if (!entry) {
                Py_DECREF(list);
                return nullptr;
            }
        } else {
            Py_INCREF(entry);
        }
        PyList_SET_ITEM(list, (Py_ssize_t)i, entry);
    }
    return list;
    END_HANDLE_TH_ERRORS
}

// Contiguous host tensors one after the other, each from a multiple of 256 bytes on, into the byte tensor `dst` on the current
// stream: through pinned memory, `stage_bytes` at a time, the first copy one of `first_piece` bytes.  The host tensors
// may change once this returns, the copies may still be running (the pinned block is torch's to keep until they are done).
void upload(std::initializer_list<at::Tensor> sources, const at::Tensor &dst, int64_t stage_bytes, int64_t first_piece,
            const c10::hip::HIPStreamMasqueradingAsCUDA &stream) {
    const at::Tensor stage = at::empty({std::min(stage_bytes, dst.numel())}, at::TensorOptions().dtype(at::kByte).pinned_memory(true));
    int64_t base = 0, sent = 0, at_ = 0;  // stage holds dst[base:]; dst[:sent] is on its way; dst[:at_] is staged
    auto send = [&]() {
        dst.narrow(0, sent, at_ - sent).copy_(stage.narrow(0, sent - base, at_ - sent), true);
        sent = at_;
    };
    for (const at::Tensor &src : sources) {
        const at::Tensor flat = src.view({-1}).view(at::kByte);
        int64_t done = 0;
        at_ = (at_ + 255) / 256 * 256;
        while (done < flat.numel()) {
            if (at_ - base >= stage.numel()) {
                send();
                stream.synchronize();  // the copies still read the stage
                base = at_;
            }
            const int64_t piece = std::min({sent == 0 ? first_piece : stage.numel(), flat.numel() - done, base + stage.numel() - at_});
            stage.narrow(0, at_ - base, piece).copy_(flat.narrow(0, done, piece));
            done += piece;
            at_ += piece;
            if (sent == 0 && dst.numel() > first_piece) send();  // (what is no longer than that goes in one)
        }
    }
    send();
}

// repack(qweight, scales, qzeros or None, k, n, groupsize, device index, stage_bytes, first_piece): a GPTQ projection's contiguous
// host tensors uploaded and rearranged on the device's current stream -> (words, scales) when that is done.  Driven from Python
// the same steps left more of the host's time around the link's (0.5 / 3.1 / 11.3 MiB: 60 -> 47 / 122 -> 108 / 281 -> 271 us).
// Subclasses are taken too, since loaders keep these tensors as a Parameter of their own: qweight and scales are read
// through views and copies only, which a subclass that runs its own operations answers as well; zero-points are read where
// they lie, and one of those, or a tensor without memory, has nothing there.
PyObject *py_repack(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 9 || !g_lib.repack) Py_RETURN_NONE;
    long long number[6];  // k, n, groupsize, device, stage_bytes, first_piece
    for (int i = 0; i < 6; ++i) {
        number[i] = PyLong_AsLongLong(args[3 + i]);
        if (number[i] == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
    }
    const int64_t k = number[0], n = number[1], g = number[2];
    if ((g != -1 && g != 128) || k <= 0 || n <= 0 || k % 128 != 0 || n % 256 != 0 || k > INT32_MAX || n > INT32_MAX ||
        number[3] < 0 || number[3] > INT8_MAX || number[4] < 256 || number[4] % 256 != 0 || number[5] < 256 || number[5] % 256 != 0)
        Py_RETURN_NONE;
    const int64_t groups = g == -1 ? 1 : k / 128, q_bytes = k / 2 * n, s_bytes = groups * n * 2;  // (q_bytes is a multiple of 16 KiB)
    const at::Tensor *host[3] = {};
    const at::ScalarType types[3] = {at::kInt, at::kHalf, at::kInt};
    const int64_t sizes[3] = {k / 8 * n, groups * n, groups * n / 8};
    for (int i = 0; i < 3; ++i) {
        if (i == 2 && args[i] == Py_None) break;
        const at::Tensor *t = THPVariable_Check(args[i]) ? &THPVariable_Unpack(args[i]) : nullptr;
        const bool read_in_place = i == 2;
        if (!t || (read_in_place && (t->unsafeGetTensorImpl()->is_python_dispatch() || !t->has_storage() || !t->storage().data() ||
                                     t->is_neg())) ||
            !t->device().is_cpu() || t->scalar_type() != types[i] || t->layout() != at::kStrided || t->numel() != sizes[i] ||
            !t->is_contiguous())
            Py_RETURN_NONE;
        host[i] = t;
    }
    const at::Tensor q = *host[0], s = *host[1], z = host[2] ? *host[2] : at::Tensor();
    at::Tensor b, tiled;
    bool done = false;
    {
        pybind11::gil_scoped_release no_gil;
        at::AutoDispatchBelowADInplaceOrView no_autograd;
        const c10::Device device(c10::DeviceType::CUDA, (c10::DeviceIndex)number[3]);
        c10::hip::HIPGuardMasqueradingAsCUDA guard(device);
        const auto stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index());
        const at::Tensor raw = at::detail::empty_cuda({q_bytes + s_bytes}, at::kByte, device, std::nullopt);
        b = at::detail::empty_cuda({k / 16, 2 * n}, at::kInt, device, std::nullopt);
        tiled = at::detail::empty_cuda({groups, n}, at::kHalf, device, std::nullopt);
        upload({q, s}, raw, number[4], number[5], stream);
        bool eights = true;
        if (z.defined()) {  // looked at while the copies run
            const uint32_t *word = reinterpret_cast<const uint32_t *>(z.data_ptr());
            uint32_t other = 0;
            for (int64_t i = 0; i < sizes[2]; ++i) other |= word[i] ^ 0x88888888u;
            eights = other == 0;
        }
        if (eights) {
            char *const at_ = static_cast<char *>(raw.data_ptr());
            done = g_lib.repack(at_, at_ + q_bytes, nullptr, (int)k, (int)n, (int)g, b.data_ptr(), tiled.data_ptr(), (int)number[3],
                                (void *)stream.stream()) == KILN_W4A16_OK;
            stream.synchronize();
        }
    }
    if (!done) Py_RETURN_NONE;
    PyObject *pb = THPVariable_Wrap(std::move(b)), *ps = THPVariable_Wrap(std::move(tiled));
    PyObject *pair = pb && ps ? PyTuple_Pack(2, pb, ps) : nullptr;
    Py_XDECREF(pb);
    Py_XDECREF(ps);
    return pair;
    END_HANDLE_TH_ERRORS
}

// set_workspaces(marlin_gemm's dictionary of them)
PyObject *py_set_workspaces(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    if (nargs != 1 || !PyDict_CheckExact(args[0])) {
        PyErr_SetString(PyExc_TypeError, "set_workspaces takes a dictionary");
        return nullptr;
    }
    Py_INCREF(args[0]);
    Py_XDECREF(g_workspaces);
    g_workspaces = args[0];
    Py_RETURN_NONE;
}

// bind(addresses of the library's functions, in the order of Library)
PyObject *py_bind(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    if (nargs != 13) {
        PyErr_SetString(PyExc_TypeError, "bind takes thirteen function addresses");
        return nullptr;
    }
    void *p[13];
    for (int i = 0; i < 13; ++i) p[i] = PyLong_AsVoidPtr(args[i]);
    if (PyErr_Occurred()) return nullptr;
    g_lib.gemm = reinterpret_cast<decltype(g_lib.gemm)>(p[0]);
    g_lib.gemm_lora = reinterpret_cast<decltype(g_lib.gemm_lora)>(p[1]);
    g_lib.swiglu = reinterpret_cast<decltype(g_lib.swiglu)>(p[2]);
    g_lib.swiglu_lora = reinterpret_cast<decltype(g_lib.swiglu_lora)>(p[3]);
    g_lib.mlp = reinterpret_cast<decltype(g_lib.mlp)>(p[4]);
    g_lib.workspace_bytes = reinterpret_cast<decltype(g_lib.workspace_bytes)>(p[5]);
    g_lib.mlp_workspace_bytes = reinterpret_cast<decltype(g_lib.mlp_workspace_bytes)>(p[6]);
    g_lib.stack_adapters = reinterpret_cast<decltype(g_lib.stack_adapters)>(p[7]);
    g_lib.quantize = reinterpret_cast<decltype(g_lib.quantize)>(p[8]);
    g_lib.takes_sides = reinterpret_cast<decltype(g_lib.takes_sides)>(p[9]);
    g_lib.gemm_sides = reinterpret_cast<decltype(g_lib.gemm_sides)>(p[10]);
    g_lib.repack = reinterpret_cast<decltype(g_lib.repack)>(p[11]);
    g_lib.takes_rank = reinterpret_cast<decltype(g_lib.takes_rank)>(p[12]);
    Py_RETURN_NONE;
}

// set_adapter_types(StackedLora, LoraProjectionWeights)
PyObject *py_set_adapter_types(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    if (nargs != 2 || !PyType_Check(args[0]) || !PyType_Check(args[1])) {
        PyErr_SetString(PyExc_TypeError, "set_adapter_types takes two classes");
        return nullptr;
    }
    Py_INCREF(args[0]);
    Py_INCREF(args[1]);
    g_stacked_type = reinterpret_cast<PyTypeObject *>(args[0]);
    g_single_type = reinterpret_cast<PyTypeObject *>(args[1]);
    Py_RETURN_NONE;
}

#define FAST(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(fn)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {FAST("linear", py_linear), FAST("linear_lora", py_linear_lora), FAST("linear_sides", py_linear_sides),
                           FAST("mlp", py_mlp), FAST("quantize", py_quantize), FAST("repack", py_repack), FAST("set_workspaces", py_set_workspaces), FAST("bind", py_bind),
                           FAST("set_adapter_types", py_set_adapter_types), {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_torch_calls", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_calls(void) {
    static const char *const names[6] = {"a_cat", "b_cat", "ranks", "scales", "a", "b"};
    for (int i = 0; i < 6; ++i)
        if (!(g_names[i] = PyUnicode_InternFromString(names[i]))) return nullptr;
    return PyModule_Create(&g_module);
}

// Operators whose GPU time is a few microseconds, from Python call to launch without Python in between: arguments checked,
// outputs and scratch taken from torch's caching allocator, the C ABI called on the current stream.  Written as Python
// functions with ctypes calls they cost 10-19 us of host time each, more than the kernels behind them take.
// The functions are those of kernels.py, which documents them; errors are the same AssertionError / SmhError.
#include <Python.h>
#include <dlfcn.h>

#include <ATen/Functions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <string>
#include <vector>

#include "../../include/smh.h"

namespace {

// the C ABI, from the library that ctypes has loaded
struct Api {
    decltype(&smh_last_error_string) last_error;
    decltype(&smh_q40_matmul) matmul;
    decltype(&smh_q40_matmul_plan) plan;
    decltype(&smh_q40_dequant) dequant;
    decltype(&smh_q40_quantize) quantize;
    decltype(&smh_q40_quantize_t) quantize_t;
    decltype(&smh_sample_topk_counts) sample_counts;
    decltype(&smh_sample_topk_rowtemp) sample_rowtemp;
    decltype(&smh_tree_step) tree_step;
    decltype(&smh_attn_workspace_bytes) attn_bytes;
    decltype(&smh_paged_attn_workspace_bytes) paged_bytes;
    decltype(&smh_shared_prefix_attn) shared_attn;
    decltype(&smh_paged_prefix_attn) paged_attn;
} api;
PyObject *smh_error = nullptr;

struct Refused {};                             // a Python error has been set

[[noreturn]] void refuse(const std::string &why) {
    PyErr_SetString(PyExc_AssertionError, why.c_str());
    throw Refused{};
}
void need(bool ok, const char *why) {
    if (!ok) refuse(why);
}
void check(int status, const char *what) {
    if (status == 0) return;
    PyErr_Format(smh_error, "%s failed with status %d: %s", what, status, api.last_error());
    throw Refused{};
}

typedef PyObject *const *Args;
bool none(PyObject *o) { return o == Py_None; }
const at::Tensor &tensor(PyObject *o, const char *what) {
    if (!THPVariable_Check(o)) refuse(std::string(what) + " must be a tensor");
    return THPVariable_Unpack(o);
}
const at::Tensor &gpu(PyObject *o, const char *what) {
    const at::Tensor &t = tensor(o, what);
    need(t.is_cuda(), "spec_mcts_amd kernels need GPU tensors (there is no CPU fallback)");
    return t;
}
PyObject *made(PyObject *o) {                  // a new object, or the error that kept it from being made
    if (o == nullptr) throw Refused{};
    return o;
}
// int(o) and float(o)
long number(PyObject *o) {
    if (PyLong_CheckExact(o)) {
        const long v = PyLong_AsLong(o);
        if (v == -1 && PyErr_Occurred()) throw Refused{};
        return v;
    }
    PyObject *i = made(PyNumber_Long(o));
    const long v = PyLong_AsLong(i);
    Py_DECREF(i);
    if (v == -1 && PyErr_Occurred()) throw Refused{};
    return v;
}
double real(PyObject *o) {
    if (PyFloat_CheckExact(o)) return PyFloat_AS_DOUBLE(o);
    PyObject *f = made(PyNumber_Float(o));
    const double v = PyFloat_AS_DOUBLE(f);
    Py_DECREF(f);
    return v;
}
// ... of whole numbers only
long whole_number(PyObject *o) {
    if (PyLong_CheckExact(o)) return number(o);
    PyObject *i = made(PyNumber_Index(o));
    const long v = PyLong_AsLong(i);
    Py_DECREF(i);
    if (v == -1 && PyErr_Occurred()) throw Refused{};
    return v;
}
// o <op> v, on the number as it was given
bool compares(PyObject *o, int op, long v) {
    PyObject *i = made(PyLong_FromLong(v));
    const int r = PyObject_RichCompareBool(o, i, op);
    Py_DECREF(i);
    if (r < 0) throw Refused{};
    return r == 1;
}
std::vector<int64_t> shape_of(PyObject *o, bool whole) {      // whole: only whole numbers; else int() of each
    PyObject *seq = made(PySequence_Fast(o, "a shape is a sequence of integers"));
    std::vector<int64_t> v;
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
    for (Py_ssize_t i = 0; i < n; ++i) {
        try {
            PyObject *x = PySequence_Fast_GET_ITEM(seq, i);
            v.push_back(whole ? whole_number(x) : number(x));
        } catch (Refused &) {
            Py_DECREF(seq);
            throw;
        }
    }
    Py_DECREF(seq);
    return v;
}
bool is(const at::Tensor &t, at::ScalarType s) { return t.scalar_type() == s; }
at::Tensor empty(at::IntArrayRef shape, at::ScalarType s, const at::Tensor &like) { return at::empty(shape, at::TensorOptions().dtype(s).device(like.device())); }
smh_stream_t stream() { return (smh_stream_t)c10::hip::getCurrentHIPStream().stream(); }
const void *ptr(PyObject *o) { return none(o) ? nullptr : gpu(o, "an optional argument").data_ptr(); }
PyObject *give(const at::Tensor &t) { return THPVariable_Wrap(t); }
void arity(Py_ssize_t n, Py_ssize_t want) {
    if (n != want) {
        PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
        throw Refused{};
    }
}

// (a, b_w, b_s, b_shape, residual, out)
PyObject *matmul_q40(Args x) {
    const at::Tensor &a = tensor(x[0], "a"), &w = tensor(x[1], "b_w"), &s = tensor(x[2], "b_s");
    need(a.is_contiguous(), "Matrix A must be contiguous");
    need(is(a, at::kHalf) && a.dim() == 2, "A must be fp16 [M, K]");
    const int64_t M = a.size(0), K = a.size(1);
    const std::vector<int64_t> bs = shape_of(x[3], false);
    need(bs.size() >= 2 && bs[0] == K, "Incompatible dimensions");
    const int64_t N = bs[1];
    need(a.is_cuda() && w.is_cuda() && s.is_cuda(), "spec_mcts_amd kernels need GPU tensors (there is no CPU fallback)");
    need(w.is_contiguous() && s.is_contiguous(), "the packed weight and its scales must be contiguous");
    need(is(w, at::kChar) && w.numel() == K * N / 2, "packed weight does not match b_shape");
    need(is(s, at::kHalf) && s.numel() == K * N / 64, "scales do not match b_shape");
    need(((uintptr_t)a.data_ptr() & 15) == 0, "A must be 16-byte aligned");
    at::Tensor c = none(x[5]) ? empty({M, N}, at::kHalf, a) : gpu(x[5], "out");
    need(c.dim() == 2 && c.size(0) == M && c.size(1) == N && c.is_contiguous() && is(c, at::kHalf), "out must be a contiguous fp16 [M, N]");
    int epi = SMH_EPI_NONE;
    if (!none(x[4])) {
        const at::Tensor &r = gpu(x[4], "residual");
        need(r.dim() == 2 && r.size(0) == M && r.size(1) == N && r.is_contiguous() && is(r, at::kHalf), "residual must be a contiguous fp16 [M, N]");
        epi = SMH_EPI_RESIDUAL;
    }
    // scratch for the K-slices' slabs, of exactly the planned size
    const int n = (int)N, ks = api.plan((int)M, (int)K, 1, &n);
    at::Tensor ws;
    size_t bytes = 0;
    if (ks > 1) {
        bytes = (size_t)ks * M * N * 4;
        ws = empty({(int64_t)bytes}, at::kByte, a);
    }
    check(api.matmul(a.data_ptr(), (int)M, (int)K, K, w.data_ptr(), s.data_ptr(), n, c.data_ptr(), N, epi, ptr(x[4]), N, ks > 1 ? ws.data_ptr() : nullptr,
                     bytes, stream()), "smh_q40_matmul");
    return give(c);
}

// (w, s, group_size, shape)
PyObject *deq_int40(Args x) {
    const at::Tensor &w = gpu(x[0], "w"), &s = gpu(x[1], "s");
    need(compares(x[2], Py_EQ, 64), "group_size must be 64");
    need(w.is_contiguous() && s.is_contiguous() && is(w, at::kChar) && is(s, at::kHalf), "w int8 and s fp16 must be contiguous");
    const std::vector<int64_t> shape = shape_of(x[3], true);
    int64_t n = 1;
    for (const int64_t d : shape) n *= d;
    need(n % 128 == 0 && w.numel() == n / 2 && s.numel() == n / 64, "w and s do not match the shape");
    at::Tensor out = empty(shape, at::kHalf, w);
    check(api.dequant(w.data_ptr(), s.data_ptr(), out.data_ptr(), n / 128, stream()), "smh_q40_dequant");
    return give(out);
}

PyObject *pair(const at::Tensor &q, const at::Tensor &s) {
    PyObject *a = give(q), *b = give(s);
    PyObject *t = PyTuple_New(2);
    PyTuple_SET_ITEM(t, 0, a);
    PyTuple_SET_ITEM(t, 1, b);
    return t;
}

// (w fp16, contiguous)
PyObject *q_int40(Args x) {
    const at::Tensor &w = gpu(x[0], "w");
    need(is(w, at::kHalf) && w.is_contiguous(), "w must be contiguous fp16");
    const int64_t n = w.numel();
    need(n % 128 == 0, "the number of values must be a multiple of 128");
    at::Tensor q = empty({n / 128, 64}, at::kChar, w), s = empty({n / 64, 1}, at::kHalf, w);
    check(api.quantize(w.data_ptr(), q.data_ptr(), s.data_ptr(), n / 64, stream()), "smh_q40_quantize");
    return pair(q, s);
}

// (v [N, K], contiguous)
PyObject *quantize_q40_t(Args x) {
    const at::Tensor &v = gpu(x[0], "v");
    need(v.dim() == 2 && v.size(0) % 128 == 0 && v.is_contiguous(), "v must be contiguous [N, K] with N a multiple of 128");
    const int type = is(v, at::kHalf) ? 0 : is(v, at::kBFloat16) ? 1 : is(v, at::kFloat) ? 2 : -1;
    need(type >= 0, "v must be fp16, bfloat16 or fp32");
    const int64_t N = v.size(0), K = v.size(1);
    at::Tensor q = empty({N * K / 128, 64}, at::kChar, v), s = empty({N * K / 64, 1}, at::kHalf, v);
    check(api.quantize_t(v.data_ptr(), type, (int)N, (int)K, q.data_ptr(), s.data_ptr(), stream()), "smh_q40_quantize_t");
    return pair(q, s);
}

// (logits, temperature, top_k, counts, uniform, out)
PyObject *sample_topk_counts(Args x) {
    const at::Tensor &logits = gpu(x[0], "logits"), &counts = gpu(x[3], "counts"), &uniform = gpu(x[4], "uniform");
    need(logits.dim() == 2 && is(logits, at::kHalf) && logits.stride(1) == 1, "logits must be fp16 [rows, vocab]");
    const int64_t rows = logits.size(0), vocab = logits.size(1);
    need(is(counts, at::kInt) && counts.is_contiguous() && counts.numel() >= rows, "counts must be int32 [rows]");
    need(is(uniform, at::kFloat) && uniform.is_contiguous(), "uniform must be contiguous fp32");
    at::Tensor out = none(x[5]) ? at::zeros({uniform.numel()}, at::TensorOptions().dtype(at::kLong).device(logits.device())) : gpu(x[5], "out");
    need(is(out, at::kLong) && out.is_contiguous() && out.numel() >= uniform.numel(), "out must be int64 with an entry per uniform number");
    const int k = (int)(compares(x[2], Py_GT, vocab) ? vocab : number(x[2]));
    if (THPVariable_Check(x[1])) {
        const at::Tensor &temp = gpu(x[1], "temperature");
        need(is(temp, at::kFloat) && temp.is_contiguous() && temp.numel() >= rows, "temperature must be fp32 [rows]");
        check(api.sample_rowtemp(logits.data_ptr(), (int)rows, (int)vocab, logits.stride(0), (const float *)temp.data_ptr(), k, (const float *)uniform.data_ptr(),
                                 (const int32_t *)counts.data_ptr(), (int64_t *)out.data_ptr(), (int)uniform.numel(), stream()), "smh_sample_topk_rowtemp");
    } else {
        check(api.sample_counts(logits.data_ptr(), (int)rows, (int)vocab, logits.stride(0), (float)real(x[1]), k, (const float *)uniform.data_ptr(),
                                (const int32_t *)counts.data_ptr(), (int64_t *)out.data_ptr(), (int)uniform.numel(), stream()), "smh_sample_topk_counts");
    }
    return give(out);
}

// (draws, output_counts, alive, curr_b, results, t_dev, pages, origin, state, terminal_seq, results_len, next_tokens, summary, eos)
PyObject *tree_step(Args x) {
    const at::Tensor &draws = gpu(x[0], "draws"), &oc = gpu(x[1], "output_counts"), &alive = gpu(x[2], "alive"), &curr = gpu(x[3], "curr_b");
    const at::Tensor &results = gpu(x[4], "results"), &t = gpu(x[5], "t_dev"), &origin = gpu(x[7], "origin"), &state = gpu(x[8], "state");
    const at::Tensor &seq = gpu(x[9], "terminal_seq"), &len = gpu(x[10], "results_len"), &next = gpu(x[11], "next_tokens"), &summary = gpu(x[12], "summary");
    need(is(results, at::kLong) && results.dim() == 2 && results.is_contiguous(), "results must be contiguous int64 [batch, steps]");
    const int64_t B = results.size(0), ld = results.size(1);
    need(is(draws, at::kLong) && draws.is_contiguous(), "draws must be contiguous int64");
    need(is(oc, at::kInt) && oc.dim() == 2 && oc.size(0) == 2 && oc.size(1) == B && oc.is_contiguous(), "output_counts must be contiguous int32 [2, batch]");
    need(is(alive, at::kByte) && alive.numel() == B && alive.is_contiguous(), "alive must be uint8 [batch]");
    need(is(curr, at::kInt) && is(t, at::kInt) && is(summary, at::kInt) && summary.numel() >= 2, "curr_b, t_dev and summary must be int32");
    need(is(origin, at::kInt) && origin.numel() >= B && is(state, at::kInt) && state.numel() == B, "origin and state must be int32 [batch]");
    need(is(len, at::kInt) && len.numel() == B && is(next, at::kLong) && next.numel() >= B, "results_len int32 [batch], next_tokens int64 [batch]");
    need(is(seq, at::kLong) && seq.is_contiguous(), "terminal_seq must be contiguous int64");
    int32_t *pages = nullptr;
    int64_t stride = 0;
    if (!none(x[6])) {
        const at::Tensor &p = gpu(x[6], "pages");
        need(is(p, at::kInt) && p.dim() == 2 && p.size(0) >= B && p.stride(1) == 1, "pages must be int32 [>= batch, positions]");
        pages = (int32_t *)p.data_ptr();
        stride = p.stride(0);
    }
    int32_t *tok = (int32_t *)oc.data_ptr();
    check(api.tree_step((const int64_t *)draws.data_ptr(), (int)draws.numel(), tok, tok + B, (uint8_t *)alive.data_ptr(), (int32_t *)curr.data_ptr(), (int)B,
                        (int64_t *)results.data_ptr(), ld, (const int32_t *)t.data_ptr(), pages, stride, (int32_t *)origin.data_ptr(),
                        (int32_t *)state.data_ptr(), (const int64_t *)seq.data_ptr(), (int)seq.numel(), number(x[13]), (int32_t *)len.data_ptr(),
                        (int64_t *)next.data_ptr(), (int32_t *)summary.data_ptr(), stream()), "smh_tree_step");
    Py_RETURN_NONE;
}

void half_rows(const at::Tensor &k, PyObject *vo, const char *why, const at::Tensor **v) {
    need(!none(vo), why);
    *v = &gpu(vo, "v");
    need(k.is_contiguous() && (*v)->is_contiguous() && is(k, at::kHalf) && is(**v, at::kHalf), why);
}

// (q, prefix_k, prefix_v, P, suffix_k, suffix_v, suffix_ks, suffix_vs, Smax, lens, lens_stride, cur_k, cur_v, n_kv_heads, out)
PyObject *shared_prefix_attn(Args x) {
    const at::Tensor &q = gpu(x[0], "q");
    need(q.is_contiguous() && is(q, at::kHalf) && q.dim() == 3, "q must be contiguous fp16 [B, H, D]");
    const int64_t B = q.size(0), H = q.size(1), D = q.size(2), P = number(x[3]);
    int64_t Hkv;
    const at::Tensor *v = nullptr;
    if (!none(x[1])) {
        const at::Tensor &k = gpu(x[1], "prefix_k");
        half_rows(k, x[2], "prefix_k and prefix_v must be contiguous fp16", &v);
        need(k.dim() >= 3 && compares(x[3], Py_LE, k.size(-3)), "P exceeds the prefix rows");
        Hkv = k.size(-2);
    } else {
        need(compares(x[3], Py_EQ, 0), "P without a prefix");
        Hkv = !none(x[13]) ? whole_number(x[13]) : !none(x[11]) ? gpu(x[11], "cur_k").size(1) : H;
    }
    int fmt = SMH_KV_NONE;
    if (!none(x[4])) {
        const at::Tensor &k = gpu(x[4], "suffix_k"), &sv = gpu(x[5], "suffix_v");
        need(k.is_contiguous() && sv.is_contiguous() && !none(x[9]), "the suffix must be contiguous and has lens");
        const at::Tensor &lens = gpu(x[9], "lens");
        need(is(lens, at::kInt), "lens must be int32");
        if (is(k, at::kHalf)) {
            fmt = SMH_KV_FP16;
        } else {
            need(is(k, at::kChar) && !none(x[6]) && !none(x[7]), "a suffix is fp16, or int8 rows with scales");
            need(is(gpu(x[6], "suffix_ks"), at::kHalf) && is(gpu(x[7], "suffix_vs"), at::kHalf), "suffix scales must be fp16");
            fmt = SMH_KV_Q40;
        }
    }
    if (!none(x[11])) half_rows(gpu(x[11], "cur_k"), x[12], "cur_k and cur_v must be contiguous fp16", &v);
    at::Tensor out = none(x[14]) ? at::empty_like(q) : gpu(x[14], "out");
    need(out.sizes() == q.sizes() && is(out, at::kHalf) && out.is_contiguous() && out.device() == q.device(), "out must be like q");
    const size_t bytes = api.attn_bytes((int)B, (int)H, (int)P);
    at::Tensor ws = empty({(int64_t)bytes}, at::kByte, q);
    check(api.shared_attn(q.data_ptr(), out.data_ptr(), (int)B, (int)H, (int)Hkv, (int)D, ptr(x[1]), ptr(x[2]), (int)P, fmt, ptr(x[4]), ptr(x[5]), ptr(x[6]), ptr(x[7]),
                          (int)number(x[8]), (const int32_t *)ptr(x[9]), (int)number(x[10]), ptr(x[11]), ptr(x[12]), ws.data_ptr(), bytes, stream()),
          "smh_shared_prefix_attn");
    return give(out);
}

// (q, pages, lens or None, pool_k, pool_v, pool_ks, pool_vs, head_major, prefix_k, prefix_v, P, prefix_head_major, cur_k, cur_v, lens_stride)
PyObject *paged_prefix_attn(Args x) {
    const at::Tensor &q = gpu(x[0], "q"), &pages = gpu(x[1], "pages"), &pk = gpu(x[3], "pool_k"), &pv = gpu(x[4], "pool_v");
    need(q.is_contiguous() && is(q, at::kHalf) && q.dim() == 3, "q must be contiguous fp16 [B, H, D]");
    const int64_t B = q.size(0), H = q.size(1), D = q.size(2);
    const int page_bytes = is(pages, at::kShort) ? 2 : is(pages, at::kInt) ? 4 : is(pages, at::kLong) ? 8 : 0;
    need(pages.dim() == 2 && pages.size(0) >= B && pages.stride(1) == 1 && page_bytes > 0, "pages must be int16, int32 or int64 [B, positions]");
    const int32_t *lens = nullptr;
    if (!none(x[2])) {
        const at::Tensor &l = gpu(x[2], "lens");
        need(is(l, at::kInt), "lens must be int32");
        lens = (const int32_t *)l.data_ptr();
    }
    need(pk.is_contiguous() && pv.is_contiguous() && pk.sizes() == pv.sizes() && pk.dim() == 3, "pool_k and pool_v must be contiguous and of one shape");
    const bool head_major = PyObject_IsTrue(x[7]) == 1, prefix_head_major = PyObject_IsTrue(x[11]) == 1;
    int fmt;
    int64_t Hkv, rows, row_stride = 0, head_stride = 0;
    if (is(pk, at::kHalf)) {
        fmt = SMH_KV_FP16;
        need(pk.size(2) == D, "pool rows must have the head dimension");
        Hkv = pk.size(head_major ? 0 : 1);
        rows = pk.size(head_major ? 1 : 0);
        if (head_major) { row_stride = D; head_stride = rows * D; }
    } else {
        fmt = SMH_KV_Q40;
        need(is(pk, at::kChar) && !none(x[5]) && !none(x[6]) && !head_major && pk.size(2) == 64, "a pool is fp16, or token-major int8 rows with scales");
        const at::Tensor &ks = gpu(x[5], "pool_ks"), &vs = gpu(x[6], "pool_vs");
        need(is(ks, at::kHalf) && is(vs, at::kHalf) && ks.is_contiguous() && vs.is_contiguous(), "pool scales must be contiguous fp16");
        Hkv = pk.size(1);
        rows = pk.size(0);
    }
    need(Hkv > 0 && H % Hkv == 0, "query heads must be a multiple of the kv heads");
    int64_t P = number(x[10]), p_row = 0, p_head = 0;
    const at::Tensor *v = nullptr;
    if (!none(x[8]) && P > 0) {
        const at::Tensor &k = gpu(x[8], "prefix_k");
        half_rows(k, x[9], "prefix_k and prefix_v must be contiguous fp16", &v);
        need(k.dim() == 3 && k.size(prefix_head_major ? 0 : 1) == Hkv && compares(x[10], Py_LE, k.size(prefix_head_major ? 1 : 0)), "the prefix does not match");
        if (prefix_head_major) { p_row = D; p_head = k.size(1) * D; }
    } else {
        P = 0;
    }
    if (!none(x[12])) {
        const at::Tensor &ck = gpu(x[12], "cur_k");
        half_rows(ck, x[13], "cur_k and cur_v must be contiguous fp16", &v);
        need(ck.dim() == 3 && ck.size(0) == B && ck.size(1) == Hkv && ck.size(2) == D, "cur_k must be [B, Hkv, D]");
    }
    at::Tensor out = at::empty_like(q);
    // (the partials of shared pages only where the call can use them)
    const size_t bytes = fmt == SMH_KV_FP16 && lens == nullptr ? api.paged_bytes((int)B, (int)H, (int)Hkv, (int)P, (int)pages.size(1))
                                                               : api.attn_bytes((int)B, (int)H, (int)P);
    at::Tensor ws = empty({(int64_t)bytes}, at::kByte, q);
    check(api.paged_attn(q.data_ptr(), out.data_ptr(), (int)B, (int)H, (int)Hkv, (int)D, P > 0 ? ptr(x[8]) : nullptr, P > 0 ? ptr(x[9]) : nullptr, (int)P, p_row, p_head,
                         fmt, pk.data_ptr(), pv.data_ptr(), ptr(x[5]), ptr(x[6]), row_stride, head_stride, rows, pages.data_ptr(), page_bytes, pages.stride(0),
                         (int)pages.size(1), lens, (int)number(x[14]), ptr(x[12]), ptr(x[13]), 0, ws.data_ptr(), bytes, stream()), "smh_paged_prefix_attn");
    return give(out);
}

// ---- what the layer calls read of a transformer block ----
struct Ref {                                   // a reference of one's own
    PyObject *o;
    explicit Ref(PyObject *made_) : o(made(made_)) {}
    Ref(Ref &&r) : o(r.o) { r.o = nullptr; }
    Ref(const Ref &) = delete;
    Ref &operator=(const Ref &) = delete;
    ~Ref() { Py_XDECREF(o); }
};
struct Names {
    PyObject *modules, *parameters, *attention, *feed_forward, *attention_norm, *ffn_norm, *weight, *eps, *prompt_len, *w, *s, *tiled, *buf;
    PyObject *caches[6], *lin[7];
    Names() {
        auto in = [](const char *n) { return made(PyUnicode_InternFromString(n)); };
        modules = in("_modules"); parameters = in("_parameters");
        attention = in("attention"); feed_forward = in("feed_forward"); attention_norm = in("attention_norm"); ffn_norm = in("ffn_norm");
        weight = in("weight"); eps = in("eps"); prompt_len = in("cache_prompt_len"); w = in("w"); s = in("s"); tiled = in("_tiled"); buf = in("buf");
        const char *c[6] = {"cache_prompt_k", "cache_prompt_v", "cache_k", "cache_k_s", "cache_v", "cache_v_s"};
        const char *l[7] = {"wq", "wk", "wv", "wo", "w1", "w2", "w3"};
        for (int i = 0; i < 6; ++i) caches[i] = in(c[i]);
        for (int i = 0; i < 7; ++i) lin[i] = in(l[i]);
    }
};
Ref attribute(PyObject *o, PyObject *name) { return Ref(PyObject_GetAttr(o, name)); }
// A submodule or parameter of an nn.Module, out of the dictionary that the module's own (Python) __getattr__ would look into.
Ref member(PyObject *o, PyObject *kind, PyObject *name) {
    PyObject *d = PyObject_GenericGetDict(o, nullptr);
    if (d == nullptr) {
        PyErr_Clear();
    } else {
        PyObject *of_kind = PyDict_GetItem(d, name) == nullptr ? PyDict_GetItem(d, kind) : nullptr;      // (borrowed)
        PyObject *v = of_kind != nullptr && PyDict_Check(of_kind) ? PyDict_GetItem(of_kind, name) : nullptr;
        Py_XINCREF(v);
        Py_DECREF(d);
        if (v != nullptr) return Ref(v);
    }
    return attribute(o, name);
}
constexpr int LAYER_WORDS = 2 + 2 + 6 + 7 * 4;

// (block, key: bytearray of LAYER_WORDS 8-byte words) -> the rows of the block's prompt cache; -1 - rows where the key was another one.
// The key is the addresses of all tensors that smh_layer takes from the block and of the checkpoint weights behind the tiled ones, the
// norms' eps, and the tiled weights as the objects they are (the caller keeps them alive); it is brought up to date.
PyObject *layer_state(Args x) {
    static const Names n;
    PyObject *block = x[0];
    need(PyByteArray_Check(x[1]) && PyByteArray_GET_SIZE(x[1]) == LAYER_WORDS * 8, "the key of a layer is a bytearray of layer_key_bytes");
    uint64_t now[LAYER_WORDS];
    int at = 0;
    auto address = [&](const Ref &t) { now[at++] = (uint64_t)(uintptr_t)tensor(t.o, "a layer's attribute").data_ptr(); };
    auto number_of = [&](const Ref &f) {
        const double v = real(f.o);
        memcpy(&now[at++], &v, 8);
    };
    const Ref att = member(block, n.modules, n.attention), ff = member(block, n.modules, n.feed_forward);
    for (PyObject *name : {n.attention_norm, n.ffn_norm}) {
        const Ref norm = member(block, n.modules, name);
        address(member(norm.o, n.parameters, n.weight));
        number_of(attribute(norm.o, n.eps));
    }
    int64_t capacity = 0;
    for (int i = 0; i < 6; ++i) {
        const Ref t = attribute(att.o, n.caches[i]);
        address(t);
        if (i == 0) capacity = tensor(t.o, "cache_prompt_k").size(1);
    }
    for (int i = 0; i < 7; ++i) {
        const Ref lin = member(i < 4 ? att.o : ff.o, n.modules, n.lin[i]);
        address(attribute(lin.o, n.w));
        address(attribute(lin.o, n.s));
        const Ref tiled = attribute(lin.o, n.tiled);
        now[at++] = (uint64_t)(uintptr_t)tiled.o;
        if (none(tiled.o)) now[at++] = 0;
        else address(attribute(tiled.o, n.buf));
    }
    const Ref rows_ = attribute(att.o, n.prompt_len);
    const long rows = number(rows_.o);
    need(rows >= 0 && rows <= capacity, "cache_prompt_len exceeds the prompt cache");
    char *key = PyByteArray_AS_STRING(x[1]);
    const bool same = memcmp(key, now, sizeof now) == 0;
    if (!same) memcpy(key, now, sizeof now);
    return PyLong_FromLong(same ? rows : -1 - rows);
}

template <PyObject *(*F)(Args), int N>
PyObject *call(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    try {
        arity(n, N);
        return F(args);
    } catch (Refused &) {
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}

// (handle of libsmh.so, the exception of failed calls)
PyObject *connect(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 2) { PyErr_SetString(PyExc_TypeError, "connect(handle, error)"); return nullptr; }
    void *lib = PyLong_AsVoidPtr(args[0]);
    if (lib == nullptr) return nullptr;
    bool ok = true;
    auto find = [&](auto &fn, const char *name) {
        fn = (std::decay_t<decltype(fn)>)dlsym(lib, name);
        if (fn == nullptr) ok = false;
    };
    find(api.last_error, "smh_last_error_string");
    find(api.matmul, "smh_q40_matmul");
    find(api.plan, "smh_q40_matmul_plan");
    find(api.dequant, "smh_q40_dequant");
    find(api.quantize, "smh_q40_quantize");
    find(api.quantize_t, "smh_q40_quantize_t");
    find(api.sample_counts, "smh_sample_topk_counts");
    find(api.sample_rowtemp, "smh_sample_topk_rowtemp");
    find(api.tree_step, "smh_tree_step");
    find(api.attn_bytes, "smh_attn_workspace_bytes");
    find(api.paged_bytes, "smh_paged_attn_workspace_bytes");
    find(api.shared_attn, "smh_shared_prefix_attn");
    find(api.paged_attn, "smh_paged_prefix_attn");
    if (!ok) { PyErr_SetString(PyExc_RuntimeError, "the library lacks an entry point: build it again"); return nullptr; }
    Py_XDECREF(smh_error);
    smh_error = args[1];
    Py_INCREF(smh_error);
    Py_RETURN_NONE;
}

#define OP(name, n) {#name, (PyCFunction)(void (*)(void))call<name, n>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"connect", (PyCFunction)(void (*)(void))connect, METH_FASTCALL, nullptr},
    OP(matmul_q40, 6), OP(deq_int40, 4), OP(q_int40, 1), OP(quantize_q40_t, 1), OP(sample_topk_counts, 6), OP(tree_step, 14),
    OP(shared_prefix_attn, 15), OP(paged_prefix_attn, 15), OP(layer_state, 2), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ops(void) {
    PyObject *m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddIntConstant(m, "layer_key_bytes", LAYER_WORDS * 8) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}

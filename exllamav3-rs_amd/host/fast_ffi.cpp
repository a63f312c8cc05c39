// exl3r._fast: the torch-tensor wrappers of exl3r/ffi.py in native code, for the calls that need no explanation.
//
// A decode call's kernel takes 2 to 4 us, and the same call through the Python wrapper took ~10 us of host time:
// a view per tensor to find its row stride, the current stream as an object, and 18 arguments through ctypes.
// Each function here takes its wrapper's arguments (all of them, in order), checks what the wrapper checks and
// makes the same C ABI call with the same arguments.  It returns the call's status, or None when anything is
// out of the ordinary -- a CPU tensor, a tensor subclass, a stream given, a layout beyond contiguous or 2-D, a
// failed check -- and the Python wrapper then does it all, with its errors.  Nothing is kept between calls.
#include <torch/csrc/autograd/python_variable.h>
#include <c10/hip/HIPStream.h>

#include <cstring>

#include "../../include/exl3r/rowops.h"

namespace {

struct Table
{
#define EXL3R_FN(name) decltype(&::name) name = nullptr
    EXL3R_FN(exl3r_rms_norm);
    EXL3R_FN(exl3r_rms_norm_res_in);
    EXL3R_FN(exl3r_silu_mul);
    EXL3R_FN(exl3r_gelu_mul);
    EXL3R_FN(exl3r_mul_sigmoid);
    EXL3R_FN(exl3r_gated_rms_norm);
    EXL3R_FN(exl3r_gated_rms_norm_had);
    EXL3R_FN(exl3r_rope);
    EXL3R_FN(exl3r_rope_table);
    EXL3R_FN(exl3r_rope_qg);
    EXL3R_FN(exl3r_rope_paged_kv);
    EXL3R_FN(exl3r_rope_paged_kv_had);
    EXL3R_FN(exl3r_argmax_sample);
    EXL3R_FN(exl3r_gumbel_sample);
    EXL3R_FN(exl3r_rms_norm_had);
    EXL3R_FN(exl3r_act_mul_had);
    EXL3R_FN(exl3r_embedding);
    EXL3R_FN(exl3r_embedding_rms_norm);
#undef EXL3R_FN
} T;

struct Decline {};   // thrown to hand the call to the Python wrapper

void need(bool ok)
{
    if (!ok) throw Decline{};
}

// A plain torch.Tensor (or Parameter) with storage on the GPU.
const at::Tensor& tensor(PyObject* o)
{
    need(THPVariable_CheckExact(o));
    const at::Tensor& t = THPVariable_Unpack(o);
    need(t.defined() && t.is_cuda() && t.has_storage() && t.layout() == at::kStrided);
    return t;
}
const at::Tensor* optional(PyObject* o) { return o == Py_None ? nullptr : &tensor(o); }

int code(const at::Tensor& t)
{
    switch (t.scalar_type())
    {
        case at::kFloat: return EXL3R_F32;
        case at::kHalf: return EXL3R_F16;
        case at::kBFloat16: return EXL3R_BF16;
        case at::kInt: return EXL3R_I32;
        case at::kLong: return EXL3R_I64;
        default: throw Decline{};
    }
}
int code(const at::Tensor* t, int none) { return t ? code(*t) : none; }
void* ptr(const at::Tensor& t) { return t.data_ptr(); }
void* ptr(const at::Tensor* t) { return t ? ptr(*t) : nullptr; }

float real(PyObject* o)
{
    need(PyFloat_CheckExact(o) || PyLong_CheckExact(o));
    const double v = PyFloat_AsDouble(o);
    if (PyErr_Occurred()) throw Decline{};
    return (float)v;
}
int64_t whole(PyObject* o)
{
    need(PyLong_CheckExact(o) || PyBool_Check(o));
    const long long v = PyLong_AsLongLong(o);
    if (PyErr_Occurred()) throw Decline{};
    return v;
}
int int32_of(PyObject* o)
{
    const int64_t v = whole(o);
    need(v >= INT32_MIN && v <= INT32_MAX);
    return (int)v;
}
bool flag(PyObject* o)
{
    need(PyBool_Check(o));
    return o == Py_True;
}
void* stream_of(const at::Tensor& t, PyObject* given)
{
    need(given == Py_None);
    return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// ffi._rows for the layouts it meets as a rule: contiguous, or 2-D with dense rows.
struct Rows
{
    int64_t rows, dim, ld;
    bool same(const Rows& o) const { return rows == o.rows && dim == o.dim; }
};
Rows rows_of(const at::Tensor& t)
{
    const int64_t d = t.dim();
    need(d >= 1 && t.numel() > 0);
    const int64_t dim = t.size(d - 1);
    if (d == 1)
    {
        return { 1, dim, dim };
    }
    if (t.is_contiguous()) return { t.numel() / dim, dim, dim };
    need(d == 2 && (dim == 1 || t.stride(1) == 1));
    const int64_t n = t.size(0);
    return { n, dim, n > 1 ? std::max(dim, t.stride(0)) : dim };
}

// The entry point's call without the interpreter lock, as ctypes makes it.
struct Unlocked
{
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};
template <class F>
PyObject* call(F&& f)
{
    int rc;
    {
        Unlocked u;
        rc = f();
    }
    return PyLong_FromLong(rc);
}

template <class F>
PyObject* guarded(Py_ssize_t given, Py_ssize_t wanted, F&& f)
{
    try
    {
        need(given == wanted);
        return f();
    }
    catch (const Decline&) {}
    catch (const std::exception&) {}
    PyErr_Clear();
    Py_RETURN_NONE;
}

#define EXL3R_PY(name, n) \
    PyObject* name##_body(PyObject* const* v); \
    PyObject* name(PyObject*, PyObject* const* v, Py_ssize_t k) { return guarded(k, n, [&] { return name##_body(v); }); } \
    PyObject* name##_body(PyObject* const* v)

// x, w, y, eps, constant_bias, constant_scale, stream
EXL3R_PY(rms_norm, 7)
{
    const auto &x = tensor(v[0]), &y = tensor(v[2]);
    const auto* w = optional(v[1]);
    const Rows rx = rows_of(x), ry = rows_of(y);
    need(rx.same(ry));
    const int xt = code(x), wt = code(w, EXL3R_F16), yt = code(y);
    const float eps = real(v[3]), cb = real(v[4]), cs = real(v[5]);
    void* s = stream_of(x, v[6]);
    return call([&] { return T.exl3r_rms_norm(ptr(x), xt, rx.ld, ptr(w), wt, ptr(y), yt, ry.ld, rx.rows, rx.dim, eps, cb, cs, s); });
}

// x, w, y, r, eps, constant_bias, constant_scale, stream
EXL3R_PY(rms_norm_res_in, 8)
{
    const auto &x = tensor(v[0]), &y = tensor(v[2]), &r = tensor(v[3]);
    const auto* w = optional(v[1]);
    const Rows rx = rows_of(x), ry = rows_of(y), rr = rows_of(r);
    need(rx.same(ry) && rx.same(rr));
    const int xt = code(x), wt = code(w, EXL3R_F16), yt = code(y), rt = code(r);
    const float eps = real(v[4]), cb = real(v[5]), cs = real(v[6]);
    void* s = stream_of(x, v[7]);
    return call([&] { return T.exl3r_rms_norm_res_in(ptr(x), xt, rx.ld, ptr(w), wt, ptr(y), yt, ry.ld, ptr(r), rt, rr.ld,
                                                     rx.rows, rx.dim, eps, cb, cs, s); });
}

// act (0 silu, 1 gelu, 2 x * sigmoid(y)), x, y, z, act_limit, stream
EXL3R_PY(act_mul, 6)
{
    const int act = int32_of(v[0]);
    const auto &x = tensor(v[1]), &y = tensor(v[2]), &z = tensor(v[3]);
    const Rows rx = rows_of(x), ry = rows_of(y), rz = rows_of(z);
    need(rx.same(ry) && rx.same(rz) && x.scalar_type() == y.scalar_type());
    const int xt = code(x), zt = code(z);
    const float limit = real(v[4]);
    void* s = stream_of(x, v[5]);
    return call([&] {
        if (act == 2) return T.exl3r_mul_sigmoid(ptr(x), ptr(y), xt, ptr(z), zt, rx.rows, rx.dim, rx.ld, ry.ld, rz.ld, s);
        return (act == 1 ? T.exl3r_gelu_mul : T.exl3r_silu_mul)(ptr(x), ptr(y), xt, ptr(z), zt, rx.rows, rx.dim, rx.ld, ry.ld,
                                                                 rz.ld, limit, s);
    });
}

// x, w, y, g, eps, constant_bias, w_groups, gate_first, gate_act, stream
EXL3R_PY(gated_rms_norm, 10)
{
    const auto &x = tensor(v[0]), &y = tensor(v[2]), &g = tensor(v[3]);
    const auto* w = optional(v[1]);
    const Rows rx = rows_of(x), ry = rows_of(y), rg = rows_of(g);
    const int groups = int32_of(v[6]);
    need(rx.same(ry) && rx.same(rg) && (!w || w->numel() == groups * rx.dim));
    const int xt = code(x), wt = code(w, EXL3R_F32), yt = code(y), gt = code(g);
    const float eps = real(v[4]), cb = real(v[5]);
    const int first = flag(v[7]), act = int32_of(v[8]);
    void* s = stream_of(x, v[9]);
    return call([&] { return T.exl3r_gated_rms_norm(ptr(x), xt, rx.ld, ptr(w), wt, groups, ptr(y), yt, ry.ld, ptr(g), gt, rg.ld,
                                                    rx.rows, rx.dim, eps, cb, first, act, s); });
}

// x, w, g, out, eps, pre_scale, y, constant_bias, w_groups, gate_first, gate_act | exact, had_scale, pre_rows, stream
EXL3R_PY(gated_rms_norm_had, 14)
{
    const auto &x = tensor(v[0]), &g = tensor(v[2]), &o = tensor(v[3]);
    const auto *w = optional(v[1]), *pre = optional(v[5]), *y = optional(v[6]);
    const Rows rx = rows_of(x), rg = rows_of(g), ro = rows_of(o);
    need(rx.same(rg) && rx.same(ro) && o.scalar_type() == at::kHalf);
    int64_t ldy = 0;
    if (y)
    {
        const Rows ry = rows_of(*y);
        need(ry.same(rx) && y->scalar_type() == at::kHalf);
        ldy = ry.ld;
    }
    const int groups = int32_of(v[8]);
    need(!w || w->numel() == groups * rx.dim);
    const int xt = code(x), wt = code(w, EXL3R_F32), gt = code(g);
    const float eps = real(v[4]), cb = real(v[7]), hs = real(v[11]);
    const int first = flag(v[9]), act = int32_of(v[10]);
    const int64_t pre_rows = whole(v[12]);
    void* s = stream_of(x, v[13]);
    return call([&] { return T.exl3r_gated_rms_norm_had(ptr(x), xt, rx.ld, ptr(w), wt, groups, ptr(g), gt, rg.ld, ptr(y), ldy,
                                                        ptr(pre), (int)pre_rows, ptr(o), ro.ld, rx.rows, rx.dim, eps, cb, first,
                                                        act, hs, s); });
}

// The q / k arguments that the RoPE wrappers share: (bsz, seq_len, heads, head_dim) with a dense innermost
// dimension and a collapsing batch stride.
struct Heads
{
    int64_t bsz, seq, h, hd, ts, hs;
};
Heads heads(const at::Tensor& t)
{
    need(t.dim() == 4 && t.stride(3) == 1 && t.numel() > 0);
    const Heads r{ t.size(0), t.size(1), t.size(2), t.size(3), t.stride(1), t.stride(2) };
    need(!(r.seq > 1 && r.bsz > 1 && t.stride(0) != r.seq * r.ts));
    return r;
}
const at::Tensor* int32_optional(PyObject* o)
{
    const auto* t = optional(o);
    need(!t || t->scalar_type() == at::kInt);
    return t;
}

// q, out_q, k, out_k, inv_freq, position, positions, q_norm, k_norm, norm_eps, norm_constant_bias, rope_mode,
// attn_factor, position_ids, stream, err_flag
EXL3R_PY(rope, 16)
{
    const auto &q = tensor(v[0]), &oq = tensor(v[1]), &inv = tensor(v[4]);
    const auto *k = optional(v[2]), *ok = optional(v[3]);
    const Heads Q = heads(q);
    need(oq.strides() == q.strides() && oq.sizes() == q.sizes());
    Heads K{ 0, 0, 0, 0, 0, 0 };
    if (k)
    {
        K = heads(*k);
        need(K.bsz == Q.bsz && K.seq == Q.seq && K.hd == Q.hd && ok && ok->strides() == k->strides());
    }
    const auto *pos = int32_optional(v[6]), *pid = int32_optional(v[13]), *qn = optional(v[7]), *kn = optional(v[8]),
               *err = optional(v[15]);
    const int position = int32_of(v[5]), mode = int32_of(v[11]), qt = code(q), nt = code(qn ? qn : kn, EXL3R_F16);
    const float eps = real(v[9]), cb = real(v[10]), attn = real(v[12]);
    void* s = stream_of(q, v[14]);
    if (inv.dim() > 1)
    {
        need(inv.dim() <= 3 && inv.scalar_type() == at::kFloat && inv.is_contiguous());
        need(inv.dim() == 2 || inv.size(0) >= Q.bsz);
        const int64_t rows = inv.size(-2), half = inv.size(-1), bs = inv.dim() == 3 ? rows * half : 0;
        return call([&] { return T.exl3r_rope_table(ptr(q), ptr(oq), Q.ts, Q.hs, (int)Q.h, ptr(k), ptr(ok), K.ts, K.hs, (int)K.h, qt,
                                                    Q.bsz, Q.seq, (int)Q.hd, (const float*)ptr(inv), rows, bs, (int)(half * 2),
                                                    position, (const int32_t*)ptr(pos), (const int32_t*)ptr(pid), ptr(qn), ptr(kn),
                                                    nt, eps, cb, mode, attn, (int32_t*)ptr(err), s); });
    }
    need(inv.dim() == 1);
    return call([&] { return T.exl3r_rope(ptr(q), ptr(oq), Q.ts, Q.hs, (int)Q.h, ptr(k), ptr(ok), K.ts, K.hs, (int)K.h, qt, Q.bsz,
                                          Q.seq, (int)Q.hd, (const float*)ptr(inv), (int)inv.size(0) * 2, position,
                                          (const int32_t*)ptr(pos), (const int32_t*)ptr(pid), ptr(qn), ptr(kn), nt, eps, cb, mode,
                                          attn, s); });
}

// inv_freq [R/2] of the wrappers that take no table of angles.
void frequencies(const at::Tensor& inv) { need(inv.dim() == 1 && inv.scalar_type() == at::kFloat); }

// qg, out_q, k, out_k, inv_freq, position, positions, q_norm, k_norm, norm_eps, norm_constant_bias, rope_mode,
// attn_factor, position_ids, stream
EXL3R_PY(rope_qg, 15)
{
    const auto &qg = tensor(v[0]), &oq = tensor(v[1]), &inv = tensor(v[4]);
    const auto *k = optional(v[2]), *ok = optional(v[3]);
    const Heads Q = heads(qg);
    const int64_t hd = Q.hd / 2;
    need(Q.hd % 2 == 0 && Q.hs == Q.hd && oq.dim() == 4 && oq.size(0) == Q.bsz && oq.size(1) == Q.seq && oq.size(2) == Q.h &&
         oq.size(3) == hd && oq.is_contiguous());
    Heads K{ 0, 0, 0, 0, 0, 0 };
    if (k)
    {
        K = heads(*k);
        need(K.bsz == Q.bsz && K.seq == Q.seq && K.hd == hd && ok && ok->strides() == k->strides());
    }
    frequencies(inv);
    const auto *pos = int32_optional(v[6]), *pid = int32_optional(v[13]), *qn = optional(v[7]), *kn = optional(v[8]);
    const int position = int32_of(v[5]), mode = int32_of(v[11]), qt = code(qg), nt = code(qn ? qn : kn, EXL3R_F16);
    const float eps = real(v[9]), cb = real(v[10]), attn = real(v[12]);
    void* s = stream_of(qg, v[14]);
    return call([&] { return T.exl3r_rope_qg(ptr(qg), Q.ts, ptr(oq), (int)Q.h, ptr(k), ptr(ok), K.ts, K.hs, (int)K.h, qt, Q.bsz, Q.seq,
                                             (int)hd, (const float*)ptr(inv), (int)inv.size(0) * 2, position,
                                             (const int32_t*)ptr(pos), (const int32_t*)ptr(pid), ptr(qn), ptr(kn), nt, eps, cb,
                                             mode, attn, s); });
}

// The paged append's arguments, from k_cache on.
struct Paged
{
    const at::Tensor &kc, &vc, &table, &lens;
};
Paged paged(PyObject* const* v, int64_t hk, int64_t hd)
{
    Paged p{ tensor(v[0]), tensor(v[1]), tensor(v[2]), tensor(v[3]) };
    need(p.kc.dim() == 4 && p.kc.sizes() == p.vc.sizes() && p.kc.size(2) == hk && p.kc.size(3) == hd && p.kc.is_contiguous() &&
         p.vc.is_contiguous());
    need(p.table.dim() == 2 && p.table.scalar_type() == at::kInt && p.lens.scalar_type() == at::kInt);
    return p;
}

// q, out_q, k, out_k, v, inv_freq, position, positions, q_norm, k_norm, norm_eps, norm_constant_bias, rope_mode,
// attn_factor, k_cache, v_cache, block_table, cache_seqlens, position_ids, err_flag, stream
// (a cs_table takes the Python wrapper)
EXL3R_PY(rope_paged_kv, 21)
{
    const auto &q = tensor(v[0]), &oq = tensor(v[1]), &k = tensor(v[2]), &vv = tensor(v[4]), &inv = tensor(v[5]);
    const auto* ok = optional(v[3]);
    const Heads Q = heads(q), K = heads(k), V = heads(vv);
    need(k.sizes() == vv.sizes() && K.bsz == Q.bsz && K.seq == Q.seq && K.hd == Q.hd);
    need(oq.strides() == q.strides() && oq.sizes() == q.sizes() && (!ok || (heads(*ok).hd == K.hd && ok->strides() == k.strides())));
    const Paged p = paged(v + 14, K.h, Q.hd);
    frequencies(inv);
    const auto *pos = int32_optional(v[7]), *pid = int32_optional(v[18]), *qn = optional(v[8]), *kn = optional(v[9]),
               *err = optional(v[19]);
    const int position = int32_of(v[6]), mode = int32_of(v[12]), qt = code(q), nt = code(qn ? qn : kn, EXL3R_F16);
    const float eps = real(v[10]), cb = real(v[11]), attn = real(v[13]);
    void* s = stream_of(q, v[20]);
    return call([&] { return T.exl3r_rope_paged_kv(ptr(q), ptr(oq), Q.ts, Q.hs, (int)Q.h, ptr(k), ptr(ok), K.ts, K.hs, ptr(vv), V.ts, V.hs,
                                                   (int)K.h, qt, Q.bsz, Q.seq, (int)Q.hd, (const float*)ptr(inv), (int)inv.size(0) * 2,
                                                   position, (const int32_t*)ptr(pos), (const int32_t*)ptr(pid), ptr(qn), ptr(kn), nt,
                                                   eps, cb, mode, attn, ptr(p.kc), ptr(p.vc), (int)p.kc.size(1), p.kc.size(0),
                                                   (const int32_t*)ptr(p.table), p.table.size(1), (const int32_t*)ptr(p.lens),
                                                   (int32_t*)ptr(err), nullptr, s); });
}

// as rope_paged_kv up to cache_seqlens, then q_post_scale, k_post_scale, v_post_scale, position_ids, err_flag, stream;
// rope_mode carries the exact flag
EXL3R_PY(rope_paged_kv_had, 24)
{
    const auto &q = tensor(v[0]), &oq = tensor(v[1]), &k = tensor(v[2]), &vv = tensor(v[4]), &inv = tensor(v[5]);
    const auto* ok = optional(v[3]);
    const Heads Q = heads(q), K = heads(k), V = heads(vv);
    need(k.sizes() == vv.sizes() && K.bsz == Q.bsz && K.seq == Q.seq && K.hd == Q.hd && Q.hs == Q.hd && K.hs == K.hd && V.hs == V.hd);
    need(oq.strides() == q.strides() && oq.sizes() == q.sizes());
    need(!ok || (ok->strides() == k.strides() && heads(*ok).hs == Q.hd));
    const Paged p = paged(v + 14, K.h, Q.hd);
    frequencies(inv);
    const auto *sq = optional(v[18]), *sk = optional(v[19]), *sv = optional(v[20]);
    const auto *pos = int32_optional(v[7]), *pid = int32_optional(v[21]), *qn = optional(v[8]), *kn = optional(v[9]),
               *err = optional(v[22]);
    const int position = int32_of(v[6]), mode = int32_of(v[12]), qt = code(q), nt = code(qn ? qn : kn, EXL3R_F16);
    const float eps = real(v[10]), cb = real(v[11]), attn = real(v[13]);
    void* s = stream_of(q, v[23]);
    return call([&] { return T.exl3r_rope_paged_kv_had(ptr(q), ptr(oq), Q.ts, (int)Q.h, ptr(k), ptr(ok), K.ts, ptr(vv), V.ts, (int)K.h, qt,
                                                       Q.bsz, Q.seq, (int)Q.hd, (const float*)ptr(inv), (int)inv.size(0) * 2, position,
                                                       (const int32_t*)ptr(pos), (const int32_t*)ptr(pid), ptr(qn), ptr(kn), nt, eps,
                                                       cb, mode, attn, ptr(p.kc), ptr(p.vc), (int)p.kc.size(1), p.kc.size(0),
                                                       (const int32_t*)ptr(p.table), p.table.size(1), (const int32_t*)ptr(p.lens),
                                                       (int32_t*)ptr(err), ptr(sq), ptr(sk), ptr(sv), nullptr, s); });
}

// logits, ids, max_logit, random (None: the argmax), stream
EXL3R_PY(sample, 5)
{
    const auto &x = tensor(v[0]), &ids = tensor(v[1]);
    const Rows r = rows_of(x);
    need(ids.scalar_type() == at::kLong && ids.numel() == r.rows);
    const int xt = code(x), max_logit = int32_of(v[2]);
    void* s = stream_of(x, v[4]);
    if (v[3] == Py_None)
        return call([&] { return T.exl3r_argmax_sample(ptr(x), xt, r.rows, r.dim, r.ld, max_logit, (int64_t*)ptr(ids), s); });
    const uint32_t random = (uint32_t)whole(v[3]);
    return call([&] { return T.exl3r_gumbel_sample(ptr(x), xt, r.rows, r.dim, r.ld, max_logit, random, (int64_t*)ptr(ids), s); });
}

// x, w, outs, pre_scales, eps, constant_bias, constant_scale, r, y, had_scale, rotate_x | exact, x_post_scale, stream
EXL3R_PY(rms_norm_had, 13)
{
    const auto& x = tensor(v[0]);
    const auto *w = optional(v[1]), *r = optional(v[7]), *y = optional(v[8]), *post = optional(v[11]);
    need(PyList_CheckExact(v[2]) && PyList_CheckExact(v[3]));
    const Py_ssize_t n = PyList_GET_SIZE(v[2]);
    need(n >= 1 && n <= 4 && PyList_GET_SIZE(v[3]) == n);
    const Rows rx = rows_of(x);
    const void* pre[4] = {};
    void* out[4] = {};
    int64_t ldo = 0;
    for (Py_ssize_t i = 0; i < n; ++i)
    {
        const auto& o = tensor(PyList_GET_ITEM(v[2], i));
        const Rows ro = rows_of(o);
        need(ro.same(rx) && o.scalar_type() == at::kHalf && (i == 0 || ro.ld == ldo));
        ldo = ro.ld;
        out[i] = ptr(o);
        pre[i] = ptr(optional(PyList_GET_ITEM(v[3], i)));
    }
    const int64_t ldr = r ? rows_of(*r).ld : 0, ldy = y ? rows_of(*y).ld : 0;
    need(!y || y->scalar_type() == at::kHalf);
    const int xt = code(x), wt = code(w, EXL3R_F16), rt = code(r, EXL3R_F16), rotate = int32_of(v[10]);
    const float eps = real(v[4]), cb = real(v[5]), cs = real(v[6]), hs = real(v[9]);
    void* s = stream_of(x, v[12]);
    return call([&] { return T.exl3r_rms_norm_had(ptr(x), xt, rx.ld, ptr(w), wt, ptr(r), rt, ldr, ptr(y), ldy, (int)n, pre, out, ldo,
                                                  rx.rows, rx.dim, eps, cb, cs, hs, rotate, ptr(post), s); });
}

// act, x, y, out, pre_scale, z, act_limit, had_scale, rotate flags, x_post_scale, y_post_scale, stream
EXL3R_PY(act_mul_had, 12)
{
    const int act = int32_of(v[0]), rotate = int32_of(v[8]);
    const auto &x = tensor(v[1]), &y = tensor(v[2]), &o = tensor(v[3]);
    const auto *pre = optional(v[4]), *z = optional(v[5]), *xp = optional(v[9]), *yp = optional(v[10]);
    const Rows rx = rows_of(x), ry = rows_of(y), ro = rows_of(o);
    need(rx.same(ry) && rx.same(ro) && x.scalar_type() == y.scalar_type() && o.scalar_type() == at::kHalf);
    int64_t ldz = 0;
    if (z)
    {
        const Rows rz = rows_of(*z);
        need(rz.same(rx) && z->scalar_type() == at::kHalf);
        ldz = rz.ld;
    }
    const int xt = code(x);
    const float limit = real(v[6]), hs = real(v[7]);
    void* s = stream_of(x, v[11]);
    return call([&] { return T.exl3r_act_mul_had(act, ptr(x), ptr(y), xt, rx.ld, ry.ld, ptr(z), ldz, ptr(pre), ptr(o), ro.ld, rx.rows,
                                                 rx.dim, limit, hs, rotate, ptr(xp), ptr(yp), s); });
}

// table, ids, out, err_flag, stream
EXL3R_PY(embedding, 5)
{
    const auto &t = tensor(v[0]), &ids = tensor(v[1]), &o = tensor(v[2]);
    const auto* err = optional(v[3]);
    need(t.dim() == 2);
    const int64_t n = ids.numel();
    const Rows ro = rows_of(o);
    need(ro.rows == n && ro.dim == t.size(1));
    const int tt = code(t), it = code(ids), ot = code(o);
    void* s = stream_of(t, v[4]);
    return call([&] { return T.exl3r_embedding(ptr(t), tt, t.size(0), t.size(1), t.stride(0), ptr(ids), it, n, ptr(o), ot, ro.ld,
                                               (int32_t*)ptr(err), s); });
}

// table, ids, h, w, y, eps, constant_bias, constant_scale, err_flag, stream
EXL3R_PY(embedding_rms_norm, 10)
{
    const auto &t = tensor(v[0]), &ids = tensor(v[1]), &y = tensor(v[4]);
    const auto *h = optional(v[2]), *w = optional(v[3]), *err = optional(v[8]);
    need(t.dim() == 2);
    const int64_t n = ids.numel();
    const Rows ry = rows_of(y);
    need(ry.rows == n && ry.dim == t.size(1));
    int64_t ldh = t.size(1);
    int ht = EXL3R_F32;
    if (h)
    {
        const Rows rh = rows_of(*h);
        need(rh.same(ry));
        ldh = rh.ld;
        ht = code(*h);
    }
    const int tt = code(t), it = code(ids), wt = code(w, EXL3R_F16), yt = code(y);
    const float eps = real(v[5]), cb = real(v[6]), cs = real(v[7]);
    void* s = stream_of(t, v[9]);
    return call([&] { return T.exl3r_embedding_rms_norm(ptr(t), tt, t.size(0), t.size(1), t.stride(0), ptr(ids), it, n, ptr(h), ht, ldh,
                                                        ptr(w), wt, ptr(y), yt, ry.ld, eps, cb, cs, (int32_t*)ptr(err), s); });
}

// bind(name, address): an entry point of the loaded library.
PyObject* bind(PyObject*, PyObject* const* v, Py_ssize_t k)
{
    const char* name = k == 2 ? PyUnicode_AsUTF8(v[0]) : nullptr;
    void* p = name ? PyLong_AsVoidPtr(v[1]) : nullptr;
    if (PyErr_Occurred()) return nullptr;
#define EXL3R_FN(n) if (name && !std::strcmp(name, #n)) { T.n = (decltype(T.n))p; Py_RETURN_TRUE; }
    EXL3R_FN(exl3r_rms_norm) EXL3R_FN(exl3r_rms_norm_res_in) EXL3R_FN(exl3r_silu_mul) EXL3R_FN(exl3r_gelu_mul)
    EXL3R_FN(exl3r_mul_sigmoid) EXL3R_FN(exl3r_gated_rms_norm) EXL3R_FN(exl3r_gated_rms_norm_had) EXL3R_FN(exl3r_rope)
    EXL3R_FN(exl3r_rope_table) EXL3R_FN(exl3r_rope_qg) EXL3R_FN(exl3r_rope_paged_kv) EXL3R_FN(exl3r_rope_paged_kv_had)
    EXL3R_FN(exl3r_argmax_sample) EXL3R_FN(exl3r_gumbel_sample) EXL3R_FN(exl3r_rms_norm_had) EXL3R_FN(exl3r_act_mul_had)
    EXL3R_FN(exl3r_embedding) EXL3R_FN(exl3r_embedding_rms_norm)
#undef EXL3R_FN
    Py_RETURN_FALSE;
}

#define EXL3R_DEF(name) { #name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr }
PyMethodDef methods[] = {
    EXL3R_DEF(bind), EXL3R_DEF(rms_norm), EXL3R_DEF(rms_norm_res_in), EXL3R_DEF(act_mul), EXL3R_DEF(gated_rms_norm),
    EXL3R_DEF(gated_rms_norm_had), EXL3R_DEF(rope), EXL3R_DEF(rope_qg), EXL3R_DEF(rope_paged_kv), EXL3R_DEF(rope_paged_kv_had),
    EXL3R_DEF(sample), EXL3R_DEF(rms_norm_had), EXL3R_DEF(act_mul_had), EXL3R_DEF(embedding), EXL3R_DEF(embedding_rms_norm),
    { nullptr, nullptr, 0, nullptr } };
PyModuleDef module = { PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr };

}  // namespace

// built_for: the torch and the interpreter it is compiled against, whose C++ and C ABIs it uses; the loader compares
// them with the ones that run.
PyMODINIT_FUNC PyInit__fast()
{
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "built_for", EXL3R_BUILT_FOR)) Py_CLEAR(m);
    return m;
}

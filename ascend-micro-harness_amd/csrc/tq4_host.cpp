// tq4_host.cpp -- the Python entry points' argument checks and launches in
// native code (CPython extension _tq4_host).
//
// A call of a few microseconds of GPU time spent 11 to 14 us of host time in
// Python: a dozen tensor checks, ctypes conversions and the stream lookup. Each
// function here takes the positional arguments of its tq4.py entry point,
// makes the same checks and calls the same C ABI entry (the address that
// ctypes resolved, so the library that tq4.py loaded). When a call is anything
// but plainly valid -- a tensor of another type, size, device or layout, a
// subclass, an argument that is not a plain number, an allocation that it does
// not make -- it returns None before any effect, and the Python code takes the
// call, with its own messages and conversions: what is refused there is refused
// there still. A status other than 0 goes back to Python as an int.
// The GIL is released around the launch, as ctypes does.
#include <ATen/ATen.h>
#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <cmath>
#include <cstring>

#include "../../include/tq4.h"
#include "../../include/tq4_kv4fp8.h"

namespace {

struct Abi {
    decltype(&tq4_reshape_and_cache_a8) reshape_and_cache_a8;
    decltype(&tq4_reshape_and_cache_bf16) reshape_and_cache_bf16;
    decltype(&tq4_reshape_scatter) reshape_scatter;
    decltype(&tq4_decode_auto_splits) decode_auto_splits;
    decltype(&tq4_paged_decode) paged_decode;
    decltype(&tq4_paged_decode_partials) paged_decode_partials;
    decltype(&tq4_splitk_combine) splitk_combine;
    decltype(&tq4_rms_reshape_and_cache) rms_reshape_and_cache;
    decltype(&tq4_icdf_quantize) icdf_quantize;
    decltype(&tq4_lloydmax_quantize) lloydmax_quantize;
    decltype(&tq4_kv4fp8_workspace_bytes) kv4fp8_workspace_bytes;
    decltype(&tq4_kv4fp8_decode) kv4fp8_decode;
    decltype(&tq4_kv4fp8_decode_raw_query) kv4fp8_decode_raw_query;
};
Abi g_abi;
bool g_bound = false;

constexpr uint32_t bit(at::ScalarType t) { return 1u << (int)t; }
constexpr uint32_t kBytes = bit(at::kChar) | bit(at::kByte);
constexpr uint32_t kF32 = bit(at::kFloat), kI32 = bit(at::kInt);
constexpr uint32_t kBf16 = bit(at::kBFloat16), kF16 = bit(at::kHalf);

// The tensor behind an argument, or nullptr: a plain contiguous device tensor
// of one of the dtypes.
const at::Tensor* plain(PyObject* o, uint32_t dtypes)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || t.layout() != at::kStrided || !t.has_storage() || !t.is_cuda())
        return nullptr;
    const int s = (int)t.scalar_type();
    if (s >= 32 || !((dtypes >> s) & 1u) || !t.is_contiguous()) return nullptr;
    return &t;
}

// Collects the arguments of one call; ok turns false at the first that is not
// plainly valid.
struct Args {
    PyObject* const* a;
    Py_ssize_t n, at = 0;
    bool ok = true;

    PyObject* next() { return at < n ? a[at++] : (ok = false, Py_None); }

    const at::Tensor* tensor(uint32_t dtypes)
    {
        const at::Tensor* t = plain(next(), dtypes);
        if (!t) ok = false;
        return t;
    }
    const at::Tensor* tensor_or_none(uint32_t dtypes)
    {
        PyObject* o = next();
        if (o == Py_None) return nullptr;
        const at::Tensor* t = plain(o, dtypes);
        if (!t) ok = false;
        return t;
    }
    // a whole number in [0, 2^31), or `none` for None
    uint32_t num(int64_t none = -1)
    {
        PyObject* o = next();
        if (o == Py_None && none >= 0) return (uint32_t)none;
        if (!PyLong_CheckExact(o)) return ok = false, 0u;
        int over = 0;
        const long long v = PyLong_AsLongLongAndOverflow(o, &over);
        if (over || v < 0 || v > 0x7fffffffll) return ok = false, 0u;
        return (uint32_t)v;
    }
    float real(double none)
    {
        PyObject* o = next();
        if (o == Py_None) return (float)none;
        if (!PyFloat_CheckExact(o)) return ok = false, 0.0f;
        return (float)PyFloat_AS_DOUBLE(o);
    }
    bool flag()
    {
        PyObject* o = next();
        if (o != Py_True && o != Py_False) ok = false;
        return o == Py_True;
    }
    // the stream argument: a torch stream, or None for the current one
    void* stream()
    {
        PyObject* o = next();
        if (!ok) return nullptr;
        if (o == Py_None) return (void*)c10::hip::getCurrentHIPStream().stream();
        PyObject* h = PyObject_GetAttrString(o, "cuda_stream");
        void* p = h && PyLong_CheckExact(h) ? PyLong_AsVoidPtr(h) : (ok = false, nullptr);
        Py_XDECREF(h);
        if (PyErr_Occurred()) {
            PyErr_Clear();
            ok = false;
        }
        return p;
    }
    bool need(bool c) { return ok = ok && c; }
};

void* ptr(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }
size_t nbytes(const at::Tensor* t) { return t ? (size_t)t->numel() * t->element_size() : 0; }
double inv_sqrt(int64_t d) { return 1.0 / std::sqrt((double)d); }
bool small(int64_t v) { return v >= 0 && v <= 0x7fffffffll; }

template <class F>
int unlocked(F&& f)
{
    int st;
    Py_BEGIN_ALLOW_THREADS st = f();
    Py_END_ALLOW_THREADS return st;
}

// f(Args) -> new reference, or nullptr for "take it in Python"; a C++
// exception before the launch is the same, unless Python code raised it (a
// dispatch mode in an allocation): that one goes to the caller.
template <class F>
PyObject* entry(PyObject* const* a, Py_ssize_t n, F&& f)
{
    try {
        Args g{a, n};
        if (g_bound) {
            if (PyObject* r = f(g)) return r;
            if (PyErr_Occurred()) return nullptr;
        }
    } catch (...) {
        if (PyErr_Occurred()) return nullptr;
    }
    Py_RETURN_NONE;
}

struct Shape3 {
    int64_t a, b, c;
};
bool shape3(const at::Tensor* t, Shape3& s)
{
    if (!t || t->dim() != 3) return false;
    s = {t->size(0), t->size(1), t->size(2)};
    return small(s.a) && small(s.b) && small(s.c) && t->numel() > 0;
}

// a * b, at most 2^63 - 1: more elements than any tensor holds, as Python's
// unbounded product would be.
uint64_t mul(uint64_t a, uint64_t b)
{
    uint64_t r;
    return __builtin_mul_overflow(a, b, &r) || r > (uint64_t)INT64_MAX ? (uint64_t)INT64_MAX : r;
}
bool at_least(const at::Tensor* t, uint64_t n) { return t && (uint64_t)t->numel() >= n; }

// The TQ4 cache of num_blocks pages (tq4.py _check_cache).
bool cache_ok(const at::Tensor* kc, const at::Tensor* vc, const at::Tensor* sc, uint64_t blocks,
              uint64_t heads, uint64_t block_size, uint64_t d)
{
    const uint64_t rows = mul(mul(blocks, heads), block_size);
    return at_least(kc, mul(rows, d) / 2) && at_least(vc, mul(rows, d) / 2) &&
           at_least(sc, mul(rows, 2));
}

// The pages of a pool given by its key cache alone (num_blocks None); -1 when
// they do not fit.
int64_t pool_pages(const at::Tensor* kc, const Shape3& s, uint32_t S)
{
    if (!kc || S == 0) return -1;
    const uint64_t pages = mul(kc->numel(), 2) / mul(mul(s.b, S), s.c);
    return small((int64_t)pages) ? (int64_t)pages : -1;
}

bool holds(const at::Tensor* t, int64_t n) { return !t || t->numel() >= n; }

// (is_a8, key, value, key_cache, value_cache, scale_cache, slot_mapping,
//  pi_signs, tables, block_size, num_blocks, tokens_per_core, inv_sqrt_len,
//  reuse_mode4_flags, stream)
PyObject* reshape_and_cache(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return entry(a, n, [](Args& g) -> PyObject* {
        const bool a8 = g.flag();
        const uint32_t in = a8 ? bit(at::kChar) : kBf16;
        const at::Tensor *k = g.tensor(in), *v = g.tensor(in), *kc = g.tensor(kBytes),
                         *vc = g.tensor(kBytes), *sc = g.tensor(kF32), *sl = g.tensor(kI32),
                         *pi = g.tensor_or_none(kF32),
                         *tb = g.tensor_or_none(a8 ? kBytes : kBf16 | bit(at::kShort));
        Shape3 s{};
        if (!g.need(shape3(k, s) && v && v->numel() == k->numel())) return nullptr;
        const uint32_t S = g.num(), P = g.num(pool_pages(kc, s, S)), tpc = g.num();
        const float isl = g.real(inv_sqrt(s.c));
        const bool reuse = g.flag();
        void* st = g.stream();
        if (!g.need(S > 0 && cache_ok(kc, vc, sc, P, s.b, S, s.c) && holds(sl, s.a) &&
                    holds(pi, s.c) && holds(tb, 32 * s.c)))
            return nullptr;
        auto call = [&](auto fn, auto* kp, auto* vp) {
            return unlocked([&] {
                return fn(st, kp, vp, (int8_t*)ptr(kc), (int8_t*)ptr(vc), (float*)ptr(sc),
                          (const int32_t*)ptr(sl), (const float*)ptr(pi),
                          (const int32_t*)ptr(tb), (uint32_t)s.a, (uint32_t)s.b, (uint32_t)s.c,
                          S, P, tpc, isl, reuse);
            });
        };
        return PyLong_FromLong(
            a8 ? call(g_abi.reshape_and_cache_a8, (const int8_t*)ptr(k), (const int8_t*)ptr(v))
               : call(g_abi.reshape_and_cache_bf16, (const uint16_t*)ptr(k),
                      (const uint16_t*)ptr(v)));
    });
}

// (key, value, key_cache, value_cache, scale_cache, slot_mapping, pi_signs,
//  cu_seqlens, launch_probe, num_requests, block_size, num_blocks, item_begin,
//  item_count, block_dim, inv_sqrt_len, stream)
PyObject* reshape_scatter(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return entry(a, n, [](Args& g) -> PyObject* {
        const at::Tensor *k = g.tensor(kBf16), *v = g.tensor(kBf16), *kc = g.tensor(kBytes),
                         *vc = g.tensor(kBytes), *sc = g.tensor(kF32), *sl = g.tensor(kI32),
                         *pi = g.tensor(kF32), *cu = g.tensor_or_none(kI32),
                         *probe = g.tensor_or_none(kI32);
        Shape3 s{};
        if (!g.need(shape3(k, s) && v && v->numel() == k->numel())) return nullptr;
        const int64_t all = cu ? cu->numel() - 1 : s.a;
        if (!g.need(small(all))) return nullptr;
        const uint32_t R = g.num(all), S = g.num(), P = g.num(pool_pages(kc, s, S));
        const uint32_t begin = g.num();
        const uint64_t every = (uint64_t)R * (uint64_t)s.b;
        if (!g.need(every <= 0x7fffffffull)) return nullptr;
        const uint32_t count = g.num((int64_t)every), grid = g.num();
        const float isl = g.real(inv_sqrt(s.c));
        void* st = g.stream();
        if (!g.need(S > 0 && cache_ok(kc, vc, sc, P, s.b, S, s.c) && holds(sl, s.a) &&
                    holds(pi, s.c) && holds(cu, (int64_t)R + 1) && holds(probe, 32) &&
                    (cu || R <= s.a)))
            return nullptr;
        return PyLong_FromLong(unlocked([&] {
            return g_abi.reshape_scatter(
                st, grid, (const uint16_t*)ptr(k), (const uint16_t*)ptr(v), (int8_t*)ptr(kc),
                (int8_t*)ptr(vc), (float*)ptr(sc), (const int32_t*)ptr(sl),
                (const float*)ptr(pi), (const int32_t*)ptr(cu), (int32_t*)ptr(probe), R,
                (uint32_t)s.b, (uint32_t)s.c, S, P, begin, count, isl);
        }));
    });
}

// The operands that paged_decode and paged_decode_partials share.
struct DecodeArgs {
    const at::Tensor *q, *kc, *vc, *sc, *bt, *cl, *pi;
    uint32_t Hkv, S, P;
    Shape3 s{};

    explicit DecodeArgs(Args& g)
        : q(g.tensor(kBf16)), kc(g.tensor(kBytes)), vc(g.tensor(kBytes)), sc(g.tensor(kF32)),
          bt(g.tensor(kI32)), cl(g.tensor(kI32)), pi(g.tensor_or_none(kF32)), Hkv(g.num()),
          S(g.num()), P(g.num())
    {
        g.need(shape3(q, s) && S > 0 && cache_ok(kc, vc, sc, P, Hkv, S, s.c) && bt && cl &&
               bt->dim() == 2 && bt->size(0) == s.a && small(bt->size(1)) &&
               cl->numel() == s.a && holds(pi, s.c));
    }
};

// (q, key_cache, value_cache, scale_cache, block_tables, context_lens, pi_signs,
//  num_kv_heads, block_size, num_blocks, out, workspace, gate, num_splits,
//  scale, inv_sqrt_len, output_stage, flags, stream) -> (status, out)
PyObject* paged_decode(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return entry(a, n, [](Args& g) -> PyObject* {
        DecodeArgs d(g);
        if (!g.ok) return nullptr;
        PyObject* out_obj = g.next();
        const at::Tensor* out = out_obj == Py_None ? nullptr : plain(out_obj, kBf16);
        const at::Tensor* ws = g.tensor_or_none(~0u);
        const at::Tensor* gate = g.tensor_or_none(kF32);
        uint32_t K = g.num();
        const float scale = g.real(inv_sqrt(d.s.c)), isl = g.real(inv_sqrt(d.s.c));
        const uint32_t stage = g.num(), flags = g.num();
        void* st = g.stream();
        const int64_t numel = d.q->numel();
        const bool rotated = flags & TQ4_DECODE_QUERY_ROTATED;
        if (!g.need((out_obj == Py_None || (out && out->numel() == numel)) &&
                    (!gate || gate->numel() == numel) &&
                    (d.pi || (stage == 0 && rotated)) && d.Hkv > 0 && d.bt->size(1) > 0))
            return nullptr;
        const uint32_t B = (uint32_t)d.s.a, mb = (uint32_t)d.bt->size(1);
        if (K == 0) K = g_abi.decode_auto_splits(B, d.Hkv, mb, d.S);
        if (!g.need(K <= 1 || ws)) return nullptr;
        at::Tensor fresh;
        if (!out) {
            fresh = at::empty_like(*d.q);
            out = &fresh;
        }
        const int rc = unlocked([&] {
            return g_abi.paged_decode(
                st, (const uint16_t*)ptr(d.q), (const int8_t*)ptr(d.kc), (const int8_t*)ptr(d.vc),
                (const float*)ptr(d.sc), (const int32_t*)ptr(d.bt), (const int32_t*)ptr(d.cl),
                (const float*)ptr(d.pi), (const float*)ptr(gate), ptr(ws), nbytes(ws),
                (uint16_t*)ptr(out), B, (uint32_t)d.s.b, d.Hkv, (uint32_t)d.s.c, d.S, d.P, mb, K,
                scale, isl, stage, flags);
        });
        if (rc != 0) return PyLong_FromLong(rc);
        if (fresh.defined()) return THPVariable_Wrap(fresh);
        Py_INCREF(out_obj);
        return out_obj;
    });
}

// (q, key_cache, value_cache, scale_cache, block_tables, context_lens, pi_signs,
//  num_kv_heads, block_size, num_blocks, num_splits, workspace, scale,
//  inv_sqrt_len, flags, stream)
PyObject* paged_decode_partials(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return entry(a, n, [](Args& g) -> PyObject* {
        DecodeArgs d(g);
        if (!g.ok) return nullptr;
        const uint32_t K = g.num();
        PyObject* ws_obj = g.next();
        const at::Tensor* ws = ws_obj == Py_None ? nullptr : plain(ws_obj, kF32);
        const float scale = g.real(inv_sqrt(d.s.c)), isl = g.real(inv_sqrt(d.s.c));
        const uint32_t flags = g.num();
        void* st = g.stream();
        const uint64_t need = mul(mul(mul(d.s.a, d.s.b), K), d.s.c + 4);
        if (!g.need(K > 0 && K <= TQ4_MAX_SPLITS && (ws_obj == Py_None || at_least(ws, need)) &&
                    (d.pi || (flags & TQ4_DECODE_QUERY_ROTATED))))
            return nullptr;
        at::Tensor fresh;
        if (!ws) {
            fresh = at::empty({d.s.a, d.s.b, (int64_t)K, d.s.c + 4},
                              d.q->options().dtype(at::kFloat));
            ws = &fresh;
        }
        const int rc = unlocked([&] {
            return g_abi.paged_decode_partials(
                st, (const uint16_t*)ptr(d.q), (const int8_t*)ptr(d.kc), (const int8_t*)ptr(d.vc),
                (const float*)ptr(d.sc), (const int32_t*)ptr(d.bt), (const int32_t*)ptr(d.cl),
                (const float*)ptr(d.pi), (float*)ptr(ws), nbytes(ws), (uint32_t)d.s.a,
                (uint32_t)d.s.b, d.Hkv, (uint32_t)d.s.c, d.S, d.P, (uint32_t)d.bt->size(1), K,
                scale, isl, flags);
        });
        if (rc != 0) return PyLong_FromLong(rc);
        if (fresh.defined()) return THPVariable_Wrap(fresh);
        Py_INCREF(ws_obj);
        return ws_obj;
    });
}

// (workspace, pi_signs, num_seqs, num_heads, head_size, num_splits, out, gate,
//  inv_sqrt_len, output_stage, stream)
PyObject* splitk_combine(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return entry(a, n, [](Args& g) -> PyObject* {
        const at::Tensor *ws = g.tensor(kF32), *pi = g.tensor_or_none(kF32);
        const uint32_t B = g.num(), Hq = g.num(), d = g.num(), K = g.num();
        PyObject* out_obj = g.next();
        const at::Tensor* out = out_obj == Py_None ? nullptr : plain(out_obj, kBf16);
        const at::Tensor* gate = g.tensor_or_none(kF32);
        if (!g.need(ws && d > 0)) return nullptr;
        const float isl = g.real(inv_sqrt(d));
        const uint32_t stage = g.num();
        void* st = g.stream();
        const uint64_t rows = (uint64_t)B * Hq;
        if (!g.need(rows > 0 && rows < (1ull << 31) && d <= 256 && K > 0 && K <= TQ4_MAX_SPLITS &&
                    at_least(ws, mul(rows * K, d + 4)) && (pi || stage == 0) &&
                    holds(pi, d) && (!gate || (uint64_t)gate->numel() == rows * d) &&
                    (out_obj == Py_None || (out && (uint64_t)out->numel() == rows * d))))
            return nullptr;
        at::Tensor fresh;
        if (!out) {
            fresh = at::empty({(int64_t)B, (int64_t)Hq, (int64_t)d},
                              ws->options().dtype(at::kBFloat16));
            out = &fresh;
        }
        const int rc = unlocked([&] {
            return g_abi.splitk_combine(st, (const float*)ptr(ws), (const float*)ptr(pi),
                                        (const float*)ptr(gate), (uint16_t*)ptr(out), B, Hq, d, K,
                                        isl, stage);
        });
        if (rc != 0) return PyLong_FromLong(rc);
        if (fresh.defined()) return THPVariable_Wrap(fresh);
        Py_INCREF(out_obj);
        return out_obj;
    });
}

// (key, value, key_cache, value_cache, scale_cache, slot_mapping, pi_signs,
//  block_size, num_blocks, inv_sqrt_len, block_dim, tokens_per_core, stream)
PyObject* rms_reshape_and_cache(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return entry(a, n, [](Args& g) -> PyObject* {
        const at::Tensor* k = g.tensor(kBf16 | kF16);
        if (!k) return nullptr;
        const at::Tensor *v = g.tensor(bit(k->scalar_type())), *kc = g.tensor(kBytes),
                         *vc = g.tensor(kBytes), *sc = g.tensor(kF32), *sl = g.tensor(kI32),
                         *pi = g.tensor(kF32);
        Shape3 s{};
        if (!g.need(shape3(k, s) && v && v->numel() == k->numel())) return nullptr;
        const uint32_t S = g.num(), P = g.num(pool_pages(kc, s, S));
        const float isl = g.real(inv_sqrt(s.c));
        const uint32_t grid = g.num(), tpc = g.num();
        void* st = g.stream();
        const uint64_t slots = (uint64_t)P * S, half = mul(mul(slots, s.b), s.c) / 2;
        if (!g.need(slots > 0 && at_least(kc, half) && at_least(vc, half) &&
                    at_least(sc, mul(slots, (2 * (uint64_t)s.b + 7) / 8 * 8)) &&
                    holds(sl, s.a) && holds(pi, s.c)))
            return nullptr;
        return PyLong_FromLong(unlocked([&] {
            return g_abi.rms_reshape_and_cache(
                st, k->scalar_type() == at::kBFloat16 ? 1 : 0, grid, ptr(k), ptr(v),
                (int8_t*)ptr(kc), (int8_t*)ptr(vc), (float*)ptr(sc), (const int32_t*)ptr(sl),
                (const float*)ptr(pi), nullptr, (uint32_t)s.a, (uint32_t)s.b, (uint32_t)s.c, S, P,
                tpc, isl);
        }));
    });
}

// The KV4/FP8 launch as tq4.py fused_decode_opt_launch fills it.
bool kv4_launch(tq4_kv4fp8_launch& L, uint64_t tokens, uint64_t heads, uint64_t kv_heads,
                uint32_t block_size, int64_t max_blocks, uint32_t splits, uint32_t heads_per_task,
                uint32_t fused_limit, float scale, float isl, uint32_t stage, uint32_t element,
                bool raw, uint32_t num_blocks)
{
    if (kv_heads == 0 || heads < kv_heads || heads_per_task == 0 || splits == 0 || splits > 8 ||
        !small(max_blocks))
        return false;
    const uint64_t group = heads / kv_heads;
    const uint64_t chunk = heads_per_task < group ? heads_per_task : group;
    const uint64_t tasks = mul(mul(mul(tokens, kv_heads), splits), (group + chunk - 1) / chunk);
    if (tasks == 0 || tasks > 0x7fffffffull || mul(tokens, heads) > 0x7fffffffull) return false;
    const uint64_t tpb = (tasks + 31) / 32, grid = (tasks + tpb - 1) / tpb;
    std::memset(&L, 0, sizeof L);
    L.grid = (uint32_t)grid;
    L.tokens = (uint32_t)tokens;
    L.heads = (uint32_t)heads;
    L.kv_heads = (uint32_t)kv_heads;
    L.head_size = 256;
    L.block_size = block_size;
    L.max_blocks = (uint32_t)max_blocks;
    L.splits = splits;
    L.heads_per_task = heads_per_task;
    L.tasks_per_block = (uint32_t)tpb;
    L.reduce_tasks_per_block = (uint32_t)((tokens * heads + grid - 1) / grid);
    L.fused_context_limit = fused_limit;
    L.scale = scale;
    L.inv_sqrt_len = isl;
    if (raw) L.prologue_vectors_per_block = L.reduce_tasks_per_block;
    L.output_stage = stage;
    L.element_type = element;
    L.probe_page = 0xFFFFFFFFu;
    L.num_blocks = num_blocks;
    return true;
}

// (raw, query, pi_signs, key_cache, value_cache, scales, block_table,
//  context_lens, kv_heads, block_size, num_blocks, gate, output_stage,
//  query_out, out, out_is_bf16, workspace, splits, heads_per_task,
//  fused_context_limit, scale, inv_sqrt_len, stream)
PyObject* kv4fp8_decode(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return entry(a, n, [](Args& g) -> PyObject* {
        const bool raw = g.flag();
        const at::Tensor* q = g.tensor(raw ? kF16 | kBf16 : kF32);
        if (!q) return nullptr;
        const at::Tensor *pi = g.tensor_or_none(kF32), *kc = g.tensor(kBytes),
                         *vc = g.tensor(kBytes), *sc = g.tensor(kF32), *bt = g.tensor(kI32),
                         *cl = g.tensor(kI32);
        const uint32_t H = g.num(), S = g.num(), P = g.num();
        const uint32_t half = raw ? bit(q->scalar_type()) : kF16 | kBf16;
        const at::Tensor* gate = g.tensor_or_none(half);
        const uint32_t stage = g.num();
        const at::Tensor* q_out = g.tensor_or_none(kF32);
        PyObject* out_obj = g.next();
        const at::Tensor* out = out_obj == Py_None ? nullptr : plain(out_obj, half);
        const bool want_bf16 = g.flag();
        const at::Tensor* ws = g.tensor(~0u);
        const uint32_t splits = g.num(), hpt = g.num(), limit = g.num();
        const float scale = g.real(1.0 / 16), isl = g.real(1.0 / 16);
        void* st = g.stream();
        Shape3 s{};
        if (!g.need(shape3(q, s) && s.c == 256 && H > 0 && S > 0 && P > 0)) return nullptr;
        const uint64_t rows = (uint64_t)P * S;
        const int64_t numel = q->numel();
        if (!g.need(at_least(kc, mul(mul(rows, H), 128)) && at_least(vc, mul(mul(rows, H), 128)) &&
                    at_least(sc, mul(rows, 8)) && bt && cl && bt->dim() == 2 && bt->size(0) == s.a &&
                    cl->numel() == s.a && (!raw || (pi && pi->numel() >= 256)) &&
                    (!gate || gate->numel() == numel) && (!q_out || q_out->numel() == numel) &&
                    (out_obj == Py_None || (out && out->numel() == numel))))
            return nullptr;
        const at::ScalarType type = raw   ? q->scalar_type()
                                    : out ? out->scalar_type()
                                          : (want_bf16 ? at::kBFloat16 : at::kHalf);
        tq4_kv4fp8_launch L;
        if (!kv4_launch(L, s.a, s.b, H, S, bt->size(1), splits, hpt, limit, scale, isl,
                        raw ? stage : 0u, type == at::kBFloat16 ? 1u : 0u, raw, P))
            return nullptr;
        if (g_abi.kv4fp8_workspace_bytes(&L) == 0) return nullptr;
        L.workspace_bytes = nbytes(ws);
        at::Tensor fresh;
        if (!out) {
            fresh = at::empty_like(*q, q->options().dtype(type));
            out = &fresh;
        }
        tq4_kv4fp8_raw_query_buffers r{};
        r.raw_query = raw ? ptr(q) : nullptr;
        r.pi_signs = ptr(pi);
        r.gate = ptr(gate);
        tq4_kv4fp8_buffers& b = r.decode;
        b.query = raw ? ptr(q_out) : ptr(q);
        b.key = ptr(kc);
        b.value = ptr(vc);
        b.scales = ptr(sc);
        b.block_table = ptr(bt);
        b.context_lengths = ptr(cl);
        b.workspace = ptr(ws);
        b.output = ptr(out);
        const int rc = unlocked([&] {
            return raw ? g_abi.kv4fp8_decode_raw_query(st, &L, &r) : g_abi.kv4fp8_decode(st, &L, &b);
        });
        if (rc != 0) return PyLong_FromLong(rc);
        if (fresh.defined()) return THPVariable_Wrap(fresh);
        Py_INCREF(out_obj);
        return out_obj;
    });
}

// (x, out, stream)
PyObject* icdf_quantize(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return entry(a, n, [](Args& g) -> PyObject* {
        const at::Tensor* x = g.tensor(kF16 | kBf16);
        if (!g.need(x && g.next() == Py_None && x->numel() > 0 && x->numel() % 1024 == 0 &&
                    small(x->numel() / 1024)))
            return nullptr;
        void* st = g.stream();
        if (!g.ok) return nullptr;
        at::Tensor out = at::empty({x->numel() / 2}, x->options().dtype(at::kByte));
        const int rc = unlocked([&] {
            return g_abi.icdf_quantize(st, x->scalar_type() == at::kBFloat16 ? 1 : 0,
                                       (const uint16_t*)ptr(x), (uint8_t*)out.data_ptr(),
                                       (uint32_t)(x->numel() / 1024));
        });
        return rc != 0 ? PyLong_FromLong(rc) : THPVariable_Wrap(out);
    });
}

// (src, bits, mode, dst, codes, stream) -> (dst, codes)
PyObject* lloydmax_quantize(PyObject*, PyObject* const* a, Py_ssize_t n)
{
    return entry(a, n, [](Args& g) -> PyObject* {
        const at::Tensor* x = g.tensor(~0u);
        const uint32_t bits = g.num(), mode = g.num();
        if (!g.need(x && (bits == 2 || bits == 4) && mode <= 5 && mode != 3 &&
                    x->scalar_type() == (mode >= 4 ? at::kByte : at::kFloat) &&
                    g.next() == Py_None && g.next() == Py_None))
            return nullptr;
        void* st = g.stream();
        const int64_t count = mode >= 4 ? x->numel() * 8 / bits : x->numel();
        if (!g.need(count > 0 && small(count))) return nullptr;
        at::Tensor codes;
        if (mode <= 2) codes = at::empty({count * bits / 8}, x->options().dtype(at::kByte));
        at::Tensor dst = at::empty({count}, x->options().dtype(at::kFloat));
        const int rc = unlocked([&] {
            return g_abi.lloydmax_quantize(
                st, ptr(x), (float*)dst.data_ptr(),
                codes.defined() ? (uint8_t*)codes.data_ptr() : nullptr, nullptr, bits, mode,
                (uint32_t)count, 1);
        });
        if (rc != 0) return PyLong_FromLong(rc);
        PyObject* d = THPVariable_Wrap(dst);
        PyObject* c = codes.defined() ? THPVariable_Wrap(codes) : (Py_INCREF(Py_None), Py_None);
        PyObject* t = d && c ? PyTuple_Pack(2, d, c) : nullptr;
        Py_XDECREF(d);
        Py_XDECREF(c);
        return t;
    });
}

// bind({name: address}) -- the loaded library's entries
PyObject* bind(PyObject*, PyObject* arg)
{
    if (!PyDict_Check(arg)) return PyErr_Format(PyExc_TypeError, "bind takes a dict");
    struct {
        const char* name;
        void** to;
    } const all[] = {
        {"tq4_reshape_and_cache_a8", (void**)&g_abi.reshape_and_cache_a8},
        {"tq4_reshape_and_cache_bf16", (void**)&g_abi.reshape_and_cache_bf16},
        {"tq4_reshape_scatter", (void**)&g_abi.reshape_scatter},
        {"tq4_decode_auto_splits", (void**)&g_abi.decode_auto_splits},
        {"tq4_paged_decode", (void**)&g_abi.paged_decode},
        {"tq4_paged_decode_partials", (void**)&g_abi.paged_decode_partials},
        {"tq4_splitk_combine", (void**)&g_abi.splitk_combine},
        {"tq4_rms_reshape_and_cache", (void**)&g_abi.rms_reshape_and_cache},
        {"tq4_icdf_quantize", (void**)&g_abi.icdf_quantize},
        {"tq4_lloydmax_quantize", (void**)&g_abi.lloydmax_quantize},
        {"tq4_kv4fp8_workspace_bytes", (void**)&g_abi.kv4fp8_workspace_bytes},
        {"tq4_kv4fp8_decode", (void**)&g_abi.kv4fp8_decode},
        {"tq4_kv4fp8_decode_raw_query", (void**)&g_abi.kv4fp8_decode_raw_query},
    };
    for (const auto& e : all) {
        PyObject* v = PyDict_GetItemString(arg, e.name);
        void* p = v ? PyLong_AsVoidPtr(v) : nullptr;
        if (!p) return PyErr_Format(PyExc_KeyError, "bind: no address for %s", e.name);
        *e.to = p;
    }
    g_bound = true;
    Py_RETURN_NONE;
}

#define TQ4_FAST(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {TQ4_FAST(reshape_and_cache),
                          TQ4_FAST(reshape_scatter),
                          TQ4_FAST(paged_decode),
                          TQ4_FAST(paged_decode_partials),
                          TQ4_FAST(splitk_combine),
                          TQ4_FAST(rms_reshape_and_cache),
                          TQ4_FAST(kv4fp8_decode),
                          TQ4_FAST(icdf_quantize),
                          TQ4_FAST(lloydmax_quantize),
                          {"bind", bind, METH_O, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_tq4_host",
                       "Native argument checks and launches of tq4.py.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tq4_host(void)
{
    PyObject* m = PyModule_Create(&kModule);
    // the torch whose headers this was built with: tq4.py binds no other
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0) Py_CLEAR(m);
    return m;
}

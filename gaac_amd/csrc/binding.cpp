// Python calls of the library's entry points (include/gaac_hip.h): gaac_amd._binding.<entry point>(arguments), raising RuntimeError with the
// library's message where an entry point returns non-zero.  Tensors are handed over as they are; a host tensor raises.  A function in the place of
// an address (the stream) is called for it once the arguments before it have been looked at: without a GPU, a host tensor is what the error names.
// What it is for: a launch has up to 47 arguments, half of them tensors.  Through ctypes, with is_cuda and data_ptr() called from Python for each
// tensor, attention() costs the host 14 us, more than the kernel takes over a short context, and a step of append and attention 24; with the
// arguments converted here 9 and 15, made here as a whole (below) 7 and 12.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty.h>
#include <algorithm>
#include <exception>
#include <tuple>
#include <type_traits>
#include <utility>
#include "../../include/gaac_hip.h"

namespace {

const char* (*g_last_error)() = nullptr;

// One argument; false with a Python error set.  Numbers convert as ctypes converts them: anything with __index__, cut to the type's bits.
bool convert(PyObject* o, void*& v) {
  if (o == Py_None) { v = nullptr; return true; }
  if (THPVariable_Check(o)) {
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda()) {
      PyErr_SetString(PyExc_RuntimeError, "gaac_amd kernels need device tensors (got a CPU tensor): there is no CPU path");
      return false;
    }
    v = t.data_ptr();
    return true;
  }
  if (PyCallable_Check(o)) {
    PyObject* r = PyObject_CallNoArgs(o);
    const bool ok = r != nullptr && PyLong_Check(r) && convert(r, v);
    if (r != nullptr && !PyLong_Check(r)) PyErr_SetString(PyExc_TypeError, "expected a function that returns an address");
    Py_XDECREF(r);
    return ok;
  }
  if (!PyLong_Check(o)) { PyErr_Format(PyExc_TypeError, "expected a tensor, an address or None, got %s", Py_TYPE(o)->tp_name); return false; }
  v = reinterpret_cast<void*>(static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(o)));
  return !PyErr_Occurred();
}
bool convert(PyObject* o, long& v) {
  if (PyFloat_Check(o)) { PyErr_SetString(PyExc_TypeError, "expected an integer, got float"); return false; }
  v = static_cast<long>(PyLong_AsUnsignedLongMask(o));
  return v != -1 || !PyErr_Occurred();
}
bool convert(PyObject* o, int& v) {
  long l;
  if (!convert(o, l)) return false;
  v = static_cast<int>(l);
  return true;
}
bool convert(PyObject* o, float& v) {
  const double d = PyFloat_AsDouble(o);
  v = static_cast<float>(d);
  return d != -1.0 || !PyErr_Occurred();
}

template <typename A> using Held = std::conditional_t<std::is_pointer_v<A>, void*, A>;      // what an argument is converted to
template <typename A> A passed(Held<A> v) { if constexpr (std::is_pointer_v<A>) return static_cast<A>(v); else return v; }

template <typename... A, size_t... I>
PyObject* invoke(const char* name, int (*fn)(A...), PyObject* const* args, std::index_sequence<I...>) {
  std::tuple<Held<A>...> held;
  try {
    if (!(convert(args[I], std::get<I>(held)) && ...)) return nullptr;
  } catch (const std::exception& e) {      // a tensor without memory
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = fn(passed<A>(std::get<I>(held))...);
  Py_END_ALLOW_THREADS
  if (rc != 0) {
    PyErr_Format(PyExc_RuntimeError, "%s failed (%d): %s", name, rc, g_last_error());
    return nullptr;
  }
  Py_RETURN_NONE;
}
template <typename... A>
PyObject* invoke(const char* name, int (*fn)(A...), PyObject* const* args, Py_ssize_t n) {
  if (fn == nullptr) { PyErr_SetString(PyExc_RuntimeError, "gaac_amd._binding.bind has not been called"); return nullptr; }
  if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
    PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, static_cast<Py_ssize_t>(sizeof...(A)), n);
    return nullptr;
  }
  return invoke(name, fn, args, std::index_sequence_for<A...>{});
}

#define GAAC_ENTRY_POINTS(X)                                                                                                              \
  X(gaac_wait_words) X(gaac_page_finish) X(gaac_cache_check)                                                                              \
  X(gaac_exponent_hist) X(gaac_bases_from_hist) X(gaac_encode_tiles) X(gaac_compact) X(gaac_tile_scan) X(gaac_page_pack)                  \
  X(gaac_row_offsets) X(gaac_decode_tiles) X(gaac_prompt_store) X(gaac_cache_prefill) X(gaac_attn_split) X(gaac_attn_combine)             \
  X(gaac_cache_append)                                                                                                                    \
  X(gaac_paged_store) X(gaac_paged_free) X(gaac_paged_release) X(gaac_paged_decode) X(gaac_paged_attn) X(gaac_bf16_attn)                  \
  X(gaac_attn_fused) X(gaac_attn_fused_static) X(gaac_static_init) X(gaac_static_reset) X(gaac_static_flags) X(gaac_attn_launch)
#define X(name)                                            \
  decltype(&::name) p_##name = nullptr;                    \
  PyObject* py_##name(PyObject*, PyObject* const* args, Py_ssize_t n) { return invoke(#name, p_##name, args, n); }
GAAC_ENTRY_POINTS(X)
#undef X

// ---------------------------------------------------------------------------------------------------- whole calls
// What CompressedKVCache, Codec and attention() do on each call, where the arguments are what a program usually has: plain tensors on the device, in the
// layout that the kernels read.  None where they are not, before anything is launched: the Python code of the call, which has the checks and messages,
// takes over, as it does where there is no binding.  Host us a call, Python / here: attention 9.0 / 7.2, over the slot cache 8.5 / 6.9, append 6.2 / 4.8 (a launch
// alone takes 3), a page's decoder 5.4 / 4.3; 4096 tokens x 8 heads encoded and expanded again 37.9 / 30.2, a prompt of 777 tokens 21.7 / 18.4.
struct Otherwise {};      // thrown: not such arguments

struct Refs {             // objects that are held until the call has been made (another thread may replace an attribute meanwhile)
  PyObject* r[64];
  int n = 0;
  ~Refs() { while (n > 0) Py_DECREF(r[--n]); }
  PyObject* operator()(PyObject* o, PyObject* name) {
    PyObject* p = PyObject_GetAttr(o, name);
    if (p == nullptr) throw Otherwise{};
    return r[n++] = p;
  }
};
#define GAAC_NAMES(X)                                                                                                                        \
  X(k) X(v) X(sm) X(codes) X(flags) X(tile_off) X(ovf) X(head_start) X(ovf_head_start) X(base3) X(base4) X(tail) X(ovf_used) X(ovf_cap)     \
  X(n_kv) X(cap) X(S) X(H) X(kind) X(tail_len) X(overflow) X(n_slots) X(per_sequence_bases) X(_scan) X(pm) X(pl) X(pa) X(epoch) X(rows) X(nslot)
#define X(name) PyObject* n_##name = nullptr;
GAAC_NAMES(X)
#undef X

constexpr long DIM = 128, TILE = 16, CODE_BYTES = 48, TILE_ESCAPES = 1280, HIST_BYTES = 256 * 64 * 4 + 32;

const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) throw Otherwise{};
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda()) throw Otherwise{};
  return t;
}
template <typename P> P* address(PyObject* o) { return static_cast<P*>(tensor(o).data_ptr()); }
long number(PyObject* o) {
  if (!PyLong_CheckExact(o)) throw Otherwise{};
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) throw Otherwise{};
  return v;
}
void* stream_of(PyObject* o) {
  void* v = nullptr;
  if (!convert(o, v)) throw Otherwise{};
  return v;
}
bool is_rows(const at::Tensor& t, int dims) { return t.dim() == dims && t.scalar_type() == at::kBFloat16 && t.size(dims - 1) == DIM; }
// rows_in_place: whether the encoder can read the rows where they lie
bool in_place(const at::Tensor& t, int head_dim, int row_dim, long& hs, long& rs) {
  hs = t.size(head_dim) > 1 ? t.stride(head_dim) : 0;
  rs = t.size(row_dim) > 1 ? t.stride(row_dim) : DIM;
  return t.stride(2) == 1 && rs >= DIM && rs % 8 == 0 && hs % 8 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}
at::Tensor bytes(const at::Tensor& like, at::IntArrayRef shape, at::ScalarType type = at::kByte) { return at::empty(shape, at::TensorOptions().dtype(type).device(like.device())); }
at::Tensor host_words(long n) { return at::empty({n}, at::TensorOptions().dtype(at::kInt).pinned_memory(true)); }

struct Failed { const char* name; int rc; };      // thrown: an entry point's refusal, with the GIL held
void must(const char* name, int rc) { if (rc != 0) throw Failed{name, rc}; }
template <typename F> PyObject* whole_call(Py_ssize_t given, Py_ssize_t n, F body) {
  if (given != n) { PyErr_Format(PyExc_TypeError, "expected %zd arguments (%zd given)", n, given); return nullptr; }
  if (p_gaac_wait_words == nullptr) { PyErr_SetString(PyExc_RuntimeError, "gaac_amd._binding.bind has not been called"); return nullptr; }
  try {
    return body();
  } catch (const Otherwise&) {
  } catch (const Failed& f) {
    PyErr_Format(PyExc_RuntimeError, "%s failed (%d): %s", f.name, f.rc, g_last_error());
    return nullptr;
  } catch (const std::exception&) {      // no memory, a tensor without any: Python meets the same and raises its own type (nothing is stored until a call's last launch)
  }
  PyErr_Clear();
  Py_RETURN_NONE;
}
struct NoGil {      // (taken back also where an exception leaves: a tensor without an address of its own, as in vmap)
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};
template <typename F> int without_gil(F f) {
  const NoGil released;
  return f();
}
PyObject* numbers(const at::Tensor& words) {
  const long n = words.numel();
  const int* w = static_cast<const int*>(words.data_ptr());
  PyObject* l = PyList_New(n);
  for (long i = 0; l != nullptr && i < n; ++i) {
    PyObject* o = PyLong_FromLong(w[i]);
    if (o == nullptr) { Py_DECREF(l); return nullptr; }
    PyList_SET_ITEM(l, i, o);
  }
  return l;
}

// attend(K, V, n_kv, ws, q, slots or None, SL or None, S_pad, scale, nsplit, tail_len or None, S_all, stream) -> out like q [B, n_q, 128]
PyObject* attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return whole_call(n, 13, [&]() -> PyObject* {
    Refs get;
    const at::Tensor& q = tensor(a[4]);
    const long n_kv = number(a[2]), S_pad = number(a[7]), nsplit = number(a[9]), S_all = number(a[11]);
    if (!is_rows(q, 3) || !q.is_contiguous() || n_kv <= 0 || q.size(1) % n_kv != 0 || q.size(1) < n_kv || q.size(1) / n_kv > 16 || !PyFloat_CheckExact(a[8])) throw Otherwise{};
    const long B = q.size(0), n_q = q.size(1);
    const bool tail = a[10] != Py_None;
    const int* slots = nullptr;
    if (a[5] != Py_None) {
      const at::Tensor& s = tensor(a[5]);
      if (s.dim() != 1 || s.size(0) != B || s.scalar_type() != at::kInt || !s.is_contiguous()) throw Otherwise{};
      slots = static_cast<const int*>(s.data_ptr());
    }
    if (number(get(a[3], n_rows)) != B * n_q || number(get(a[3], n_nslot)) != nsplit || B == 0) throw Otherwise{};
    struct Store { uint8_t *sm, *cd; int *fl, *to; uint8_t* ov; int* hs; uint8_t *b3, *b4; void* tail; long nb; } st[2];
    for (int i = 0; i < 2; ++i) {
      PyObject* o = a[i];
      Store& s = st[i];
      s.sm = address<uint8_t>(get(o, n_sm)); s.cd = address<uint8_t>(get(o, n_codes)); s.fl = address<int>(get(o, n_flags)); s.to = address<int>(get(o, n_tile_off));
      s.ov = address<uint8_t>(get(o, n_ovf)); s.hs = address<int>(get(o, tail ? n_head_start : n_ovf_head_start));
      PyObject* b3 = get(o, n_base3);
      s.nb = tensor(b3).size(0); s.b3 = address<uint8_t>(b3); s.b4 = address<uint8_t>(get(o, n_base4));
      s.tail = tail ? address<void>(get(o, n_tail)) : nullptr;
    }
    const int* SL = a[6] == Py_None ? nullptr : address<int>(a[6]);
    const int* TL = tail ? address<int>(a[10]) : nullptr;
    auto *pm = address<unsigned long long>(get(a[3], n_pm)), *pl = address<unsigned long long>(get(a[3], n_pl)), *pa = address<unsigned long long>(get(a[3], n_pa));
    unsigned* epoch = address<unsigned>(get(a[3], n_epoch));
    const float scale = static_cast<float>(PyFloat_AS_DOUBLE(a[8]));
    void* stream = stream_of(a[12]);
    at::Tensor out = bytes(q, {B, n_q, DIM}, at::kBFloat16);
    must("gaac_attn_fused", without_gil([&] {
      return p_gaac_attn_fused(st[0].sm, st[0].cd, st[0].fl, st[0].to, st[0].ov, st[0].hs, st[0].b3, st[0].b4, st[1].sm, st[1].cd, st[1].fl, st[1].to, st[1].ov, st[1].hs,
                               st[1].b3, st[1].b4, q.data_ptr(), slots, static_cast<int>(B), static_cast<int>(n_q), static_cast<int>(n_kv), SL, static_cast<int>(S_pad), scale,
                               static_cast<int>(nsplit), static_cast<int>(st[0].nb), st[0].tail, st[1].tail, TL, tail ? static_cast<int>(TILE) : 0, static_cast<int>(S_all), pm, pl, pa,
                               epoch, out.data_ptr(), stream);
    }));
    return THPVariable_Wrap(out);
  });
}

struct CacheStore { void* tail; uint8_t *b3, *b4, *sm, *cd; int* fl; uint8_t* ov; int *to, *used; };
CacheStore cache_store(Refs& get, PyObject* o) {
  return {address<void>(get(o, n_tail)), address<uint8_t>(get(o, n_base3)), address<uint8_t>(get(o, n_base4)), address<uint8_t>(get(o, n_sm)), address<uint8_t>(get(o, n_codes)),
          address<int>(get(o, n_flags)), address<uint8_t>(get(o, n_ovf)), address<int>(get(o, n_tile_off)), address<int>(get(o, n_ovf_used))};
}

// token_append(cache, slots, k, v, stream) -> True
PyObject* token_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return whole_call(n, 5, [&]() -> PyObject* {
    Refs get;
    const at::Tensor &slots = tensor(a[1]), &k = tensor(a[2]), &v = tensor(a[3]);
    const long n_kv = number(get(a[0], n_n_kv)), cap = number(get(a[0], n_cap));
    if (!is_rows(k, 3) || !is_rows(v, 3) || k.sizes() != v.sizes() || k.size(1) != n_kv || !k.is_contiguous() || !v.is_contiguous()) throw Otherwise{};
    if (slots.scalar_type() != at::kInt || slots.numel() != k.size(0) || !slots.is_contiguous() || k.size(0) == 0) throw Otherwise{};
    PyObject *ko = get(a[0], n_k), *vo = get(a[0], n_v);
    const CacheStore K = cache_store(get, ko), V = cache_store(get, vo);
    int *tail_len = address<int>(get(a[0], n_tail_len)), *S = address<int>(get(a[0], n_S)), *overflow = address<int>(get(a[0], n_overflow));
    const long ovf_cap = number(get(ko, n_ovf_cap)), nb = tensor(get(ko, n_base3)).size(0);
    void* stream = stream_of(a[4]);
    must("gaac_cache_append", without_gil([&] {
      return p_gaac_cache_append(static_cast<int*>(slots.data_ptr()), static_cast<int>(k.size(0)), static_cast<int>(n_kv), k.data_ptr(), v.data_ptr(), tail_len, S, static_cast<int>(cap),
                                 static_cast<int>(ovf_cap), static_cast<int>(nb), K.tail, K.b3, K.b4, K.sm, K.cd, K.fl, K.ov, K.to, K.used, V.tail, V.b3, V.b4, V.sm, V.cd, V.fl, V.ov,
                                 V.to, V.used, overflow, stream);
    }));
    Py_RETURN_TRUE;
  });
}

// prompt_store(cache, slot, k, v, stream) -> the heads' escape totals, of K and then of V
PyObject* prompt_store(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return whole_call(n, 5, [&]() -> PyObject* {
    Refs get;
    const at::Tensor &k = tensor(a[2]), &v = tensor(a[3]);
    const long slot = number(a[1]), n_kv = number(get(a[0], n_n_kv)), cap = number(get(a[0], n_cap)), n_slots = number(get(a[0], n_n_slots));
    if (!is_rows(k, 3) || !is_rows(v, 3) || k.sizes() != v.sizes() || k.size(1) != n_kv || k.size(0) < TILE || k.size(0) > cap || slot < 0 || slot >= n_slots) throw Otherwise{};
    long k_hs, k_rs, v_hs, v_rs;
    if (!in_place(k, 1, 0, k_hs, k_rs) || !in_place(v, 1, 0, v_hs, v_rs)) throw Otherwise{};
    const long L = k.size(0), nt = 2 * n_kv * (L / TILE);
    PyObject *ko = get(a[0], n_k), *vo = get(a[0], n_v);
    const int calibrate = PyObject_IsTrue(get(a[0], n_per_sequence_bases));
    if (calibrate < 0) throw Otherwise{};
    const CacheStore K = cache_store(get, ko), V = cache_store(get, vo);
    int *tail_len = address<int>(get(a[0], n_tail_len)), *S = address<int>(get(a[0], n_S)), *head_start = address<int>(get(ko, n_head_start));
    const long ovf_cap = number(get(ko, n_ovf_cap)), nb = tensor(get(ko, n_base3)).size(0);
    const at::Tensor& scan = tensor(get(a[0], n__scan));
    const long scan_row = scan.size(2);
    void* stream = stream_of(a[4]);
    // scratch: escape slots | exponent counts (hist_bytes in kv_cache.py) | tile sizes | head sizes
    const long tables = 2 * n_kv * std::max(std::min((L + 255) / 256, std::max(std::min(256 / (2 * n_kv), 64l), 1l)), (L + 65534) / 65535);
    const long at_hist = nt * TILE_ESCAPES, at_sizes = at_hist + (calibrate ? tables * HIST_BYTES : 0);
    at::Tensor scratch = bytes(k, {at_sizes + 4 * (nt + 2 * n_kv)}), totals = host_words(2 * n_kv);
    uint8_t* base = static_cast<uint8_t*>(scratch.data_ptr());
    int* words = static_cast<int*>(totals.data_ptr());
    must("gaac_prompt_store", without_gil([&] {
      return p_gaac_prompt_store(k.data_ptr(), v.data_ptr(), k_hs, k_rs, v_hs, v_rs, static_cast<int>(L), static_cast<int>(n_kv), static_cast<int>(slot * n_kv), static_cast<int>(cap),
                                 static_cast<int>(ovf_cap), static_cast<int>(nb), calibrate, tail_len, S, head_start, K.tail, K.b3, K.b4, K.sm, K.cd, K.fl, K.ov, K.to, K.used,
                                 V.tail, V.b3, V.b4, V.sm, V.cd, V.fl, V.ov, V.to, V.used, base + at_hist, at_sizes - at_hist, base,
                                 reinterpret_cast<int*>(base + at_sizes), reinterpret_cast<int*>(base + at_sizes + 4 * nt),
                                 static_cast<unsigned long long*>(scan.data_ptr()) + slot * n_kv * scan_row, scan.stride(0), static_cast<int>(scan_row), 0, words, stream);
    }));
    must("gaac_wait_words", without_gil([&] { return p_gaac_wait_words(words, static_cast<int>(2 * n_kv), stream); }));
    return numbers(totals);
  });
}

// page_encode(x, kind, base3, base4, n_kv, bytes of room a row, stream)
//   -> (sm, codes, flags, ovf_off, ovf or None where the room was too small, head_start, tile_off, the heads' totals, slots | sizes of the tiles | of the heads)
PyObject* page_encode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return whole_call(n, 7, [&]() -> PyObject* {
    const at::Tensor &x = tensor(a[0]), &b3 = tensor(a[2]), &b4 = tensor(a[3]);
    const long kind = number(a[1]), n_kv = number(a[4]), row_room = number(a[5]);
    long hs, rs;
    if (x.dim() != 3 || x.size(2) != DIM || x.itemsize() != 2 || x.size(0) == 0 || x.size(1) == 0 || !in_place(x, 0, 1, hs, rs)) throw Otherwise{};
    const long H = x.size(0), S = x.size(1), tiles = (S + TILE - 1) / TILE, S_pad = tiles * TILE, nt = H * tiles, room = row_room * H * S + 8;
    const int Hi = static_cast<int>(H), Si = static_cast<int>(S), Pi = static_cast<int>(S_pad);
    if (S_pad >= 1l << 31 || H >= 1l << 31) throw Otherwise{};
    void* stream = stream_of(a[6]);
    // each buffer is made when the next launch needs it
    at::Tensor sm = bytes(x, {H, S_pad * DIM}), cd = bytes(x, {H, S_pad * CODE_BYTES}), fl = bytes(x, {H, S_pad}, at::kInt), slots = bytes(x, {nt * TILE_ESCAPES + 4 * (nt + H)});
    uint8_t* slot = static_cast<uint8_t*>(slots.data_ptr());
    int *sizes = reinterpret_cast<int*>(slot + nt * TILE_ESCAPES), *heads = sizes + nt;
    must("gaac_encode_tiles", without_gil([&] {
      return p_gaac_encode_tiles(static_cast<int>(kind), x.data_ptr(), hs, rs, Hi, Si, Pi, static_cast<uint8_t*>(b3.data_ptr()), static_cast<uint8_t*>(b4.data_ptr()), static_cast<int>(n_kv),
                                 nullptr, static_cast<uint8_t*>(sm.data_ptr()), static_cast<uint8_t*>(cd.data_ptr()), static_cast<int*>(fl.data_ptr()), slot, sizes, stream);
    }));
    at::Tensor totals = host_words(H), off = bytes(x, {H, tiles}, at::kInt), ovf_off = bytes(x, {H, S}, at::kInt), start = bytes(x, {H + 1}, at::kInt), ovf = bytes(x, {room});
    int* words = static_cast<int*>(totals.data_ptr());
    must("gaac_page_finish", without_gil([&] {
      return p_gaac_page_finish(slot, sizes, static_cast<int*>(fl.data_ptr()), Hi, Si, Pi, static_cast<int*>(off.data_ptr()), heads, words, static_cast<int*>(start.data_ptr()),
                                static_cast<uint8_t*>(ovf.data_ptr()), room, static_cast<int*>(ovf_off.data_ptr()), stream);
    }));
    must("gaac_wait_words", without_gil([&] { return p_gaac_wait_words(words, Hi, stream); }));
    long total = 0;
    for (long h = 0; h < H; ++h) total += words[h];
    const bool fits = total + 8 <= room && total < (1l << 31) - 1;
    PyObject* list = numbers(totals);
    if (list == nullptr) return nullptr;
    PyObject* stream_view = fits ? THPVariable_Wrap(ovf.narrow(0, 0, total + 8)) : Py_NewRef(Py_None);
    return Py_BuildValue("(NNNNNNNNN)", THPVariable_Wrap(sm), THPVariable_Wrap(cd), THPVariable_Wrap(fl), THPVariable_Wrap(ovf_off), stream_view, THPVariable_Wrap(start),
                         THPVariable_Wrap(off), list, THPVariable_Wrap(slots));
  });
}

// page_decode(page, stream) -> bf16 [H, S, 128]
PyObject* page_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return whole_call(n, 2, [&]() -> PyObject* {
    Refs get;
    const long H = number(get(a[0], n_H)), S = number(get(a[0], n_S)), n_kv = number(get(a[0], n_n_kv));
    PyObject* kind = get(a[0], n_kind);
    if (!PyUnicode_CheckExact(kind) || H <= 0 || S <= 0) throw Otherwise{};
    const at::Tensor& sm = tensor(get(a[0], n_sm));
    if (sm.dim() != 2) throw Otherwise{};
    const auto at = [&](PyObject* name) { return tensor(get(a[0], name)).data_ptr(); };
    auto *cd = at(n_codes), *fl = at(n_flags), *off = at(n_tile_off), *ovf = at(n_ovf), *start = at(n_ovf_head_start), *b3 = at(n_base3), *b4 = at(n_base4);
    void* stream = stream_of(a[1]);
    at::Tensor out = bytes(sm, {H, S, DIM}, at::kBFloat16);
    must("gaac_decode_tiles", without_gil([&] {
      return p_gaac_decode_tiles(PyUnicode_CompareWithASCIIString(kind, "k") == 0 ? 0 : 1, static_cast<uint8_t*>(sm.data_ptr()), static_cast<uint8_t*>(cd), static_cast<int*>(fl),
                                 static_cast<int*>(off), static_cast<uint8_t*>(ovf), static_cast<int*>(start), static_cast<uint8_t*>(b3), static_cast<uint8_t*>(b4),
                                 static_cast<int>(n_kv), nullptr, static_cast<int>(H), static_cast<int>(S), static_cast<int>(sm.size(1) / DIM), out.data_ptr(), S * DIM, DIM, stream);
    }));
    return THPVariable_Wrap(out);
  });
}
#define GAAC_WHOLE_CALLS(X) X(attend) X(token_append) X(prompt_store) X(page_encode) X(page_decode)

// bind(path): the entry points of the library at path (the product or one of its measurement builds); AttributeError names a missing one
PyObject* bind(PyObject*, PyObject* path) {
  const char* file = PyUnicode_AsUTF8(path);
  if (file == nullptr) return nullptr;
  void* lib = dlopen(file, RTLD_NOW | RTLD_LOCAL);
  if (lib == nullptr) { PyErr_SetString(PyExc_RuntimeError, dlerror()); return nullptr; }
  const auto find = [&](const char* name) {
    void* p = dlsym(lib, name);
    if (p == nullptr && !PyErr_Occurred()) PyErr_Format(PyExc_AttributeError, "%s: undefined symbol: %s", file, name);
    return p;
  };
#define X(name) p_##name = reinterpret_cast<decltype(p_##name)>(find(#name));
  GAAC_ENTRY_POINTS(X)
#undef X
  g_last_error = reinterpret_cast<const char* (*)()>(find("gaac_last_error"));
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

#define X(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr},
#define Y(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr},
PyMethodDef methods[] = {GAAC_ENTRY_POINTS(X) GAAC_WHOLE_CALLS(Y){"bind", bind, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
#undef X
#undef Y
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() {
#define X(name) if ((n_##name = PyUnicode_InternFromString(#name)) == nullptr) return nullptr;
  GAAC_NAMES(X)
#undef X
  PyObject* m = PyModule_Create(&module);
  if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", GAAC_TORCH_VERSION) != 0) { Py_DECREF(m); return nullptr; }      // whose headers these are
  return m;
}

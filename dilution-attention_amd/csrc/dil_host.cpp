// Native host side of the Python layer (module dilution._host): the argument
// checks, allocations and library calls of the operator's entry points in one
// call each, through the C ABI of libdilution_hip.so (include/dilution_hip.h).
//
// What bounds a short call is the host: a B1 H4 T512 training pass is about 100
// us of kernels and took 204-228 us to issue, about 45 us of it per direction in
// Python (ctypes arguments, slices, checks); a decode step took 23 us to issue 3
// launches of about 4.  Here a direction costs its launches and allocations.
//
// The library is not linked: its entry points come as addresses from the ctypes
// handle (bind), so that DILUTION_HIP_LIB picks the build for both.
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/utils/pybind.h>
#include <pybind11/pybind11.h>
#include <pybind11/stl.h>

#include <array>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/dilution_hip.h"

namespace py = pybind11;

namespace {

// ---------------------------------------------------------------------------
// the library's entry points

struct Api {
  decltype(&dil_status_string) status_string = nullptr;
  decltype(&dil_forward_key_pass) forward_key_pass = nullptr;
  decltype(&dil_forward_workspace_bytes) forward_workspace_bytes = nullptr;
  decltype(&dil_forward_rows_group) forward_rows_group = nullptr;
  decltype(&dil_backward_workspace_bytes) backward_workspace_bytes = nullptr;
  decltype(&dil_backward_rows) backward_rows = nullptr;
  decltype(&dil_prefill_workspace_bytes) prefill_workspace_bytes = nullptr;
  decltype(&dil_prefill_rows) prefill_rows = nullptr;
  decltype(&dil_decode_workspace_bytes) decode_workspace_bytes = nullptr;
  decltype(&dil_decode_step_variant) decode_step_variant = nullptr;
  decltype(&dil_rows_linear) rows_linear = nullptr;
  decltype(&dil_rows_linear_qkv) rows_linear_qkv = nullptr;
};
Api api;
bool bound = false;
std::string why_unbound = "not loaded";

template <typename F>
void take(F& f, const py::dict& addresses, const char* name) {
  f = reinterpret_cast<F>(addresses[name].cast<uintptr_t>());
}

void bind(const py::dict& a) {
  take(api.status_string, a, "dil_status_string");
  take(api.forward_key_pass, a, "dil_forward_key_pass");
  take(api.forward_workspace_bytes, a, "dil_forward_workspace_bytes");
  take(api.forward_rows_group, a, "dil_forward_rows_group");
  take(api.backward_workspace_bytes, a, "dil_backward_workspace_bytes");
  take(api.backward_rows, a, "dil_backward_rows");
  take(api.prefill_workspace_bytes, a, "dil_prefill_workspace_bytes");
  take(api.prefill_rows, a, "dil_prefill_rows");
  take(api.decode_workspace_bytes, a, "dil_decode_workspace_bytes");
  take(api.decode_step_variant, a, "dil_decode_step_variant");
  take(api.rows_linear, a, "dil_rows_linear");
  take(api.rows_linear_qkv, a, "dil_rows_linear_qkv");
  bound = true;
}

void need_library() {
  if (!bound) throw std::runtime_error("dilution HIP kernels are not available: " + why_unbound);
}

void check_status(int status, const char* what) {
  if (status != 0)
    throw std::runtime_error(std::string(what) + " failed with status " + std::to_string(status) + ": " +
                             api.status_string(status));
}

// The library call without the interpreter's lock, as a ctypes call runs.
template <typename F>
void launch(const char* what, F&& f) {
  int status;
  {
    py::gil_scoped_release free;
    status = f();
  }
  check_status(status, what);
}

// ---------------------------------------------------------------------------
// types, widths, precisions

constexpr int kCheckpointRows = 32;

int type_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return 0;
    case at::kBFloat16: return 1;
    case at::kHalf: return 2;
    default: return -1;
  }
}
at::ScalarType supported(at::ScalarType t) { return type_code(t) < 0 ? at::kFloat : t; }

int precision_code(const std::string& p) {
  if (p == "ieee") return 0;
  if (p == "tf32") return 1;
  if (p == "bf16") return 2;
  throw py::value_error("dot_precision must be one of ieee, tf32, bf16");
}

std::string dims(const at::Tensor& x) {
  std::string s = "(";
  for (int64_t i = 0; i < x.dim(); ++i) s += (i ? ", " : "") + std::to_string(x.size(i));
  return s + (x.dim() == 1 ? ",)" : ")");
}

void check_head_dim(int64_t d, const std::string* precision) {
  if (d & (d - 1)) throw py::value_error("head_dim must be a power of two");
  if (d != 16 && d != 32 && d != 64 && d != 128 && d != 256)
    throw py::value_error("head_dim must be one of (16, 32, 64, 128, 256) on the gfx950 kernels (head_dim_supported(); "
                          "got " + std::to_string(d) + ")");
  if (precision != nullptr && d == 256 && *precision != "bf16")
    throw py::value_error("head_dim " + std::to_string(d) + " runs with dot_precision='bf16' only on the gfx950 kernels "
                          "(head_dim_supported(); got '" + *precision + "')");
}

void check_device(std::initializer_list<const at::Tensor*> ts) {
  const at::Device dev = (*ts.begin())->device();
  for (const at::Tensor* t : ts) {
    if (!t->is_cuda()) throw std::runtime_error("dilution HIP kernels need tensors on the GPU (no CPU path)");
    if (t->device() != dev)
      throw py::value_error("all tensors must be on one device, got " + dev.str() + " and " + t->device().str());
  }
}

// ---------------------------------------------------------------------------
// layouts

// Whether the kernels read (or write) this (B, H, T, D) tensor where it lies
// (the layout rules of dil_rows).  Rows that are apart also have to lie within
// 2^31 bytes, which the one-pass backward's 32-bit offsets cover.
bool strided_rows(const at::Tensor& x) {
  const int64_t lane = 16 / x.element_size();
  const int64_t b = x.size(0), h = x.size(1), t = x.size(2), d = x.size(3);
  const int64_t sb = x.stride(0), sh = x.stride(1), st = x.stride(2), sd = x.stride(3);
  return sd == 1 && st >= d && st < (int64_t{1} << 20) && st % lane == 0 && (b == 1 || sb % lane == 0) &&
         (h == 1 || sh % lane == 0) && (st == d || t * st * x.element_size() < (int64_t{1} << 31)) &&
         reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
}

// x in `type` as the kernels can read it: x itself when its type and layout
// allow (views of a fused projection do), else a contiguous copy.  flat: rows
// head_dim apart.
at::Tensor operand(const at::Tensor& x, at::ScalarType type, bool flat) {
  at::Tensor y = x.scalar_type() == type ? x : x.to(type);
  if (flat) y = y.contiguous();
  return strided_rows(y) ? y : y.clone(at::MemoryFormat::Contiguous);
}

// (batch, heads) as the kernels count slices: as they are within dil_rows'
// limits, else every slice a batch of its own.
std::pair<int64_t, int64_t> slice_dims(int64_t batch, int64_t heads) {
  if (heads < (int64_t{1} << 16) && batch * heads * heads < (int64_t{1} << 32)) return {batch, heads};
  return {batch * heads, 1};
}
at::Tensor sliced(const at::Tensor& x, std::pair<int64_t, int64_t> d) {
  if (x.size(0) == d.first && x.size(1) == d.second) return x;
  return x.contiguous().view({d.first, d.second, x.size(2), x.size(3)});
}

// A new tensor in `type` whose memory order follows x: (B, T, H, D) when x's rows
// are stepped over heads first (the views of a (B, T, H * D) projection), so
// that its view back to (B, T, H * D) needs no copy; else contiguous.
at::Tensor empty_as(const at::Tensor& x, at::ScalarType type) {
  const auto o = x.options().dtype(type);
  if (x.size(1) > 1 && x.size(2) > 1 && x.stride(1) < x.stride(2))
    return at::empty({x.size(0), x.size(2), x.size(1), x.size(3)}, o).transpose(1, 2);
  return at::empty({x.size(0), x.size(1), x.size(2), x.size(3)}, o);
}

// The kernels built for rows head_dim apart only: the ablation variants, and
// head_dim 256 (no registers for a row stride).
struct Variant {
  int bid, share;
  float shift;
  bool production() const { return bid == 0 && share == 1; }
};
Variant variant_of(const py::tuple& v) { return {v[0].cast<int>(), v[1].cast<int>(), v[2].cast<float>()}; }
bool flat_only(const Variant& v, int64_t head_dim) { return head_dim > 128 || !v.production(); }

dil_rows row_ref(const at::Tensor& x) { return dil_rows{x.data_ptr(), x.stride(0), x.stride(1), x.stride(2)}; }
float* f32(const at::Tensor& x) { return static_cast<float*>(x.data_ptr()); }

at::Tensor workspace(int64_t bytes, const at::Tensor& like) {
  return at::empty({bytes > 1 ? bytes : 1}, like.options().dtype(at::kByte));
}

// ---------------------------------------------------------------------------
// forward: (out (B, H, T, D), rmax, rden, ssum, total, pk or None, carry or None)

using Maybe = std::optional<at::Tensor>;

std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, Maybe, Maybe> forward(
    const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const std::string& dot_precision, bool keep_carry,
    bool save_pk, double budget_gib, const py::tuple& variant, uintptr_t stream) {
  const int prec = precision_code(dot_precision);
  if (q.dim() != 4 || !q.sizes().equals(k.sizes()) || !q.sizes().equals(v.sizes()))
    throw py::value_error("q, k, v must share one (B, H, T, D) shape, got " + dims(q) + ", " + dims(k) + ", " + dims(v));
  const int64_t batch = q.size(0), heads = q.size(1), seq = q.size(2), d = q.size(3), n = batch * heads;
  check_head_dim(d, &dot_precision);
  check_device({&q, &k, &v});
  need_library();
  const Variant var = variant_of(variant);
  const at::ScalarType type = supported(at::promote_types(at::promote_types(q.scalar_type(), k.scalar_type()), v.scalar_type()));
  const int tc = type_code(type);
  const bool flat = flat_only(var, d);
  c10::DeviceGuard guard(q.device());
  const auto o = q.options().dtype(at::kFloat);
  const int64_t nb = (seq + kCheckpointRows - 1) / kCheckpointRows;
  at::Tensor out = at::empty({batch, heads, seq, d}, o);
  at::Tensor rmax = at::empty({n, seq}, o), rden = at::empty({n, seq}, o), ssum = at::empty({n, seq}, o);
  at::Tensor total = at::empty({batch, heads, seq}, o);
  Maybe pk, carry;
  if (save_pk) pk = at::empty({n, seq, d}, o);
  int64_t rows = n;
  if (keep_carry) {
    carry = at::empty({n, nb, seq}, o);
  } else if (!var.production() || !api.forward_key_pass(seq, 0, static_cast<int>(d), tc, prec)) {
    // the three-pass forward reads the checkpoints it writes: the slices go
    // in groups whose (rows, T/32, T) scratch fits the budget.  The key pass
    // writes none without aux and takes every slice in one call.
    const int64_t per_row = std::max<int64_t>(nb * seq * 4, 1);
    rows = std::max<int64_t>(1, std::min(n, static_cast<int64_t>(budget_gib * 1073741824.0) / per_row));
    carry = at::empty({rows, nb, seq}, o);
  }
  const at::Tensor ws = workspace(api.forward_workspace_bytes(rows, seq, static_cast<int>(d), tc, prec, save_pk), q);
  const auto sd = rows >= n ? slice_dims(batch, heads) : std::make_pair(n, int64_t{1});   // (n, 1): groups of slices
  const at::Tensor qs = sliced(operand(q, type, flat), sd), ks = sliced(operand(k, type, flat), sd),
                   vs = sliced(operand(v, type, flat), sd);
  launch("dil_forward", [&]() -> int {
    for (int64_t a = 0; a < n; a += rows) {
      const int64_t c = std::min(rows, n - a);
      dil_rows rq = row_ref(qs), rk = row_ref(ks), rv = row_ref(vs);
      auto advance = [&](dil_rows& r, const at::Tensor& x) {
        r.data = static_cast<const char*>(r.data) + a * x.stride(0) * x.element_size();
      };
      if (rows < n) {
        advance(rq, qs);
        advance(rk, ks);
        advance(rv, vs);
      }
      const int status = api.forward_rows_group(
          &rq, &rk, &rv, rows < n ? c : sd.first, sd.second, n, seq, static_cast<int>(d), tc, prec, var.bid, var.share,
          var.shift, f32(out) + a * seq * d, f32(rmax) + a * seq, f32(rden) + a * seq, f32(ssum) + a * seq,
          carry ? f32(*carry) : nullptr, f32(total) + a * seq, pk ? f32(*pk) + a * seq * d : nullptr, ws.data_ptr(),
          ws.numel(), reinterpret_cast<void*>(stream));
      if (status != 0) return status;
    }
    return 0;
  });
  return {out, rmax, rden, ssum, total, pk, carry};
}

// ---------------------------------------------------------------------------
// backward: (dq, dk, dv)

std::tuple<at::Tensor, at::Tensor, at::Tensor> backward(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
                                                        const at::Tensor& out, const at::Tensor& rmax,
                                                        const at::Tensor& rden, const at::Tensor& carry,
                                                        const at::Tensor& ssum, const at::Tensor& pk,
                                                        const at::Tensor& dout, const std::string& dot_precision,
                                                        const py::tuple& variant, uintptr_t stream) {
  need_library();
  const int prec = precision_code(dot_precision);
  // what a saved-tensor hook gave back, too
  check_device({&q, &k, &v, &out, &rmax, &rden, &carry, &ssum, &pk, &dout});
  const Variant var = variant_of(variant);
  const int64_t batch = q.size(0), heads = q.size(1), seq = q.size(2), d = q.size(3), n = batch * heads;
  const at::ScalarType type = supported(at::promote_types(at::promote_types(q.scalar_type(), k.scalar_type()), v.scalar_type()));
  const at::ScalarType dtype = supported(dout.scalar_type());
  const int tc = type_code(type);
  const bool flat = flat_only(var, d);
  c10::DeviceGuard guard(q.device());
  const auto sd = slice_dims(batch, heads);
  const at::Tensor qs = sliced(operand(q, type, flat), sd), ks = sliced(operand(k, type, flat), sd),
                   vs = sliced(operand(v, type, flat), sd),
                   ds = sliced(operand(dout.reshape(q.sizes()), dtype, false), sd), of = out.contiguous();
  // the gradients in the memory order of their inputs
  at::Tensor dq = sliced(empty_as(q, type), sd), dk = sliced(empty_as(k, type), sd), dv = sliced(empty_as(v, type), sd);
  const at::Tensor ws = workspace(api.backward_workspace_bytes(n, seq, static_cast<int>(d), tc, prec), q);
  launch("dil_backward", [&]() -> int {
    const dil_rows r[7] = {row_ref(qs), row_ref(ks), row_ref(vs), row_ref(ds), row_ref(dq), row_ref(dk), row_ref(dv)};
    return api.backward_rows(&r[0], &r[1], &r[2], &r[3], f32(of), f32(rmax), f32(rden), f32(ssum), f32(carry), f32(pk),
                             sd.first, sd.second, seq, static_cast<int>(d), tc, type_code(dtype), tc, prec, var.bid,
                             var.share, var.shift, &r[4], &r[5], &r[6], ws.data_ptr(), ws.numel(),
                             reinterpret_cast<void*>(stream));
  });
  auto finish = [&](const at::Tensor& g, const at::Tensor& x) {
    const at::Tensor y = g.sizes().equals(x.sizes()) ? g : g.view(x.sizes());
    return y.scalar_type() == x.scalar_type() ? y : y.to(x.scalar_type());
  };
  return {finish(dq, q), finish(dk, k), finish(dv, v)};
}

// ---------------------------------------------------------------------------
// caches

// Shapes of a decode / prefill call against its cache (kernels.py:1003-1021):
// contiguous (B, H, capacity, D) K and V, a contiguous (B, H, capacity) fp32
// demand, q of the same (B, H, ., D).  Returns the capacity.
int64_t check_cache(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& committed) {
  if (k.dim() != 4 || !k.sizes().equals(v.sizes()))
    throw py::value_error("k_cache and v_cache must both be (B, H, capacity, D)");
  const int64_t b = k.size(0), h = k.size(1), capacity = k.size(2), d = k.size(3);
  if (q.dim() != 4 || q.size(0) != b || q.size(1) != h || q.size(3) != d)
    throw py::value_error("queries " + dims(q) + " do not match the cache " + dims(k));
  if (committed.dim() != 3 || committed.size(0) != b || committed.size(1) != h || committed.size(2) != capacity)
    throw py::value_error("committed must be (B, H, capacity) = (" + std::to_string(b) + ", " + std::to_string(h) + ", " +
                          std::to_string(capacity) + "), got " + dims(committed));
  if (committed.scalar_type() != at::kFloat) throw py::value_error("committed must be float32");
  if (!k.is_contiguous() || !v.is_contiguous() || !committed.is_contiguous())
    throw py::value_error("k_cache, v_cache and committed must be contiguous");
  return capacity;
}
int cache_type(const at::Tensor& k, const at::Tensor& v) {
  const int tc = type_code(k.scalar_type());
  if (tc < 0 || v.scalar_type() != k.scalar_type())
    throw py::value_error("k_cache and v_cache must share a float dtype");
  return tc;
}

// (out, rmax, rden, ssum, carry or None)
std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, Maybe> prefill_chunk(
    const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& committed, int64_t start,
    const std::string& dot_precision, bool keep_carry, const Maybe& into, uintptr_t stream) {
  const int prec = precision_code(dot_precision);
  const int64_t capacity = check_cache(q, k, v, committed);
  const int64_t batch = q.size(0), heads = q.size(1), chunk = q.size(2), d = q.size(3), n = batch * heads;
  check_head_dim(d, &dot_precision);
  if (start < 0 || start + chunk > capacity)
    throw py::value_error("rows [" + std::to_string(start) + ", " + std::to_string(start + chunk) +
                          ") outside cache capacity " + std::to_string(capacity));
  check_device({&q, &k, &v, &committed});
  need_library();
  const int tc = cache_type(k, v);
  c10::DeviceGuard guard(q.device());
  const auto o = q.options().dtype(at::kFloat);
  const auto sd = slice_dims(batch, heads);
  const at::Tensor qs = sliced(operand(q, k.scalar_type(), flat_only(Variant{0, 1, 1.f}, d)), sd);
  at::Tensor out = into ? *into : at::empty({batch, heads, chunk, d}, o);
  const at::Tensor orows = out.size(0) == sd.first && out.size(1) == sd.second ? out : out.view({sd.first, sd.second, chunk, d});
  at::Tensor rmax = at::empty({n, chunk}, o), rden = at::empty({n, chunk}, o), ssum = at::empty({n, chunk}, o);
  // a caller that keeps no checkpoints passes none where the library needs none
  Maybe carry;
  if (keep_carry || !api.forward_key_pass(chunk, start, static_cast<int>(d), tc, prec))
    carry = at::empty({n, (chunk + kCheckpointRows - 1) / kCheckpointRows, start + chunk}, o);
  const at::Tensor ws = workspace(api.prefill_workspace_bytes(n, chunk, start, static_cast<int>(d), tc, prec), q);
  launch("dil_prefill_chunk", [&]() -> int {
    const dil_rows rq = row_ref(qs), ro = row_ref(orows);
    return api.prefill_rows(&rq, k.data_ptr(), v.data_ptr(), sd.first, sd.second, chunk, start, capacity,
                            static_cast<int>(d), tc, prec, f32(committed), &ro, type_code(out.scalar_type()), f32(rmax),
                            f32(rden), f32(ssum), carry ? f32(*carry) : nullptr, ws.data_ptr(), ws.numel(),
                            reinterpret_cast<void*>(stream));
  });
  return {out, rmax, rden, ssum, carry};
}

at::Tensor decode_step(const at::Tensor& q1, const at::Tensor& k, const at::Tensor& v, const at::Tensor& committed,
                       int64_t length, const py::tuple& variant, uintptr_t stream) {
  if (q1.dim() != 4) throw py::value_error("q1 must be (B, H, 1, D), got " + dims(q1));
  const int64_t batch = q1.size(0), heads = q1.size(1), d = q1.size(3), n = batch * heads;
  if (q1.size(2) != 1) throw py::value_error("decode step takes exactly one query row per (batch, head)");
  if (d & (d - 1)) throw py::value_error("head_dim must be a power of two");
  const int64_t capacity = check_cache(q1, k, v, committed);
  if (length < 1 || length > capacity)
    throw py::value_error("length " + std::to_string(length) + " outside cache capacity " + std::to_string(capacity));
  check_head_dim(d, nullptr);
  check_device({&q1, &k, &v, &committed});
  need_library();
  const int tc = cache_type(k, v);
  const Variant var = variant_of(variant);
  c10::DeviceGuard guard(q1.device());
  // q1 keeps its own dtype: the kernels read it as fp32 and store the output
  // in it (kernels.py:953, 1029)
  const at::ScalarType qt = supported(q1.scalar_type());
  const at::Tensor qf = (q1.scalar_type() == qt ? q1 : q1.to(qt)).contiguous();
  at::Tensor out = at::empty({batch, heads, 1, d}, q1.options().dtype(qt));
  const at::Tensor ws = workspace(api.decode_workspace_bytes(n, length, static_cast<int>(d)), q1);
  launch("dil_decode_step", [&]() -> int {
    return api.decode_step_variant(qf.data_ptr(), k.data_ptr(), v.data_ptr(), f32(committed), out.data_ptr(), n, capacity,
                                   length, static_cast<int>(d), tc, type_code(qt), var.bid, var.share, var.shift,
                                   ws.data_ptr(), ws.numel(), reinterpret_cast<void*>(stream));
  });
  return q1.scalar_type() == qt ? out : out.to(q1.scalar_type());
}

// ---------------------------------------------------------------------------
// the decode step's few-row projections

enum { kPlain = 0, kResid = 1, kNorm = 2, kSwiglu = 3 };

const void* ptr(const Maybe& t) { return t ? t->data_ptr() : nullptr; }

at::Tensor rows_linear(const at::Tensor& x, const at::Tensor& w1, int mode, const Maybe& w2, const Maybe& g,
                       const Maybe& resid, double eps, const Maybe& into, uintptr_t stream) {
  if (x.dim() != 2 || w1.dim() != 2) throw py::value_error("rows_linear takes x (rows, K) and a weight (N, K)");
  const int64_t rows = x.size(0), kk = x.size(1), n = w1.size(0);
  auto plain = [&](const at::Tensor& t) {
    return t.scalar_type() == at::kBFloat16 && t.is_contiguous() && t.device() == x.device();
  };
  if (!plain(x) || !plain(w1) || (w2 && !plain(*w2)) || (g && !plain(*g)) || (resid && !plain(*resid)))
    throw py::value_error("rows_linear takes contiguous bf16 tensors on one device");
  // the kernel indexes every operand with the rows, N and K given here
  if (w1.size(1) != kk) throw py::value_error("rows_linear: weight " + dims(w1) + " does not match x " + dims(x));
  if (w2 && !w2->sizes().equals(w1.sizes()))
    throw py::value_error("rows_linear: w2 " + dims(*w2) + " must have w1's shape " + dims(w1));
  if (g && (g->dim() != 1 || g->size(0) != kk))
    throw py::value_error("rows_linear: the norm weight must have shape (" + std::to_string(kk) + ",), got " + dims(*g));
  if (resid && (resid->dim() != 2 || resid->size(0) != rows || resid->size(1) != n))
    throw py::value_error("rows_linear: resid must have shape (" + std::to_string(rows) + ", " + std::to_string(n) +
                          "), got " + dims(*resid));
  if ((mode == kNorm || mode == kSwiglu) && !g)
    throw py::value_error("rows_linear: the normed modes need the norm weight g");
  if (mode == kSwiglu && !w2) throw py::value_error("rows_linear: the SwiGLU mode needs w2");
  if (mode == kResid && !resid) throw py::value_error("rows_linear: the residual mode needs resid");
  check_device({&x});
  need_library();
  at::Tensor out;
  if (into) {
    out = *into;
    if (out.dim() != 2 || out.size(0) != rows || out.size(1) != n || !plain(out))
      throw py::value_error("out must be a contiguous bf16 (rows, N) tensor on the inputs' device");
  } else {
    out = at::empty({rows, n}, x.options());
  }
  c10::DeviceGuard guard(x.device());
  launch("dil_rows_linear", [&]() -> int {
    return api.rows_linear(x.data_ptr(), w1.data_ptr(), ptr(w2), ptr(g), ptr(resid), out.data_ptr(), rows, n, kk, mode, 1,
                           static_cast<float>(eps), reinterpret_cast<void*>(stream));
  });
  return out;
}

at::Tensor rows_linear_qkv(const at::Tensor& x, const at::Tensor& w, const at::Tensor& g, double eps, const at::Tensor& kc,
                           const at::Tensor& vc, const Maybe& pos_dev, int64_t pos, uintptr_t stream) {
  if (x.dim() != 2 || kc.dim() != 4)
    throw py::value_error("rows_linear_qkv takes x (B, d_model) and (B, H, capacity, D) caches");
  const int64_t rows = x.size(0), kk = x.size(1), batch = kc.size(0), heads = kc.size(1), capacity = kc.size(2), d = kc.size(3);
  for (const at::Tensor* t : {&x, &w, &g, &kc, &vc})
    if (t->scalar_type() != at::kBFloat16 || !t->is_contiguous() || t->device() != x.device())
      throw py::value_error("rows_linear_qkv takes contiguous bf16 tensors on one device");
  if (batch != rows || !vc.sizes().equals(kc.sizes()) || w.dim() != 2 || w.size(0) != 3 * heads * d || w.size(1) != kk)
    throw py::value_error("rows_linear_qkv: x, w and the caches disagree in shape");
  if (g.dim() != 1 || g.size(0) != kk)
    throw py::value_error("rows_linear_qkv: the norm weight must have shape (" + std::to_string(kk) + ",), got " + dims(g));
  check_device({&x});
  need_library();
  if (pos_dev && (pos_dev->scalar_type() != at::kLong || pos_dev->numel() != 1 || pos_dev->device() != x.device()))
    throw py::value_error("a device position is a one-element int64 tensor on the inputs' device");
  c10::DeviceGuard guard(x.device());
  at::Tensor q = at::empty({rows, heads * d}, x.options());
  launch("dil_rows_linear_qkv", [&]() -> int {
    return api.rows_linear_qkv(x.data_ptr(), w.data_ptr(), g.data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(), rows,
                               heads, d, capacity, pos_dev ? static_cast<const int64_t*>(pos_dev->data_ptr()) : nullptr,
                               pos, kk, 1, static_cast<float>(eps), reinterpret_cast<void*>(stream));
  });
  return q;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "native host side of the dilution-attention entry points";
  // torch's own error types (out of memory among them) for what ATen throws
  py::register_local_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const c10::Error&) {
      torch::translate_exception_to_python(p);
    }
  });
  m.def("bind", &bind, "take the library's entry points, {name: address}");
  m.def("unavailable", [](const std::string& why) { why_unbound = why; }, "the reason a call gives without bind");
  m.def("strided_rows", &strided_rows);
  m.def("slice_dims", &slice_dims);
  m.def("empty_as", &empty_as);
  m.def("forward", &forward);
  m.def("backward", &backward);
  m.def("prefill_chunk", &prefill_chunk);
  m.def("decode_step", &decode_step);
  m.def("rows_linear", &rows_linear);
  m.def("rows_linear_qkv", &rows_linear_qkv);
}

// extern "C" entry points of libdilution_hip.so (declared in include/dilution_hip.h).
// Argument checks that need no device access happen here; every launch is
// asynchronous on the caller's stream.
#include <hip/hip_runtime.h>

#include <initializer_list>

#include "../../include/dilution_hip.h"
#include "dil_internal.hpp"
#include "dil_variant.hpp"

namespace {

bool valid_head_dim(int d) { return d == 16 || d == 32 || d == 64 || d == 128 || d == 256; }
// head_dim 256 runs with bf16 operands only: the fp32 and split-operand tiles
// of the row-parallel output pass exceed the 160 KB of LDS at that width
bool valid_head_dim(int d, int precision) { return valid_head_dim(d) && (d < 256 || precision == 2); }
bool valid_dtype(int t) { return t == 0 || t == 1 || t == 2; }
bool valid_precision(int p) { return p == 0 || p == 1 || p == 2; }

// True when every pointer is non-null (a required argument).
template <typename... Ps>
bool all_set(const Ps*... ps) {
  return ((ps != nullptr) && ...);
}

// The layout rules of dil_rows: data 16-byte aligned, every stride that is
// stepped over a multiple of 16 bytes, rows at least head_dim elements apart
// (so a chunk past the last row lies past the resource that covers the rows)
// and less than 2^20 (the 32-bit offsets within a group of 512 rows).
bool valid_rows(const dil_rows* r, int64_t batch, int64_t heads, int head_dim, int dtype) {
  if (r == nullptr || r->data == nullptr) return false;
  const int64_t es = dtype == 0 ? 4 : 2;
  auto step_ok = [&](int64_t size, int64_t stride) { return size == 1 || (stride >= 0 && stride * es % 16 == 0); };
  return reinterpret_cast<uintptr_t>(r->data) % 16 == 0 && step_ok(batch, r->batch_stride) &&
         step_ok(heads, r->head_stride) && r->row_stride * es % 16 == 0 && r->row_stride >= head_dim &&
         r->row_stride < (int64_t{1} << 20);
}
// slices at equal steps (one batch, one head, or batches that follow the heads)
bool even_slices(const dil_rows* r, int64_t batch, int64_t heads) {
  return batch == 1 || heads == 1 || r->batch_stride == heads * r->head_stride;
}
// The view of slices of `rows` rows.  A single row has no next one: its stride
// (any, as torch leaves the strides of dimensions of size 1) is head_dim, so that
// the forms built for rows head_dim apart take it.
dil::RowsView view_of(const dil_rows* r, int64_t batch, int64_t heads, int64_t rows, int head_dim) {
  const int64_t row_stride = rows == 1 ? head_dim : r->row_stride;
  if (even_slices(r, batch, heads))
    return dil::flat_rows(heads == 1 ? r->batch_stride : r->head_stride, row_stride);
  const uint32_t h = static_cast<uint32_t>(heads);
  const uint32_t magic = static_cast<uint32_t>(((uint64_t{1} << 32) + h - 1) / h);
  return dil::RowsView{h, magic, r->batch_stride, r->head_stride, row_stride};
}
// slices are counted in 32 bits by the views, and their batch found by one
// multiplication (RowsView)
bool valid_slices(int64_t batch, int64_t heads) {
  return batch >= 1 && heads >= 1 && heads < (int64_t{1} << 16) && batch * heads < (int64_t{1} << 31) &&
         batch * heads * heads < (int64_t{1} << 32);
}

int run_forward(const dil::ForwardArgs& a) {
  if (!valid_head_dim(a.head_dim, a.prec)) return dil::kErrHeadDim;
  if (!valid_dtype(a.dtype) || !valid_dtype(a.out_dtype)) return dil::kErrDtype;
  if (!valid_precision(a.prec)) return dil::kErrPrecision;
  if (a.n < 1 || a.C < 1) return dil::kErrShape;
  // carry may be null when the call takes the key pass (dil::forward checks)
  if (!all_set(a.q, a.k, a.v, static_cast<const void*>(a.out), static_cast<const void*>(a.rmax),
               static_cast<const void*>(a.rden), static_cast<const void*>(a.ssum),
               static_cast<const void*>(a.total), static_cast<const void*>(a.workspace)))
    return dil::kErrShape;
  if (a.workspace_bytes < dil::forward_workspace_least(a.n, a.C, a.Tk, a.head_dim, a.dtype, a.prec,
                                                       a.pk != nullptr, a.key_pass))
    return dil::kErrWorkspace;
  return dil::forward(a);
}

int run_backward(const dil::BackwardArgs& a) {
  if (!valid_head_dim(a.head_dim, a.prec)) return dil::kErrHeadDim;
  if (!valid_dtype(a.dtype) || !valid_dtype(a.dout_dtype) || !valid_dtype(a.grad_dtype))
    return dil::kErrDtype;
  if (!valid_precision(a.prec)) return dil::kErrPrecision;
  if (a.n < 1 || a.T < 1) return dil::kErrShape;
  if (!all_set(a.q, a.k, a.v, a.dout, static_cast<const void*>(a.out), static_cast<const void*>(a.rmax),
               static_cast<const void*>(a.rden), static_cast<const void*>(a.ssum),
               static_cast<const void*>(a.carry), static_cast<const void*>(a.pk),
               static_cast<const void*>(a.dq), static_cast<const void*>(a.dk),
               static_cast<const void*>(a.dv), static_cast<const void*>(a.workspace)))
    return dil::kErrShape;
  if (a.workspace_bytes < dil::backward_workspace_bytes(a.n, a.T, a.head_dim, a.dtype, a.prec))
    return dil::kErrWorkspace;
  return dil::backward(a);
}

}  // namespace

namespace dil {

int check_variant(const Variant& v, int head_dim) {
  if (v.bid < 0 || v.bid >= kNumBids || v.share < SHARE_NONE || v.share > SHARE_EXCL || !(v.shift > 0.f))
    return kErrVariant;
  (void)head_dim;                            // every variant is built for every valid head_dim
  return 0;
}

}  // namespace dil

namespace {

// The arguments of a whole-sequence forward beside its inputs and their layout.
void fill_forward(dil::ForwardArgs& a, int64_t n, int64_t seq, int head_dim, int dtype, int precision, int bid,
                  int share, float shift, float* out, float* rmax, float* rden, float* ssum, float* carry,
                  float* committed_total, float* pk, void* workspace, int64_t workspace_bytes, void* stream) {
  a.key_pass = dil::forward_key_pass_requested();
  a.n = a.call_n = n;
  a.C = seq;
  a.Tk = seq;
  a.q0 = 0;
  a.head_dim = head_dim;
  a.dtype = dtype;
  a.prec = precision;
  a.out = out;
  a.out_dtype = 0;
  a.rmax = rmax;
  a.rden = rden;
  a.ssum = ssum;
  a.carry = carry;
  a.demand_in = nullptr;
  a.din_sn = 0;
  a.total = committed_total;
  a.tot_sn = seq;
  a.pk = pk;
  a.var = dil::Variant{bid, share, shift};
  a.workspace = workspace;
  a.workspace_bytes = workspace_bytes;
  a.stream = stream;
}

// The arguments of a prefill chunk beside its queries, outputs and their layouts.
void fill_prefill(dil::ForwardArgs& a, const void* k_cache, const void* v_cache, int64_t n, int64_t chunk,
                  int64_t start, int64_t capacity, int head_dim, int dtype, int precision, float* committed,
                  float* rmax, float* rden, float* ssum, float* carry, void* workspace,
                  int64_t workspace_bytes, void* stream) {
  a.key_pass = dil::forward_key_pass_requested();
  a.k = k_cache;
  a.v = v_cache;
  a.kv = a.vv = dil::flat_rows(capacity * head_dim, head_dim);
  a.n = a.call_n = n;
  a.C = chunk;
  a.Tk = start + chunk;
  a.q0 = start;
  a.head_dim = head_dim;
  a.dtype = dtype;
  a.prec = precision;
  a.rmax = rmax;
  a.rden = rden;
  a.ssum = ssum;
  a.carry = carry;
  a.demand_in = committed;
  a.din_sn = capacity;
  a.total = committed;
  a.tot_sn = capacity;
  a.pk = nullptr;
  a.workspace = workspace;
  a.workspace_bytes = workspace_bytes;
  a.stream = stream;
}

void fill_backward(dil::BackwardArgs& a, const float* out, const float* rmax, const float* rden,
                   const float* ssum, const float* carry, const float* pk, int64_t n, int64_t seq, int head_dim,
                   int dtype, int dout_dtype, int grad_dtype, int precision, int bid, int share, float shift,
                   void* workspace, int64_t workspace_bytes, void* stream) {
  a.out = out;
  a.rmax = rmax;
  a.rden = rden;
  a.ssum = ssum;
  a.carry = carry;
  a.pk = pk;
  a.n = n;
  a.T = seq;
  a.head_dim = head_dim;
  a.dtype = dtype;
  a.dout_dtype = dout_dtype;
  a.grad_dtype = grad_dtype;
  a.prec = precision;
  a.var = dil::Variant{bid, share, shift};
  a.workspace = workspace;
  a.workspace_bytes = workspace_bytes;
  a.stream = stream;
}

}  // namespace

extern "C" {

int dil_abi_version(void) { return 4; }

const char* dil_status_string(int status) {
  switch (status) {
    case 0: return "success";
    case dil::kErrHeadDim:
      return "head_dim must be one of 16, 32, 64, 128, or 256 with bf16 operands (the bid / share "
             "variants: 16-128)";
    case dil::kErrDtype: return "unsupported dtype code";
    case dil::kErrWorkspace: return "workspace smaller than the size query returned";
    case dil::kErrShape: return "invalid shape or length";
    case dil::kErrPrecision: return "dot_precision must be one of ieee, tf32, bf16";
    case dil::kErrVariant:
      return "operator variant out of range (bid 0-7, share 0-2, shift > 0)";
    case dil::kErrScratch:
      return "the call needs more scratch than dil_decode_step_noalloc holds "
             "(DIL_NOALLOC_SCRATCH_BYTES); use dil_decode_step with a workspace";
    default: break;
  }
  if (status > 0) return hipGetErrorString(static_cast<hipError_t>(status));
  return "unknown status";
}

int64_t dil_decode_workspace_bytes(int64_t n, int64_t length, int head_dim) {
  return dil::decode_workspace_bytes(n, length, head_dim);
}

int dil_decode_step_variant(const void* q1, const void* k_cache, const void* v_cache,
                            float* committed, void* out, int64_t n, int64_t capacity,
                            int64_t length, int head_dim, int dtype, int q_dtype, int bid,
                            int share, float shift, void* workspace, int64_t workspace_bytes,
                            void* stream) {
  if (!valid_head_dim(head_dim)) return dil::kErrHeadDim;
  if (!valid_dtype(dtype) || !valid_dtype(q_dtype)) return dil::kErrDtype;
  if (n < 1 || length < 1 || length > capacity) return dil::kErrShape;
  if (!all_set(q1, k_cache, v_cache, static_cast<const void*>(committed), static_cast<const void*>(out),
               static_cast<const void*>(workspace)))
    return dil::kErrShape;
  if (workspace_bytes < dil::decode_workspace_bytes(n, length, head_dim)) return dil::kErrWorkspace;
  dil::DecodeArgs a{};
  a.q1 = q1;
  a.q_sn = head_dim;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.kv_sn = capacity * head_dim;
  a.committed = committed;
  a.c_sn = capacity;
  a.out = out;
  a.o_sn = head_dim;
  a.workspace = workspace;
  a.workspace_bytes = workspace_bytes;
  a.n = n;
  a.length = length;
  a.head_dim = head_dim;
  a.dtype = dtype;
  a.q_dtype = q_dtype;
  a.var = dil::Variant{bid, share, shift};
  a.stream = stream;
  return dil::decode_step(a);
}

int dil_decode_step(const void* q1, const void* k_cache, const void* v_cache, float* committed,
                    void* out, int64_t n, int64_t capacity, int64_t length, int head_dim,
                    int dtype, int q_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  return dil_decode_step_variant(q1, k_cache, v_cache, committed, out, n, capacity, length,
                                 head_dim, dtype, q_dtype, 0, 1, 1.f, workspace, workspace_bytes,
                                 stream);
}

int dil_decode_step_dlen(const void* q1, const void* k_cache, const void* v_cache, float* committed,
                         void* out, int64_t n, int64_t capacity, const int64_t* length,
                         int64_t max_length, int head_dim, int dtype, int q_dtype, void* workspace,
                         int64_t workspace_bytes, void* stream) {
  if (!valid_head_dim(head_dim)) return dil::kErrHeadDim;
  if (!valid_dtype(dtype) || !valid_dtype(q_dtype)) return dil::kErrDtype;
  if (n < 1 || max_length < 1 || max_length > capacity) return dil::kErrShape;
  if (!all_set(q1, k_cache, v_cache, static_cast<const void*>(committed), static_cast<const void*>(out),
               static_cast<const void*>(length), static_cast<const void*>(workspace)))
    return dil::kErrShape;
  if (workspace_bytes < dil::decode_workspace_bytes(n, max_length, head_dim)) return dil::kErrWorkspace;
  dil::DecodeArgs a{};
  a.q1 = q1;
  a.q_sn = head_dim;
  a.k_cache = k_cache;
  a.v_cache = v_cache;
  a.kv_sn = capacity * head_dim;
  a.committed = committed;
  a.c_sn = capacity;
  a.out = out;
  a.o_sn = head_dim;
  a.workspace = workspace;
  a.workspace_bytes = workspace_bytes;
  a.n = n;
  a.length = max_length;
  a.dlen = length;
  a.head_dim = head_dim;
  a.dtype = dtype;
  a.q_dtype = q_dtype;
  a.var = dil::Variant{0, 1, 1.f};
  a.stream = stream;
  return dil::decode_step(a);
}

int64_t dil_forward_workspace_bytes(int64_t n, int64_t seq, int head_dim, int dtype,
                                    int precision, int want_pk) {
  return dil::forward_workspace_bytes(n, seq, seq, head_dim, dtype, precision, want_pk,
                                      dil::forward_key_pass_requested());
}

int dil_forward_variant(const void* q, const void* k, const void* v, int64_t n, int64_t seq,
                        int head_dim, int dtype, int precision, int bid, int share, float shift,
                        float* out, float* rmax, float* rden, float* ssum, float* carry,
                        float* committed_total, float* pk, void* workspace, int64_t workspace_bytes,
                        void* stream) {
  dil::ForwardArgs a{};
  a.q = q;
  a.k = k;
  a.v = v;
  a.qv = a.kv = a.vv = a.ov = dil::flat_rows(seq * head_dim, head_dim);
  fill_forward(a, n, seq, head_dim, dtype, precision, bid, share, shift, out, rmax, rden, ssum, carry,
               committed_total, pk, workspace, workspace_bytes, stream);
  return run_forward(a);
}

int dil_forward_rows_group(const dil_rows* q, const dil_rows* k, const dil_rows* v, int64_t batch, int64_t heads,
                           int64_t call_slices, int64_t seq, int head_dim, int dtype, int precision, int bid,
                           int share, float shift, float* out, float* rmax, float* rden, float* ssum,
                           float* carry, float* committed_total, float* pk, void* workspace,
                           int64_t workspace_bytes, void* stream) {
  if (!valid_head_dim(head_dim, precision)) return dil::kErrHeadDim;
  if (!valid_dtype(dtype)) return dil::kErrDtype;
  if (!valid_slices(batch, heads) || call_slices < batch * heads || seq < 1) return dil::kErrShape;
  for (const dil_rows* r : {q, k, v})
    if (!valid_rows(r, batch, heads, head_dim, dtype)) return dil::kErrShape;
  dil::ForwardArgs a{};
  a.q = q->data;
  a.k = k->data;
  a.v = v->data;
  a.qv = view_of(q, batch, heads, seq, head_dim);
  a.kv = view_of(k, batch, heads, seq, head_dim);
  a.vv = view_of(v, batch, heads, seq, head_dim);
  a.ov = dil::flat_rows(seq * head_dim, head_dim);
  fill_forward(a, batch * heads, seq, head_dim, dtype, precision, bid, share, shift, out, rmax, rden, ssum,
               carry, committed_total, pk, workspace, workspace_bytes, stream);
  a.call_n = call_slices;
  return run_forward(a);
}

int dil_forward_rows(const dil_rows* q, const dil_rows* k, const dil_rows* v, int64_t batch, int64_t heads,
                     int64_t seq, int head_dim, int dtype, int precision, int bid, int share, float shift,
                     float* out, float* rmax, float* rden, float* ssum, float* carry, float* committed_total,
                     float* pk, void* workspace, int64_t workspace_bytes, void* stream) {
  return dil_forward_rows_group(q, k, v, batch, heads, batch * heads, seq, head_dim, dtype, precision, bid, share,
                                shift, out, rmax, rden, ssum, carry, committed_total, pk, workspace,
                                workspace_bytes, stream);
}

int dil_forward(const void* q, const void* k, const void* v, int64_t n, int64_t seq,
                int head_dim, int dtype, int precision, float* out, float* rmax, float* rden,
                float* ssum, float* carry, float* committed_total, float* pk, void* workspace,
                int64_t workspace_bytes, void* stream) {
  return dil_forward_variant(q, k, v, n, seq, head_dim, dtype, precision, 0, 1, 1.f, out, rmax,
                             rden, ssum, carry, committed_total, pk, workspace, workspace_bytes,
                             stream);
}

int dil_forward_key_pass(int64_t chunk, int64_t start, int head_dim, int dtype, int precision) {
  if (!valid_head_dim(head_dim) || !valid_dtype(dtype) || !valid_precision(precision) || chunk < 1 ||
      start < 0)
    return 0;
  return dil::forward_takes_key_pass(chunk, start + chunk, start, head_dim, precision, dil::Variant{},
                                     dil::forward_key_pass_requested())
             ? 1
             : 0;
}

int64_t dil_prefill_workspace_bytes(int64_t n, int64_t chunk, int64_t start, int head_dim,
                                    int dtype, int precision) {
  return dil::forward_workspace_bytes(n, chunk, start + chunk, head_dim, dtype, precision, 0,
                                      dil::forward_key_pass_requested());
}

int dil_prefill_chunk(const void* q_chunk, const void* k_cache, const void* v_cache, int64_t n,
                      int64_t chunk, int64_t start, int64_t capacity, int head_dim, int dtype,
                      int precision, float* committed, float* out, float* rmax, float* rden,
                      float* ssum, float* carry, void* workspace, int64_t workspace_bytes,
                      void* stream) {
  if (!valid_head_dim(head_dim, precision)) return dil::kErrHeadDim;
  if (!valid_dtype(dtype)) return dil::kErrDtype;
  if (!valid_precision(precision)) return dil::kErrPrecision;
  if (chunk < 1 || start < 0 || start + chunk > capacity) return dil::kErrShape;
  dil::ForwardArgs a{};
  a.q = q_chunk;
  a.qv = a.ov = dil::flat_rows(chunk * head_dim, head_dim);
  a.out = out;
  a.out_dtype = 0;
  fill_prefill(a, k_cache, v_cache, n, chunk, start, capacity, head_dim, dtype, precision, committed, rmax,
               rden, ssum, carry, workspace, workspace_bytes, stream);
  return run_forward(a);
}

int dil_prefill_rows(const dil_rows* q_chunk, const void* k_cache, const void* v_cache, int64_t batch,
                     int64_t heads, int64_t chunk, int64_t start, int64_t capacity, int head_dim, int dtype,
                     int precision, float* committed, const dil_rows* out, int out_dtype, float* rmax,
                     float* rden, float* ssum, float* carry, void* workspace, int64_t workspace_bytes,
                     void* stream) {
  if (!valid_head_dim(head_dim, precision)) return dil::kErrHeadDim;
  if (!valid_dtype(dtype) || !valid_dtype(out_dtype)) return dil::kErrDtype;
  if (!valid_slices(batch, heads) || chunk < 1 || start < 0 || start + chunk > capacity) return dil::kErrShape;
  if (!valid_rows(q_chunk, batch, heads, head_dim, dtype) ||
      !valid_rows(out, batch, heads, head_dim, out_dtype))
    return dil::kErrShape;
  dil::ForwardArgs a{};
  a.q = q_chunk->data;
  a.qv = view_of(q_chunk, batch, heads, chunk, head_dim);
  a.out = const_cast<void*>(out->data);
  a.ov = view_of(out, batch, heads, chunk, head_dim);
  a.out_dtype = out_dtype;
  fill_prefill(a, k_cache, v_cache, batch * heads, chunk, start, capacity, head_dim, dtype, precision,
               committed, rmax, rden, ssum, carry, workspace, workspace_bytes, stream);
  return run_forward(a);
}

int64_t dil_backward_workspace_bytes(int64_t n, int64_t seq, int head_dim, int dtype,
                                     int precision) {
  return dil::backward_workspace_bytes(n, seq, head_dim, dtype, precision);
}

int dil_backward_variant(const void* q, const void* k, const void* v, const void* dout,
                         const float* out, const float* rmax, const float* rden,
                         const float* ssum, const float* carry, const float* pk, int64_t n,
                         int64_t seq, int head_dim, int dtype, int dout_dtype, int grad_dtype,
                         int precision, int bid, int share, float shift, void* dq, void* dk,
                         void* dv, void* workspace, int64_t workspace_bytes, void* stream) {
  dil::BackwardArgs a{};
  a.q = q;
  a.k = k;
  a.v = v;
  a.dout = dout;
  a.dq = dq;
  a.dk = dk;
  a.dv = dv;
  a.qv = a.kv = a.vv = a.dov = a.gqv = a.gkv = a.gvv = dil::flat_rows(seq * head_dim, head_dim);
  fill_backward(a, out, rmax, rden, ssum, carry, pk, n, seq, head_dim, dtype, dout_dtype, grad_dtype, precision,
                bid, share, shift, workspace, workspace_bytes, stream);
  return run_backward(a);
}

int dil_backward_rows(const dil_rows* q, const dil_rows* k, const dil_rows* v, const dil_rows* dout,
                      const float* out, const float* rmax, const float* rden, const float* ssum,
                      const float* carry, const float* pk, int64_t batch, int64_t heads, int64_t seq,
                      int head_dim, int dtype, int dout_dtype, int grad_dtype, int precision, int bid, int share,
                      float shift, const dil_rows* dq, const dil_rows* dk, const dil_rows* dv, void* workspace,
                      int64_t workspace_bytes, void* stream) {
  if (!valid_head_dim(head_dim, precision)) return dil::kErrHeadDim;
  if (!valid_dtype(dtype) || !valid_dtype(dout_dtype) || !valid_dtype(grad_dtype)) return dil::kErrDtype;
  if (!valid_slices(batch, heads) || seq < 1) return dil::kErrShape;
  for (const dil_rows* r : {q, k, v})
    if (!valid_rows(r, batch, heads, head_dim, dtype)) return dil::kErrShape;
  for (const dil_rows* r : {dq, dk, dv})
    if (!valid_rows(r, batch, heads, head_dim, grad_dtype)) return dil::kErrShape;
  if (!valid_rows(dout, batch, heads, head_dim, dout_dtype)) return dil::kErrShape;
  dil::BackwardArgs a{};
  a.q = q->data;
  a.k = k->data;
  a.v = v->data;
  a.dout = dout->data;
  a.dq = const_cast<void*>(dq->data);
  a.dk = const_cast<void*>(dk->data);
  a.dv = const_cast<void*>(dv->data);
  a.qv = view_of(q, batch, heads, seq, head_dim);
  a.kv = view_of(k, batch, heads, seq, head_dim);
  a.vv = view_of(v, batch, heads, seq, head_dim);
  a.dov = view_of(dout, batch, heads, seq, head_dim);
  a.gqv = view_of(dq, batch, heads, seq, head_dim);
  a.gkv = view_of(dk, batch, heads, seq, head_dim);
  a.gvv = view_of(dv, batch, heads, seq, head_dim);
  fill_backward(a, out, rmax, rden, ssum, carry, pk, batch * heads, seq, head_dim, dtype, dout_dtype, grad_dtype,
                precision, bid, share, shift, workspace, workspace_bytes, stream);
  return run_backward(a);
}

int dil_backward(const void* q, const void* k, const void* v, const void* dout,
                 const float* out, const float* rmax, const float* rden, const float* ssum,
                 const float* carry, const float* pk, int64_t n, int64_t seq, int head_dim,
                 int dtype, int dout_dtype, int grad_dtype, int precision, void* dq, void* dk,
                 void* dv, void* workspace, int64_t workspace_bytes, void* stream) {
  return dil_backward_variant(q, k, v, dout, out, rmax, rden, ssum, carry, pk, n, seq, head_dim,
                              dtype, dout_dtype, grad_dtype, precision, 0, 1, 1.f, dq, dk, dv,
                              workspace, workspace_bytes, stream);
}

}  // extern "C"

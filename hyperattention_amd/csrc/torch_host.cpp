// Host path of the HyperAttention module on torch tensors: one call from Python per forward, the autograd node
// and its backward in C++.
//
// The kernels of a short sequence run for 10 to 50 us; argument blocks filled field by field from Python and a
// Python autograd function cost 20 to 70 us per forward and 200 to 390 us per forward + backward, so those calls
// waited for the host.  Here a forward is a handful of allocations from torch's caching allocator and one call
// of the C ABI (include/hyperattn.h), and a backward runs on autograd's thread without the interpreter lock.
//
// Python binding: hyperattention_amd/_host (see hyper_attention.py, which is the only caller).
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <cmath>
#include <optional>
#include <vector>

#include "../../include/hyperattn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The exception the reference raises for the same mistake (negative statuses), RuntimeError for HIP errors.
// Autograd's threads do not hold the interpreter lock; python_error carries the exception over to the caller.
[[noreturn]] void fail(PyObject* type, const char* message) {
  pybind11::gil_scoped_acquire gil;
  PyErr_SetString(type, message);
  python_error e;
  e.persist();
  throw e;
}

void check(int status) {
  if (status == 0) return;
  PyObject* types[] = {PyExc_ValueError, PyExc_AssertionError, PyExc_AssertionError, PyExc_AssertionError,
                       PyExc_NotImplementedError, PyExc_ValueError};
  if (status < 0) fail(-status <= 6 ? types[-status - 1] : PyExc_RuntimeError, ha_last_error());
  fail(PyExc_RuntimeError, ("HIP error " + std::to_string(status) + ": " + ha_last_error()).c_str());
}

void require(bool ok, const char* message) {
  if (!ok) fail(PyExc_AssertionError, message);
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// The kernels move rows in 16-byte pieces: last dimension contiguous, rows aligned, no zero or negative strides
// along the rows.
bool readable(const Tensor& t) {
  if (t.stride(3) != 1 || (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15)) return false;
  for (int i = 0; i < 3; ++i)
    if (t.stride(i) & 7) return false;
  return t.stride(2) > 0;
}
Tensor as_readable(const Tensor& t) { return readable(t) ? t : t.contiguous(); }

// A row's address is its head's plus 32 bits, the row number times a stride below 16 MiB (include/hyperattn.h).  With
// gradients wider views are copied; a forward alone leaves them to the library, which refuses them.
bool addressable(const Tensor& t) {
  return t.stride(2) < (int64_t(1) << 23) && (t.size(2) - 1) * t.stride(2) * 2 + 256 <= (int64_t(1) << 32);
}
Tensor as_addressable(const Tensor& t) { return readable(t) && addressable(t) ? t : t.contiguous(); }

// The backward is built for head dims 64 and 128; others up to 128 run in zero-padded copies of q, k, v and the output's
// gradient, made for it in one launch, whose gradients' wanted columns are copied out in another.
int64_t built_dim(int64_t d) { return d <= 64 ? 64 : 128; }
Tensor rows_of(const Tensor& like, int64_t d) { return at::empty({like.size(0), like.size(1), like.size(2), d}, like.options()); }
ha_row_copy row_copy(const Tensor& from, const Tensor& to) {
  return {from.data_ptr(), to.data_ptr(), from.size(0), from.size(1), from.size(2), from.size(3), to.size(3),
          from.stride(0), from.stride(1), from.stride(2), to.stride(0), to.stride(1), to.stride(2)};
}

struct Config {
  double scale;
  bool causal;
  int64_t projs, block, sample, min_seq;
  bool smooth;
};

ha_dtype dtype_code(const Tensor& t) { return t.scalar_type() == at::kHalf ? HA_F16 : HA_BF16; }

ha_forward_args forward_args(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& proj, const Tensor& sampled,
                             const Config& c) {
  ha_forward_args a = {};
  a.q = q.data_ptr();
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  a.proj = proj.data_ptr();
  a.sampled_idx = sampled.defined() ? (const int32_t*)sampled.data_ptr() : nullptr;
  a.batch = q.size(0); a.heads = q.size(1); a.kv_heads = k.size(1); a.n = q.size(2); a.d = q.size(3); a.dv = v.size(3);
  a.lsh_num_projs = c.projs; a.block_size = c.block; a.sample_size = c.sample; a.min_seq_len = c.min_seq;
  a.smooth_block = c.smooth; a.causal = c.causal; a.scale = (float)c.scale; a.dtype = dtype_code(q);
  a.q_stride_b = q.stride(0); a.q_stride_h = q.stride(1); a.q_stride_n = q.stride(2);
  a.k_stride_b = k.stride(0); a.k_stride_h = k.stride(1); a.k_stride_n = k.stride(2);
  a.v_stride_b = v.stride(0); a.v_stride_h = v.stride(1); a.v_stride_n = v.stride(2);
  return a;
}

Tensor bytes_on(const Tensor& like, int64_t nbytes) {
  return at::empty({std::max<int64_t>(nbytes, 256)}, like.options().dtype(at::kByte));
}

Tensor attach_workspace(ha_forward_args& a, const Tensor& like) {
  const int64_t nbytes = ha_forward_workspace_bytes(&a);
  if (nbytes < 0) check((int)nbytes);
  Tensor ws = bytes_on(like, nbytes);
  a.workspace = ws.data_ptr();
  a.workspace_bytes = ws.numel();
  return ws;
}

// A top-level leaf (causal, the whole sequence within min_seq_len) returns the exact kernel's log-sum-exp with its
// rows padded to a multiple of 128 (hyper_attention.py:52-58); the kernel writes the padding's zeros.
bool is_leaf(const Config& c, int64_t n) { return c.causal && n <= c.min_seq; }
int64_t lse_rows(const Config& c, int64_t n) { return is_leaf(c, n) ? (n + 127) / 128 * 128 : n; }

std::pair<Tensor, Tensor> infer(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& proj, const Tensor& sampled,
                                const Config& c) {
  const int64_t b = q.size(0), h = q.size(1), n = q.size(2);
  Tensor out = at::empty({b, h, n, v.size(3)}, q.options());
  Tensor lse = at::empty({b, h, lse_rows(c, n)}, q.options().dtype(at::kFloat));
  ha_forward_args a = forward_args(q, k, v, proj, sampled, c);
  a.out = out.data_ptr();
  a.lse = (float*)lse.data_ptr();
  a.lse_rows = lse.size(2);
  Tensor ws = attach_workspace(a, q);
  check(ha_forward(&a, stream_of(q)));
  return {out, lse};
}

// ------------------------------------------------------------------------------------------- with gradients
// The attention calls a forward is made of, on segments of the whole (batch, heads, n, d) tensors: one call
// without causal mask, one exact causal call, or (hyper_attention.py:51-96) exact causal attention on the leaves
// plus one un-masked call per level on (second-half queries, first-half keys).
struct Call {
  bool hashed, causal;
  int64_t n, segs, seg_stride, q_off;
  int level;  // of the un-masked calls of the recursion (0 = whole sequence); -1: not packed
};

std::vector<Call> calls_of(int64_t n, const Config& c) {
  if (!c.causal) return {{!(c.min_seq > n), false, n, 1, n, 0, -1}};
  std::vector<int64_t> len{n};
  while (len.back() > c.min_seq) len.push_back(len.back() / 2);
  const int levels = (int)len.size() - 1;
  std::vector<Call> calls{{false, true, len[levels], int64_t(1) << levels, len[levels], 0, -1}};
  for (int j = 0; j < levels; ++j)
    calls.push_back({!(c.min_seq > len[j + 1]), false, len[j + 1], int64_t(1) << j, len[j], len[j + 1], j});
  return calls;
}

ha_attn_operands operands(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out, const Tensor& lse,
                          const Config& c, const Call& call) {
  ha_attn_operands t = {};
  t.q = q.data_ptr(); t.k = k.data_ptr(); t.v = v.data_ptr(); t.out = out.data_ptr(); t.lse = (float*)lse.data_ptr();
  t.batch = q.size(0); t.heads = q.size(1); t.n_q = t.n_k = call.n; t.d = q.size(3); t.dv = v.size(3);
  t.q_stride_b = q.stride(0); t.q_stride_h = q.stride(1); t.q_stride_n = q.stride(2);
  t.k_stride_b = k.stride(0); t.k_stride_h = k.stride(1); t.k_stride_n = k.stride(2);
  t.v_stride_b = v.stride(0); t.v_stride_h = v.stride(1); t.v_stride_n = v.stride(2);
  t.o_stride_b = out.stride(0); t.o_stride_h = out.stride(1); t.o_stride_n = out.stride(2);
  t.lse_stride_b = lse.stride(0); t.lse_stride_h = lse.stride(1);
  t.segs = call.segs; t.seg_stride_rows = call.seg_stride; t.q_seg_offset = call.q_off; t.k_seg_offset = 0;
  if (call.level >= 0) {  // out and lse hold the rows the call writes and nothing else, segment after segment
    t.o_seg_stride_rows = call.n;
    t.o_seg_offset = 0;
  }
  t.kv_group = q.size(1) / k.size(1);
  t.scale = (float)c.scale;
  t.dtype = dtype_code(q);
  return t;
}

ha_block_attn_args block_args(const ha_attn_operands& t, const Tensor& ws, int64_t q_idx_at, int64_t k_idx_at,
                              const Tensor& sampled, const Config& c) {
  ha_block_attn_args a = {};
  a.t = t;
  const int64_t kv_heads = t.heads / t.kv_group, rows = t.segs * t.n_q;
  a.q_idx = (const char*)ws.data_ptr() + q_idx_at;
  a.k_idx = (const char*)ws.data_ptr() + k_idx_at;
  a.idx_type = HA_IDX_I32;
  a.q_idx_stride_b = t.heads * rows; a.q_idx_stride_h = rows; a.q_idx_stride_n = 1;
  a.k_idx_stride_b = kv_heads * rows; a.k_idx_stride_h = rows; a.k_idx_stride_n = 1;
  a.sampled_idx = sampled.defined() ? sampled.data_ptr() : nullptr;
  if (sampled.defined() && sampled.dim() > 1) {  // a list per k/v head: hyper_attention.py lets it through without mask
    a.sampled_stride_h = c.sample;
    a.sampled_stride_b = sampled.dim() > 2 ? kv_heads * c.sample : 0;
  }
  a.block_size = c.block; a.sample_size = c.sample; a.smooth_block = c.smooth;
  return a;
}

// What a forward leaves for its backward besides tensors.
struct Saved : torch::CustomClassHolder {
  Config c;
  Tensor proj, sampled;                     // for the forward alone (the backward's sample list is saved with the tensors)
  std::vector<Call> calls;
  std::vector<int64_t> q_idx_at, k_idx_at;  // per call: byte offsets of its orders in the sort's workspace
  int64_t n;                                // rows of the caller's tensors (an odd n runs with one row more)
};

class Attention : public torch::autograd::Function<Attention> {
 public:
  static variable_list forward(AutogradContext* ctx, const Tensor& q_in, const Tensor& k_in, const Tensor& v_in,
                               c10::intrusive_ptr<Saved> s) {
    const Config& c = s->c;
    Tensor q = q_in, k = k_in, v = v_in;
    int64_t n = s->n = q.size(2);
    if (c.causal && n > c.min_seq && (n & 1)) {
      // the recursion appends a zero row to an odd length (hyper_attention.py:61-64): no query before it sees its
      // key, its own result is dropped, and only n itself can be odd in a plan the kernels take
      q = at::constant_pad_nd(q, {0, 0, 0, 1});
      k = at::constant_pad_nd(k, {0, 0, 0, 1});
      v = at::constant_pad_nd(v, {0, 0, 0, 1});
      ++n;
    }
    const int64_t b = q.size(0), h = q.size(1), d = q.size(3);
    void* const stream = stream_of(q);
    s->calls = calls_of(n, c);
    const int levels = (int)s->calls.size() - 1;
    const bool any_hashed = std::any_of(s->calls.begin(), s->calls.end(), [](const Call& x) { return x.hashed; });
    s->q_idx_at.assign(s->calls.size(), -1);
    s->k_idx_at.assign(s->calls.size(), -1);
    const auto f32 = q.options().dtype(at::kFloat);
    // the first call's result; the levels' results packed: a level writes the second halves of its segments, n/2
    // rows per head
    Tensor o0 = at::empty({b, h, n, d}, q.options()), lse0 = at::empty({b, h, lse_rows(c, n)}, f32);
    Tensor o_un, lse_un;
    if (levels) {
      o_un = at::empty({levels, b, h, n / 2, d}, q.options());
      lse_un = at::empty({levels, b, h, n / 2}, f32);
    }
    Tensor ws;
    if (any_hashed) {
      ha_forward_args a = forward_args(q, k, v, s->proj, s->sampled, c);
      ws = attach_workspace(a, q);
      int64_t at_q[48], at_k[48];
      int nlev = 0;
      if (c.causal) {  // with the leaves, beside which rows are hashed and ranked: forward + backward of 24 x 4096 234.6 -> 231.6 us,
                       // 8 x 32768 862 -> 850, 4 x 12 x 10240 1432 -> 1401; d = 128 and long sequences the same
        const ha_attn_operands t = operands(q, k, v, o0, lse0, c, s->calls[0]);
        check(ha_forward_sort_leaves(&a, &t, at_q, at_k, &nlev, stream));
      } else {
        check(ha_forward_sort(&a, at_q, at_k, &nlev, stream));
      }
      for (size_t i = 0; i < s->calls.size(); ++i)
        if (s->calls[i].hashed) {
          const int j = std::max(s->calls[i].level, 0);
          s->q_idx_at[i] = at_q[j];
          s->k_idx_at[i] = at_k[j];
        }
    }
    for (size_t i = any_hashed && c.causal ? 1 : 0; i < s->calls.size(); ++i) {
      const Call& call = s->calls[i];
      Tensor o = i ? o_un.select(0, call.level) : o0, l = i ? lse_un.select(0, call.level) : lse0;
      ha_attn_operands t = operands(q, k, v, o, l, c, call);
      if (call.hashed) {
        ha_block_attn_args a = block_args(t, ws, s->q_idx_at[i], s->k_idx_at[i], s->sampled, c);
        check(ha_block_attn_fwd(&a, stream));
      } else {
        if (!levels) t.lse_rows = lse0.size(2);
        check(ha_flash_attn_fwd(&t, call.causal, stream));
      }
    }
    Tensor out = o0, lse = lse0, lse0_shifted = lse0, lse_un_shifted;
    if (levels) {
      // one pass merges the leaf and level results of every row with the reference's arithmetic and writes, for
      // the backward, each call's log-sum-exp shifted by the logarithm of its total merge weight
      out = at::empty_like(o0);
      lse = at::empty_like(lse0);
      lse0_shifted = at::empty_like(lse0);
      lse_un_shifted = at::empty_like(lse_un);
      const void* o_ptr[48];
      const float* l_ptr[48];
      float* s_ptr[48];
      for (int j = 0; j < levels; ++j) {
        o_ptr[j] = o_un.select(0, j).data_ptr();
        l_ptr[j] = (const float*)lse_un.select(0, j).data_ptr();
        s_ptr[j] = (float*)lse_un_shifted.select(0, j).data_ptr();
      }
      check(ha_lse_merge_levels(o0.data_ptr(), (const float*)lse0.data_ptr(), o_ptr, l_ptr, s_ptr,
                                (float*)lse0_shifted.data_ptr(), out.data_ptr(), (float*)lse.data_ptr(), levels, b * h, n, d,
                                dtype_code(q), 1, stream));
    }
    if (n != s->n) {
      out = out.narrow(2, 0, s->n);
      lse = lse.narrow(2, 0, s->n);
    }
    // The sample list too: the backward reads it with the forward's log-sum-exps, so a list that was changed in place
    // in between has to be an error.
    ctx->save_for_backward({q, k, v, o0, lse0_shifted, o_un, lse_un_shifted, ws, any_hashed ? s->sampled : Tensor()});
    s->proj.reset();
    s->sampled.reset();
    ctx->saved_data["s"] = c10::IValue::make_capsule(s);
    ctx->mark_non_differentiable({lse});
    ctx->set_materialize_grads(false);
    return {out, lse};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list result(4);
    Tensor dout = grads[0];
    if (!dout.defined()) return result;
    const variable_list saved = ctx->get_saved_variables();
    Tensor q = saved[0], k = saved[1], v = saved[2];
    const auto s = c10::static_intrusive_pointer_cast<Saved>(ctx->saved_data["s"].toCapsule());
    const Config& c = s->c;
    c10::OptionalDeviceGuard guard(q.device());
    void* const stream = stream_of(q);
    const int64_t n = q.size(2);
    dout = n != s->n ? at::constant_pad_nd(dout, {0, 0, 0, n - s->n}) : as_addressable(dout);
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    const int64_t d = q.size(3), wide = built_dim(d);
    Tensor dq_wide = dq, dk_wide = dk, dv_wide = dv;
    if (d != wide) {
      const Tensor pq = rows_of(q, wide), pk = rows_of(k, wide), pv = rows_of(v, wide), pdout = rows_of(dout, wide);
      const ha_row_copy copies[] = {row_copy(q, pq), row_copy(k, pk), row_copy(v, pv), row_copy(dout, pdout)};
      check(ha_copy_rows(copies, 4, stream));
      q = pq; k = pk; v = pv; dout = pdout;
      dq_wide = rows_of(q, wide); dk_wide = rows_of(k, wide); dv_wide = rows_of(v, wide);
    }
    // A call's gradients are linear in the output gradient it is given, and that enters only through
    // P = exp(s - lse): weighting a row's output gradient by the call's merge weight w equals giving the call the
    // log-sum-exp lse - log(w).  So every call gets the output gradient as it is and the shifted log-sum-exps.
    // The first call writes every row of dq, dk and dv, the levels add to their segments.
    int64_t nbytes = 0;
    std::vector<ha_attn_operands> ops;
    for (size_t i = 0; i < s->calls.size(); ++i) {
      const Call& call = s->calls[i];
      ops.push_back(operands(q, k, v, i ? saved[5].select(0, call.level) : saved[3],
                             i ? saved[6].select(0, call.level) : saved[4], c, call));
      int64_t m;
      if (call.hashed) {
        const ha_block_attn_args a = block_args(ops.back(), saved[7], s->q_idx_at[i], s->k_idx_at[i], saved[8], c);
        m = ha_block_attn_bwd_workspace_bytes(&a);
      } else {
        m = ha_attn_bwd_workspace_bytes(&ops.back(), 0);
      }
      if (m < 0) check((int)m);
      nbytes = std::max(nbytes, m);
    }
    Tensor ws = bytes_on(q, nbytes);  // one workspace for all calls: they run one after the other on the stream
    for (size_t i = 0; i < s->calls.size(); ++i) {
      ha_attn_grads g = {};
      g.out_d = d;
      g.dout = dout.data_ptr(); g.dq = dq_wide.data_ptr(); g.dk = dk_wide.data_ptr(); g.dv = dv_wide.data_ptr();
      g.do_stride_b = dout.stride(0); g.do_stride_h = dout.stride(1); g.do_stride_n = dout.stride(2);
      g.dq_stride_b = dq_wide.stride(0); g.dq_stride_h = dq_wide.stride(1); g.dq_stride_n = dq_wide.stride(2);
      g.dk_stride_b = dk_wide.stride(0); g.dk_stride_h = dk_wide.stride(1); g.dk_stride_n = dk_wide.stride(2);
      g.dv_stride_b = dv_wide.stride(0); g.dv_stride_h = dv_wide.stride(1); g.dv_stride_n = dv_wide.stride(2);
      g.accumulate = i > 0;
      g.workspace = ws.data_ptr();
      g.workspace_bytes = ws.numel();
      if (s->calls[i].hashed) {
        ha_block_attn_args a = block_args(ops[i], saved[7], s->q_idx_at[i], s->k_idx_at[i], saved[8], c);
        check(ha_block_attn_bwd(&a, &g, stream));
      } else {
        check(ha_flash_attn_bwd(&ops[i], s->calls[i].causal, &g, stream));
      }
    }
    if (d != wide) {
      const ha_row_copy copies[] = {row_copy(dq_wide, dq), row_copy(dk_wide, dk), row_copy(dv_wide, dv)};
      check(ha_copy_rows(copies, 3, stream));
    }
    if (n != s->n) {
      dq = dq.narrow(2, 0, s->n);
      dk = dk.narrow(2, 0, s->n);
      dv = dv.narrow(2, 0, s->n);
    }
    result[0] = dq;
    result[1] = dk;
    result[2] = dv;
    return result;
  }
};

bool wants_grad(const Tensor& q, const Tensor& k, const Tensor& v) {
  return at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
}

// HyperAttention.forward without the residual estimator.  Returns (attn, lse), or nothing where the head dims have
// to be padded first: not multiples of 8, or gradients wanted and a value dim of its own.
std::optional<std::pair<Tensor, Tensor>> forward(const Tensor& query, const Tensor& key, const Tensor& value, const Tensor& proj,
                                                 const std::optional<Tensor>& sampled_idx, double scale, bool causal,
                                                 int64_t projs, int64_t block, int64_t sample, int64_t min_seq, bool smooth) {
  require(query.dim() == 4 && key.dim() == 4 && value.dim() == 4, "query, key and value are (batch, heads, seq_len, dim)");
  require(query.size(2) == key.size(2), "query and key have different sequence lengths");
  require(value.size(2) == key.size(2) && value.size(1) == key.size(1) && value.size(0) == key.size(0) &&
              query.size(0) == key.size(0) && query.size(3) == key.size(3),
          "query, key and value do not fit together");
  // what the attention calls of a pass with gradients are given is the quotient
  require(key.size(1) > 0 && query.size(1) % key.size(1) == 0, "the key/value heads must divide the query heads");
  const bool grad = wants_grad(query, key, value);
  // no length is below a negative min_seq_len, so the causal recursion would not end; without mask there is nothing to
  // end, and a call with gradients hashes, as with zero
  require(min_seq >= 0 || (grad && !causal), "min_seq_len must not be negative");
  min_seq = std::max<int64_t>(min_seq, 0);
  require(query.is_cuda() && key.device() == query.device() && value.device() == query.device(), "tensors must be on one GPU");
  require(query.scalar_type() == at::kHalf || query.scalar_type() == at::kBFloat16, "Only support fp16 and bf16");
  require(key.scalar_type() == query.scalar_type() && value.scalar_type() == query.scalar_type(),
          "All tensors must have the same type");
  const int64_t d = query.size(3), dv = value.size(3);
  require(d <= 128 && dv <= 128, "FlashAttention only support head dimensions up to 128");
  if (d % 8 || dv % 8 || (grad && d != dv)) return std::nullopt;
  // the runtime's device is the tensors' one in all but a few programs: ask before paying for a guard
  c10::OptionalDeviceGuard guard;
  if (c10::hip::current_device() != query.device().index()) guard.reset_device(query.device());
  Config c{scale != 0. ? scale : 1. / std::sqrt((double)d), causal, projs, block, sample, min_seq, smooth};
  // A pass that hashes nothing does not read the projection, wherever it is; one exact call with gradients does not ask
  // for its type either.
  const std::vector<Call> calls = calls_of(query.size(2) + (causal && query.size(2) > min_seq ? query.size(2) & 1 : 0), c);
  const bool hashed = std::any_of(calls.begin(), calls.end(), [](const Call& x) { return x.hashed; });
  if (hashed || !grad || calls.size() > 1) {
    require(proj.scalar_type() == query.scalar_type(), "All three tensors must have the same type");
    require(proj.numel() == d * projs, "the projection does not fit the head dim");
  }
  require(!hashed || proj.device() == query.device(), "the projection must be on the tensors' GPU");
  const Tensor p = proj.is_contiguous() ? proj : proj.contiguous();
  const Tensor sampled = sampled_idx ? *sampled_idx : Tensor();
  const int64_t n = query.size(2);
  const bool leaf = is_leaf(c, n);
  Tensor out, lse;
  if (grad) {
    auto s = c10::make_intrusive<Saved>();
    s->c = c;
    s->proj = p;
    s->sampled = sampled;
    const variable_list r = Attention::apply(as_addressable(query), as_addressable(key), as_addressable(value), s);
    out = r[0];
    lse = r[1];
  } else {
    std::tie(out, lse) = infer(as_readable(query), as_readable(key), as_readable(value), p, sampled, c);
  }
  return std::make_pair(out, leaf ? lse : lse.unsqueeze(-1));
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.def("abi_version", [] { return ha_abi_version(); });
  m.def("forward", [](const Tensor& query, const Tensor& key, const Tensor& value, const Tensor& proj,
                      const std::optional<Tensor>& sampled_idx, double scale, bool causal, int64_t projs, int64_t block,
                      int64_t sample, int64_t min_seq, bool smooth) {
    try {
      return forward(query, key, value, proj, sampled_idx, scale, causal, projs, block, sample, min_seq, smooth);
    } catch (python_error& e) {
      e.restore();
      throw pybind11::error_already_set();
    }
  });
}

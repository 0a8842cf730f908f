// Host side of the operators as a Python extension: tensors in, C ABI calls out, autograd nodes in C++.
//
// A small call is bounded by its host path, not by its kernels: through ctypes and Python autograd nodes a step at B4 T512
// H12 D64 took 190 us for 50 us of kernels.  Every entry point here takes the tensors as the public Python
// functions received them, in their own layout (head_first or not: the strides are swapped, no view is made), checks
// that it can handle them, allocates the results, calls include/fox_attn.h and, when a gradient can be asked for, records a
// C++ autograd node.  It returns None for anything else -- invalid arguments, tensors that need a copy first, another
// current device -- and the Python function then goes through its general path, which raises the documented errors.
#include <ATen/TracerMode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/InferenceMode.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <atomic>
#include <cmath>
#include <map>
#include <mutex>
#include <optional>

#include "../../include/fox_attn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check(int rc, const char* what) {
  TORCH_CHECK(rc == FOX_OK, what, " failed (code ", rc, "): ", fox_last_error());
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

int dtype_code(const Tensor& t) { return t.scalar_type() == at::kBFloat16 ? FOX_DTYPE_BF16 : FOX_DTYPE_FP16; }

bool head_dim_ok(int64_t d) { return d == 16 || d == 32 || d == 64 || d == 128; }

// What the kernels ask of a 16-bit tensor: unit inner stride, 16-byte aligned base, outer strides in whole 16-byte vectors.
bool vectors_ok(const Tensor& t) {
  const auto s = t.strides();
  const size_t n = s.size();
  if (s[n - 1] != 1 || (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15)) return false;
  for (size_t i = 0; i + 1 < n; ++i)
    if (s[i] & 7) return false;
  return true;
}

// (B, H, T, D) if head_first, else (B, T, H, D)
fox_view view_of(const Tensor& t, bool head_first) {
  return fox_view{t.data_ptr(), t.stride(0), t.stride(head_first ? 1 : 2), t.stride(head_first ? 2 : 1)};
}

Tensor empty_bytes_like(const Tensor& t, int64_t bytes) { return at::empty({bytes}, t.options().dtype(at::kByte)); }
Tensor empty_floats(const Tensor& t, int64_t n) { return at::empty({n}, t.options().dtype(at::kFloat)); }

// Arrival counters for kernels whose last workgroup finishes the work of all: kCounters zeros per stream, which every such kernel leaves zero
// again.  Launches on one stream follow each other, so the block of a stream has one user at a time, whichever threads feed the stream.  Only
// for torch's own streams, which live as long as the process (the handle of another stream may come back as a different stream), at most
// kCounterBlocks of them per device, and not during capture (a graph may be replayed beside its stream).  Null: the caller takes the way without
// counters.  kCounters is the most that fox_attn_decode_counters asks for: at least two workgroups for each, on at most as many as there are CUs.
constexpr int64_t kCounters = 128;
constexpr size_t kCounterBlocks = 64;
uint32_t* arrival_counters(const Tensor& like, int64_t n) {
  const c10::hip::HIPStream stream = c10::hip::getCurrentHIPStream(like.device().index());
  const bool torch_owned = stream.id() == 0 || (stream.id() & 1);
  if (n > kCounters || !torch_owned || c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return nullptr;
  static std::mutex mutex;
  static auto* devices = new std::map<int, std::map<int64_t, Tensor>>;   // (not destroyed: the device may be gone before static objects are)
  const std::lock_guard<std::mutex> lock(mutex);
  auto& blocks = (*devices)[like.device().index()];
  auto it = blocks.find(stream.id());
  if (it == blocks.end()) {
    if (blocks.size() >= kCounterBlocks) return nullptr;
    const c10::InferenceMode no_inference(false);
    it = blocks.emplace(stream.id(), at::zeros({kCounters}, like.options().dtype(at::kInt))).first;
  }
  return (uint32_t*)it->second.mutable_data_ptr();
}

// ---------------------------------------------------------------------------------------------------------------
// attention
// ---------------------------------------------------------------------------------------------------------------
struct Attention {   // one call, in the caller's layout
  bool head_first = false, is_logit = false, auto_threshold = false;
  double sm_scale = 0;
  int64_t B = 0, H = 0, M = 0, N = 0, D = 0;
  Tensor seq_start, threshold;   // undefined when absent; threshold is (B, H) contiguous fp32
  // norm and gate in the epilogue
  bool epilogue = false;
  Tensor gate, weight;           // gate undefined for the plain norm; weight fp32 contiguous
  int act = FOX_ACT_NONE;
  double eps = 0;

  fox_dims dims(const Tensor& q) const {
    return fox_dims{(int32_t)B, (int32_t)H, (int32_t)M, (int32_t)N, (int32_t)D, dtype_code(q)};
  }
  int64_t gs_h(const Tensor& g) const { return g.stride(head_first ? 1 : 2); }
  int64_t gs_n(const Tensor& g) const { return g.stride(head_first ? 2 : 1); }
  const int64_t* seq_ptr() const { return seq_start.defined() ? seq_start.const_data_ptr<int64_t>() : nullptr; }
  const float* thr_ptr() const { return threshold.defined() ? threshold.const_data_ptr<float>() : nullptr; }
};

struct Forward {     // what a forward leaves behind
  Tensor out;        // o, or y with an epilogue
  Tensor o, log_fgate, rstd;
  Tensor rows;       // fp32: log_lambda (B,H,N), then at lse_at() the log-normaliser (B,H,M)
};

int64_t lse_at(const Attention& a) { return (a.B * a.H * a.N + 3) / 4 * 4; }

int gate_dtype(const Tensor& g) {
  switch (g.scalar_type()) {
    case at::kBFloat16: return FOX_DTYPE_BF16;
    case at::kHalf: return FOX_DTYPE_FP16;
    case at::kFloat: return FOX_DTYPE_FP32;
    default: return -1;
  }
}

Forward run_forward(Attention& a, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g) {
  Forward f;
  void* stream = stream_of(q);
  const fox_dims dims = a.dims(q);
  const fox_view qv = view_of(q, a.head_first), kv = view_of(k, a.head_first), vv = view_of(v, a.head_first);
  Tensor norm_scratch;
  if (a.auto_threshold) {
    a.threshold = at::empty({a.B, a.H}, q.options().dtype(at::kFloat));
    norm_scratch = at::empty({a.B, a.H, 3}, q.options().dtype(at::kInt));
  }
  // log_lambda (B,H,N) and the log-normaliser (B,H,M) come from one allocation, which the backward keeps; key splits have their own
  int64_t ws_bytes = 0;
  check(fox_attn_fwd_plan(&dims, a.threshold.defined(), nullptr, nullptr, &ws_bytes), "fox_attn_fwd_plan");
  const int64_t at_l = lse_at(a);
  f.rows = empty_floats(q, at_l + a.B * a.H * a.M);
  Tensor ws;
  if (ws_bytes > 0) ws = empty_bytes_like(q, ws_bytes);
  float* base = f.rows.mutable_data_ptr<float>();
  // short rows and small grids: the forward takes the gates as they are; else their cumulative sums come from a scan in front of it
  // (logits: with logsigmoid fused in; the fp32 log gates are a by-product)
  int32_t from_gates = 0;
  check(fox_attn_fwd_takes_gates(&dims, a.threshold.defined(), &from_gates), "fox_attn_fwd_takes_gates");
  fox_gates gates{g.const_data_ptr(), a.is_logit, a.is_logit ? gate_dtype(g) : FOX_DTYPE_FP32, g.stride(0), a.gs_h(g), a.gs_n(g), nullptr};
  if (a.is_logit) {
    f.log_fgate = at::empty({a.B, a.H, a.N}, q.options().dtype(at::kFloat));
    gates.log_fgate = f.log_fgate.mutable_data_ptr<float>();
  }
  if (a.auto_threshold) {
    float* thr = a.threshold.mutable_data_ptr<float>();
    uint32_t* scratch = (uint32_t*)norm_scratch.mutable_data_ptr();
    if (from_gates) check(fox_auto_threshold(&dims, &qv, &kv, (float)a.sm_scale, thr, scratch, stream), "fox_auto_threshold");
    else check(fox_auto_threshold_scan(&dims, &qv, &kv, (float)a.sm_scale, thr, scratch, &gates, a.seq_ptr(), base, stream), "fox_auto_threshold_scan");
  } else if (!from_gates && a.is_logit) {
    check(fox_gate_cumsum_fwd(gates.g, gates.dtype, gates.stride_b, gates.stride_h, gates.stride_n, a.seq_ptr(), gates.log_fgate, base, dims.B,
                              dims.H, dims.N, stream), "fox_gate_cumsum_fwd");
  } else if (!from_gates) {
    check(fox_cumsum_fwd(g.const_data_ptr<float>(), gates.stride_b, gates.stride_h, gates.stride_n, a.seq_ptr(), base, dims.B, dims.H, dims.N,
                         stream), "fox_cumsum_fwd");
  }
  fox_fwd_args args{};
  args.dims = dims;
  args.q = qv;
  args.k = kv;
  args.v = vv;
  args.log_lambda = base;
  args.lse = base + at_l;
  args.seq_start = a.seq_ptr();
  args.threshold = a.thr_ptr();
  args.sm_scale = (float)a.sm_scale;
  args.workspace = ws_bytes > 0 ? ws.mutable_data_ptr() : nullptr;
  args.workspace_bytes = ws_bytes;
  if (!a.epilogue) {
    f.out = f.o = at::empty_like(q);
    args.o = view_of(f.o, a.head_first);
    if (from_gates) check(fox_attn_fwd_gates(&args, &gates, nullptr, stream), "fox_attn_fwd_gates");
    else check(fox_attn_fwd(&args, stream), "fox_attn_fwd");
    return f;
  }
  // o and y as rows of heads * head_dim per token: what the norm's backward and the output projection read
  f.o = at::empty({a.B, a.M, a.H, a.D}, q.options());
  f.out = at::empty({a.B, a.M, a.H, a.D}, q.options());
  f.rstd = at::empty({a.B, a.M, a.H}, q.options().dtype(at::kFloat));
  args.o = view_of(f.o, false);
  fox_fwd_epilogue epi{};
  if (a.gate.defined()) epi.gate = view_of(a.gate, a.head_first);
  epi.y = view_of(f.out, false);
  epi.weight = a.weight.const_data_ptr<float>();
  epi.rstd = f.rstd.mutable_data_ptr<float>();
  epi.eps = (float)a.eps;
  epi.activation = a.act;
  if (from_gates) check(fox_attn_fwd_gates(&args, &gates, &epi, stream), "fox_attn_fwd_gates");
  else check(fox_attn_fwd_norm_gate(&args, &epi, stream), "fox_attn_fwd_norm_gate");
  if (a.head_first) {
    f.o = f.o.transpose(1, 2);
    f.out = f.out.transpose(1, 2);
  }
  return f;
}

// One query row without a graph or a threshold: nobody needs the cumulative sums, so the kernel takes the gates themselves.
bool decodes_from_gates(const Attention& a) {
  return a.M == 1 && !a.is_logit && !a.auto_threshold && !a.threshold.defined() && !a.epilogue;
}
Tensor run_decode(const Attention& a, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g) {
  fox_fwd_args args{};
  args.dims = a.dims(q);
  int64_t ws_bytes = 0;
  check(fox_attn_decode_workspace_bytes(&args.dims, &ws_bytes), "fox_attn_decode_workspace_bytes");
  Tensor out = at::empty_like(q), ws;
  args.q = view_of(q, a.head_first);
  args.k = view_of(k, a.head_first);
  args.v = view_of(v, a.head_first);
  args.o = view_of(out, a.head_first);
  args.seq_start = a.seq_ptr();
  args.sm_scale = (float)a.sm_scale;
  if (ws_bytes > 0) {
    ws = empty_bytes_like(q, ws_bytes);
    args.workspace = ws.mutable_data_ptr();
    args.workspace_bytes = ws_bytes;
  }
  int32_t counters = 0;
  check(fox_attn_decode_counters(&args.dims, &counters), "fox_attn_decode_counters");
  uint32_t* arrived = counters > 0 ? arrival_counters(q, counters) : nullptr;
  check(fox_attn_decode_counted(&args, g.const_data_ptr<float>(), g.stride(0), a.gs_h(g), a.gs_n(g), arrived, stream_of(q)), "fox_attn_decode");
  return out;
}

// The list that takes the pruning bounds of every backward while record_pruning_bounds() is active; the interpreter lock guards it.
PyObject* g_bounds = nullptr;
std::atomic<bool> g_bounds_on{false};

// Room for the bounds of one backward, handed to the kernels and to the list.
void record_bounds(const Attention& a, const Tensor& q, fox_bwd_args& args) {
  int32_t block_m = 0, block_n = 0, kv_n = 0, kv_m = 0;
  check(fox_tile_config(args.dims.D, &block_m, &block_n, &kv_n, &kv_m), "fox_tile_config");
  const auto ints = q.options().dtype(at::kInt);
  Tensor first = at::zeros({a.B, a.H, (a.M + block_m - 1) / block_m}, ints), end = at::full({a.B, a.H, (a.N + 63) / 64}, -1, ints);
  const pybind11::gil_scoped_acquire gil;
  if (!g_bounds) return;
  args.q_first_block = first.mutable_data_ptr<int32_t>();
  args.kv_end_row = end.mutable_data_ptr<int32_t>();
  pybind11::dict d;
  d["dq_first_block"] = pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(first));
  d["kv_end_row"] = pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(end));
  pybind11::reinterpret_borrow<pybind11::list>(g_bounds).append(d);   // (keeps both tensors alive past the launches)
}

// dq, dk, dv and the gradient of the gates, in the layout of the inputs.  g: the gate logits, undefined for log gates, of which the
// backward needs the strides only
variable_list run_backward(const Attention& a, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, at::IntArrayRef g_strides,
                           const Tensor& o, const Tensor& rows, Tensor d_o) {
  if (!vectors_ok(d_o)) d_o = d_o.contiguous();
  void* stream = stream_of(q);
  const int64_t n_c = a.B * a.H * a.N, n_l = a.B * a.H * a.M;
  // one allocation for the fp32 temporaries: rowsum(o * do) and the row sums of dS (B,H,M each), then dlog_lambda (B,H,N)
  Tensor tmp = empty_floats(q, 2 * n_l + n_c);
  float* t = tmp.mutable_data_ptr<float>();
  Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
  Tensor dg = a.is_logit ? at::empty_like(g)
                         : at::empty_strided({a.B, a.head_first ? a.H : a.N, a.head_first ? a.N : a.H}, g_strides, tmp.options());
  fox_bwd_args args{};
  args.dims = a.dims(q);
  args.q = view_of(q, a.head_first);
  args.k = view_of(k, a.head_first);
  args.v = view_of(v, a.head_first);
  args.o = view_of(o, a.head_first);
  args.d_o = view_of(d_o, a.head_first);
  args.dq = view_of(dq, a.head_first);
  args.dk = view_of(dk, a.head_first);
  args.dv = view_of(dv, a.head_first);
  args.log_lambda = rows.const_data_ptr<float>();
  args.lse = args.log_lambda + lse_at(a);
  args.seq_start = a.seq_ptr();
  args.threshold = a.thr_ptr();
  args.sm_scale = (float)a.sm_scale;
  args.delta = t;
  args.drow = t + n_l;
  args.dlog_lambda = t + 2 * n_l;
  if (a.threshold.defined() && g_bounds_on.load(std::memory_order_relaxed)) record_bounds(a, q, args);
  if (!a.is_logit) {
    args.dlog_fgate = dg.mutable_data_ptr<float>();
    args.dlog_fgate_stride_b = dg.stride(0);
    args.dlog_fgate_stride_h = a.gs_h(dg);
    args.dlog_fgate_stride_n = a.gs_n(dg);
    check(fox_attn_bwd(&args, stream), "fox_attn_bwd");
  } else {
    check(fox_attn_bwd_logits(&args, g.const_data_ptr(), gate_dtype(g), g.stride(0), a.gs_h(g), a.gs_n(g), dg.mutable_data_ptr(),
                              dg.stride(0), a.gs_h(dg), a.gs_n(dg), stream), "fox_attn_bwd_logits");
  }
  return {dq, dk, dv, dg};
}

// dx, dg (undefined without a gate) and dweight (fp32) of the per-head RMS norm over rows of G heads of D elements
void run_norm_backward(const Tensor& x, const Tensor& gate, const Tensor& w32, const Tensor& rstd, const Tensor& dy, int64_t rows,
                       int64_t G, int64_t D, int act, double eps, Tensor& dx, Tensor& dgate, Tensor& dw) {
  dw = empty_floats(x, G * D);
  int64_t ws_bytes = 0;
  check(fox_norm_gate_workspace_bytes(rows, (int32_t)G, (int32_t)D, &ws_bytes), "fox_norm_gate_workspace_bytes");
  Tensor ws = empty_bytes_like(x, ws_bytes);
  fox_norm_gate_args n{};
  n.rows = rows;
  n.G = (int32_t)G;
  n.D = (int32_t)D;
  n.dtype = dtype_code(x);
  n.activation = act;
  n.eps = (float)eps;
  n.x = x.const_data_ptr();
  n.x_stride_row = G * D;
  if (gate.defined()) {
    n.g = gate.const_data_ptr();
    n.g_stride_row = G * D;
    n.dg = dgate.mutable_data_ptr();
    n.dg_stride_row = G * D;
  }
  n.weight = w32.const_data_ptr<float>();
  n.rstd = const_cast<float*>(rstd.const_data_ptr<float>());
  n.dy = dy.const_data_ptr();
  n.dy_stride_row = G * D;
  n.dx = dx.mutable_data_ptr();
  n.dx_stride_row = G * D;
  n.dweight = dw.mutable_data_ptr<float>();
  n.workspace = (float*)ws.mutable_data_ptr();
  check(fox_norm_gate_bwd(&n, stream_of(x)), "fox_norm_gate_bwd");
}

// Rows of heads * head_dim per token: (B, M, H, D) memory, whatever the logical order of the axes.  The strides have to be exactly
// those, also on an axis of length 1, since the kernels get them as they are.
bool heads_adjacent(const Tensor& t, bool head_first) {
  const fox_view v = view_of(t, head_first);
  const int64_t H = t.size(head_first ? 1 : 2), M = t.size(head_first ? 2 : 1), D = t.size(3);
  return t.stride(3) == 1 && v.stride_h == D && v.stride_t == H * D && v.stride_b == M * H * D && !(reinterpret_cast<uintptr_t>(v.ptr) & 15);
}
Tensor make_heads_adjacent(const Tensor& t, bool head_first) {
  if (heads_adjacent(t, head_first)) return t;
  const auto n = t.sizes();
  Tensor c = at::empty({n[0], n[head_first ? 2 : 1], n[head_first ? 1 : 2], n[3]}, t.options());
  if (head_first) c = c.transpose(1, 2);
  return c.copy_(t);
}

// Saved-tensor hooks may hand a tensor back with other strides than it was saved with; each backward brings what it reads into
// the layout that its kernel assumes.
Tensor packed(const Tensor& t) { return t.defined() ? t.contiguous() : t; }
Tensor vectors(const Tensor& t) { return vectors_ok(t) ? t : t.contiguous(); }

struct AttentionNode : public torch::autograd::Function<AttentionNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g,
                               const std::optional<Tensor>& gate, const std::optional<Tensor>& weight, Attention* a) {
    Forward f = run_forward(*a, q, k, v, g);
    ctx->save_for_backward({q, k, v, a->is_logit ? g : Tensor(), f.o, f.rows, a->seq_start, a->threshold, a->gate, a->weight, f.rstd});
    auto& d = ctx->saved_data;
    d["hf"] = a->head_first;
    d["logit"] = a->is_logit;
    d["scale"] = a->sm_scale;
    if (a->epilogue) {
      d["act"] = (int64_t)a->act;
      d["eps"] = a->eps;
      d["wtype"] = (int64_t)weight->scalar_type();
    }
    if (!a->is_logit) {
      // the gradient in the layout of the caller's gates when they are a permuted dense tensor: autograd takes it as it is
      if (g.is_non_overlapping_and_dense()) d["gs"] = g.strides();
      else d["gs"] = at::IntArrayRef{g.size(1) * g.size(2), g.size(2), 1};
      return {f.out};
    }
    Tensor log_fgate = a->head_first ? f.log_fgate : f.log_fgate.transpose(1, 2);
    ctx->mark_non_differentiable({log_fgate});
    return {f.out, log_fgate};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    auto& d = ctx->saved_data;
    const Tensor q = vectors(s[0]), k = vectors(s[1]), v = vectors(s[2]);
    Attention a;
    a.head_first = d["hf"].toBool();
    a.is_logit = d["logit"].toBool();
    a.sm_scale = d["scale"].toDouble();
    a.B = q.size(0);
    a.H = q.size(a.head_first ? 1 : 2);
    a.M = q.size(a.head_first ? 2 : 1);
    a.N = k.size(a.head_first ? 2 : 1);
    a.D = q.size(3);
    a.seq_start = packed(s[6]);
    a.threshold = packed(s[7]);
    const c10::DeviceGuard guard(q.device());
    if (!grads[0].defined()) return variable_list(7);
    Tensor d_o = grads[0], dgate, dweight;
    if (s[9].defined()) {   // the norm's backward first: its dx is the gradient of o
      const Tensor o = make_heads_adjacent(s[4], a.head_first), dy = make_heads_adjacent(grads[0], a.head_first);
      const Tensor gate = s[8].defined() ? make_heads_adjacent(s[8], a.head_first) : Tensor();
      auto rows_like = [&](void) {
        Tensor t = at::empty({a.B, a.M, a.H, a.D}, q.options());
        return a.head_first ? t.transpose(1, 2) : t;
      };
      d_o = rows_like();
      if (gate.defined()) dgate = rows_like();
      Tensor dw;
      run_norm_backward(o, gate, packed(s[9]), packed(s[10]), dy, a.B * a.M, a.H, a.D, (int)d["act"].toInt(), d["eps"].toDouble(), d_o, dgate, dw);
      dweight = dw.to((at::ScalarType)d["wtype"].toInt());
    }
    const std::vector<int64_t> g_strides = a.is_logit ? std::vector<int64_t>() : d["gs"].toIntVector();
    variable_list r = run_backward(a, q, k, v, s[3], g_strides, vectors(s[4]), packed(s[5]), d_o);
    return {r[0], r[1], r[2], r[3], dgate, dweight, Tensor()};
  }
};

// ---------------------------------------------------------------------------------------------------------------
// per-head RMS norm and token shift
// ---------------------------------------------------------------------------------------------------------------
struct NormNode : public torch::autograd::Function<NormNode> {
  static Tensor run(const Tensor& x, const Tensor& gate, const Tensor& w32, int act, double eps, int64_t G, Tensor& rstd) {
    const int64_t width = x.size(-1), rows = x.numel() / width;
    Tensor y = at::empty_like(x, x.options(), at::MemoryFormat::Contiguous);
    rstd = at::empty({rows, G}, x.options().dtype(at::kFloat));
    fox_norm_gate_args n{};
    n.rows = rows;
    n.G = (int32_t)G;
    n.D = (int32_t)(width / G);
    n.dtype = dtype_code(x);
    n.activation = act;
    n.eps = (float)eps;
    n.x = x.const_data_ptr();
    n.x_stride_row = width;
    if (gate.defined()) {
      n.g = gate.const_data_ptr();
      n.g_stride_row = width;
    }
    n.weight = w32.const_data_ptr<float>();
    n.y = y.mutable_data_ptr();
    n.y_stride_row = width;
    n.rstd = rstd.mutable_data_ptr<float>();
    check(fox_norm_gate_fwd(&n, stream_of(x)), "fox_norm_gate_fwd");
    return y;
  }

  static Tensor forward(AutogradContext* ctx, const Tensor& x, const std::optional<Tensor>& opt_gate, const Tensor& weight,
                        int64_t act, double eps, int64_t G) {
    const Tensor gate = opt_gate.value_or(Tensor()), w32 = weight.detach().to(at::kFloat).contiguous();
    Tensor rstd;
    Tensor y = run(x, gate, w32, (int)act, eps, G, rstd);
    ctx->save_for_backward({x, gate, w32, rstd});
    ctx->saved_data["act"] = act;
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["G"] = G;
    ctx->saved_data["wtype"] = (int64_t)weight.scalar_type();
    return y;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    auto& d = ctx->saved_data;
    if (!grads[0].defined()) return variable_list(6);
    const Tensor x = packed(s[0]), gate = packed(s[1]);
    const c10::DeviceGuard guard(x.device());
    const int64_t G = d["G"].toInt(), width = x.size(-1);
    Tensor dy = grads[0];
    if (!dy.is_contiguous() || !vectors_ok(dy)) dy = dy.contiguous();
    Tensor dx = at::empty_like(x), dg, dw;
    if (gate.defined()) dg = at::empty_like(gate);
    run_norm_backward(x, gate, packed(s[2]), packed(s[3]), dy, x.numel() / width, G, width / G, (int)d["act"].toInt(), d["eps"].toDouble(), dx, dg, dw);
    return {dx, dg, dw.to((at::ScalarType)d["wtype"].toInt()), Tensor(), Tensor(), Tensor()};
  }
};

struct ShiftNode : public torch::autograd::Function<ShiftNode> {
  static fox_shift_args args(const Tensor& x, const Tensor& prev_w, const Tensor& curr_w) {
    fox_shift_args a{};
    a.B = (int32_t)x.size(0);
    a.T = (int32_t)x.size(1);
    a.H = (int32_t)x.size(2);
    a.D = (int32_t)x.size(3);
    a.dtype = dtype_code(x);
    a.x = x.const_data_ptr();
    a.x_stride_b = x.stride(0);
    a.x_stride_t = x.stride(1);
    a.x_stride_h = x.stride(2);
    a.prev_weight = prev_w.const_data_ptr<float>();
    a.curr_weight = curr_w.const_data_ptr<float>();
    a.w_stride_b = prev_w.stride(0);
    a.w_stride_t = prev_w.stride(1);
    a.w_stride_h = prev_w.stride(2);
    return a;
  }
  static Tensor run(const Tensor& x, const Tensor& prev_w, const Tensor& curr_w) {
    Tensor out = at::empty_like(x);   // x is dense: the same strides
    fox_shift_args a = args(x, prev_w, curr_w);
    a.out = out.mutable_data_ptr();
    check(fox_token_shift_fwd(&a, stream_of(x)), "fox_token_shift_fwd");
    return out;
  }
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& prev_w, const Tensor& curr_w) {
    ctx->save_for_backward({x, prev_w, curr_w});
    return run(x, prev_w, curr_w);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    if (!grads[0].defined()) return variable_list(3);
    // one set of strides for x, dout and dx, one for the weights and their gradients
    const Tensor x = s[0].is_non_overlapping_and_dense() ? vectors(s[0]) : s[0].contiguous();
    const bool weights_ok = s[1].strides() == s[2].strides() && s[1].is_non_overlapping_and_dense();
    const Tensor prev_w = weights_ok ? s[1] : s[1].contiguous(), curr_w = weights_ok ? s[2] : s[2].contiguous();
    const c10::DeviceGuard guard(x.device());
    Tensor dout = grads[0];
    if (dout.strides() != x.strides() || (reinterpret_cast<uintptr_t>(dout.const_data_ptr()) & 15))
      dout = at::empty_like(x).copy_(dout);
    Tensor dx = at::empty_like(x), dprev = at::empty_like(prev_w), dcurr = at::empty_like(curr_w);
    fox_shift_args a = args(x, prev_w, curr_w);
    a.dout = dout.const_data_ptr();
    a.dx = dx.mutable_data_ptr();
    a.dprev_weight = dprev.mutable_data_ptr<float>();
    a.dcurr_weight = dcurr.mutable_data_ptr<float>();
    check(fox_token_shift_bwd(&a, stream_of(x)), "fox_token_shift_bwd");
    return {dx, dprev, dcurr};
  }
};

// ---------------------------------------------------------------------------------------------------------------
// Python entry points (METH_FASTCALL: the arguments come as a plain array).  Each returns None when the call is not one it
// handles.  The interpreter lock is free while they allocate, launch and build the graph: a launch may wait for room in a
// queue, and threads that drive other streams or devices must not wait with it (the argument array keeps its objects alive).
// ---------------------------------------------------------------------------------------------------------------
// Whether this thread runs under a function transform (vmap, grad, jvp, ...) or a Python dispatch mode.  The operators have no
// rules for transforms, and the general path's autograd nodes refuse to run under one, whether or not their tensors are wrapped;
// a mode sees, replaces or refuses the tensor operations of the general path.
bool under_transform_or_mode() {
  const auto keys = c10::impl::tls_local_dispatch_key_set().included_;
  return keys.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || keys.has(c10::DispatchKey::Python);
}

const Tensor* tensor_of(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;   // Tensor or Parameter: the general path's results keep other subclasses
  const Tensor& t = THPVariable_Unpack(o);
  // tensors with a dispatch of their own and the wrappers of functional transforms have no plain storage, negated views and zero
  // tensors hold other values than their memory; a dual tensor's tangent and a trace would be lost: all of these go through the
  // general path, which handles or refuses them
  if (t.key_set().has(c10::DispatchKey::Python) || !t.has_storage() || t.is_neg() || t._is_zerotensor() ||
      t._fw_grad(0).defined() || at::tracer::impl::is_dispatch_enabled() || under_transform_or_mode())
    return nullptr;
  return &t;
}

bool on_current_gpu(const Tensor& t) { return t.is_cuda() && t.device().index() == c10::hip::current_device(); }

bool sixteen_bit(const Tensor& t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }

bool needs_graph(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t && t->defined() && t->requires_grad()) return true;
  return false;
}

PyObject* none() { Py_RETURN_NONE; }

// The truth value of a Python flag, whatever type it comes in (bool, 0/1, numpy.bool_); false: it has none.
bool flag(PyObject* o, bool& value) {
  const int r = PyObject_IsTrue(o);
  if (r < 0) PyErr_Clear();   // the general path raises it again
  value = r > 0;
  return r >= 0;
}

std::optional<Tensor> some(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

// Fills `a` from the arguments both attention entry points share; false: not a call for the native path.
bool parse_attention(Attention& a, const Tensor* q, const Tensor* k, const Tensor* v, const Tensor* g, PyObject* head_first,
                     PyObject* seq_start, PyObject* sm_scale, PyObject* threshold, PyObject* is_logit) {
  if (!q || !k || !v || !g) return false;
  if (q->dim() != 4 || k->dim() != 4 || v->dim() != 4 || g->dim() != 3) return false;
  if (!on_current_gpu(*q) || k->device() != q->device() || v->device() != q->device() || g->device() != q->device()) return false;
  const auto dt = q->scalar_type();
  if (!sixteen_bit(*q) || k->scalar_type() != dt || v->scalar_type() != dt) return false;
  if (!flag(is_logit, a.is_logit) || !flag(head_first, a.head_first)) return false;
  if (a.is_logit ? gate_dtype(*g) < 0 : g->scalar_type() != at::kFloat) return false;
  const int ih = a.head_first ? 1 : 2, it = a.head_first ? 2 : 1;
  a.B = q->size(0);
  a.H = q->size(ih);
  a.M = q->size(it);
  a.N = k->size(it);
  a.D = q->size(3);
  if (!head_dim_ok(a.D) || a.B < 1 || a.H < 1 || a.M < 1 || a.M > a.N || a.N > INT32_MAX || a.B * a.H > INT32_MAX) return false;
  if (k->size(0) != a.B || k->size(ih) != a.H || k->size(3) != a.D || v->sizes() != k->sizes()) return false;
  if (g->size(0) != a.B || g->size(ih) != a.H || g->size(it) != a.N) return false;
  if (!vectors_ok(*q) || !vectors_ok(*k) || !vectors_ok(*v)) return false;
  if (seq_start != Py_None) {
    const Tensor* s = tensor_of(seq_start);
    if (!s || s->dim() != 1 || s->size(0) != a.B || s->device() != q->device() || s->scalar_type() != at::kLong || !s->is_contiguous())
      return false;
    a.seq_start = *s;
  }
  if (threshold != Py_None) {
    if (PyUnicode_Check(threshold)) {
      if (PyUnicode_CompareWithASCIIString(threshold, "auto") != 0) return false;
      a.auto_threshold = true;
    } else {
      const Tensor* t = tensor_of(threshold);
      if (!t || t->scalar_type() != at::kFloat || t->device() != q->device() || t->dim() > 2) return false;
      if (at::GradMode::is_enabled() && t->requires_grad()) return false;   // an input of the node there, with no gradient
      if (t->dim() == 2 && t->size(0) == a.B && t->size(1) == a.H && t->is_contiguous()) {
        a.threshold = t->detach();
      } else {
        if (t->dim() >= 1 && t->size(-1) != a.H && t->size(-1) != 1) return false;
        if (t->dim() == 2 && t->size(0) != a.B && t->size(0) != 1) return false;
        a.threshold = t->detach().expand({a.B, a.H}).contiguous();
      }
    }
  }
  if (sm_scale == Py_None) {
    a.sm_scale = 1.0 / std::sqrt((double)a.D);
  } else {
    a.sm_scale = PyFloat_AsDouble(sm_scale);
    if (a.sm_scale == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
  }
  return true;
}

// (out,) or, from the gate logits, (out, log_fgate)
PyObject* finish_attention(Attention& a, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& gate,
                           const Tensor& weight) {
  variable_list out;
  {
    const pybind11::gil_scoped_release no_gil;
    if (needs_graph({&q, &k, &v, &g, &gate, &weight})) {
      out = AttentionNode::apply(q, k, v, g, some(gate), some(weight), &a);
    } else {
      const at::NoGradGuard no_grad;
      if (decodes_from_gates(a)) {
        out.push_back(run_decode(a, q, k, v, g));
      } else {
        Forward f = run_forward(a, q, k, v, g);
        out.push_back(f.out);
        if (a.is_logit) out.push_back(a.head_first ? f.log_fgate : f.log_fgate.transpose(1, 2));
      }
    }
  }
  if (!a.is_logit) return THPVariable_Wrap(out[0]);
  PyObject* pair = PyTuple_New(2);
  if (!pair) return nullptr;
  PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(out[0]));
  PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(out[1]));
  return pair;
}

// attention(q, k, v, gates, head_first, seq_start, sm_scale, threshold, gates_are_logits)
PyObject* py_attention(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 9, "attention takes 9 arguments");
  Attention a;
  const Tensor *q = tensor_of(o[0]), *k = tensor_of(o[1]), *v = tensor_of(o[2]), *g = tensor_of(o[3]);
  if (!parse_attention(a, q, k, v, g, o[4], o[5], o[6], o[7], o[8])) return none();
  return finish_attention(a, *q, *k, *v, *g, Tensor(), Tensor());
  END_HANDLE_TH_ERRORS
}

// attention_norm_gate(q, k, v, gates, gate, weight, activation, eps, head_first, seq_start, sm_scale, threshold, gates_are_logits)
PyObject* py_attention_norm_gate(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 13, "attention_norm_gate takes 13 arguments");
  Attention a;
  const Tensor *q = tensor_of(o[0]), *k = tensor_of(o[1]), *v = tensor_of(o[2]), *g = tensor_of(o[3]), *w = tensor_of(o[5]);
  if (!parse_attention(a, q, k, v, g, o[8], o[9], o[10], o[11], o[12])) return none();
  Tensor gate;
  if (o[4] != Py_None) {
    const Tensor* t = tensor_of(o[4]);
    if (!t || t->sizes() != q->sizes() || t->scalar_type() != q->scalar_type() || t->device() != q->device() ||
        !heads_adjacent(*t, a.head_first))
      return none();
    gate = *t;
  }
  if (!w || w->dim() != 1 || w->size(0) != a.H * a.D || w->device() != q->device() || !w->is_floating_point()) return none();
  a.epilogue = true;
  a.gate = gate;
  a.weight = w->detach().to(at::kFloat).contiguous();
  a.act = (int)PyLong_AsLong(o[6]);
  a.eps = PyFloat_AsDouble(o[7]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return none();
  }
  return finish_attention(a, *q, *k, *v, *g, gate, *w);
  END_HANDLE_TH_ERRORS
}

// norm(x, gate or None, weight, activation, eps, num_groups)
PyObject* py_norm(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 6, "norm takes 6 arguments");
  const Tensor *x = tensor_of(o[0]), *w = tensor_of(o[2]);
  if (!x || !w || x->dim() < 1 || x->numel() == 0 || !on_current_gpu(*x) || !sixteen_bit(*x) || !x->is_contiguous() || !vectors_ok(*x)) return none();
  Tensor gate;
  if (o[1] != Py_None) {
    const Tensor* t = tensor_of(o[1]);
    if (!t || t->sizes() != x->sizes() || t->scalar_type() != x->scalar_type() || t->device() != x->device() || !t->is_contiguous() || !vectors_ok(*t))
      return none();
    gate = *t;
  }
  const long act = PyLong_AsLong(o[3]), G = PyLong_AsLong(o[5]);
  const double eps = PyFloat_AsDouble(o[4]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return none();
  }
  const int64_t width = x->size(-1);
  if (G < 1 || width % G || !head_dim_ok(width / G)) return none();
  if (w->dim() != 1 || w->size(0) != width || w->device() != x->device() || !w->is_floating_point()) return none();
  Tensor y;
  {
    const pybind11::gil_scoped_release no_gil;
    if (needs_graph({x, &gate, w})) {
      y = NormNode::apply(*x, some(gate), *w, (int64_t)act, eps, (int64_t)G);
    } else {
      const at::NoGradGuard no_grad;
      Tensor rstd;
      y = NormNode::run(*x, gate, w->detach().to(at::kFloat).contiguous(), (int)act, eps, G, rstd);
    }
  }
  return THPVariable_Wrap(y);
  END_HANDLE_TH_ERRORS
}

// token_shift(x, prev_weight, curr_weight)
PyObject* py_token_shift(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 3, "token_shift takes 3 arguments");
  const Tensor *x = tensor_of(o[0]), *p = tensor_of(o[1]), *c = tensor_of(o[2]);
  if (!x || !p || !c || x->dim() != 4 || p->dim() != 3 || x->numel() == 0 || !on_current_gpu(*x) || !sixteen_bit(*x) || !vectors_ok(*x) ||
      !x->is_non_overlapping_and_dense() || !head_dim_ok(x->size(3)))
    return none();
  if (p->scalar_type() != at::kFloat || c->scalar_type() != at::kFloat || p->device() != x->device() || c->device() != x->device()) return none();
  if (p->sizes() != x->sizes().slice(0, 3) || c->sizes() != p->sizes() || p->strides() != c->strides() || !p->is_non_overlapping_and_dense())
    return none();
  Tensor out;
  {
    const pybind11::gil_scoped_release no_gil;
    if (needs_graph({x, p, c})) {
      out = ShiftNode::apply(*x, *p, *c);
    } else {
      const at::NoGradGuard no_grad;
      out = ShiftNode::run(*x, *p, *c);
    }
  }
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// qk_norm_threshold(q_weight, k_weight, num_heads, head_dim, seq_len, tolerance, shared)
PyObject* py_qk_norm_threshold(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 7, "qk_norm_threshold takes 7 arguments");
  const Tensor *q = tensor_of(o[0]), *k = tensor_of(o[1]);
  // (a tensor as tolerance would have to be read back from the device here; the general path adds it)
  if (!PyFloat_Check(o[5]) && !PyLong_Check(o[5])) return none();
  const long H = PyLong_AsLong(o[2]), D = PyLong_AsLong(o[3]);
  const double T = PyFloat_AsDouble(o[4]), tolerance = PyFloat_AsDouble(o[5]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return none();
  }
  bool shared = false;
  if (!flag(o[6], shared)) return none();
  if (!q || !k || H < 1 || D < 1 || !(T > 0) || !on_current_gpu(*q) || k->device() != q->device() || q->dim() != 1 || q->sizes() != k->sizes() ||
      q->size(0) != (shared ? D : H * D) || q->scalar_type() != at::kFloat || k->scalar_type() != at::kFloat || !q->is_contiguous() || !k->is_contiguous())
    return none();
  Tensor thr;
  {
    const pybind11::gil_scoped_release no_gil;
    const at::NoGradGuard no_grad;
    thr = shared ? at::empty({}, q->options()) : at::empty({H}, q->options());
    check(fox_qk_norm_threshold(q->const_data_ptr<float>(), k->const_data_ptr<float>(), shared ? 1 : (int32_t)H, (int32_t)D, T, tolerance,
                                thr.mutable_data_ptr<float>(), stream_of(*q)), "fox_qk_norm_threshold");
  }
  return THPVariable_Wrap(thr);
  END_HANDLE_TH_ERRORS
}

// cache_append(k_buf, v_buf, g_buf, k, v, g, old) -> views of the filled part of the three buffers
PyObject* py_cache_append(PyObject*, PyObject* const* o, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(n == 7, "cache_append takes 7 arguments");
  const Tensor* t[6];
  for (int i = 0; i < 6; ++i) {
    t[i] = tensor_of(o[i]);
    if (!t[i] || t[i]->dim() != (i % 3 == 2 ? 3 : 4) || t[i]->numel() == 0 || !on_current_gpu(*t[i])) return none();
    if (i % 3 == 2 ? t[i]->scalar_type() != at::kFloat : !sixteen_bit(*t[i]) || !vectors_ok(*t[i])) return none();
    // what the copies of the general path would record or refuse, or may not do in one pass
    if (at::GradMode::is_enabled() && t[i]->requires_grad()) return none();
    if (i < 3 && t[i]->is_inference() && !c10::InferenceMode::is_enabled()) return none();
    if (i >= 3 && (t[i]->storage().is_alias_of(t[0]->storage()) || t[i]->storage().is_alias_of(t[1]->storage()) ||
                   t[i]->storage().is_alias_of(t[2]->storage())))
      return none();
  }
  const Tensor &kb = *t[0], &vb = *t[1], &gb = *t[2], &k = *t[3], &v = *t[4], &g = *t[5];
  const int64_t old = PyLong_AsLongLong(o[6]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return none();
  }
  const int64_t B = k.size(0), H = k.size(1), T = k.size(2), D = k.size(3);
  if (v.sizes() != k.sizes() || g.sizes() != k.sizes().slice(0, 3) || kb.sizes() != vb.sizes() || gb.sizes() != kb.sizes().slice(0, 3) ||
      kb.size(0) != B || kb.size(1) != H || kb.size(3) != D || kb.scalar_type() != k.scalar_type() || vb.scalar_type() != v.scalar_type() ||
      D % 8 || old < 0 || old + T > kb.size(2) || T > (1 << 30) || B * H * T * (D / 8) > INT32_MAX)
    return none();
  fox_cache_append_args a{};
  a.B = (int32_t)B; a.H = (int32_t)H; a.T = (int32_t)T; a.D = (int32_t)D;
  a.old = old;
  a.k = view_of(k, true);
  a.v = view_of(v, true);
  a.g = g.const_data_ptr<float>();
  a.g_stride_b = g.stride(0); a.g_stride_h = g.stride(1); a.g_stride_n = g.stride(2);
  a.k_buf = view_of(kb, true);
  a.v_buf = view_of(vb, true);
  a.g_buf = gb.mutable_data_ptr<float>();
  a.g_buf_stride_b = gb.stride(0); a.g_buf_stride_h = gb.stride(1); a.g_buf_stride_n = gb.stride(2);
  {
    const pybind11::gil_scoped_release no_gil;
    check(fox_cache_append(&a, stream_of(k)), "fox_cache_append");
  }
  PyObject* out = PyTuple_New(3);
  if (!out) return nullptr;
  for (int i = 0; i < 3; ++i) {
    if (!t[i]->is_inference()) t[i]->unsafeGetTensorImpl()->bump_version();   // an in-place write, as copy_ is
    PyTuple_SET_ITEM(out, i, THPVariable_Wrap(t[i]->narrow(2, 0, old + T)));
  }
  return out;
  END_HANDLE_TH_ERRORS
}

// record_bounds(list or None)
PyObject* py_record_bounds(PyObject*, PyObject* list) {
  if (list != Py_None && !PyList_Check(list)) {
    PyErr_SetString(PyExc_TypeError, "record_bounds takes a list or None");
    return nullptr;
  }
  PyObject* old = g_bounds;
  g_bounds = list == Py_None ? nullptr : list;
  Py_XINCREF(g_bounds);
  g_bounds_on.store(g_bounds != nullptr, std::memory_order_relaxed);
  Py_XDECREF(old);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"record_bounds", (PyCFunction)py_record_bounds, METH_O, nullptr},
    {"cache_append", (PyCFunction)(void (*)(void))py_cache_append, METH_FASTCALL, nullptr},
    {"qk_norm_threshold", (PyCFunction)(void (*)(void))py_qk_norm_threshold, METH_FASTCALL, nullptr},
    {"attention", (PyCFunction)(void (*)(void))py_attention, METH_FASTCALL, nullptr},
    {"attention_norm_gate", (PyCFunction)(void (*)(void))py_attention_norm_gate, METH_FASTCALL, nullptr},
    {"norm", (PyCFunction)(void (*)(void))py_norm, METH_FASTCALL, nullptr},
    {"token_shift", (PyCFunction)(void (*)(void))py_token_shift, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_fox_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fox_torch() { return PyModule_Create(&module_def); }

// Host path of the Python shim in native code: landmark_hip/_native.so, loaded by landmark_hip/_lib.py.
//
// A training step on a short sequence or a decode step keeps the GPU busy for 20-100 us, and the same calls made from
// Python -- a descriptor per tensor, a conversion per argument, an autograd node that has to take the interpreter lock
// in the engine's thread -- take as long or longer.  Here an entry point of the shim is one call: arguments are read
// from the tensors, outputs and workspaces come from torch's allocator, the launches go through the C ABI of
// include/lmk.h (liblandmark_hip.so) on torch's current stream, and the backward is a C++ autograd node.
//
// Errors keep their Python types: AssertionError for what the shim asserts, LmkError for a code of the C ABI.
#include <Python.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/lmk.h"

namespace {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

PyObject* g_lmk_error = nullptr;                         // landmark_hip._lib.LmkError

struct Failed {                                          // an error on its way to Python
  int code;                                              // of the C ABI; 0: an AssertionError
  std::string text;
};
void need(bool ok, const char* text) {
  if (!ok) throw Failed{0, text};
}
void check(int code) {
  if (code != 0) throw Failed{code, lmk_strerror(code)};
}
void set_python_error(const Failed& f) {                 // with the interpreter lock held
  if (f.code == 0 || g_lmk_error == nullptr) {
    PyErr_SetString(f.code == 0 ? PyExc_AssertionError : PyExc_RuntimeError, f.text.c_str());
    return;
  }
  PyObject* e = PyObject_CallFunction(g_lmk_error, "is", f.code, f.text.c_str());
  if (e == nullptr) return;
  PyErr_SetObject(g_lmk_error, e);
  Py_DECREF(e);
}

// Runs f without the interpreter lock.
template <class F>
auto without_gil(F&& f) {
  struct Release {
    PyThreadState* s = PyEval_SaveThread();
    ~Release() { PyEval_RestoreThread(s); }
  } release;
  return f();
}

// Calls that torch has to see as one operation: torch.jit.trace would record no more of what is done here than the
// allocation of the outputs, and a forward-mode gradient of an input would be lost where a Function without a jvp refuses
// it.  Such a call is left to an autograd Function, in Python.
bool left_to_a_function(std::initializer_list<Tensor> inputs) {
  if (torch::jit::tracer::isTracing()) return true;
  for (const Tensor& t : inputs)
    if (t.defined() && t._fw_grad(/*level=*/0).defined()) return true;
  return false;
}

// ---- what the kernels take
int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return LMK_DTYPE_BF16;
    case at::kHalf: return LMK_DTYPE_F16;
    default: return -1;
  }
}
lmk_tensor4 t4(const Tensor& t) {
  const auto s = t.strides();
  need(s.size() == 4 && s[3] == 1, "a tensor of four dimensions, the last one dense");
  return lmk_tensor4{t.data_ptr(), s[0], s[1], s[2]};
}
// Tensors the kernels can read in place (unit stride along D, rows walked forwards, 16-byte aligned) as they are,
// others as a contiguous copy.
Tensor kernel_ready(const Tensor& t) {
  const auto s = t.strides();
  const bool ok = s[3] == 1 && s[2] > 0 && ((s[0] | s[1] | s[2]) & 7) == 0 &&
                  (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
  return ok ? t : t.contiguous();
}
void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor bytes_on(const Tensor& like, size_t n) {
  return at::empty({(int64_t)n}, like.options().dtype(at::kByte));
}
bool same_shape(const Tensor& a, const Tensor& b) { return a.sizes() == b.sizes(); }

// ---- attention
// How a block of tokens is stored: BLOCKS = tensors as they are, any block of 2..128 tokens; PADDED = rows of `block`
// slots of which `block_real` hold tokens (all of them for a native block size).
struct Shape {
  int B, H, Lq, Lk, D, n_prefix, block, block_real, dtype;
  bool blocks;
  float scale;
};

Shape shape_of(const Tensor& q, const Tensor& k, int n_prefix, double scale, int block, int block_real, bool blocks) {
  return Shape{(int)q.size(0), (int)q.size(1), (int)q.size(2), (int)k.size(2), (int)q.size(3), n_prefix, block, block_real,
               dtype_code(q), blocks, (float)scale};
}

// (o, statistics): statistics (2, B*H, Lq) fp32, the forward's L and M.
std::pair<Tensor, Tensor> forward(const Shape& s, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& group_scale) {
  Tensor o = at::empty_like(q);                          // keeps q's memory layout
  Tensor st = at::empty({2, (int64_t)s.B * s.H, s.Lq}, q.options().dtype(at::kFloat));
  const lmk_tensor4 tq = t4(q), tk = t4(k), tv = t4(v), to = t4(o);
  float* L = st.data_ptr<float>();
  float* M = L + (int64_t)s.B * s.H * s.Lq;
  void* stream = stream_of(q);
  if (group_scale.defined())
    check(lmk_attn_fwd_group_scale(&tq, &tk, &tv, &to, L, M, group_scale.data_ptr<float>(), s.B, s.H, s.Lq, s.Lk, s.D, s.scale,
                                   s.block, s.n_prefix, s.dtype, stream));
  else if (s.blocks)
    check(lmk_attn_fwd_blocks(&tq, &tk, &tv, &to, L, M, s.B, s.H, s.Lq, s.Lk, s.D, s.scale, s.block, s.n_prefix, s.dtype, stream));
  else
    check(lmk_attn_fwd_padded(&tq, &tk, &tv, &to, L, M, s.B, s.H, s.Lq, s.Lk, s.D, s.scale, s.block, s.block_real, s.n_prefix,
                              s.dtype, stream));
  return {o, st};
}

struct HandoverLimits {                                  // HANDOVER_MAX_BYTES, HANDOVER_MIN_KEYS of attention.py
  int64_t max_bytes, min_keys;
};

variable_list backward(const Shape& s, const HandoverLimits& limits, const Tensor& q, const Tensor& k, const Tensor& v,
                       const Tensor& o, const float* l, const float* m, const Tensor& dout, const Tensor& group_scale) {
  Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);   // each in its input's layout
  size_t nbytes;
  if (group_scale.defined()) {
    nbytes = lmk_attn_bwd_group_scale_workspace_bytes(s.B, s.H, s.Lq, s.Lk, s.block);
  } else if (s.blocks) {
    nbytes = lmk_attn_bwd_blocks_workspace_bytes(s.B, s.H, s.Lq, s.Lk, s.block);
  } else {
    nbytes = lmk_attn_bwd_workspace_bytes(s.B, s.H, s.Lq, s.Lk, s.block);
    if (s.block_real == s.block) {
      const size_t ho = lmk_attn_bwd_handover_workspace_bytes(s.B, s.H, s.Lq, s.Lk, s.block);
      if (ho > 0 && (int64_t)ho <= limits.max_bytes && s.Lk >= limits.min_keys) nbytes = ho;   // the size picks the kernels
    }
  }
  Tensor ws = bytes_on(q, nbytes);
  const lmk_tensor4 tq = t4(q), tk = t4(k), tv = t4(v), to = t4(o), tdo = t4(dout), tdq = t4(dq), tdk = t4(dk), tdv = t4(dv);
  void* stream = stream_of(q);
  if (group_scale.defined())
    check(lmk_attn_bwd_group_scale(&tq, &tk, &tv, &to, &tdo, l, m, group_scale.data_ptr<float>(), &tdq, &tdk, &tdv,
                                   ws.data_ptr(), nbytes, s.B, s.H, s.Lq, s.Lk, s.D, s.scale, s.block, s.n_prefix, s.dtype, stream));
  else if (s.blocks)
    check(lmk_attn_bwd_blocks(&tq, &tk, &tv, &to, &tdo, l, m, &tdq, &tdk, &tdv, ws.data_ptr(), nbytes, s.B, s.H, s.Lq, s.Lk,
                              s.D, s.scale, s.block, s.n_prefix, s.dtype, stream));
  else
    check(lmk_attn_bwd_padded(&tq, &tk, &tv, &to, &tdo, l, m, &tdq, &tdk, &tdv, ws.data_ptr(), nbytes, s.B, s.H, s.Lq, s.Lk,
                              s.D, s.scale, s.block, s.block_real, s.n_prefix, s.dtype, stream));
  return {dq, dk, dv};
}

// Runs a backward's body in the engine's thread; an error of ours leaves as the Python exception it stands for.
template <class F>
variable_list node_body(F&& f) {
  try {
    return f();
  } catch (const Failed& e) {
    PyGILState_STATE g = PyGILState_Ensure();
    set_python_error(e);
    python_error err;
    err.persist();
    PyGILState_Release(g);
    throw err;
  }
}

// A tensor saved for the backward.  Saved-tensor hooks may hand back any other in its place: one that is not what was saved
// is refused before a kernel is given its address.
struct Saved {
  SavedVariable x;
  at::DimVector shape;
  at::ScalarType type = at::kFloat;
  at::Device device = at::kCPU;

  Saved() = default;
  Saved(const Tensor& t, bool is_output) : x(t, is_output), shape(t.sizes()), type(t.scalar_type()), device(t.device()) {}
  Tensor unpack(std::shared_ptr<torch::autograd::Node> saved_for = nullptr) const {
    Tensor t = x.unpack(std::move(saved_for));
    need(t.defined() && t.sizes() == shape && t.scalar_type() == type && t.device() == device,
         "saved-tensor hooks must hand back the shape, type and device that were saved");
    return t;
  }
};

struct AttentionBackward : public torch::autograd::Node {
  Saved q, k, v, o, st, gs;
  bool has_gs = false;
  Shape s;
  HandoverLimits limits;

  // The tensors the backward works on: unpacked and released by one thread at a time, as torch's generated nodes do it.
  // (Hooks may run meanwhile, so no thread may wait here with the interpreter lock held.)
  struct Unpacked {
    Tensor q, k, v, o, st, gs;
  };
  Unpacked unpack(std::shared_ptr<Node> self) {
    std::lock_guard<std::mutex> lock(mutex_);
    return {q.unpack(), k.unpack(), v.unpack(), o.unpack(std::move(self)), st.unpack(), has_gs ? gs.unpack() : Tensor()};
  }

  variable_list apply(variable_list&& grads) override {
    return node_body([&] {
      // an output that no gradient reaches: zeros, as an autograd Function is given
      const Tensor dout = grads[0].defined() ? grads[0] : input_metadata(0).zeros_like();
      need(s.Lq % s.block_real == 0 && s.Lk % s.block_real == 0, "Backward supported only for full blocks");
      const Unpacked t = unpack(getptr());
      at::AutoDispatchBelowADInplaceOrView guard;
      c10::DeviceGuard device(t.q.device());
      const Tensor stats = t.st.contiguous(), factors = has_gs ? t.gs.contiguous() : Tensor();
      const float* L = stats.data_ptr<float>();
      return backward(s, limits, t.q, t.k, t.v, t.o, L, L + (int64_t)s.B * s.H * s.Lq, kernel_ready(dout), factors);
    });
  }
  std::string name() const override { return "FusedLandmarkAttentionBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (Saved* s : {&q, &k, &v, &o, &st, &gs}) s->x.reset_data();
  }
};

// fused_landmark_attention for landmarks at fixed stride, head dims 64 and 128.
Tensor attention(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, const Tensor& gs_in, bool has_scale, double scale,
                 int64_t block, HandoverLimits limits) {
  need(q_in.dim() == 4 && k_in.dim() == 4 && v_in.dim() == 4, "q, k, v are (batch, heads, rows, head dim)");
  const int64_t Lq = q_in.size(2), Lk = k_in.size(2), D = q_in.size(3);
  need(block > 0 && (Lk - Lq) % block == 0, "the keys in front of the first query must be whole blocks");
  need(k_in.size(0) == q_in.size(0) && k_in.size(1) == q_in.size(1) && k_in.size(3) == D && same_shape(k_in, v_in),
       "k and v must have the same shape, and q's batch, heads and head dim");
  need(D <= 128, "FlashAttention only support head dimensions up to 128");
  need(q_in.scalar_type() == k_in.scalar_type() && q_in.scalar_type() == v_in.scalar_type(), "All tensors must have the same type");
  need(q_in.is_cuda() && k_in.is_cuda() && v_in.is_cuda(), "q, k, v must be on the GPU");
  need(dtype_code(q_in) >= 0, "HIP kernels are built for bf16 and fp16");
  need(D == 64 || D == 128, "HIP kernels are built for head dims (64, 128)");
  const int n_prefix = (int)((Lk - Lq) / block);
  const bool native = block == 32 || block == 64 || block == 128, has_gs = gs_in.defined();
  if (has_gs) {
    need(block >= 2 && block <= 128, "group dropout: blocks of 2..128 tokens");
    need(gs_in.dim() == 4 && gs_in.size(0) == q_in.size(0) && gs_in.size(1) == q_in.size(1) && gs_in.size(2) == Lk / block &&
             gs_in.size(3) == Lq && gs_in.scalar_type() == at::kFloat && gs_in.device() == q_in.device(),
         "group_scale is (B, H, Lk / block_size, Lq) fp32 on q's device");
  }
  if (!has_scale) scale = 1.0 / std::sqrt((double)D);
  c10::DeviceGuard device(q_in.device());
  Tensor q, k, v, gs;
  std::pair<Tensor, Tensor> r;
  const bool differentiate =
      at::GradMode::is_enabled() && (q_in.requires_grad() || k_in.requires_grad() || v_in.requires_grad());
  Shape s;
  {
    at::AutoDispatchBelowADInplaceOrView guard;
    q = kernel_ready(q_in);
    k = kernel_ready(k_in);
    v = kernel_ready(v_in);
    if (has_gs) gs = gs_in.contiguous();
    s = shape_of(q, k, n_prefix, scale, (int)block, (int)block, !native);
    r = forward(s, q, k, v, gs);
  }
  if (differentiate) {
    auto node = std::shared_ptr<AttentionBackward>(new AttentionBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(q_in, k_in, v_in));
    // a tensor that was copied into kernel layout is saved as that copy, and has no history of its own
    node->q = Saved(q, false);
    node->k = Saved(k, false);
    node->v = Saved(v, false);
    node->st = Saved(r.second, false);
    node->has_gs = has_gs;
    if (has_gs) node->gs = Saved(gs, false);
    node->s = s;
    node->limits = limits;
    torch::autograd::set_history(r.first, node);
    node->o = Saved(r.first, true);
  }
  return r.first;
}

// ---- rotary embedding
struct Tables {
  Tensor cos, sin;
};
// (n_pos, D) views of the tables the kernels can read: unit stride along D, 16-byte aligned rows, one row stride.
Tables tables(const Tensor& cos_in, const Tensor& sin_in, at::ScalarType dtype) {
  Tensor cos = cos_in.dim() == 2 ? cos_in : cos_in.reshape({-1, cos_in.size(-1)});
  Tensor sin = sin_in.dim() == 2 ? sin_in : sin_in.reshape({-1, sin_in.size(-1)});
  need(cos.scalar_type() == dtype && sin.scalar_type() == dtype, "rotary tables must be in the model dtype (llama_mem.py:121-124)");
  need(same_shape(cos, sin), "the rotary tables must have one shape");
  auto aligned = [](const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; };
  if (cos.stride(1) != 1 || cos.stride(0) % 8 || !aligned(cos)) cos = cos.contiguous();
  if (sin.stride(1) != 1 || sin.stride(0) != cos.stride(0) || !aligned(sin)) {
    sin = sin.contiguous();
    cos = cos.contiguous();
  }
  return {cos, sin};
}

// q may be undefined; `transposed`: the rotation the gradient takes.
std::pair<Tensor, Tensor> rotate(const Tensor& q_in, const Tensor& k_in, const Tables& t, const Tensor& pos, bool transposed) {
  const Tensor k = kernel_ready(k_in), q = q_in.defined() ? kernel_ready(q_in) : Tensor();
  Tensor ko = at::empty_like(k), qo = q.defined() ? at::empty_like(q) : Tensor();
  const int B = (int)k.size(0), H = (int)k.size(1), L = (int)k.size(2), D = (int)k.size(3);
  const int64_t pos_stride = (pos.size(0) == B && B > 1) ? L : 0;
  const lmk_tensor4 tk = t4(k), tko = t4(ko);
  lmk_tensor4 tq = {}, tqo = {};
  if (q.defined()) {
    tq = t4(q);
    tqo = t4(qo);
  }
  check(lmk_rotate_qk(&tk, &tko, q.defined() ? &tq : nullptr, q.defined() ? &tqo : nullptr, t.cos.data_ptr(),
                                t.sin.data_ptr(), t.cos.stride(0), t.cos.size(0), pos.data_ptr<int64_t>(), pos_stride, B, H, L, D,
                                dtype_code(k), transposed ? 1 : 0, stream_of(k)));
  return {qo, ko};
}

struct RotaryArgs {
  Tables t;
  Tensor pos;
};
struct RotaryBackward : public torch::autograd::Node {
  Saved cos, sin, pos;
  bool has_q = false;

  variable_list apply(variable_list&& grads) override {
    return node_body([&]() -> variable_list {
      Tensor cos_, sin_, pos_;
      {
        std::lock_guard<std::mutex> lock(mutex_);          // against release_variables in another thread
        cos_ = cos.unpack();
        sin_ = sin.unpack();
        pos_ = pos.unpack();
      }
      at::AutoDispatchBelowADInplaceOrView guard;
      const RotaryArgs args = {tables(cos_, sin_, cos_.scalar_type()), pos_.contiguous()};
      const Tensor &gk = grads[has_q ? 1 : 0], gq = has_q ? grads[0] : Tensor();
      if (!gk.defined() && !gq.defined()) return has_q ? variable_list{Tensor(), Tensor()} : variable_list{Tensor()};
      c10::DeviceGuard device((gk.defined() ? gk : gq).device());
      if (!has_q) return {rotate(Tensor(), gk, args.t, args.pos, true).second};
      if (!gk.defined()) return {rotate(Tensor(), gq, args.t, args.pos, true).second, Tensor()};
      auto r = rotate(gq, gk, args.t, args.pos, true);
      return {r.first, r.second};
    });
  }
  std::string name() const override { return "RotaryEmbeddingBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (Saved* s : {&cos, &sin, &pos}) s->x.reset_data();
  }
};

// What rotate() takes besides the rows x, checked and laid out as the kernel reads it.
RotaryArgs rotary_args(const Tensor& x, const Tensor& cos, const Tensor& sin, const Tensor& pos) {
  need(x.dim() == 4 && x.is_cuda() && dtype_code(x) >= 0, "k is (batch, heads, rows, head dim), bf16 or fp16, on the GPU");
  need(pos.dim() == 2 && pos.size(1) == x.size(2) && (pos.size(0) == 1 || pos.size(0) == x.size(0)),
       "position_ids is (1, rows) or (batch, rows)");
  need(pos.scalar_type() == at::kLong && pos.device() == x.device(), "position_ids is int64 on k's device");
  return {tables(cos, sin, x.scalar_type()), pos.contiguous()};
}

// apply_rotary_pos_emb; q undefined or of k's shape
std::pair<Tensor, Tensor> rotary(const Tensor& q, const Tensor& k, const Tensor& cos, const Tensor& sin, const Tensor& pos) {
  need(!q.defined() || (q.scalar_type() == k.scalar_type() && q.device() == k.device()), "q and k must have one type and device");
  c10::DeviceGuard device(k.device());
  const bool has_q = q.defined();
  RotaryArgs a;
  std::pair<Tensor, Tensor> r;
  {
    at::AutoDispatchBelowADInplaceOrView guard;
    a = rotary_args(k, cos, sin, pos);
    r = rotate(q, k, a.t, a.pos, false);
  }
  if (at::GradMode::is_enabled() && (k.requires_grad() || (has_q && q.requires_grad()))) {
    auto node = std::shared_ptr<RotaryBackward>(new RotaryBackward(), torch::autograd::deleteNode);
    node->set_next_edges(has_q ? torch::autograd::collect_next_edges(q, k) : torch::autograd::collect_next_edges(k));
    node->cos = Saved(a.t.cos, false);
    node->sin = Saved(a.t.sin, false);
    node->pos = Saved(a.pos, false);
    node->has_q = has_q;
    if (has_q) torch::autograd::set_history(r.first, node);
    torch::autograd::set_history(r.second, node);
  }
  return r;
}

// ---- the mem-cache step
// Where a cache's new rows go: the buffers and the row of the first new token.
struct Append {
  Tensor k_nopos, k_buf, v_buf;
  int64_t row;
};

// One step of the mem-cache path over the first S rows of k_cache, v_cache: (out, idx), and the append.  `shared`: one
// selection per head.
std::pair<Tensor, Tensor> mem_cache_step(const Tensor& q_in, const Tensor& kc_in, const Tensor& vc_in, int64_t S,
                                         const Tensor& kl_in, const Tensor& vl_in, const Tensor& cos, const Tensor& sin,
                                         int block, int top_k, bool has_scale, double scale, bool shared, Tensor ws, bool reuse,
                                         const Append* append) {
  need(q_in.dim() == 4 && kc_in.dim() == 4 && vc_in.dim() == 4 && kl_in.dim() == 4 && vl_in.dim() == 4,
       "queries, cache and new keys and values are (batch, heads, rows, head dim)");
  const int B = (int)q_in.size(0), H = (int)q_in.size(1), T = (int)q_in.size(2), D = (int)q_in.size(3);
  need(kc_in.size(0) == B && kc_in.size(1) == H && kc_in.size(3) == D && same_shape(kc_in, vc_in) &&
           q_in.scalar_type() == kc_in.scalar_type() && q_in.scalar_type() == vc_in.scalar_type() && q_in.is_cuda() &&
           kc_in.is_cuda() && vc_in.is_cuda(),
       "the cache must have the queries' batch, heads, head dim and type, and be on the GPU");
  need(same_shape(kl_in, q_in) && same_shape(vl_in, q_in) && kl_in.scalar_type() == q_in.scalar_type() &&
           vl_in.scalar_type() == q_in.scalar_type() && kl_in.is_cuda() && vl_in.is_cuda(),
       "the new keys and values must have the queries' shape and type, and be on the GPU");
  const int dtype = dtype_code(q_in);
  need(dtype >= 0, "HIP kernels are built for bf16 and fp16");
  need(block > 0 && (S % block == 0 || T + S % block <= block), "new chunk and cached tail must fit one block (llama_mem.py:330)");
  if (!has_scale) scale = 1.0 / std::sqrt((double)D);
  at::AutoDispatchBelowADInplaceOrView guard;
  c10::DeviceGuard device(q_in.device());
  const Tensor q = kernel_ready(q_in), kc = kernel_ready(kc_in), vc = kernel_ready(vc_in), kl = kernel_ready(kl_in),
               vl = kernel_ready(vl_in);
  const Tables t = tables(cos, sin, q.scalar_type());
  const int64_t k = std::min<int64_t>(top_k, S / block), inc = S % block;
  const size_t rbytes = lmk_retrieve_workspace_bytes(B, H, T, (int)S, D, block);
  if (!ws.defined()) ws = bytes_on(q, rbytes);
  need(ws.scalar_type() == at::kByte && ws.is_contiguous() && (size_t)ws.numel() >= rbytes && ws.device() == q.device(),
       "workspace: contiguous uint8, at least lmk_retrieve_workspace_bytes long, on the queries' device");
  Tensor idx = at::empty({B, H, shared ? 1 : T, std::max<int64_t>(k, 0)}, q.options().dtype(at::kLong));
  const lmk_tensor4 tq = t4(q), tkc = t4(kc), tvc = t4(vc), tkl = t4(kl), tvl = t4(vl);
  const void *pc = t.cos.data_ptr(), *ps = t.sin.data_ptr();
  const int64_t cs = t.cos.stride(0), n_pos = t.cos.size(0);
  void* stream = stream_of(q);

  Tensor kn;
  lmk_tensor4 tkn = {}, tkd = {}, tvd = {};
  if (append != nullptr) {
    need(append->k_nopos.dim() == 4 && same_shape(append->k_nopos, q_in) && append->k_nopos.scalar_type() == q.scalar_type() &&
             append->k_nopos.is_cuda(),
         "the keys to append must have the queries' shape and type, and be on the GPU");
    need(append->row >= S && append->row + T <= append->k_buf.size(2), "no room for the new rows");
    kn = kernel_ready(append->k_nopos);
    tkn = t4(kn);
    auto at_row = [&](const Tensor& buf) {
      lmk_tensor4 d = t4(buf);
      d.ptr = static_cast<char*>(d.ptr) + 2 * append->row * d.stride_row;
      return d;
    };
    tkd = at_row(append->k_buf);
    tvd = at_row(append->v_buf);
  }

  if (!shared) {
    const size_t abytes = lmk_attend_workspace_bytes(B, H, T, (int)S, D, block) +
                          lmk_gather_blocks_workspace_bytes(B, H, T, (int)(S / block), D, block, top_k, 0);
    Tensor aws = bytes_on(q, abytes), out = at::empty_like(q);
    const lmk_tensor4 tout = t4(out);
    if (append != nullptr)
      check(lmk_retrieve_attend_append(&tq, &tkc, &tvc, &tkl, &tvl, &tkn, &tkd, &tvd, pc, ps, cs, n_pos, idx.data_ptr<int64_t>(),
                                       &tout, ws.data_ptr(), rbytes, reuse ? 1 : 0, aws.data_ptr(), abytes, B, H, T, (int)S, D,
                                       (float)scale, block, top_k, dtype, stream));
    else
      check(lmk_retrieve_and_attend(&tq, &tkc, &tvc, &tkl, &tvl, pc, ps, cs, n_pos, idx.data_ptr<int64_t>(), &tout, ws.data_ptr(),
                                    rbytes, reuse ? 1 : 0, aws.data_ptr(), abytes, B, H, T, (int)S, D, (float)scale, block, top_k,
                                    dtype, stream));
    return {out, idx};
  }
  // one selection per head: the selected blocks, rotated, and the local window form one sequence for the fused forward
  check(lmk_retrieve_topk_shared(&tq, &tkc, pc, ps, cs, n_pos, idx.data_ptr<int64_t>(), nullptr, ws.data_ptr(), rbytes, B, H, T,
                                 (int)S, D, block, top_k, dtype, stream));
  const int64_t rows = k * block + inc + T;
  Tensor win = at::empty({2, B, H, rows, D}, q.options());
  const Tensor k_win = win.select(0, 0), v_win = win.select(0, 1);
  const Tensor q_win = inc ? at::empty({B, H, inc + T, D}, q.options()) : q;
  const lmk_tensor4 tqw = t4(q_win), tkw = t4(k_win), tvw = t4(v_win);
  check(lmk_gather_window(&tq, &tkc, &tvc, idx.data_ptr<int64_t>(), &tkl, &tvl, pc, ps, cs, n_pos, inc ? &tqw : nullptr, &tkw,
                          &tvw, B, H, T, (int)S, D, block, top_k, dtype, stream));
  Tensor o = forward(shape_of(q_win, k_win, (int)k, scale, block, block, false), q_win, k_win, v_win, Tensor()).first;
  if (append != nullptr) check(lmk_cache_append(&tkn, &tvl, &tkd, &tvd, B, H, T, D, stream));
  return {inc ? o.narrow(2, inc, T) : o, idx};
}

// ---- the ring cache (MemLMCacheStorage): buffers (B, slots, block, nh, hs), tail (B, nh, block, hs)
struct Ring {
  Tensor k, v, tail_k, tail_v;
  int tail, filled, oldest, top_k, method;
};

// attention of a chunk over the ring and itself: (y, slots), slots undefined while the ring holds no block
std::pair<Tensor, Tensor> ring_attend(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, const Tensor& cos,
                                      const Tensor& sin, const Ring& r, int64_t start, bool has_scale, double scale) {
  need(q_in.dim() == 4 && q_in.is_cuda() && q_in.scalar_type() == r.k.scalar_type() && same_shape(k_in, q_in) &&
           same_shape(v_in, q_in) && k_in.scalar_type() == q_in.scalar_type() && v_in.scalar_type() == q_in.scalar_type() &&
           k_in.is_cuda() && v_in.is_cuda(),
       "q, k, v must have one shape, the cache's type, and be on the GPU");
  const int B = (int)q_in.size(0), H = (int)q_in.size(1), T = (int)q_in.size(2), D = (int)q_in.size(3), block = (int)r.k.size(2);
  need(B <= r.k.size(0) && H == r.k.size(3) && D == r.k.size(4), "the chunk must have the cache's heads and head dim");
  need(start >= r.tail, "the tokens behind the last complete block need positions of their own");
  if (!has_scale) scale = 1.0 / std::sqrt((double)D);
  const int dtype = dtype_code(q_in);
  need(dtype >= 0, "HIP kernels are built for bf16 and fp16");
  at::AutoDispatchBelowADInplaceOrView guard;
  c10::DeviceGuard device(q_in.device());
  const Tensor q = kernel_ready(q_in), k = kernel_ready(k_in), v = kernel_ready(v_in);
  const Tables t = tables(cos, sin, q.scalar_type());
  const lmk_tensor4 tq = t4(q), tk = t4(k), tv = t4(v);
  const void *pc = t.cos.data_ptr(), *ps = t.sin.data_ptr();
  const int64_t cs = t.cos.stride(0), n_pos = t.cos.size(0), W = r.tail + T;
  void* stream = stream_of(q);
  Tensor q_win = q, k_win = k, v_win = v, win;
  if (r.tail > 0) {
    // the tokens behind the last complete block open the chunk's first block, their keys rotated at start - tail ..,
    // zero rows standing in for their queries
    win = at::empty({3, B, H, W, D}, q.options());
    q_win = win.select(0, 0);
    k_win = win.select(0, 1);
    v_win = win.select(0, 2);
    const lmk_tensor4 tlk = t4(r.tail_k), tlv = t4(r.tail_v), a = t4(q_win), b = t4(k_win), c = t4(v_win);
    check(lmk_ring_local_window(&tq, &tlk, &tlv, &tk, &tv, pc, ps, cs, n_pos, &a, &b, &c, B, H, T, r.tail, start - r.tail, D,
                                dtype, stream));
  }
  auto fwd = forward(shape_of(q_win, k_win, 0, scale, block, block, true), q_win, k_win, v_win, Tensor());
  const Tensor o_loc = r.tail > 0 ? fwd.first.narrow(2, r.tail, T) : fwd.first;
  if (r.filled == 0 || r.top_k == 0) return {o_loc, Tensor()};
  auto ring4 = [](const Tensor& x) { return lmk_tensor4{x.data_ptr(), x.stride(0), x.stride(3), x.stride(2)}; };
  const lmk_tensor4 rk = ring4(r.k), rv = ring4(r.v), to = t4(o_loc);
  std::vector<int64_t> shape = {B};
  if (r.method != LMK_SELECT_MAX_OVER_HEADS) shape.push_back(H);
  if (r.method != LMK_SELECT_MAX_OVER_TOKENS) shape.push_back(T);
  shape.push_back(r.top_k);
  Tensor slots = at::empty(shape, q.options().dtype(at::kLong));
  const size_t nbytes = lmk_retrieve_workspace_bytes(B, H, T, r.filled * block, D, block);
  const size_t pbytes = lmk_gather_blocks_workspace_bytes(B, H, T, r.filled, D, block, r.top_k, r.method == LMK_SELECT_MAX_OVER_TOKENS);
  Tensor ws = bytes_on(q, nbytes), picks = bytes_on(q, pbytes), out = at::empty_like(q);
  check(lmk_ring_retrieve_topk(&tq, &rk, pc, ps, cs, n_pos, slots.data_ptr<int64_t>(), ws.data_ptr(), nbytes, B, H, T, r.filled, D,
                               block, r.top_k, r.oldest, r.method, dtype, stream));
  const float* L = fwd.second.data_ptr<float>() + r.tail;
  const lmk_tensor4 tout = t4(out);
  check(lmk_ring_gather_attend_blocks(&tq, &rk, &rv, slots.data_ptr<int64_t>(), pc, ps, cs, n_pos, &to, L, L + (int64_t)B * H * W, W,
                                      &tout, pbytes ? picks.data_ptr() : nullptr, pbytes, B, H, T, r.filled, D, (float)scale, block,
                                      r.top_k, r.oldest, r.method, dtype, stream));
  return {out, slots};
}

// ---- Python
Tensor tensor_arg(PyObject* o) {                         // None: an undefined tensor
  if (o == Py_None) return Tensor();
  if (!THPVariable_Check(o)) throw Failed{0, "expected a tensor"};
  return THPVariable_Unpack(o);
}
int64_t int_arg(PyObject* o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
double float_arg(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return v;
}
void count(Py_ssize_t n, Py_ssize_t want) { need(n == want, "wrong number of arguments"); }

PyObject* tuple_of(std::initializer_list<Tensor> ts) {
  PyObject* t = PyTuple_New((Py_ssize_t)ts.size());
  Py_ssize_t i = 0;
  for (const Tensor& x : ts) {
    PyObject* o = x.defined() ? THPVariable_Wrap(x) : Py_NewRef(Py_None);
    PyTuple_SET_ITEM(t, i++, o);
  }
  return t;
}

template <class F>
PyObject* guarded(F&& f) {
  HANDLE_TH_ERRORS
  try {
    return f();
  } catch (const Failed& e) {
    set_python_error(e);
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

PyObject* py_set_error_class(PyObject*, PyObject* cls) {
  Py_XDECREF(g_lmk_error);
  g_lmk_error = Py_NewRef(cls);
  Py_RETURN_NONE;
}

// attention(q, k, v, group_scale | None, sm_scale | None, block, handover_max_bytes, handover_min_keys) -> out, or None for
// a call that an autograd Function has to make
PyObject* py_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    count(n, 8);
    const Tensor q = tensor_arg(a[0]), k = tensor_arg(a[1]), v = tensor_arg(a[2]), gs = tensor_arg(a[3]);
    const bool has_scale = a[4] != Py_None;
    const double scale = has_scale ? float_arg(a[4]) : 0.0;
    const int64_t block = int_arg(a[5]);
    const HandoverLimits limits = {int_arg(a[6]), int_arg(a[7])};
    if (left_to_a_function({q, k, v, gs})) Py_RETURN_NONE;
    return THPVariable_Wrap(without_gil([&] { return attention(q, k, v, gs, has_scale, scale, block, limits); }));
  });
}

// attn_fwd(q, k, v, group_scale | None, n_prefix, sm_scale, block, block_real, blocks) -> (o, L, M)
PyObject* py_attn_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    count(n, 9);
    const Tensor q = tensor_arg(a[0]), k = tensor_arg(a[1]), v = tensor_arg(a[2]), gs = tensor_arg(a[3]);
    const Shape s = shape_of(q, k, (int)int_arg(a[4]), float_arg(a[5]), (int)int_arg(a[6]), (int)int_arg(a[7]), a[8] == Py_True);
    Tensor L, M;
    const Tensor o = without_gil([&] {
      at::AutoDispatchBelowADInplaceOrView guard;
      c10::DeviceGuard device(q.device());
      auto r = forward(s, q, k, v, gs);
      L = r.second.select(0, 0);
      M = r.second.select(0, 1);
      return r.first;
    });
    return tuple_of({o, L, M});
  });
}

// attn_bwd(q, k, v, o, do, L, M, group_scale | None, n_prefix, sm_scale, block, block_real, blocks, handover_max_bytes,
//          handover_min_keys) -> (dq, dk, dv)
PyObject* py_attn_bwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    count(n, 15);
    Tensor t[8];
    for (int i = 0; i < 8; ++i) t[i] = tensor_arg(a[i]);
    const Shape s = shape_of(t[0], t[1], (int)int_arg(a[8]), float_arg(a[9]), (int)int_arg(a[10]), (int)int_arg(a[11]), a[12] == Py_True);
    const HandoverLimits limits = {int_arg(a[13]), int_arg(a[14])};
    const variable_list g = without_gil([&] {
      at::AutoDispatchBelowADInplaceOrView guard;
      c10::DeviceGuard device(t[0].device());
      return backward(s, limits, t[0], t[1], t[2], t[3], t[5].data_ptr<float>(), t[6].data_ptr<float>(), t[4], t[7]);
    });
    return tuple_of({g[0], g[1], g[2]});
  });
}

// rotary(q | None, k, cos, sin, position_ids) -> (q_embed | None, k_embed), or None for a call that an autograd Function
// has to make
PyObject* py_rotary(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    count(n, 5);
    const Tensor q = tensor_arg(a[0]), k = tensor_arg(a[1]), cos = tensor_arg(a[2]), sin = tensor_arg(a[3]), pos = tensor_arg(a[4]);
    if (left_to_a_function({q, k, cos, sin})) Py_RETURN_NONE;
    const auto r = without_gil([&] { return rotary(q, k, cos, sin, pos); });
    return tuple_of({r.first, r.second});
  });
}

// rotate(x, cos, sin, position_ids) -> x_embed: the launch alone, without autograd
PyObject* py_rotate(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    count(n, 4);
    const Tensor x = tensor_arg(a[0]), cos = tensor_arg(a[1]), sin = tensor_arg(a[2]), pos = tensor_arg(a[3]);
    return THPVariable_Wrap(without_gil([&] {
      at::AutoDispatchBelowADInplaceOrView guard;
      c10::DeviceGuard device(x.device());
      const RotaryArgs r = rotary_args(x, cos, sin, pos);
      return rotate(Tensor(), x, r.t, r.pos, false).second;
    }));
  });
}

// mem_cache_step(q, k_cache, v_cache, cached_rows, k_loc, v_loc, cos, sin, block, top_k, sm_scale | None, shared,
//                workspace | None, reuse_landmark_keys, k_append | None) -> (out, idx)
// With k_append the new rows are stored behind the cached ones: k_cache and v_cache are then the cache's buffers.
PyObject* py_mem_cache_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    count(n, 15);
    const Tensor q = tensor_arg(a[0]), kc = tensor_arg(a[1]), vc = tensor_arg(a[2]), kl = tensor_arg(a[4]), vl = tensor_arg(a[5]),
                 cos = tensor_arg(a[6]), sin = tensor_arg(a[7]), ws = tensor_arg(a[12]), kn = tensor_arg(a[14]);
    const int64_t S = int_arg(a[3]), block = int_arg(a[8]), top_k = int_arg(a[9]);
    const bool has_scale = a[10] != Py_None, shared = a[11] == Py_True, reuse = a[13] == Py_True;
    const double scale = has_scale ? float_arg(a[10]) : 0.0;
    const auto r = without_gil([&] {
      const Append append = {kn, kc, vc, S};
      return mem_cache_step(q, kc, vc, S, kl, vl, cos, sin, (int)block, (int)top_k, has_scale, scale, shared, ws, reuse,
                            kn.defined() ? &append : nullptr);
    });
    return tuple_of({r.first, r.second});
  });
}

// retrieve_workspace_bytes(B, H, T, S, D, block)
PyObject* py_retrieve_workspace_bytes(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    count(n, 6);
    return PyLong_FromSize_t(lmk_retrieve_workspace_bytes((int)int_arg(a[0]), (int)int_arg(a[1]), (int)int_arg(a[2]),
                                                          (int)int_arg(a[3]), (int)int_arg(a[4]), (int)int_arg(a[5])));
  });
}

// cache_append(k, v, k_buf, v_buf, row): rows of k and v (B, H, T, D) into the buffers from `row` on
PyObject* py_cache_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    count(n, 5);
    const Tensor k_in = tensor_arg(a[0]), v_in = tensor_arg(a[1]), kb = tensor_arg(a[2]), vb = tensor_arg(a[3]);
    const int64_t row = int_arg(a[4]);
    without_gil([&] {
      at::AutoDispatchBelowADInplaceOrView guard;
      c10::DeviceGuard device(k_in.device());
      const Tensor k = kernel_ready(k_in), v = kernel_ready(v_in);
      need(row >= 0 && row + k.size(2) <= kb.size(2), "no room for the new rows");
      lmk_tensor4 tk = t4(k), tv = t4(v), tkd = t4(kb), tvd = t4(vb);
      tkd.ptr = static_cast<char*>(tkd.ptr) + 2 * row * tkd.stride_row;
      tvd.ptr = static_cast<char*>(tvd.ptr) + 2 * row * tvd.stride_row;
      check(lmk_cache_append(&tk, &tv, &tkd, &tvd, (int)k.size(0), (int)k.size(1), (int)k.size(2), (int)k.size(3), stream_of(k)));
      return 0;
    });
    Py_RETURN_NONE;
  });
}

// ring_attend(q, k, v, cos, sin, ring_k, ring_v, tail_k, tail_v, tail, filled, oldest, top_k, method, start, sm_scale | None)
//   -> (y, slots | None)
PyObject* py_ring_attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    count(n, 16);
    Tensor t[9];
    for (int i = 0; i < 9; ++i) t[i] = tensor_arg(a[i]);
    const Ring ring = {t[5], t[6], t[7], t[8], (int)int_arg(a[9]), (int)int_arg(a[10]), (int)int_arg(a[11]), (int)int_arg(a[12]),
                       (int)int_arg(a[13])};
    const int64_t start = int_arg(a[14]);
    const bool has_scale = a[15] != Py_None;
    const double scale = has_scale ? float_arg(a[15]) : 0.0;
    const auto r = without_gil([&] { return ring_attend(t[0], t[1], t[2], t[3], t[4], ring, start, has_scale, scale); });
    return tuple_of({r.first, r.second});
  });
}

// ring_store(k, v, is_mem, tail_k, tail_v, tail_is_mem, ring_k, ring_v, tail, next_slot)
PyObject* py_ring_store(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    count(n, 10);
    Tensor t[8];
    for (int i = 0; i < 8; ++i) t[i] = tensor_arg(a[i]);
    const int tail = (int)int_arg(a[8]), next = (int)int_arg(a[9]);
    without_gil([&] {
      const Tensor &rk = t[6], &rv = t[7];
      for (const Tensor& x : t)                          // one kernel reads and writes them all
        need(x.defined() && x.device() == rk.device(), "keys, values and is_mem must be on the cache's device");
      need(rk.is_cuda(), "the cache must be on the GPU");
      need(t[0].dim() == 4 && same_shape(t[0], t[1]) && t[0].size(0) <= rk.size(0) && t[0].size(1) == rk.size(3) &&
               t[0].size(3) == rk.size(4) && same_shape(rk, rv) && rk.strides() == rv.strides(),
           "keys and values must have one shape, and the cache's heads and head dim");
      need(t[2].dim() == 2 && t[2].size(0) == t[0].size(0) && t[2].size(1) == t[0].size(2) && t[2].scalar_type() == at::kBool,
           "is_mem is (batch, rows), bool");
      at::AutoDispatchBelowADInplaceOrView guard;
      c10::DeviceGuard device(t[0].device());
      const Tensor k = kernel_ready(t[0]), v = kernel_ready(t[1]), marks = t[2].stride(1) == 1 ? t[2] : t[2].contiguous();
      const lmk_tensor4 tk = t4(k), tv = t4(v), tlk = t4(t[3]), tlv = t4(t[4]);
      check(lmk_ring_store(&tk, &tv, marks.data_ptr(), marks.stride(0), &tlk, &tlv, t[5].data_ptr(), t[5].stride(0), rk.data_ptr(),
                           rv.data_ptr(), rk.stride(0), rk.stride(1), rk.stride(2), rk.stride(3), (int)k.size(0), (int)k.size(1),
                           (int)k.size(2), (int)k.size(3), (int)rk.size(2), (int)rk.size(1), tail, next, stream_of(k)));
      return 0;
    });
    Py_RETURN_NONE;
  });
}

// The attention node as Python sees it: an autograd node with `saved_tensors` (q, k, v, o, L, M, and the group factors if
// there are any), as a Python autograd Function has them.
PyObject* py_saved_tensors(PyObject* self, void*) {
  return guarded([&]() -> PyObject* {
    auto node = std::static_pointer_cast<AttentionBackward>(reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata);
    const auto t = without_gil([&] { return node->unpack(node); });
    if (!node->has_gs) return tuple_of({t.q, t.k, t.v, t.o, t.st.select(0, 0), t.st.select(0, 1)});
    return tuple_of({t.q, t.k, t.v, t.o, t.st.select(0, 0), t.st.select(0, 1), t.gs});
  });
}
PyTypeObject g_attention_node_type;
using namespace torch::autograd;                         // names inside the macro
PyGetSetDef g_attention_node_properties[] = {
    THP_FUNCTION_DEFAULT_PROPERTIES,
    {"saved_tensors", py_saved_tensors, nullptr, nullptr, nullptr},
    {nullptr, nullptr, nullptr, nullptr, nullptr},
};

#define LMK_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f)), METH_FASTCALL, nullptr
PyMethodDef g_methods[] = {
    {"set_error_class", py_set_error_class, METH_O, nullptr},
    {"attention", LMK_FAST(py_attention)},
    {"attn_fwd", LMK_FAST(py_attn_fwd)},
    {"attn_bwd", LMK_FAST(py_attn_bwd)},
    {"rotary", LMK_FAST(py_rotary)},
    {"rotate", LMK_FAST(py_rotate)},
    {"mem_cache_step", LMK_FAST(py_mem_cache_step)},
    {"retrieve_workspace_bytes", LMK_FAST(py_retrieve_workspace_bytes)},
    {"cache_append", LMK_FAST(py_cache_append)},
    {"ring_attend", LMK_FAST(py_ring_attend)},
    {"ring_store", LMK_FAST(py_ring_store)},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  PyTypeObject* node = torch::autograd::_initFunctionPyTypeObject(
      g_attention_node_type, "landmark_hip.FusedLandmarkAttentionBackward", g_attention_node_properties, nullptr);
  torch::autograd::registerCppFunction(typeid(AttentionBackward), node);
  return PyModule_Create(&g_module);
}

// The launch path of the public Python calls as one native call each
// (tilemix_amd/_host.so, a CPython extension module).
//
// A call that needs nothing but its launches -- fp16 tensors on one GPU, 16-byte
// vectors along the head dim, supported block sizes, no bias, default switches --
// is checked, given its workspace and launched here.  Every other call returns
// None and takes the Python path, which validates, copies, pads and raises as it
// always did; so does a call whose launch fails.  The checks below are those of
// the Python path plus the conditions under which it would copy.
//
// Why: a 256-token call has ~12 us of GPU work, and the Python path (attribute
// reads, ~60 ctypes fields, six allocations, two device contexts) took ~70 us of
// host time per call; this one takes ~9 us.
//
// The GPU library stays free of torch: its entry points are bound by address
// (bind(), from the ctypes handle of tilemix_amd/_native.py).
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <pybind11/gil.h>

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <cstdlib>
#include <cstring>

#include "tilemix_hip.h"

namespace {

struct Library {
  decltype(&tilemix_quant_per_block_int8_many) quant = nullptr;
  decltype(&tilemix_attn_fwd) attn = nullptr;
  decltype(&tilemix_attn_fwd_uniform) attn_uniform = nullptr;
  decltype(&tilemix_rms_norm_f16) rms_norm = nullptr;
  decltype(&tilemix_rotary_f16) rotary = nullptr;
  decltype(&tilemix_silu_mul_f16) silu_mul = nullptr;
} g_lib;

PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "bind() takes the addresses of the six entry points");
    return nullptr;
  }
  void* at[6];
  for (int i = 0; i < 6; ++i) {
    at[i] = PyLong_AsVoidPtr(args[i]);
    if (at[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
      return nullptr;
    }
  }
  g_lib.quant = reinterpret_cast<decltype(g_lib.quant)>(at[0]);
  g_lib.attn = reinterpret_cast<decltype(g_lib.attn)>(at[1]);
  g_lib.attn_uniform = reinterpret_cast<decltype(g_lib.attn_uniform)>(at[2]);
  g_lib.rms_norm = reinterpret_cast<decltype(g_lib.rms_norm)>(at[3]);
  g_lib.rotary = reinterpret_cast<decltype(g_lib.rotary)>(at[4]);
  g_lib.silu_mul = reinterpret_cast<decltype(g_lib.silu_mul)>(at[5]);
  Py_RETURN_NONE;
}

// built_for(): what this module was compiled against -- the ABI version and the sizes of the
// parameter structs (as tilemix_params_size numbers them), and torch.  tilemix_amd/_native.py
// compares them with what is loaded before it binds anything.
PyObject* built_for(PyObject*, PyObject* const*, Py_ssize_t) {
  return Py_BuildValue("(i(nnnn)s)", TILEMIX_ABI_VERSION, static_cast<Py_ssize_t>(sizeof(tilemix_quant_params)),
                       static_cast<Py_ssize_t>(sizeof(tilemix_attn_params)),
                       static_cast<Py_ssize_t>(sizeof(tilemix_rmsnorm_params)),
                       static_cast<Py_ssize_t>(sizeof(tilemix_rotary_params)), TILEMIX_TORCH);
}

// ---- arguments ----------------------------------------------------------------

// A torch.Tensor (no subclass) on a GPU whose storage the call may read directly.
const at::Tensor* plain_tensor(PyObject* o, at::ScalarType dtype) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.scalar_type() != dtype || t.layout() != at::kStrided || t.is_neg() ||
      at::isTensorSubclassLike(t))
    return nullptr;
  return &t;
}

// An int argument that fits 32 bits (bools are accepted, as Python's int() does).
bool int_arg(PyObject* o, int& out) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  const long v = PyLong_AsLongAndOverflow(o, &overflow);
  if (overflow != 0 || v < INT32_MIN || v > INT32_MAX) return false;
  out = static_cast<int>(v);
  return true;
}

bool aligned(const void* p, uintptr_t bytes) { return reinterpret_cast<uintptr_t>(p) % bytes == 0; }

// A switch in the environment: -1 if it is set to anything but "0" or "1".
int env_switch(const char* name, int unset) {
  const char* v = std::getenv(name);
  if (v == nullptr || v[0] == '\0') return unset;
  return std::strcmp(v, "1") == 0 ? 1 : std::strcmp(v, "0") == 0 ? 0 : -1;
}
bool env_set(const char* name) {
  const char* v = std::getenv(name);
  return v != nullptr && v[0] != '\0';
}

// ---- attention ------------------------------------------------------------------

constexpr int64_t kSpan = int64_t(1) << 31;

// One fp16 operand as [tokens, heads, dim] rows.
struct Operand {
  const at::Tensor* t = nullptr;
  int64_t tokens = 0, heads = 0, dim = 0, token_stride = 0, head_stride = 0;

  // Read as it lies: 16-byte vectors, `rows` token strides below 2 GiB, and tokens no closer than
  // their rows are long (the kernels bound a sequence's reads by its length times the stride).
  bool direct(int64_t rows) const {
    return token_stride % 8 == 0 && head_stride % 8 == 0 && token_stride >= dim &&
           aligned(t->const_data_ptr(), 16) && rows * token_stride * 2 < kSpan;
  }
};

struct Call {
  Operand q, k, v;
  const at::Tensor* map = nullptr;
  const int32_t* cu_q = nullptr;  // null: uniform lengths
  const int32_t* cu_k = nullptr;
  int batch = 0, seqlen = 0;      // longest sequence (uniform: every one)
  int block_m = 0, block_n = 0, block_n_mask = 0, blkq = 0, blkk = 0;
  bool causal = false, fp16_v = false;
  bool out_like_q = false;        // the output takes q's strides (else token-major)
  double sm_scale = 0;
  int mode = 0;
};

// The workspace of one quantised operand inside the call's buffer.
struct Quantised {
  int64_t codes = 0, scale = 0, scale16 = 0, cu = 0, rows = 0;
};

int64_t up256(int64_t n) { return (n + 255) / 256 * 256; }

// The output [tokens, heads, dim], or an undefined tensor if the call is not one
// that this path serves.
at::Tensor launch(const Call& c) {
  const int64_t d = c.q.dim, kv_rows = int64_t(c.seqlen) + 64;
  // (An empty TILEMIX_FORCE_CONFIG forces nothing; an empty TILEMIX_HIP_FUSED_Q_QUANT means off.)
  if (g_lib.attn == nullptr || env_set("TILEMIX_FORCE_CONFIG") || std::getenv("TILEMIX_HIP_FUSED_Q_QUANT") != nullptr)
    return {};
  if (c.k.tokens != c.v.tokens || c.k.heads != c.v.heads || c.k.dim != d || c.v.dim != d || d <= 0 || d > 128 ||
      d % 16 != 0)
    return {};
  if (c.q.heads <= 0 || c.k.heads <= 0 || c.q.heads % c.k.heads != 0 || c.q.heads > INT32_MAX) return {};
  const at::Device device = c.q.t->device();
  if (c.k.t->device() != device || c.v.t->device() != device || c.map->device() != device) return {};
  if (c.batch <= 0 || c.seqlen <= 0 || c.mode < 0 || c.mode > 2) return {};
  if ((c.block_m != 64 && c.block_m != 128 && c.block_m != 256 && c.block_m != 512) ||
      (c.block_n != 64 && c.block_n != 128 && c.block_n != 256))
    return {};
  if (c.block_n_mask <= 0 || c.block_n_mask % c.block_n != 0 ||
      (int64_t(c.seqlen) + c.block_n_mask - 1) / c.block_n_mask > 64)
    return {};
  if (!c.map->is_contiguous() ||
      c.map->numel() != c.k.heads * ((int64_t(c.seqlen) + c.block_m - 1) / c.block_m))
    return {};
  if (c.blkq <= 0 || c.blkk <= 0 || c.blkk % 4 != 0) return {};
  if (!c.q.direct(128) || !c.k.direct(kv_rows) || !c.v.direct(kv_rows)) return {};

  const bool int8 = c.mode != TILEMIX_ROUTING_FP16;
  const bool int8_v = int8 && !c.fp16_v;
  // Q is quantised by the attention kernel's 128-row workgroups (one BLKQ = 128
  // block each); block_m 64 with mixed routing on int8 V codes runs 64-row ones.
  const bool fused_q = int8 && c.blkq == 128 && (c.block_m >= 128 || c.fp16_v || c.mode != TILEMIX_ROUTING_MIXED);
  const bool uniform = c.cu_q == nullptr;

  const c10::DeviceGuard guard(device);
  void* const stream = c10::hip::getCurrentHIPStream(device.index()).stream();
  const auto options = at::TensorOptions().device(device);
  at::Tensor out = c.out_like_q ? at::empty_like(*c.q.t)
                                : at::empty({c.q.tokens, c.q.heads, d}, options.dtype(at::kHalf));
  // The kernel writes four columns at a time.
  if (out.stride(2) != 1 || out.stride(0) % 4 != 0 || out.stride(1) % 4 != 0 || !aligned(out.const_data_ptr(), 8))
    return {};

  tilemix_attn_params p{};
  tilemix_quant_params quant[3]{};
  Quantised at_[3];
  const Operand* operands[3];
  int count = 0, of_q = -1, of_k = -1, of_v = -1;
  at::Tensor work;
  if (int8) {
    if (!fused_q) operands[of_q = count++] = &c.q;
    operands[of_k = count++] = &c.k;
    if (int8_v) operands[of_v = count++] = &c.v;
    int64_t bytes = 0;
    for (int i = 0; i < count; ++i) {
      const Operand& x = *operands[i];
      const int blk = i == of_q ? c.blkq : c.blkk;
      Quantised& w = at_[i];
      // sum_b ceil(L_b / blk) <= ceil(tokens / blk) + batch
      w.rows = (x.tokens + blk - 1) / blk + c.batch;
      w.codes = bytes;
      w.scale = w.codes + up256(x.tokens * x.heads * d);
      w.scale16 = w.scale + up256(w.rows * x.heads * 4);
      w.cu = w.scale16 + up256(w.rows * x.heads * 2);
      bytes = w.cu + (uniform ? 0 : up256((int64_t(c.batch) + 1) * 4));
      if (kv_rows * x.heads * d >= kSpan) return {};  // the codes' own token stride
    }
    work = at::empty({bytes}, options.dtype(at::kByte));
    unsigned char* const base = static_cast<unsigned char*>(work.data_ptr());
    for (int i = 0; i < count; ++i) {
      const Operand& x = *operands[i];
      const Quantised& w = at_[i];
      tilemix_quant_params& s = quant[i];
      s.input = x.t->const_data_ptr();
      s.output = reinterpret_cast<int8_t*>(base + w.codes);
      s.scale = reinterpret_cast<float*>(base + w.scale);
      s.scale_half = base + w.scale16;
      s.cu_seqlens = i == of_q ? c.cu_q : c.cu_k;
      s.cu_seqlens_scale = uniform ? nullptr : reinterpret_cast<int32_t*>(base + w.cu);
      s.stride_in_token = x.token_stride;
      s.stride_in_head = x.head_stride;
      s.stride_out_token = x.heads * d;
      s.stride_out_head = d;
      s.scale_rows_capacity = w.rows;
      s.sm_scale = 1.0f;
      s.heads = static_cast<int32_t>(x.heads);
      s.head_dim = static_cast<int32_t>(d);
      s.blk_tokens = i == of_q ? c.blkq : c.blkk;
      s.batch = c.batch;
      s.max_seqlen = c.seqlen;
    }
    if (fused_q) {
      p.q_quant_in_kernel = 1;
    } else {
      p.q8 = quant[of_q].output;
      p.sq = quant[of_q].scale_half;
      p.cu_q_scale = quant[of_q].cu_seqlens_scale;
      p.stride_q8_token = quant[of_q].stride_out_token;
      p.stride_q8_head = d;
    }
    p.k8 = quant[of_k].output;
    p.sk = quant[of_k].scale_half;
    p.cu_k_scale = quant[of_k].cu_seqlens_scale;
    p.stride_k8_token = quant[of_k].stride_out_token;
    p.stride_k8_head = d;
    if (int8_v) {
      p.v8 = quant[of_v].output;
      p.sv = quant[of_v].scale_half;
      p.cu_v_scale = quant[of_v].cu_seqlens_scale;
      p.stride_v8_token = quant[of_v].stride_out_token;
      p.stride_v8_head = d;
    }
  }
  p.q = c.q.t->const_data_ptr();
  p.k = c.k.t->const_data_ptr();
  p.v = c.v.t->const_data_ptr();
  p.out = out.data_ptr();
  p.precision_bitmask = static_cast<const uint64_t*>(c.map->const_data_ptr());
  p.cu_seqlens_q = c.cu_q;
  p.cu_seqlens_k = c.cu_k;
  p.stride_q_token = c.q.token_stride;
  p.stride_q_head = c.q.head_stride;
  p.stride_k_token = c.k.token_stride;
  p.stride_k_head = c.k.head_stride;
  p.stride_v_token = c.v.token_stride;
  p.stride_v_head = c.v.head_stride;
  p.stride_o_token = out.stride(0);
  p.stride_o_head = out.stride(1);
  p.sm_scale = static_cast<float>(c.sm_scale);
  p.heads_q = static_cast<int32_t>(c.q.heads);
  p.heads_k = static_cast<int32_t>(c.k.heads);
  p.head_dim = static_cast<int32_t>(d);
  p.batch = c.batch;
  p.max_seqlen_q = p.max_seqlen_k = c.seqlen;
  p.block_m = c.block_m;
  p.block_n = c.block_n;
  p.block_n_mask = c.block_n_mask;
  p.blkq = c.blkq;
  p.blkk = c.blkk;
  p.causal = c.causal ? 1 : 0;
  p.routing_mode = c.mode;
  p.int8_use_fp16_v = c.fp16_v ? 1 : 0;

  int status = 0;
  Py_BEGIN_ALLOW_THREADS;  // a launch may wait for room in the queue
  if (count > 0) status = g_lib.quant(quant, count, uniform ? c.seqlen : 0, stream);
  if (status == 0) status = uniform ? g_lib.attn_uniform(&p, c.seqlen, stream) : g_lib.attn(&p, stream);
  Py_END_ALLOW_THREADS;
  return status == 0 ? out : at::Tensor();
}

// packed(q, k, v, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, bitmask, block_m, block_n,
//        block_n_mask, BLKQ, BLKK, causal, sm_scale | None, mode, scalar_scales, int8_use_fp16_v)
PyObject* packed(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c;
  int max_k = 0;
  if (n != 18) Py_RETURN_NONE;
  Operand* const xs[3] = {&c.q, &c.k, &c.v};
  for (int i = 0; i < 3; ++i) {
    const at::Tensor* t = plain_tensor(a[i], at::kHalf);
    if (t == nullptr || t->dim() != 3 || t->stride(2) != 1) Py_RETURN_NONE;
    *xs[i] = Operand{t, t->size(0), t->size(1), t->size(2), t->stride(0), t->stride(1)};
  }
  const at::Tensor* const cu_q = plain_tensor(a[3], at::kInt);
  const at::Tensor* const cu_k = plain_tensor(a[4], at::kInt);
  c.map = plain_tensor(a[7], at::kUInt64);
  if (cu_q == nullptr || cu_k == nullptr || c.map == nullptr) Py_RETURN_NONE;
  if (!cu_q->is_contiguous() || !cu_k->is_contiguous() || cu_q->numel() != cu_k->numel() ||
      cu_q->numel() > INT32_MAX || cu_q->device() != c.q.t->device() || cu_k->device() != c.q.t->device())
    Py_RETURN_NONE;
  if (!int_arg(a[5], c.seqlen) || !int_arg(a[6], max_k) || max_k != c.seqlen || !int_arg(a[8], c.block_m) ||
      !int_arg(a[9], c.block_n) || !int_arg(a[10], c.block_n_mask) || !int_arg(a[11], c.blkq) ||
      !int_arg(a[12], c.blkk) || !int_arg(a[15], c.mode))
    Py_RETURN_NONE;
  const int causal = PyObject_IsTrue(a[13]), scalar_scales = PyObject_IsTrue(a[16]), fp16_v = PyObject_IsTrue(a[17]);
  if (causal < 0 || scalar_scales < 0 || fp16_v < 0) return nullptr;
  if (scalar_scales != 0 && (c.block_m != c.blkq || c.block_n != c.blkk)) Py_RETURN_NONE;
  if (a[14] == Py_None) {
    c.sm_scale = std::pow(static_cast<double>(c.q.dim), -0.5);
  } else if (PyFloat_Check(a[14])) {
    c.sm_scale = PyFloat_AS_DOUBLE(a[14]);
  } else {
    Py_RETURN_NONE;
  }
  c.cu_q = static_cast<const int32_t*>(cu_q->const_data_ptr());
  c.cu_k = static_cast<const int32_t*>(cu_k->const_data_ptr());
  c.batch = static_cast<int>(cu_q->numel()) - 1;
  c.causal = causal != 0;
  c.fp16_v = fp16_v != 0;
  c.out_like_q = true;
  at::Tensor out = launch(c);
  if (!out.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// dense(q, k, v, block_m, block_n, block_n_mask | None, causal, scale, precision_map) on [B, H, T, D] tensors;
// the routing mode and the V format come from the environment as in tilemix_varlen_attention.
PyObject* dense(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c;
  if (n != 9) Py_RETURN_NONE;
  const char* const mode = std::getenv("TILEMIX_BITMASK_ROUTING_MODE");
  if (mode == nullptr || mode[0] == '\0' || std::strcmp(mode, "mixed") == 0) c.mode = TILEMIX_ROUTING_MIXED;
  else if (std::strcmp(mode, "fp16") == 0) c.mode = TILEMIX_ROUTING_FP16;
  else if (std::strcmp(mode, "int8") == 0) c.mode = TILEMIX_ROUTING_INT8;
  else Py_RETURN_NONE;
  const int fp16_v = env_switch("TILEMIX_SCORE_ONLY_PV", 1);
  if (fp16_v < 0) Py_RETURN_NONE;
  c.fp16_v = fp16_v != 0;
  int64_t batch = 0, tokens = 0;
  Operand* const xs[3] = {&c.q, &c.k, &c.v};
  for (int i = 0; i < 3; ++i) {
    const at::Tensor* t = plain_tensor(a[i], at::kHalf);
    if (t == nullptr || t->dim() != 4 || t->stride(3) != 1) Py_RETURN_NONE;
    if (i == 0) {
      batch = t->size(0);
      tokens = t->size(2);
    }
    // rows b T + t at one token stride: a token-major tensor, or one sequence in any layout
    const int64_t token_stride = tokens == 1 && batch != 1 ? t->stride(0) : t->stride(2);
    if (t->size(0) != batch || t->size(2) != tokens || (batch != 1 && t->stride(0) != tokens * token_stride))
      Py_RETURN_NONE;
    *xs[i] = Operand{t, batch * tokens, t->size(1), t->size(3), token_stride, t->stride(1)};
  }
  if (batch <= 0 || tokens <= 0 || batch * tokens > INT32_MAX) Py_RETURN_NONE;
  c.map = plain_tensor(a[8], at::kUInt64);
  if (c.map == nullptr || !int_arg(a[3], c.block_m) || !int_arg(a[4], c.block_n)) Py_RETURN_NONE;
  c.block_n_mask = c.block_n;
  if (a[5] != Py_None && !int_arg(a[5], c.block_n_mask)) Py_RETURN_NONE;
  const int causal = PyObject_IsTrue(a[6]);
  if (causal < 0) return nullptr;
  if (!PyFloat_Check(a[7])) Py_RETURN_NONE;
  c.sm_scale = PyFloat_AS_DOUBLE(a[7]);
  c.causal = causal != 0;
  c.batch = static_cast<int>(batch);
  c.seqlen = static_cast<int>(tokens);
  c.blkq = 128;
  c.blkk = 64;
  const at::Tensor out = launch(c);
  if (!out.defined()) Py_RETURN_NONE;
  // [B * T, H, D] as [B, H, T, D]
  return THPVariable_Wrap(out.view({batch, tokens, c.q.heads, c.q.dim}).permute({0, 2, 1, 3}));
  END_HANDLE_TH_ERRORS
}

// ---- quantisation API ---------------------------------------------------------------

// quantize(x, cu_seqlens, max_seqlen, blk, ... three times at most): codes, fp16 scales cut to their
// rows and int32 scale-row prefix of each tensor, as quantize_q(k)v_for_tilemix returns them.
PyObject* quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n < 4 || n > 12 || n % 4 != 0 || g_lib.quant == nullptr) Py_RETURN_NONE;
  const int count = static_cast<int>(n / 4);
  tilemix_quant_params quant[3]{};
  at::Tensor codes[3], scale16[3];
  int64_t rows[3];
  int64_t entries = 0, scale_bytes = 0;
  const at::Tensor* first = nullptr;
  for (int i = 0; i < count; ++i) {
    const at::Tensor* const x = plain_tensor(a[4 * i], at::kHalf);
    const at::Tensor* const cu = plain_tensor(a[4 * i + 1], at::kInt);
    tilemix_quant_params& s = quant[i];
    if (x == nullptr || cu == nullptr || x->dim() != 3 || x->stride(2) != 1 || !cu->is_contiguous() ||
        cu->numel() < 2 || cu->numel() > INT32_MAX || !int_arg(a[4 * i + 2], s.max_seqlen) ||
        !int_arg(a[4 * i + 3], s.blk_tokens))
      Py_RETURN_NONE;
    if (i == 0) {
      first = x;
      entries = cu->numel();
    }
    if (x->device() != first->device() || cu->device() != first->device() || cu->numel() != entries) Py_RETURN_NONE;
    if (s.max_seqlen < 0 || s.blk_tokens <= 0 || x->size(1) <= 0 || x->size(1) > INT32_MAX || x->size(2) <= 0 ||
        x->size(2) % 8 != 0 || x->size(2) > 256 || x->stride(0) % 8 != 0 || x->stride(1) % 8 != 0 ||
        !aligned(x->const_data_ptr(), 16))
      Py_RETURN_NONE;
    s.input = x->const_data_ptr();
    s.cu_seqlens = static_cast<const int32_t*>(cu->const_data_ptr());
    s.stride_in_token = x->stride(0);
    s.stride_in_head = x->stride(1);
    s.stride_out_token = x->size(1) * x->size(2);
    s.stride_out_head = x->size(2);
    s.heads = static_cast<int32_t>(x->size(1));
    s.head_dim = static_cast<int32_t>(x->size(2));
    s.batch = static_cast<int32_t>(entries - 1);
    s.sm_scale = 1.0f;
    rows[i] = (x->size(0) + s.blk_tokens - 1) / s.blk_tokens + s.batch;
    s.scale_rows_capacity = rows[i];
    scale_bytes += up256(rows[i] * s.heads * 4);
  }
  const c10::DeviceGuard guard(first->device());
  const auto options = at::TensorOptions().device(first->device());
  const at::Tensor scale = at::empty({scale_bytes}, options.dtype(at::kByte));  // the launch's fp32 scales
  const at::Tensor prefixes = at::empty({count, entries}, options.dtype(at::kInt));
  unsigned char* scale_at = static_cast<unsigned char*>(scale.data_ptr());
  for (int i = 0; i < count; ++i) {
    tilemix_quant_params& s = quant[i];
    codes[i] = at::empty(THPVariable_Unpack(a[4 * i]).sizes(), options.dtype(at::kChar));
    scale16[i] = at::empty({rows[i], s.heads}, options.dtype(at::kHalf));
    s.output = static_cast<int8_t*>(codes[i].data_ptr());
    s.scale = reinterpret_cast<float*>(scale_at);
    s.scale_half = scale16[i].data_ptr();
    s.cu_seqlens_scale = static_cast<int32_t*>(prefixes.data_ptr()) + i * entries;
    scale_at += up256(rows[i] * s.heads * 4);
  }
  void* const stream = c10::hip::getCurrentHIPStream(first->device().index()).stream();
  int status = 0;
  at::Tensor ends;
  {
    // The row counts come back in one copy (waits for the launch).
    pybind11::gil_scoped_release no_gil;
    status = g_lib.quant(quant, count, 0, stream);
    if (status == 0) ends = prefixes.cpu();
  }
  if (status != 0) Py_RETURN_NONE;
  const int32_t* const end = static_cast<const int32_t*>(ends.const_data_ptr());
  PyObject* const result = PyTuple_New(3 * count);
  if (result == nullptr) return nullptr;
  for (int i = 0; i < count; ++i) {
    PyTuple_SET_ITEM(result, 3 * i, THPVariable_Wrap(codes[i]));
    PyTuple_SET_ITEM(result, 3 * i + 1, THPVariable_Wrap(scale16[i].narrow(0, 0, end[(i + 1) * entries - 1])));
    PyTuple_SET_ITEM(result, 3 * i + 2, THPVariable_Wrap(prefixes.select(0, i)));
  }
  return result;
  END_HANDLE_TH_ERRORS
}

// ---- prefill helpers ---------------------------------------------------------------

// rms_norm(x, weight, eps): rows of x at one stride.
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || g_lib.rms_norm == nullptr || !PyFloat_Check(a[2])) Py_RETURN_NONE;
  const at::Tensor* const x = plain_tensor(a[0], at::kHalf);
  const at::Tensor* const w = plain_tensor(a[1], at::kHalf);
  if (x == nullptr || w == nullptr || x->dim() < 1 || !x->is_contiguous() || x->numel() == 0) Py_RETURN_NONE;
  const int64_t cols = x->size(-1);
  if (w->dim() != 1 || w->size(0) != cols || w->stride(0) != 1 || w->device() != x->device() || cols > INT32_MAX)
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(x->device());
  at::Tensor out = at::empty(x->sizes(), at::TensorOptions().device(x->device()).dtype(at::kHalf));
  tilemix_rmsnorm_params p{};
  p.x = x->const_data_ptr();
  p.weight = w->const_data_ptr();
  p.out = out.data_ptr();
  p.rows = x->numel() / cols;
  p.stride_x = p.stride_out = cols;
  p.cols = static_cast<int32_t>(cols);
  p.eps = static_cast<float>(PyFloat_AS_DOUBLE(a[2]));
  void* const stream = c10::hip::getCurrentHIPStream(x->device().index()).stream();
  int status = 0;
  Py_BEGIN_ALLOW_THREADS;
  status = g_lib.rms_norm(&p, stream);
  Py_END_ALLOW_THREADS;
  if (status != 0) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// rotary(q, k, cos, sin): rotary_token_major's operands.
PyObject* rotary(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || g_lib.rotary == nullptr) Py_RETURN_NONE;
  const at::Tensor* x[4];
  for (int i = 0; i < 4; ++i) {
    x[i] = plain_tensor(a[i], at::kHalf);
    if (x[i] == nullptr || x[i]->dim() != (i < 2 ? 4 : 3) || x[i]->numel() == 0 || x[i]->stride(-1) != 1 ||
        x[i]->device() != x[0]->device() || x[i]->_fw_grad(0).defined())
      Py_RETURN_NONE;
  }
  const at::Tensor &q = *x[0], &k = *x[1], &cos = *x[2], &sin = *x[3];
  const int64_t b = q.size(0), hq = q.size(1), t = q.size(2), d = q.size(3), hk = k.size(1);
  if (d % 2 != 0 || k.size(0) != b || k.size(2) != t || k.size(3) != d || cos.size(1) != t || cos.size(2) != d ||
      sin.sizes() != cos.sizes() || (cos.size(0) != 1 && cos.size(0) != b) || b > INT32_MAX || t > INT32_MAX ||
      hq > INT32_MAX || hk > INT32_MAX || d > INT32_MAX)
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(q.device());
  const auto options = at::TensorOptions().device(q.device()).dtype(at::kHalf);
  const at::Tensor oq = at::empty({b, t, hq, d}, options), ok = at::empty({b, t, hk, d}, options);
  tilemix_rotary_params p{};
  p.q = q.const_data_ptr();
  p.k = k.const_data_ptr();
  p.cos = cos.const_data_ptr();
  p.sin = sin.const_data_ptr();
  p.q_out = oq.data_ptr();
  p.k_out = ok.data_ptr();
  p.stride_q_batch = q.stride(0);
  p.stride_q_head = q.stride(1);
  p.stride_q_token = q.stride(2);
  p.stride_k_batch = k.stride(0);
  p.stride_k_head = k.stride(1);
  p.stride_k_token = k.stride(2);
  p.stride_cos_batch = cos.size(0) > 1 ? cos.stride(0) : 0;
  p.stride_cos_token = cos.stride(1);
  p.stride_sin_batch = sin.size(0) > 1 ? sin.stride(0) : 0;
  p.stride_sin_token = sin.stride(1);
  p.batch = static_cast<int32_t>(b);
  p.tokens = static_cast<int32_t>(t);
  p.heads_q = static_cast<int32_t>(hq);
  p.heads_k = static_cast<int32_t>(hk);
  p.head_dim = static_cast<int32_t>(d);
  void* const stream = c10::hip::getCurrentHIPStream(q.device().index()).stream();
  int status = 0;
  Py_BEGIN_ALLOW_THREADS;
  status = g_lib.rotary(&p, stream);
  Py_END_ALLOW_THREADS;
  if (status != 0) Py_RETURN_NONE;
  PyObject* const rq = THPVariable_Wrap(oq.transpose(1, 2));
  PyObject* const rk = rq == nullptr ? nullptr : THPVariable_Wrap(ok.transpose(1, 2));
  PyObject* const both = rk == nullptr ? nullptr : PyTuple_Pack(2, rq, rk);
  Py_XDECREF(rq);
  Py_XDECREF(rk);
  return both;
  END_HANDLE_TH_ERRORS
}

// silu_mul(gate, up): contiguous operands of one shape.
PyObject* silu_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || g_lib.silu_mul == nullptr) Py_RETURN_NONE;
  const at::Tensor* const gate = plain_tensor(a[0], at::kHalf);
  const at::Tensor* const up = plain_tensor(a[1], at::kHalf);
  if (gate == nullptr || up == nullptr || gate->sizes() != up->sizes() || !gate->is_contiguous() ||
      !up->is_contiguous() || up->device() != gate->device())
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(gate->device());
  at::Tensor out = at::empty(gate->sizes(), at::TensorOptions().device(gate->device()).dtype(at::kHalf));
  void* const stream = c10::hip::getCurrentHIPStream(gate->device().index()).stream();
  int status = 0;
  Py_BEGIN_ALLOW_THREADS;
  if (gate->numel() > 0)
    status = g_lib.silu_mul(gate->const_data_ptr(), up->const_data_ptr(), out.data_ptr(), gate->numel(), stream);
  Py_END_ALLOW_THREADS;
  if (status != 0) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef method(const char* name) {
  return PyMethodDef{name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, nullptr};
}

PyMethodDef g_methods[] = {method<built_for>("built_for"),
                           method<bind>("bind"),     method<packed>("packed"),     method<dense>("dense"),
                           method<quantize>("quantize"),
                           method<rms_norm>("rms_norm"), method<rotary>("rotary"), method<silu_mul>("silu_mul"),
                           PyMethodDef{nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&g_module); }

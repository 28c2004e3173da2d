// Per-block symmetric int8 quantisation (Q per BLKQ tokens, K per BLKK tokens).
//
// Follows quant_per_block_int8_kernel (attention/triton/quant_per_block_varlen.py:6-45):
//   x    = fp32(x) * sm_scale                      (:38-39)
//   s    = max|x| / 127.                           (:40, IEEE fp32 division)
//   t    = x / s ; t += 0.5 * (t >= 0 ? 1 : -1)    (:41-42)
//   code = int8(t)  (truncation)                   (:43)
// plus the host-side scale bookkeeping of per_block_int8_single (:55-63),
// done on the device so no device->host copy is needed to size the output.
//
// One workgroup owns one (tensor, sequence, block, head).  Up to kQuantMany tensors
// (K and V, or Q, K and V of one call) go out in one launch.  Blocks of up to
// kRegRows row groups (BLK * D <= 16384 for the usual widths: every Q/K/V block
// of the hot path) are read from HBM once and held in registers between the max
// pass and the code pass; larger blocks are streamed twice.
//
// What bounds it: HBM (2 bytes read, 1 written per element), closely followed by
// VALU issue, so the arithmetic is kept small: a thread's rows differ by a
// uniform stride (no division per 16-byte chunk), the block maximum is taken on
// packed 16-bit magnitudes, and a code costs 5.5 instructions (mixed-precision
// FMAs straight from the fp16 operand, conversions that write their byte).  Heads are the fastest
// block index, so the workgroups in flight read neighbouring 256-byte rows.
// Against a kernel with a 32-bit division per chunk, fp32 maxima reduced through
// LDS, the scale-row prefix (and its barrier) before the loads, and ~12 instructions
// per code: K of 8 x 4096 x 8 heads x 128 25.0 -> 18.5 us (5.5 TB/s), Q of 8 x 4096 x 24
// x 128 65 -> 49 us (6.1 TB/s), K of 8 x 2048 13.6 -> 10.7 us, of 1 x 1000 5.5 -> 4.1 us.
//
// Small blocks, and workgroups past the end of their sequence, last as long as
// their chain of scalar loads and divisions before the first row (or the exit).  Divisors
// come as multipliers from the host, a launch of one tensor reads its arguments at
// once, the maximum takes one barrier.  With the divisions, a tensor chosen after a
// load and two barriers (us): 8192 tokens x 8 heads x 128 in blocks of 1 101 -> 60, of 4
// 28.0 -> 17.7, of 64 6.5 -> 5.8; 200 prompts of 5 tokens and one of 8000, blocks of 64
// 161 -> 48.  The loads of a block's rows are unconditional (a row past the block is its
// first one again), so that they go out together: as conditional ones the first was
// waited for alone, and K and V of 8192 tokens x 8 heads x 128 took 11.4 us instead of 10.5.
#include "attn_common.h"

#include <algorithm>
#include <type_traits>

namespace tmx {

namespace {

constexpr int kQuantThreads = 256;
constexpr int kRegRows = 8;    // row groups a thread holds in registers
constexpr int kQuantMany = 3;  // tensors per launch
// Workgroups of a launch along x: HIP takes less than 2^32 threads there.
constexpr int64_t kQuantGrid = (int64_t(1) << 32) / kQuantThreads - 1;

struct QuantTensor {
  const f16* in;
  int8_t* out;
  float* scale;
  f16* scale_half;
  const int32_t* cu;
  int32_t* cu_scale;
  int64_t si_t, si_h, so_t, so_h;
  int64_t capacity;
  FastDiv by_heads, by_chunks, by_blk;  // heads, 8-element chunks per row, tokens per block
  float sm_scale;
  int rpi;        // rows the workgroup reads per step
  int uni_rows;   // uni > 0: scale rows per sequence
  int first_blk;  // first block of this launch
};

struct QuantKArgs {
  QuantTensor t[kQuantMany];
  int first[kQuantMany];  // first workgroup of each tensor within a sequence's (past the grid: no such tensor)
  int uni;                // > 0: every sequence has this many tokens (cu is not read)
};

__device__ __forceinline__ uint32_t pk_max_u16(uint32_t x, uint32_t y) {
  uint32_t r;
  asm("v_pk_max_u16 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
  return r;
}

// Maximum over the wave (every lane gets it): lanes l ^ 32 and l ^ 16 by
// permlane swaps, the rest of a 16-lane row by DPP moves.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
  const auto p = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  v = max((uint32_t)p[0], (uint32_t)p[1]);
  const auto q = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = max((uint32_t)q[0], (uint32_t)q[1]);
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false));  // row_ror 8
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false));  // row_ror 4
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4e, 0xf, 0xf, false));   // quad_perm 2 3 0 1
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xb1, 0xf, 0xf, false));   // quad_perm 1 0 3 2
  return v;
}

__device__ __forceinline__ int wave_sum_i(int v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// MANY: several tensors.  (A launch of one reads its arguments without waiting for
// the choice of the tensor.)
template <bool MANY>
__global__ void __launch_bounds__(kQuantThreads) quant_per_block_int8_kernel(const QuantKArgs args) {
  __shared__ uint32_t red[2][kQuantThreads / 64];
  __shared__ int red_rows[kQuantThreads / 64];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int id = blockIdx.x, b = blockIdx.y;
  const int tensor = MANY ? (id >= args.first[1]) + (id >= args.first[2]) : 0;
  const QuantTensor a = args.t[tensor];  // a copy: by reference each argument's load waits for its use
  const int uni = args.uni;
  const int t = MANY ? id - args.first[tensor] : id;
  const int row = fast_div(t, a.by_heads), heads = a.by_heads.d, h = t - row * heads;
  const int blk = a.first_blk + row;

  int start = b * uni, len = uni;
  if (uni <= 0) {
    start = a.cu[b];
    len = a.cu[b + 1] - start;
  }
  const int blk_tokens = a.by_blk.d;
  const int rows = min(blk_tokens, len - blk * blk_tokens);  // <= 0: no such block in this sequence

  // Scale-row base of sequence b (the sum of ceil(L / blk) over the earlier ones):
  // each wave's part goes to LDS after the block's loads have gone out, and the thread
  // that stores the scale adds them behind the maximum's barrier.  The sum is a chain
  // of loads, so all four waves share it and each keeps four loads in flight: by one
  // wave alone, a load at a time, 4096 sequences of 16 tokens x 8 heads x 128 take 126 us
  // instead of 73, 8192 of 4 tokens 367 instead of 170.
  auto scale_rows = [&](int n) { return n > 0 ? fast_div(n - 1, a.by_blk) + 1 : 0; };
  auto sum_scale_rows = [&]() {
    if (uni > 0) return;
    int part = 0;
    if (b > wave * 64) {
      for (int b0 = tid; b0 < b; b0 += 4 * kQuantThreads) {
        int len4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int bb = min(b0 + i * kQuantThreads, b);
          len4[i] = a.cu[bb + 1] - a.cu[bb];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) part += b0 + i * kQuantThreads < b ? scale_rows(len4[i]) : 0;
      }
      part = wave_sum_i(part);
    }
    if (lane == 0) red_rows[wave] = part;
  };
  auto scale_base = [&]() -> int {  // behind a barrier after sum_scale_rows
    if (uni > 0) return b * a.uni_rows;
    int base = 0;
#pragma unroll
    for (int w = 0; w < kQuantThreads / 64; ++w) base += red_rows[w];
    return base;
  };
  auto publish = [&](int base) {
    if (blk == 0 && h == 0 && a.cu_scale != nullptr) {
      a.cu_scale[b + 1] = base + scale_rows(len);
      if (b == 0) a.cu_scale[0] = 0;
    }
  };
  if (rows <= 0) {
    if (blk == 0 && h == 0) {
      sum_scale_rows();
      __syncthreads();
      if (tid == 0) publish(scale_base());
    }
    return;
  }

  const int rpi = a.rpi;
  const int r0 = fast_div(tid, a.by_chunks), col = (tid - r0 * a.by_chunks.d) << 3;
  const bool used = r0 < rpi;  // the chunks per row need not divide the workgroup
  const int64_t tok0 = (int64_t)start + (int64_t)blk * blk_tokens;
  const f16* in_row0 = a.in + tok0 * a.si_t + (int64_t)h * a.si_h + col;
  const f16* in = in_row0 + (int64_t)r0 * a.si_t;
  int8_t* out = a.out + (tok0 + r0) * a.so_t + (int64_t)h * a.so_h + col;
  const int64_t in_step = (int64_t)rpi * a.si_t, out_step = (int64_t)rpi * a.so_t;

  const float sm = a.sm_scale;
  // sm_scale == 1 (the hot path: quantize_q(k)_for_tilemix): the quotient is
  // taken from an IEEE reciprocal with one correction step (div_by_recip),
  // equal to the IEEE division on the whole fp16 domain; other scales divide
  // directly.
  const bool unit_scale = sm == 1.0f;
  auto encode = [&](const u32x4& x, float s, float rs, int8_t* dst) {
    float v[8];
    if (unit_scale) {
      // rs is 0 for an all-zero block, whose codes then come out as 0.
#pragma unroll
      for (int e = 0; e < 4; ++e) quotient_pair(x[e], s, rs, v + 2 * e);
    } else {
      const f16x8 xv = __builtin_bit_cast(f16x8, x);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float t = ((float)xv[e] * sm) / s;
        v[e] = s == 0.0f ? 0.0f : t + ((t >= 0.0f) ? 0.5f : -0.5f);
      }
    }
    *reinterpret_cast<uint2*>(dst) = trunc_bytes(v);
  };
  // max|x * sm| over the block from the lane's largest magnitude (packed 16-bit
  // patterns without their signs order like the values; RN(x * sm) is monotonic
  // in |x|).  The maximum ignores NaNs, whose patterns lie above infinity's: a
  // block that holds one takes its maximum again from the values below.
  auto block_max = [&](uint32_t m2, int pass) -> uint32_t {
    const uint32_t m = wave_max_u32(max(m2 & 0xffffu, m2 >> 16));
    if (lane == 0) red[pass][wave] = m;
    __syncthreads();
    uint32_t r = red[pass][0];
#pragma unroll
    for (int w = 1; w < kQuantThreads / 64; ++w) r = max(r, red[pass][w]);
    return r;
  };
  constexpr uint32_t kInf = 0x7c00u;
  auto magnitudes = [](const u32x4& x, uint32_t m2) {
#pragma unroll
    for (int e = 0; e < 4; ++e) m2 = pk_max_u16(m2, x[e] & 0x7fff7fffu);
    return m2;
  };
  auto finite_magnitudes = [&](const u32x4& x, uint32_t m2) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t lo = x[e] & 0x7fffu, hi = (x[e] >> 16) & 0x7fffu;
      m2 = pk_max_u16(m2, (lo > kInf ? 0u : lo) | ((hi > kInf ? 0u : hi) << 16));
    }
    return m2;
  };
  auto scale_of = [&](uint32_t m) -> float {
    const float amax = fmaxf(0.0f, fabsf((float)__builtin_bit_cast(f16, (uint16_t)m) * sm));
    return amax / 127.0f;  // IEEE division (no fast-math in this build)
  };
  auto finish = [&](float s) {
    if (tid == 0) {
      const int base = scale_base();
      const int64_t row = (int64_t)base + blk;
      if (row < a.capacity) {
        a.scale[row * heads + h] = s;
        if (a.scale_half != nullptr) a.scale_half[row * heads + h] = (f16)s;
      }
      publish(base);
    }
  };

  auto in_registers = [&](auto nreg) {
    constexpr int kN = decltype(nreg)::value;
    u32x4 xs[kN];
    uint32_t m2 = 0;
#pragma unroll
    for (int i = 0; i < kN; ++i)  // past the block: its first row once more, which leaves the maximum as it is
      xs[i] = *reinterpret_cast<const u32x4*>(used && r0 + i * rpi < rows ? in + i * in_step : in_row0);
    sum_scale_rows();
#pragma unroll
    for (int i = 0; i < kN; ++i) m2 = magnitudes(xs[i], m2);
    uint32_t m = block_max(m2, 0);
    if (m > kInf) {
      m2 = 0;
#pragma unroll
      for (int i = 0; i < kN; ++i) m2 = finite_magnitudes(xs[i], m2);
      m = block_max(m2, 1);
    }
    const float s = scale_of(m);
    const float rs = s == 0.0f ? 0.0f : 1.0f / s;
#pragma unroll
    for (int i = 0; i < kN; ++i)
      if (used && r0 + i * rpi < rows) encode(xs[i], s, rs, out + i * out_step);
    finish(s);
  };
  if (rows <= rpi * (kRegRows / 2)) {
    in_registers(std::integral_constant<int, kRegRows / 2>{});
  } else if (rows <= rpi * kRegRows) {
    in_registers(std::integral_constant<int, kRegRows>{});
  } else {
    uint32_t m2 = 0;
    for (int i = 0; used && r0 + i * rpi < rows; ++i)
      m2 = magnitudes(*reinterpret_cast<const u32x4*>(in + i * in_step), m2);
    sum_scale_rows();
    uint32_t m = block_max(m2, 0);
    if (m > kInf) {
      m2 = 0;
      for (int i = 0; used && r0 + i * rpi < rows; ++i)
        m2 = finite_magnitudes(*reinterpret_cast<const u32x4*>(in + i * in_step), m2);
      m = block_max(m2, 1);
    }
    const float s = scale_of(m);
    const float rs = s == 0.0f ? 0.0f : 1.0f / s;
    for (int i = 0; used && r0 + i * rpi < rows; ++i)
      encode(*reinterpret_cast<const u32x4*>(in + i * in_step), s, rs, out + i * out_step);
    finish(s);
  }
}

int check_quant(const tilemix_quant_params& p, bool uniform) {
  if (!p.input || !p.output || !p.scale || (!uniform && !p.cu_seqlens)) {
    set_error("tilemix_quant_per_block_int8: null tensor pointer");
    return TILEMIX_E_INVALID;
  }
  if (p.heads <= 0 || p.batch < 0 || p.blk_tokens <= 0 || p.max_seqlen < 0) {
    set_error("tilemix_quant_per_block_int8: invalid sizes (heads=%d batch=%d blk=%d max_seqlen=%d)",
              p.heads, p.batch, p.blk_tokens, p.max_seqlen);
    return TILEMIX_E_INVALID;
  }
  if (p.head_dim <= 0 || p.head_dim % 8 != 0 || p.head_dim > 256) {
    set_error("tilemix_quant_per_block_int8: head_dim must be a positive multiple of 8 <= 256, got %d",
              p.head_dim);
    return TILEMIX_E_INVALID;
  }
  if ((reinterpret_cast<uintptr_t>(p.input) & 15) || (p.stride_in_token & 7) || (p.stride_in_head & 7) ||
      (reinterpret_cast<uintptr_t>(p.output) & 7) || (p.stride_out_token & 7) || (p.stride_out_head & 7)) {
    set_error("tilemix_quant_per_block_int8: input must be 16-byte aligned with strides multiple of 8 "
              "elements; output 8-byte aligned with strides multiple of 8");
    return TILEMIX_E_INVALID;
  }
  return TILEMIX_OK;
}

}  // namespace

int launch_quant(const tilemix_quant_params* ps, int count, int uniform_seqlen, hipStream_t stream) {
  if (count < 1 || count > kQuantMany || uniform_seqlen < 0) {
    set_error("tilemix_quant_per_block_int8: 1 to %d tensors and a non-negative uniform length, got %d and %d",
              kQuantMany, count, uniform_seqlen);
    return TILEMIX_E_INVALID;
  }
  QuantKArgs a{};
  a.uni = uniform_seqlen;
  int64_t total = 0, blocks[kQuantMany];
  for (int i = 0; i < count; ++i) {
    const tilemix_quant_params& p = ps[i];
    const int status = check_quant(p, uniform_seqlen > 0);
    if (status != TILEMIX_OK) return status;
    if (p.batch != ps[0].batch) {
      set_error("tilemix_quant_per_block_int8: the tensors of one launch share the batch, got %d and %d",
                ps[0].batch, p.batch);
      return TILEMIX_E_INVALID;
    }
    // The kernel numbers tokens in 32 bits (cu_seqlens does so by its type).
    if ((int64_t)uniform_seqlen * p.batch > INT32_MAX) {
      set_error("tilemix_quant_per_block_int8: %d sequences of %d tokens exceed the 32-bit token index", p.batch,
                uniform_seqlen);
      return TILEMIX_E_INVALID;
    }
    const int max_seqlen = uniform_seqlen > 0 ? uniform_seqlen : p.max_seqlen;
    // With no tokens, one block per sequence still publishes cu_seqlens_scale.
    const int64_t nblk = std::max<int64_t>(1, ((int64_t)max_seqlen + p.blk_tokens - 1) / p.blk_tokens);
    if (p.batch > 0 && (nblk > kQuantGrid || p.heads > kQuantGrid)) {
      set_error("tilemix_quant_per_block_int8: at most %lld blocks in a sequence and heads, got %lld and %d",
                (long long)kQuantGrid, (long long)nblk, p.heads);
      return TILEMIX_E_INVALID;
    }
    blocks[i] = nblk;
    QuantTensor& t = a.t[i];
    t.in = static_cast<const f16*>(p.input);
    t.out = p.output;
    t.scale = p.scale;
    t.scale_half = static_cast<f16*>(p.scale_half);
    t.cu = p.cu_seqlens;
    t.cu_scale = p.cu_seqlens_scale;
    t.si_t = p.stride_in_token;
    t.si_h = p.stride_in_head;
    t.so_t = p.stride_out_token;
    t.so_h = p.stride_out_head;
    t.capacity = p.scale_rows_capacity;
    t.sm_scale = p.sm_scale;
    t.by_heads = make_fast_div(p.heads);
    t.by_chunks = make_fast_div(p.head_dim / 8);
    t.by_blk = make_fast_div(p.blk_tokens);
    t.rpi = kQuantThreads / (p.head_dim / 8);
    t.uni_rows = uniform_seqlen > 0 ? (uniform_seqlen - 1) / p.blk_tokens + 1 : 0;
    t.first_blk = 0;
    a.first[i] = (int)std::min<int64_t>(total, INT32_MAX);
    total += nblk * p.heads;
  }
  if (ps[0].batch == 0) return TILEMIX_OK;
  auto launch = [&](const QuantKArgs& args, int64_t groups, bool many) -> int {
    const dim3 grid((unsigned)groups, (unsigned)ps[0].batch);
    if (many)
      hipLaunchKernelGGL((quant_per_block_int8_kernel<true>), grid, dim3(kQuantThreads), 0, stream, args);
    else
      hipLaunchKernelGGL((quant_per_block_int8_kernel<false>), grid, dim3(kQuantThreads), 0, stream, args);
    const hipError_t err = hipGetLastError();
    if (err == hipSuccess) return TILEMIX_OK;
    set_error("tilemix_quant_per_block_int8: launch failed: %s", hipGetErrorString(err));
    return TILEMIX_E_LAUNCH;
  };
  if (total <= kQuantGrid) {
    for (int i = count; i < kQuantMany; ++i) a.first[i] = INT32_MAX;
    return launch(a, total, count > 1);
  }
  // One tensor, and as many of its blocks as a launch takes, at a time.
  for (int i = 0; i < count; ++i) {
    QuantKArgs one = a;
    one.t[0] = a.t[i];
    const int64_t step = kQuantGrid / ps[i].heads;
    for (int64_t first = 0; first < blocks[i]; first += step) {
      one.t[0].first_blk = (int)first;
      const int status = launch(one, std::min(step, blocks[i] - first) * ps[i].heads, false);
      if (status != TILEMIX_OK) return status;
    }
  }
  return TILEMIX_OK;
}

}  // namespace tmx

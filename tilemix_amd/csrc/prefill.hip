// Prefill helper kernels of the LLaMA glue: RMSNorm, token-major split-half
// rotary embedding of Q and K, SiLU(gate) * up.  All three are HBM-streaming
// kernels (one read of every input, one write of every output, 16-byte
// accesses); the formulas follow models/tilemix_llama.py:718-869.
#include "attn_common.h"

#include <math.h>

#include <algorithm>

namespace tmx {

namespace {

// Materialise an fp32 result before its conversion to fp16: the reference
// rounds to fp32 and then to fp16, which the compiler would otherwise fuse
// into one mixed-precision instruction (a single rounding).  Products of two
// fp16 values are exact in fp32 and need no barrier.
__device__ __forceinline__ float keep32(float x) {
  asm volatile("" : "+v"(x));
  return x;
}

// RN(h * s) of the low / high fp16 half of h2 (one rounding; the addend -0 keeps
// the sign of a zero product).
__device__ __forceinline__ float mul_half(uint32_t h2, float s, bool high) {
  float r;
  if (high)
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h2), "v"(s), "v"(-0.0f));
  else
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(h2), "v"(s), "v"(-0.0f));
  return r;
}
// acc + h * h of the low / high fp16 half of h2 in fp32.
__device__ __forceinline__ float add_square(uint32_t h2, float acc, bool high) {
  float r;
  if (high)
    asm("v_fma_mix_f32 %0, %1, %1, %2 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "=v"(r) : "v"(h2), "v"(acc));
  else
    asm("v_fma_mix_f32 %0, %1, %1, %2 op_sel_hi:[1,1,0]" : "=v"(r) : "v"(h2), "v"(acc));
  return r;
}

// ---- RMSNorm (reference :718-797) ------------------------------------------
// The sum of squares adds separately rounded products (the reference's
// reduction is built without FMA contraction; the square of an fp16 value is
// exact in fp32, so one mixed-precision FMA per value gives the same sum), in
// this kernel's own order.  One wave per row; rows of up to 16 * 64 eight-element
// chunks (cols <= 8192) stay in registers between the sum of squares and the
// output pass, longer rows are read twice.
//
// Bound by HBM (4 bytes per value).  The kernel is instantiated per number of
// chunks a lane holds (NCH), so that a row takes only the registers it needs and
// more waves keep loads in flight, and the fp32 work is two instructions per
// value (an fp16 product of two fp16 values is their exact fp32 product rounded
// once).  Against one instantiation for every width with fp32 multiplies and adds
// (us): 32768 x 3072 88 -> 78 (5.2 TB/s, a large copy's rate), 8192 x 2048 15.6 -> 12.8,
// 2048 x 3072 7.8 -> 7.0, 4096 x 8192 23.5 -> 22.9.
constexpr int kNormWaves = 4;
constexpr int kNormChunks = 16;  // chunks per lane of the longest rows that are read in chunks
constexpr int kNormStep = 4;     // chunks in flight per lane where a row is read twice

struct NormArgs {
  const f16* x;
  const f16* w;
  f16* out;
  int64_t rows, sx, so;
  int cols;
  float inv_cols, eps;
};

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ f16 norm_one(float x, float rs, f16 w) {
  const f16 hn = (f16)keep32(x * rs);        // fp16(fp32(x) * rsqrt(var + eps))
  return (f16)((float)w * (float)hn);        // fp16(fp32(w) * fp32(hn))
}

// NCH: 8-element chunks a lane holds; 0: none.  Rows longer than 16 chunks a lane, and
// the rows that are not 16-byte aligned, go element by element.  ALIGNED: every
// row is (asking each row costs 64 rows of 3072 3.54 instead of 3.46 us).  Of rows 3076
// elements apart every other one is aligned: 2048 of them 18.3 us element by element,
// 16.3 so; 16384 71.7 and 63.8.  With more than 8 chunks a lane the registers that
// hold an aligned row would cost the other rows the waves that hide their loads (16384
// rows, us: 6402 wide 329 -> 199, 7753 396 -> 261, 5120 of 5124 186 -> 130), so NCH = 0 reads
// its aligned rows twice; up to 8 chunks that gains nothing (4096 of 4100 86 -> 91).
template <int NCH, bool ALIGNED>
__global__ void __launch_bounds__(kNormWaves * 64) rmsnorm_kernel(const NormArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * kNormWaves + (threadIdx.x >> 6);
  if (row >= a.rows) return;
  const f16* xr = a.x + row * a.sx;
  f16* orow = a.out + row * a.so;
  const int chunks = a.cols >> 3;          // full 8-element chunks
  const int tail0 = chunks << 3;           // first element of the ragged tail
  float ss = 0.0f;
  auto aligned_row = [&]() {
    return ((reinterpret_cast<uintptr_t>(xr) | reinterpret_cast<uintptr_t>(orow) | reinterpret_cast<uintptr_t>(a.w)) &
            15) == 0;
  };
  auto factor = [&]() {
    const float var = wave_sum(ss) * a.inv_cols;
    return 1.0f / sqrtf(var + a.eps);
  };
  auto store_chunk = [&](int c, const u32x4& x, float rs) {
    const f16x8 wv = *reinterpret_cast<const f16x8*>(a.w + c * 8);
    f16x8 hn;
#pragma unroll
    for (int e = 0; e < 8; ++e) hn[e] = (f16)mul_half(x[e >> 1], rs, e & 1);
    *reinterpret_cast<f16x8*>(orow + c * 8) = wv * hn;
  };
  if (NCH > 0 && (ALIGNED || aligned_row())) {
    u32x4 xv[NCH > 0 ? NCH : 1];
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = i * 64 + lane;
      xv[i] = (u32x4){};
      if (c < chunks) xv[i] = *reinterpret_cast<const u32x4*>(xr + c * 8);
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = add_square(xv[i][e >> 1], ss, e & 1);
    for (int c = tail0 + lane; c < a.cols; c += 64) ss += (float)xr[c] * (float)xr[c];
    const float rs = factor();
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = i * 64 + lane;
      if (c < chunks) store_chunk(c, xv[i], rs);
    }
    for (int c = tail0 + lane; c < a.cols; c += 64) orow[c] = norm_one((float)xr[c], rs, a.w[c]);
  } else if (NCH == 0 && chunks <= kNormChunks * 64 && aligned_row()) {
    // the same sums, kNormStep chunks at a time
    auto each_step = [&](auto&& use) {
      for (int c0 = lane; c0 < chunks; c0 += 64 * kNormStep) {
        u32x4 xv[kNormStep];
#pragma unroll
        for (int i = 0; i < kNormStep; ++i) {
          xv[i] = (u32x4){};
          if (c0 + i * 64 < chunks) xv[i] = *reinterpret_cast<const u32x4*>(xr + (c0 + i * 64) * 8);
        }
        use(c0, xv);
      }
    };
    each_step([&](int, const u32x4(&xv)[kNormStep]) {
#pragma unroll
      for (int i = 0; i < kNormStep; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = add_square(xv[i][e >> 1], ss, e & 1);
    });
    for (int c = tail0 + lane; c < a.cols; c += 64) ss += (float)xr[c] * (float)xr[c];
    const float rs = factor();
    each_step([&](int c0, const u32x4(&xv)[kNormStep]) {
#pragma unroll
      for (int i = 0; i < kNormStep; ++i)
        if (c0 + i * 64 < chunks) store_chunk(c0 + i * 64, xv[i], rs);
    });
    for (int c = tail0 + lane; c < a.cols; c += 64) orow[c] = norm_one((float)xr[c], rs, a.w[c]);
  } else {
    for (int c = lane; c < a.cols; c += 64) ss += (float)xr[c] * (float)xr[c];
    const float rs = factor();
    for (int c = lane; c < a.cols; c += 64) orow[c] = norm_one((float)xr[c], rs, a.w[c]);
  }
}

// ---- rotary (reference :808-847) -------------------------------------------
// One thread per pair of 8-element chunks (d, d + D/2) of a (b, t, h) row: the two
// chunks are each other's rotation partners, so a row is read once.  Heads of Q and
// then K are the fastest row index, so the rows of a token read its cos / sin from
// cache.  Output rows are token-major.  Bound by HBM (4 bytes per value) at large
// token counts, by the launch and one round of loads at small ones.
// Kernel in us, against one thread per chunk that loads its partner chunk too / 16 head
// slots per token that keep cos / sin over several heads, Q and K in turn (slots
// idle with few heads, several rounds with many): 24 + 8 heads x 128, 16 tokens 2.63 /
// 3.53 / 2.41, 2048 9.1 / 7.1 / 6.2, 32768 104 / 98.3 / 95.0 (5.7 TB/s);
// 4 + 1 heads x 128, 16384 tokens 10.9 / 19.2 / 8.8; 14 + 2 x 64, 2048 3.97 / 4.54 / 3.22.
// Two, three or four heads per thread with all slots in use were no faster.
struct RotaryArgs {
  const f16* q;
  const f16* k;
  const f16* cs;
  const f16* sn;
  f16* oq;
  f16* ok;
  int64_t qz, qh, qt, kz, kh, kt, cz, ct, sz, st;
  int64_t rows;  // batch * tokens * (hq + hk)
  int t, hq, hk, d;
  // rotary_kernel: 8-element chunk pairs per row, rows per token, tokens
  FastDiv by_pairs, by_heads, by_tokens;
  int per_wg;  // rows of a workgroup, at most 256 / pairs
};

__device__ __forceinline__ f16 rope_one(float x, float xr, float c, float s, float sign) {
  const f16 a = (f16)(x * c);
  const f16 b = (f16)((xr * sign) * s);
  return (f16)keep32((float)a + (float)b);
}

__device__ __forceinline__ f16x8 rope8(const f16x8& x, const f16x8& xr, const f16x8& c, const f16x8& s, float sign) {
  f16x8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = rope_one((float)x[e], (float)xr[e], (float)c[e], (float)s[e], sign);
  return o;
}

__global__ void __launch_bounds__(256) rotary_kernel(const RotaryArgs a) {
  const int half = a.d >> 1;
  const int rl = fast_div(threadIdx.x, a.by_pairs), d0 = (threadIdx.x - rl * a.by_pairs.d) * 8;
  const int64_t row = (int64_t)blockIdx.x * a.per_wg + rl;
  if (rl >= a.per_wg || row >= a.rows) return;
  const int bt = fast_div((int)row, a.by_heads), h = (int)row - bt * a.by_heads.d, hk = h - a.hq;
  const int b = fast_div(bt, a.by_tokens), t = bt - b * a.t;
  const f16* cs = a.cs + b * a.cz + t * a.ct + d0;
  const f16* sn = a.sn + b * a.sz + t * a.st + d0;
  const f16* x = (hk < 0 ? a.q + b * a.qz + t * a.qt + h * a.qh : a.k + b * a.kz + t * a.kt + hk * a.kh) + d0;
  f16* o = (hk < 0 ? a.oq + ((int64_t)bt * a.hq + h) * a.d : a.ok + ((int64_t)bt * a.hk + hk) * a.d) + d0;
  const f16x8 c0 = *reinterpret_cast<const f16x8*>(cs), c1 = *reinterpret_cast<const f16x8*>(cs + half);
  const f16x8 s0 = *reinterpret_cast<const f16x8*>(sn), s1 = *reinterpret_cast<const f16x8*>(sn + half);
  // cos and sin go out first: the other way round 32768 tokens of 32 + 8 heads x 64 take 66.3
  // instead of 62.8 us.
  asm volatile("" ::: "memory");
  const f16x8 x0 = *reinterpret_cast<const f16x8*>(x), x1 = *reinterpret_cast<const f16x8*>(x + half);
  *reinterpret_cast<f16x8*>(o) = rope8(x0, x1, c0, s0, -1.0f);
  *reinterpret_cast<f16x8*>(o + half) = rope8(x1, x0, c1, s1, 1.0f);
}

// Generic element-wise variant (any even head_dim, any alignment).
__global__ void __launch_bounds__(256) rotary_kernel_scalar(const RotaryArgs a) {
  for (int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x; gid < a.rows * a.d; gid += (int64_t)gridDim.x * 256) {
    const int d = (int)(gid % a.d);
    int64_t r = gid / a.d;
    const int H = a.hq + a.hk;
    const int h = (int)(r % H);
    r /= H;
    const int t = (int)(r % a.t);
    const int64_t b = r / a.t;
    const int half = a.d >> 1;
    const int dr = (d + half) % a.d;
    const float sign = d < half ? -1.0f : 1.0f;
    const f16* src;
    f16* dst;
    if (h < a.hq) {
      src = a.q + b * a.qz + (int64_t)h * a.qh + (int64_t)t * a.qt;
      dst = a.oq + ((b * a.t + t) * a.hq + h) * a.d;
    } else {
      src = a.k + b * a.kz + (int64_t)(h - a.hq) * a.kh + (int64_t)t * a.kt;
      dst = a.ok + ((b * a.t + t) * a.hk + (h - a.hq)) * a.d;
    }
    const float c = (float)a.cs[b * a.cz + (int64_t)t * a.ct + d];
    const float s = (float)a.sn[b * a.sz + (int64_t)t * a.st + d];
    dst[d] = rope_one((float)src[d], (float)src[dr], c, s, sign);
  }
}

// ---- SiLU * up (reference :850-869) -----------------------------------------
// g / den (den >= 1): a Newton step on the hardware reciprocal, Markstein's
// correction of the quotient, and the fix-up instruction for infinities and NaNs.
// Correctly rounded, but for den = 2 - 2^-23 with a reciprocal that is not the nearest
// (one ulp then, which no fp16 result shows as exp is exact enough there).  A
// quotient too small for its remainder to be exact lies far below half of fp16's
// smallest value and becomes 0 either way; a denominator of infinity (exp(-g)
// overflows) is such a case.  The full IEEE division adds
// scaling steps for ranges that do not occur here; every gate gives the same fp16
// value, whichever reciprocal within one ulp the instruction returns.  2048 x 8192: 19.5 -> 18.4 us; 32768 x 8192 is HBM-bound either way
// (276 -> 273 us, 5.9 TB/s).
__device__ __forceinline__ float silu_div(float g, float den) {
  float r = __builtin_amdgcn_rcpf(den);
  r = __builtin_fmaf(__builtin_fmaf(-den, r, 1.0f), r, r);
  const float q = g * r;
  return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-q, den, g), r, q), den, g);
}
__device__ __forceinline__ f16 silu_mul_one(f16 g16, f16 u16) {
  const float g = (float)g16;
  const f16 act = (f16)keep32(silu_div(g, keep32(1.0f + expf(-g))));
  return act * u16;  // fp16 product: the exact fp32 product rounded once
}

__global__ void __launch_bounds__(256) silu_mul_kernel(const f16* g, const f16* u, f16* o, int64_t n) {
  const int64_t i8 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i8 + 8 <= n) {
    const f16x8 gv = *reinterpret_cast<const f16x8*>(g + i8);
    const f16x8 uv = *reinterpret_cast<const f16x8*>(u + i8);
    f16x8 ov;
#pragma unroll
    for (int e = 0; e < 8; ++e) ov[e] = silu_mul_one(gv[e], uv[e]);
    *reinterpret_cast<f16x8*>(o + i8) = ov;
  } else {
    for (int64_t i = i8; i < n; ++i) o[i] = silu_mul_one(g[i], u[i]);
  }
}

__global__ void __launch_bounds__(256) silu_mul_kernel_scalar(const f16* g, const f16* u, f16* o, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) o[i] = silu_mul_one(g[i], u[i]);
}

int check_launch(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return TILEMIX_E_LAUNCH;
  }
  return TILEMIX_OK;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

template <bool ALIGNED>
static void launch_norm(const NormArgs& a, hipStream_t stream) {
  const int lane_chunks = (a.cols / 8 + 63) / 64;  // per lane
  const dim3 grid((unsigned)((a.rows + kNormWaves - 1) / kNormWaves)), block(kNormWaves * 64);
  switch (lane_chunks > (ALIGNED ? kNormChunks : 8) ? 0
          : lane_chunks > 8                         ? kNormChunks
          : lane_chunks > 6                         ? 8
                                                    : (lane_chunks + 1) / 2 * 2) {
    case 2:
      hipLaunchKernelGGL((rmsnorm_kernel<2, ALIGNED>), grid, block, 0, stream, a);
      break;
    case 4:
      hipLaunchKernelGGL((rmsnorm_kernel<4, ALIGNED>), grid, block, 0, stream, a);
      break;
    case 6:
      hipLaunchKernelGGL((rmsnorm_kernel<6, ALIGNED>), grid, block, 0, stream, a);
      break;
    case 8:
      hipLaunchKernelGGL((rmsnorm_kernel<8, ALIGNED>), grid, block, 0, stream, a);
      break;
    case kNormChunks:
      hipLaunchKernelGGL((rmsnorm_kernel<kNormChunks, true>), grid, block, 0, stream, a);
      break;
    default:
      hipLaunchKernelGGL((rmsnorm_kernel<0, false>), grid, block, 0, stream, a);
  }
}

int launch_rmsnorm(const tilemix_rmsnorm_params& p, hipStream_t stream) {
  if (p.x == nullptr || p.weight == nullptr || p.out == nullptr) {
    set_error("tilemix_rms_norm_f16: null tensor pointer");
    return TILEMIX_E_INVALID;
  }
  if (p.rows < 0 || p.cols <= 0 || p.stride_x < p.cols || p.stride_out < p.cols || !(p.eps >= 0.0f)) {
    set_error("tilemix_rms_norm_f16: invalid shape (rows %lld, cols %d, strides %lld/%lld, eps %g)",
              (long long)p.rows, p.cols, (long long)p.stride_x, (long long)p.stride_out, (double)p.eps);
    return TILEMIX_E_INVALID;
  }
  if (p.rows == 0) return TILEMIX_OK;
  NormArgs a;
  a.x = static_cast<const f16*>(p.x);
  a.w = static_cast<const f16*>(p.weight);
  a.out = static_cast<f16*>(p.out);
  a.rows = p.rows;
  a.sx = p.stride_x;
  a.so = p.stride_out;
  a.cols = p.cols;
  a.inv_cols = 1.0f / (float)p.cols;  // the mean's factor, as fp32(1/N)
  a.eps = p.eps;
  const bool aligned = aligned16(p.x) && aligned16(p.out) && aligned16(p.weight) &&
                       (p.rows == 1 || ((p.stride_x | p.stride_out) & 7) == 0);
  if (aligned)
    launch_norm<true>(a, stream);
  else
    launch_norm<false>(a, stream);
  return check_launch("tilemix_rms_norm_f16");
}

int launch_rotary(const tilemix_rotary_params& p, hipStream_t stream) {
  if (p.q == nullptr || p.k == nullptr || p.cos == nullptr || p.sin == nullptr || p.q_out == nullptr ||
      p.k_out == nullptr) {
    set_error("tilemix_rotary_f16: null tensor pointer");
    return TILEMIX_E_INVALID;
  }
  if (p.batch < 0 || p.tokens < 0 || p.heads_q <= 0 || p.heads_k <= 0 || p.head_dim <= 0 || (p.head_dim & 1)) {
    set_error("tilemix_rotary_f16: invalid shape (batch %d, tokens %d, heads %d/%d, head_dim %d)", p.batch,
              p.tokens, p.heads_q, p.heads_k, p.head_dim);
    return TILEMIX_E_INVALID;
  }
  RotaryArgs a;
  a.q = static_cast<const f16*>(p.q);
  a.k = static_cast<const f16*>(p.k);
  a.cs = static_cast<const f16*>(p.cos);
  a.sn = static_cast<const f16*>(p.sin);
  a.oq = static_cast<f16*>(p.q_out);
  a.ok = static_cast<f16*>(p.k_out);
  a.qz = p.stride_q_batch;
  a.qh = p.stride_q_head;
  a.qt = p.stride_q_token;
  a.kz = p.stride_k_batch;
  a.kh = p.stride_k_head;
  a.kt = p.stride_k_token;
  a.cz = p.stride_cos_batch;
  a.ct = p.stride_cos_token;
  a.sz = p.stride_sin_batch;
  a.st = p.stride_sin_token;
  a.t = p.tokens;
  a.hq = p.heads_q;
  a.hk = p.heads_k;
  a.d = p.head_dim;
  const int64_t heads = (int64_t)p.heads_q + p.heads_k;
  a.rows = (int64_t)p.batch * p.tokens * heads;
  if (a.rows == 0) return TILEMIX_OK;
  constexpr int64_t kMaxGroups = (1 << 24) - 1;  // of 256 threads: HIP takes less than 2^32 along x
  // Whole tokens where that idles at most an eighth of the workgroup: its output then
  // starts at a line's start more often (32768 tokens of 20 + 4 heads x 80 47.9 -> 44.8 us).
  a.per_wg = std::max(1, 256 / std::max(1, p.head_dim / 16));
  const int64_t whole = a.per_wg / heads * heads;
  if (whole * 8 >= (int64_t)a.per_wg * 7) a.per_wg = (int)whole;
  const int64_t groups = (a.rows - 1) / a.per_wg + 1;
  // 16-byte chunks need head_dim % 16 == 0 (so both halves are chunk aligned)
  // and every row start 16-byte aligned.
  const bool vec = (p.head_dim % 16) == 0 && p.head_dim <= 16 * 256 && a.rows <= INT32_MAX && groups <= kMaxGroups &&
                   aligned16(p.q) && aligned16(p.k) && aligned16(p.cos) && aligned16(p.sin) && aligned16(p.q_out) &&
                   aligned16(p.k_out) &&
                   ((a.qz | a.qh | a.qt | a.kz | a.kh | a.kt | a.cz | a.ct | a.sz | a.st) & 7) == 0;
  if (vec) {
    const int pairs = p.head_dim / 16;
    a.by_pairs = make_fast_div(pairs);
    a.by_heads = make_fast_div(p.heads_q + p.heads_k);
    a.by_tokens = make_fast_div(p.tokens);
    hipLaunchKernelGGL(rotary_kernel, dim3((unsigned)groups), dim3(256), 0, stream, a);
  } else {
    const int64_t all = std::min((a.rows * p.head_dim + 255) / 256, kMaxGroups);
    hipLaunchKernelGGL(rotary_kernel_scalar, dim3((unsigned)all), dim3(256), 0, stream, a);
  }
  return check_launch("tilemix_rotary_f16");
}

int launch_silu_mul(const void* gate, const void* up, void* out, int64_t n, hipStream_t stream) {
  if (gate == nullptr || up == nullptr || out == nullptr || n < 0) {
    set_error("tilemix_silu_mul_f16: null tensor pointer or negative size");
    return TILEMIX_E_INVALID;
  }
  if (n == 0) return TILEMIX_OK;
  const f16* g = static_cast<const f16*>(gate);
  const f16* u = static_cast<const f16*>(up);
  f16* o = static_cast<f16*>(out);
  if (aligned16(gate) && aligned16(up) && aligned16(out)) {
    const int64_t threads = (n + 7) / 8;
    hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, g, u, o, n);
  } else {
    hipLaunchKernelGGL(silu_mul_kernel_scalar, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, g, u, o, n);
  }
  return check_launch("tilemix_silu_mul_f16");
}

}  // namespace tmx

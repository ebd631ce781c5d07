// Piece 2: the KV compressor (gated softmax pool over `ratio` tokens + RMSNorm) and the
// interleaved RoPE it is followed by.
//
//   latent[b, g, :] = RMSNorm( dtype( sum_r kv[b, g*ratio + r, :] * softmax_r(gate[b, g*ratio + r, :]) ) )
//   -- src/mzoo/archs/owlet1/cache.py:142-172 (DeepseekV41Compressor.forward, fp32 pooling),
//      owlet1/norm_rope.py:25-30 (RMSNorm: h * rsqrt(mean(h^2) + eps), dtype, weight * h).
//   ratio 1: latent = RMSNorm(dtype(kv)) (the un-gated per-token projection).
//   rope: owlet1/norm_rope.py:126-145 (pairs (even, odd) of the trailing rope channels,
//   fp32 math, inverse = conjugate rotation).
//
// Bit-exact by construction against the CPU restatement (oracle/compressor.py): both
// evaluate the same float32 operation sequence --
//   exp: n = rint(x*log2e), r = (x - n*ln2_hi) - n*ln2_lo, degree-7 Taylor in Horner form,
//        times 2^n through the exponent field (two steps below 2^-126); no fused ops;
//   softmax over r: running max, exp(g_r - max), sum from 0 in r order, divide;
//   pooled: sum from 0 in r order of kv_r * p_r;
//   RMSNorm: lane l of the wave sums channels l, l+64, ... in order from 0, then the xor
//   butterfly (32, 16, 8, 4, 2, 1); var = sum / D; rsqrt = 1 / sqrt (correctly rounded).
// Layout: one wave per (b, group), lane l owning channels l + 64 i (coalesced 256 B rows), or
// one workgroup per group where the ratio is large.
#include "common.h"

namespace mzk {
namespace {

constexpr int kMaxPerLane = 16;  // D <= 1024
constexpr int kPoolAhead = 2;    // channels per lane loaded together (2 * ratio registers each)

// Blocks along the grid's x, which takes fewer than 2^32 threads (2^21 blocks of 1024); the rest
// along y.
constexpr int64_t kGridX = int64_t(1) << 21;
inline dim3 grid_xy(int64_t blocks) {
  const int64_t x = blocks < kGridX ? blocks : kGridX;
  return dim3(static_cast<unsigned>(x), static_cast<unsigned>((blocks + x - 1) / x));
}
__device__ __forceinline__ int64_t block_xy() { return static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x; }

// The pooled value of one channel over R tokens held in registers: the operations and order
// above; exp(g_r - max) is formed once and used in the sum and in the weight.
template <int R>
__device__ __forceinline__ float pool_channel(const float (&k)[R], const float (&g)[R]) {
  float m = g[0];
#pragma unroll
  for (int r = 1; r < R; ++r) m = fmaxf(m, g[r]);
  float e[R];
  float s = 0.0f;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    e[r] = exp_pinned(g[r] - m);
    s = s + e[r];
  }
  float acc = 0.0f;
#pragma unroll
  for (int r = 0; r < R; ++r) acc = acc + k[r] * div_rn(e[r], s);
  return acc;
}

// Ratios 1, 2 and 4, and 3 and 5 from wave_groups() groups: one wave per group, kPoolAhead
// channels' whole groups loaded into registers before the first is used.  It was bound by
// latency -- loops that read each gate three times from the cache, one load in flight, and
// formed each exp twice; now by the divisions and exps (some 55 operations per token and
// channel), about twice its memory time.
// 8192 tokens x 576 channels: ratio 4 35.9 -> 14.0 us, ratio 2 24.3 -> 13.6 us (4 channels
// ahead 14.2, 8 15.3, 16 15.4).
template <int ODT, int WDT, int RATIO>
__global__ void __launch_bounds__(256) compress_kernel(const float* __restrict__ kv, const float* __restrict__ gate,
                                                       int64_t B, int64_t n_groups, int ratio, int D,
                                                       int64_t tokens_per_batch, const void* __restrict__ weight,
                                                       float eps, void* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int64_t rid = block_xy() * 4 + (threadIdx.x >> 6);
  if (rid >= B * n_groups) return;  // whole waves
  const int64_t b = rid / n_groups;
  const int64_t g = rid - b * n_groups;
  const float* kvb = kv + (b * tokens_per_batch + g * ratio) * D;
  const float* gtb = gate ? gate + (b * tokens_per_batch + g * ratio) * D : nullptr;

  float h[kMaxPerLane];
  float ss = 0.0f;
  constexpr int R = RATIO, A = kPoolAhead;
  static_assert(kMaxPerLane % A == 0, "whole batches of channels");
#pragma unroll
  for (int i0 = 0; i0 < kMaxPerLane; i0 += A) {
    if (64 * i0 < D) {  // uniform
      float k[A][R], g[A][R];
#pragma unroll
      for (int a = 0; a < A; ++a) {
        // channels at or beyond D read channel D - 1 and are dropped
        const int d = lane + 64 * (i0 + a) < D ? lane + 64 * (i0 + a) : D - 1;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          k[a][r] = kvb[r * D + d];
          g[a][r] = R > 1 ? gtb[r * D + d] : 0.0f;
        }
      }
#pragma unroll
      for (int a = 0; a < A; ++a) {
        h[i0 + a] = 0.0f;
        if (64 * (i0 + a) < D) {  // uniform
          const float v = round_to_dtype<ODT>(R > 1 ? pool_channel<R>(k[a], g[a]) : k[a][0]);
          if (lane + 64 * (i0 + a) < D) {
            h[i0 + a] = v;
            ss = ss + v * v;
          }
        }
      }
    } else {
#pragma unroll
      for (int a = 0; a < A; ++a) h[i0 + a] = 0.0f;
    }
  }
  // xor butterfly: every lane ends with the same total
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) ss = ss + __shfl_xor(ss, m, 64);
  const float var = div_rn(ss, static_cast<float>(D));
  const float inv = div_rn(1.0f, sqrt_rn(var + eps));
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) {
    const int d = lane + 64 * i;
    if (d < D) {
      const float normed = round_to_dtype<ODT>(h[i] * inv);
      const float w = load_as_f32<WDT>(weight, d);
      store_from_f32<ODT>(out, rid * D + d, w * normed);
    }
  }
}

// Any other ratio, and ratios 3 and 5 of fewer groups: one workgroup per group, thread d owns
// channel d and walks the group's tokens in order, kTokensAhead of them loaded together; the
// channels meet in LDS, where wave 0 sums their squares in the pinned order.  A group of 128
// tokens in one wave took 9 channels x 128 tokens x 3 dependent reads per lane in turn: 8192
// tokens x 576 channels at ratio 128 889 -> 62.8 us, at ratio 8 59 -> 14.5 (16 tokens ahead:
// 59.5 and 23.6 us; 4: 72 and 16.1).
constexpr int kTokensAhead = 8;

// Ratios 3 and 5 in the wave form: from here, a wave or more for each SIMD, it keeps the chip
// busy, and it reads a short group's tokens once, where the workgroup form requests 8 at a time
// three times over.  Workgroup -> wave form, us: ratio 3, 576 channels, 1000 groups 9.2 -> 8.6 (682:
// 7.5 -> 8.6), 2730 24.1 -> 13.4, 21845 188 -> 68; 1024 channels, 1000 groups 13.4 -> 13.1 (682: 10.8 ->
// 12.7); ratio 5, 1024 channels, 1638 groups 26.7 -> 23.5 (1200: 20.3 -> 22.7), 13107 197 -> 123.
constexpr int64_t wave_groups(int ratio) { return 256 * (ratio + 1); }

template <int ODT, int WDT>
__global__ void __launch_bounds__(64 * kMaxPerLane)
    compress_wide_kernel(const float* __restrict__ kv, const float* __restrict__ gate, int64_t groups, int64_t n_groups,
                         int ratio, int D, int64_t tokens_per_batch, const void* __restrict__ weight, float eps,
                         void* __restrict__ out) {
  __shared__ float h_lds[64 * kMaxPerLane];
  __shared__ float inv_lds;
  const int64_t rid = block_xy();
  if (rid >= groups) return;
  const int64_t b = rid / n_groups;
  const int64_t g = rid - b * n_groups;
  const int d = threadIdx.x < D ? threadIdx.x : D - 1;  // (threads beyond D: a channel again, dropped)
  const float* k = kv + (b * tokens_per_batch + g * ratio) * D + d;
  const float* gt = gate + (b * tokens_per_batch + g * ratio) * D + d;
  // kTokensAhead tokens from p on, of which `left` are the group's (beyond them its last, not
  // used).  The walks count the tokens left and move the pointer: the count cannot wrap at any
  // ratio, and the addresses stay 32-bit offsets (a 64-bit token number took 8192 tokens of 576 channels
  // at ratio 128 from 62.8 to 70.7 us, at ratio 8 from 15.4 to 16.6; so counted 63.4 and 15.8).
  const int step = kTokensAhead * D;
  auto ahead = [&](const float* p, int left, float (&v)[kTokensAhead]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kTokensAhead; ++j) v[j] = p[(j < left ? j : left - 1) * D];
  };
  float gv[kTokensAhead], kvv[kTokensAhead];
  const float* at = gt;
  float m = gt[0];
  for (int left = ratio; left > 0; left -= kTokensAhead, at += step) {
    ahead(at, left, gv);
#pragma unroll
    for (int j = 0; j < kTokensAhead; ++j)
      if (j < left) m = fmaxf(m, gv[j]);
  }
  at = gt;
  float s = 0.0f;
  for (int left = ratio; left > 0; left -= kTokensAhead, at += step) {
    ahead(at, left, gv);
#pragma unroll
    for (int j = 0; j < kTokensAhead; ++j)
      if (j < left) s = s + exp_pinned(gv[j] - m);
  }
  at = gt;
  float acc = 0.0f;
  for (int left = ratio; left > 0; left -= kTokensAhead, at += step, k += step) {
    ahead(at, left, gv);
    ahead(k, left, kvv);
#pragma unroll
    for (int j = 0; j < kTokensAhead; ++j)
      if (j < left) acc = acc + kvv[j] * div_rn(exp_pinned(gv[j] - m), s);
  }
  const float v = round_to_dtype<ODT>(acc);  // latent.to(dtype) before the norm
  h_lds[threadIdx.x] = v;
  __syncthreads();
  if (threadIdx.x < 64) {
    float ss = 0.0f;
    for (int c = threadIdx.x; c < D; c += 64) ss = ss + h_lds[c] * h_lds[c];
#pragma unroll
    for (int x = 32; x >= 1; x >>= 1) ss = ss + __shfl_xor(ss, x, 64);
    const float var = div_rn(ss, static_cast<float>(D));
    if (threadIdx.x == 0) inv_lds = div_rn(1.0f, sqrt_rn(var + eps));
  }
  __syncthreads();
  if (threadIdx.x < D) {
    const float normed = round_to_dtype<ODT>(v * inv_lds);
    store_from_f32<ODT>(out, rid * D + d, load_as_f32<WDT>(weight, d) * normed);
  }
}

// DeepseekV41RMSNorm (owlet1/norm_rope.py:25-30) of any width: one wave per row, the sum
// of squares in the pinned order above (lane l sums channels l, l+64, ... from 0, then the
// xor butterfly), var = sum / D, inv = 1 / sqrt(var + eps); normed = IDT(h * inv) (the
// ".to(input_dtype)"), out = ODT(weight * normed).  Two passes over the row (L2-resident).
template <int IDT, int WDT, int ODT>
__global__ void __launch_bounds__(256) rms_norm_kernel(const void* __restrict__ x, int64_t rows, int D,
                                                       int64_t x_stride, const void* __restrict__ weight, float eps,
                                                       void* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // whole waves
  const int64_t base = row * x_stride;
  float ss = 0.0f;
  for (int d = lane; d < D; d += 64) {
    const float v = load_as_f32<IDT>(x, base + d);
    ss = ss + v * v;
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) ss = ss + __shfl_xor(ss, m, 64);
  const float var = div_rn(ss, static_cast<float>(D));
  const float inv = div_rn(1.0f, sqrt_rn(var + eps));
  for (int d = lane; d < D; d += 64) {
    const float normed = round_to_dtype<IDT>(load_as_f32<IDT>(x, base + d) * inv);
    store_from_f32<ODT>(out, row * D + d, load_as_f32<WDT>(weight, d) * normed);
  }
}

template <int IDT, int WDT>
int launch_rms_norm_o(int odt, const void* x, int64_t rows, int D, int64_t xs, const void* w, float eps, void* out,
                      hipStream_t s) {
  const unsigned grid = static_cast<unsigned>((rows + 3) / 4);
  switch (odt) {
    case MZK_F32: rms_norm_kernel<IDT, WDT, MZK_F32><<<grid, 256, 0, s>>>(x, rows, D, xs, w, eps, out); break;
    case MZK_BF16: rms_norm_kernel<IDT, WDT, MZK_BF16><<<grid, 256, 0, s>>>(x, rows, D, xs, w, eps, out); break;
    case MZK_F16: rms_norm_kernel<IDT, WDT, MZK_F16><<<grid, 256, 0, s>>>(x, rows, D, xs, w, eps, out); break;
    default: set_last_error("rms_norm: unsupported out dtype %d", odt); return MZK_EINVAL;
  }
  return MZK_OK;
}

template <int IDT>
int launch_rms_norm(int wdt, int odt, const void* x, int64_t rows, int D, int64_t xs, const void* w, float eps,
                    void* out, hipStream_t s) {
  switch (wdt) {
    case MZK_F32: return launch_rms_norm_o<IDT, MZK_F32>(odt, x, rows, D, xs, w, eps, out, s);
    case MZK_BF16: return launch_rms_norm_o<IDT, MZK_BF16>(odt, x, rows, D, xs, w, eps, out, s);
    case MZK_F16: return launch_rms_norm_o<IDT, MZK_F16>(odt, x, rows, D, xs, w, eps, out, s);
    default: set_last_error("rms_norm: unsupported weight dtype %d", wdt); return MZK_EINVAL;
  }
}

// rows x D (dtype DT); cos/sin [rows / heads, rd/2] fp32, broadcast over `heads`
// consecutive rows.  Nope channels are copied through unchanged.
template <int DT>
__global__ void rope_kernel(const void* __restrict__ x, const float* __restrict__ cosv, const float* __restrict__ sinv,
                            int64_t rows, int D, int rd, int heads, int inverse, void* __restrict__ y) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int half = rd / 2;
  const int per_row = (D - rd) + half;  // nope channels + rope pairs
  if (t >= rows * per_row) return;
  const int64_t row = t / per_row;
  const int k = static_cast<int>(t - row * per_row);
  const int64_t base = row * D;
  if (k < D - rd) {
    store_from_f32<DT>(y, base + k, load_as_f32<DT>(x, base + k));
    return;
  }
  const int i = k - (D - rd);
  const int64_t crow = row / heads;
  const float c = cosv[crow * half + i];
  const float s = inverse ? -sinv[crow * half + i] : sinv[crow * half + i];
  const float ev = load_as_f32<DT>(x, base + (D - rd) + 2 * i);
  const float od = load_as_f32<DT>(x, base + (D - rd) + 2 * i + 1);
  store_from_f32<DT>(y, base + (D - rd) + 2 * i, ev * c - od * s);
  store_from_f32<DT>(y, base + (D - rd) + 2 * i + 1, ev * s + od * c);
}

template <int ODT, int WDT>
void launch_compress_r(const float* kv, const float* gate, int64_t B, int64_t n, int ratio, int D, int64_t tpb,
                       const void* w, float eps, void* out, hipStream_t s) {
  const dim3 grid = grid_xy((B * n + 3) / 4);
  const bool wide = (ratio == 3 || ratio == 5) && B * n < wave_groups(ratio);
  switch (wide ? 0 : ratio) {
    case 1: compress_kernel<ODT, WDT, 1><<<grid, 256, 0, s>>>(kv, gate, B, n, ratio, D, tpb, w, eps, out); break;
    case 2: compress_kernel<ODT, WDT, 2><<<grid, 256, 0, s>>>(kv, gate, B, n, ratio, D, tpb, w, eps, out); break;
    case 3: compress_kernel<ODT, WDT, 3><<<grid, 256, 0, s>>>(kv, gate, B, n, ratio, D, tpb, w, eps, out); break;
    case 4: compress_kernel<ODT, WDT, 4><<<grid, 256, 0, s>>>(kv, gate, B, n, ratio, D, tpb, w, eps, out); break;
    case 5: compress_kernel<ODT, WDT, 5><<<grid, 256, 0, s>>>(kv, gate, B, n, ratio, D, tpb, w, eps, out); break;
    default:
      compress_wide_kernel<ODT, WDT><<<grid_xy(B * n), (D + 63) / 64 * 64, 0, s>>>(kv, gate, B * n, n, ratio, D, tpb, w, eps,
                                                                                   out);
  }
}

template <int ODT>
int launch_compress_w(int wdt, const float* kv, const float* gate, int64_t B, int64_t n, int ratio, int D, int64_t tpb,
                      const void* w, float eps, void* out, hipStream_t s) {
  switch (wdt) {
    case MZK_F32: launch_compress_r<ODT, MZK_F32>(kv, gate, B, n, ratio, D, tpb, w, eps, out, s); break;
    case MZK_BF16: launch_compress_r<ODT, MZK_BF16>(kv, gate, B, n, ratio, D, tpb, w, eps, out, s); break;
    case MZK_F16: launch_compress_r<ODT, MZK_F16>(kv, gate, B, n, ratio, D, tpb, w, eps, out, s); break;
    default: set_last_error("compress: unsupported weight dtype %d", wdt); return MZK_EINVAL;
  }
  return MZK_OK;
}

template <int DT>
void launch_rope(const void* x, const float* c, const float* sn, int64_t rows, int D, int rd, int heads, int inverse,
                 void* y, hipStream_t s) {
  const int64_t n = rows * ((D - rd) + rd / 2);
  rope_kernel<DT><<<static_cast<unsigned>((n + 255) / 256), 256, 0, s>>>(x, c, sn, rows, D, rd, heads, inverse, y);
}

}  // namespace
}  // namespace mzk

using namespace mzk;

extern "C" int mzk_compress(const float* kv, const float* gate, int64_t B, int64_t n_groups, int ratio, int D,
                            int64_t tokens_per_batch, const void* norm_weight, int weight_dtype, float eps, void* out,
                            int out_dtype, void* stream) {
  MZK_CHECK_ARG(B >= 0 && n_groups >= 0 && ratio >= 1 && D >= 1 && D <= 64 * kMaxPerLane,
                "compress: bad sizes (ratio >= 1, 1 <= D <= %d)", 64 * kMaxPerLane);
  MZK_CHECK_ARG(tokens_per_batch >= n_groups * ratio, "compress: tokens_per_batch < n_groups * ratio");
  if (B * n_groups == 0) return MZK_OK;
  MZK_CHECK_ARG(kv && norm_weight && out && (ratio == 1 || gate), "compress: null pointer");
  int rc;
  hipStream_t s = as_stream(stream);
  switch (out_dtype) {
    case MZK_F32: rc = launch_compress_w<MZK_F32>(weight_dtype, kv, gate, B, n_groups, ratio, D, tokens_per_batch,
                                                  norm_weight, eps, out, s); break;
    case MZK_BF16: rc = launch_compress_w<MZK_BF16>(weight_dtype, kv, gate, B, n_groups, ratio, D, tokens_per_batch,
                                                    norm_weight, eps, out, s); break;
    case MZK_F16: rc = launch_compress_w<MZK_F16>(weight_dtype, kv, gate, B, n_groups, ratio, D, tokens_per_batch,
                                                  norm_weight, eps, out, s); break;
    default: set_last_error("compress: unsupported out dtype %d", out_dtype); return MZK_EINVAL;
  }
  if (rc) return rc;
  MZK_LAUNCH_CHECK("compress");
  return MZK_OK;
}

extern "C" int mzk_rope(const void* x, int dtype, const float* cos_t, const float* sin_t, int64_t rows, int D,
                        int rope_dim, int heads, int inverse, void* y, void* stream) {
  MZK_CHECK_ARG(rows >= 0 && D >= 1 && rope_dim >= 0 && rope_dim <= D && rope_dim % 2 == 0 && heads >= 1,
                "rope: bad sizes (even rope_dim <= D, heads >= 1)");
  if (rows == 0) return MZK_OK;
  MZK_CHECK_ARG(x && y && (rope_dim == 0 || (cos_t && sin_t)), "rope: null pointer");
  MZK_DISPATCH_DT(dtype, launch_rope, x, cos_t, sin_t, rows, D, rope_dim, heads, inverse, y, as_stream(stream));
  MZK_LAUNCH_CHECK("rope");
  return MZK_OK;
}

extern "C" int mzk_rms_norm(const void* x, int x_dtype, int64_t rows, int D, int64_t x_row_stride,
                            const void* weight, int weight_dtype, float eps, void* out, int out_dtype, void* stream) {
  MZK_CHECK_ARG(rows >= 0 && D >= 1 && x_row_stride >= D, "rms_norm: bad sizes (D >= 1, row stride >= D)");
  if (rows == 0) return MZK_OK;
  MZK_CHECK_ARG(x && weight && out, "rms_norm: null pointer");
  hipStream_t s = as_stream(stream);
  int rc;
  switch (x_dtype) {
    case MZK_F32: rc = launch_rms_norm<MZK_F32>(weight_dtype, out_dtype, x, rows, D, x_row_stride, weight, eps, out, s); break;
    case MZK_BF16: rc = launch_rms_norm<MZK_BF16>(weight_dtype, out_dtype, x, rows, D, x_row_stride, weight, eps, out, s); break;
    case MZK_F16: rc = launch_rms_norm<MZK_F16>(weight_dtype, out_dtype, x, rows, D, x_row_stride, weight, eps, out, s); break;
    default: set_last_error("rms_norm: unsupported input dtype %d", x_dtype); return MZK_EINVAL;
  }
  if (rc) return rc;
  MZK_LAUNCH_CHECK("rms_norm");
  return MZK_OK;
}

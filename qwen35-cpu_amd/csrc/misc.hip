// Small kernels: embedding gather, stand-alone activation ops used by the
// kernel-level ABI entries, and the reference-shaped DeltaNet row update.
#include "q35_device.h"
#include "q35_internal.h"

namespace q35 {
namespace {

// dequantize_embedding_row for the identity-basis DOT4 head
// (src/runtime/gguf_matrix.inl:21-26, q4_dot4.cpp:31-40): x = half(d[r]) * (u - 8).
__global__ void embed_kernel(const q35_q4_0_block_x8 *embed, int nb, const int32_t *tokens,
                             float *x, int hidden, int32_t *counts, long long counts_stride,
                             const int32_t *slots, const uint8_t *count_input, bool g16) {
  const int r = blockIdx.x;
  const int token = tokens[r];
  const int rt = token >> 3, row = token & 7;
  for (int k = threadIdx.x; k < hidden; k += blockDim.x) {
    const int b = k >> 5, kk = k & 31;
    if (g16) {
      // Q4G16Tile: d[half][row] then the DOT4 codes (q4_g16_dequantize_row, q4_g16.cpp:98-103)
      const uint8_t *tile = reinterpret_cast<const uint8_t *>(embed) + (static_cast<size_t>(rt) * nb + b) * 160;
      const uint16_t dh = *reinterpret_cast<const uint16_t *>(tile + 2 * (8 * (kk >> 4) + row));
      const int u = (tile[32 + 32 * (kk >> 3) + 4 * row + (kk & 3)] >> (4 * ((kk & 7) >> 2))) & 15;
      x[static_cast<size_t>(r) * hidden + k] = half_bits_to_float(dh) * static_cast<float>(u - 8);
      continue;
    }
    const q35_q4_0_block_x8 &w = embed[static_cast<size_t>(rt) * nb + b];
    const int u = (w.qs[32 * (kk >> 3) + 4 * row + (kk & 3)] >> (4 * ((kk & 7) >> 2))) & 15;
    x[static_cast<size_t>(r) * hidden + k] = half_bits_to_float(w.d[row]) * static_cast<float>(u - 8);
  }
  if (threadIdx.x == 0 && counts != nullptr && count_input != nullptr && count_input[r])
    counts[static_cast<long long>(slots[r]) * counts_stride + token] += 1;
}

__global__ void rms_norm_kernel(const float *x, const float *w, float *y, int width, float eps,
                                float offset) {
  __shared__ float scratch[8];
  const int r = blockIdx.x;
  const float *xr = x + static_cast<size_t>(r) * width;
  float ss = 0.0F;
  for (int i = threadIdx.x; i < width; i += 256) ss += xr[i] * xr[i];
  ss = block_sum<4>(ss, scratch);
  const float inv = 1.0F / sqrtf(ss / static_cast<float>(width) + eps);
  for (int i = threadIdx.x; i < width; i += 256)
    y[static_cast<size_t>(r) * width + i] = xr[i] * inv * (w[i] + offset);
}

__global__ void l2_normalize_kernel(float *x, int width, float eps, float scale) {
  __shared__ float scratch[8];
  float *xr = x + static_cast<size_t>(blockIdx.x) * width;
  float ss = 0.0F;
  for (int i = threadIdx.x; i < width; i += 256) ss += xr[i] * xr[i];
  ss = block_sum<4>(ss, scratch);
  const float m = scale / sqrtf(ss + eps);
  __syncthreads();
  for (int i = threadIdx.x; i < width; i += 256) xr[i] *= m;
}

// causal_conv1d_silu_f32 (activation.cpp:164-222): kernel-major weights
// [kernel][channels], the ring of kernel - 1 past inputs per channel in
// `state` (position p in slot (ring + p) mod (kernel - 1), the call's first
// token being position 0). The sum of a token: the product of its own
// input's tap, then the history oldest first, one fmaf per tap (written out, so
// that every form below rounds alike).
//
// The history of a token is the call's own input rows except for its first
// kernel - 1 tokens, so tokens need not run in order: a thread takes V
// adjacent channels of kConvRun consecutive tokens, the last taps in
// registers, and the launch is bound by the two streams (inputs in, outputs
// out). Only the first run (tokens below kConvRun >= kernel - 1) reads the
// ring, and the same threads then write the ring's new rows, so no other
// workgroup touches it. 1500 tokens of 8192 channels: one thread per channel
// walking every token through the ring in memory took 1250 us (0.08 TB/s),
// this form 21.0 us (4.7 TB/s).
constexpr int kConvRun = 8;
// Kernels other than 4 re-read their taps token by token, so a run takes as
// long as walking about 12 tokens through the ring. Runs against the walk:
// kernel 5 over 1000 channels 9.6 against 7.7 us at 8 tokens, 9.7 against 10.2
// at 12, 9.7 against 12.8 at 16; kernel 9 over 6144 channels 13.8 against 10.1,
// 14.3 and 18.4; over 64 channels they meet at 13. Below this the walk is taken.
constexpr int kConvGeneralMin = 13;

template <int V>
struct ConvVec {
  float v[V];
};
template <int V>
__device__ __forceinline__ ConvVec<V> conv_load(const float *p) {
  ConvVec<V> r;
  if constexpr (V == 4) {
    const q35_f32x4 x = *reinterpret_cast<const q35_f32x4 *>(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) r.v[e] = x[e];
  } else {
    r.v[0] = *p;
  }
  return r;
}
template <int V>
__device__ __forceinline__ void conv_store(float *p, const ConvVec<V> &r) {
  if constexpr (V == 4)
    *reinterpret_cast<q35_f32x4 *>(p) = q35_f32x4{r.v[0], r.v[1], r.v[2], r.v[3]};
  else
    *p = r.v[0];
}

// K: the kernel size (taps in registers), or 0 for any size up to
// kConvRun + 1 (taps re-read through the caches).
template <int V, int K>
__global__ void conv1d_silu_runs_kernel(float *state, int ring, const float *input, long long stride, const float *w,
                                        float *out, int batch, int channels, int kernel, int begin, int end) {
  const int c = begin + V * static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (c >= end) return;
  const int hist = K > 0 ? K - 1 : kernel - 1;
  const int t0 = static_cast<int>(blockIdx.y) * kConvRun, t1 = min(t0 + kConvRun, batch);
  // input of position p >= -hist: before 0 from the ring
  auto past = [&](int p) {
    return conv_load<V>(p >= 0 ? input + p * stride + c : state + static_cast<size_t>((ring + p + hist) % hist) * channels + c);
  };
  auto finish = [&](int t, const ConvVec<V> &sum) {
    ConvVec<V> y;
#pragma unroll
    for (int e = 0; e < V; ++e) y.v[e] = silu_times(sum.v[e], 1.0F);
    conv_store<V>(out + static_cast<size_t>(t) * channels + c, y);
  };
  if constexpr (K > 0) {
    ConvVec<V> wk[K], x[K - 1 + kConvRun];  // x[i]: position t0 - (K - 1) + i
#pragma unroll
    for (int k = 0; k < K; ++k) wk[k] = conv_load<V>(w + static_cast<size_t>(k) * channels + c);
#pragma unroll
    for (int i = 0; i < K - 1 + kConvRun; ++i) x[i] = past(min(t0 - (K - 1) + i, batch - 1));
#pragma unroll
    for (int i = 0; i < kConvRun; ++i) {
      if (t0 + i >= t1) break;
      ConvVec<V> sum;
#pragma unroll
      for (int e = 0; e < V; ++e) {
        sum.v[e] = x[K - 1 + i].v[e] * wk[K - 1].v[e];
#pragma unroll
        for (int k = 0; k < K - 1; ++k) sum.v[e] = fmaf(x[i + k].v[e], wk[k].v[e], sum.v[e]);
      }
      finish(t0 + i, sum);
    }
  } else {
    for (int t = t0; t < t1; ++t) {
      const ConvVec<V> x = past(t), wl = conv_load<V>(w + static_cast<size_t>(hist) * channels + c);
      ConvVec<V> sum;
#pragma unroll
      for (int e = 0; e < V; ++e) sum.v[e] = x.v[e] * wl.v[e];
      for (int k = 0; k < hist; ++k) {
        const ConvVec<V> h = past(t - hist + k), wt = conv_load<V>(w + static_cast<size_t>(k) * channels + c);
#pragma unroll
        for (int e = 0; e < V; ++e) sum.v[e] = fmaf(h.v[e], wt.v[e], sum.v[e]);
      }
      finish(t, sum);
    }
  }
  if (t0 == 0)
    for (int p = max(0, batch - hist); p < batch; ++p)
      conv_store<V>(state + static_cast<size_t>((ring + p) % hist) * channels + c, conv_load<V>(input + p * stride + c));
}

// The same with one thread per channel walking the tokens in order through
// the ring: for outputs that overlap the inputs (each token's input is read
// before its output is written), for kernels longer than a run, and for the
// few tokens where runs of a general kernel size are slower.
__global__ void conv1d_silu_kernel(float *state, int ring, const float *input, long long stride, const float *w,
                                   float *out, int batch, int channels, int kernel, int begin, int end) {
  const int c = begin + static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (c >= end) return;
  const int hist = kernel - 1;
  for (int t = 0; t < batch; ++t) {
    const float x = input[t * stride + c];
    float sum = x * w[static_cast<size_t>(hist) * channels + c];
    for (int k = 0; k < hist; ++k)
      sum = fmaf(state[static_cast<size_t>((ring + k) % hist) * channels + c],
                 w[static_cast<size_t>(k) * channels + c], sum);
    if (hist) state[static_cast<size_t>(ring) * channels + c] = x;
    out[static_cast<size_t>(t) * channels + c] = silu_times(sum, 1.0F);
    if (hist) ring = (ring + 1) % hist;
  }
}

__global__ void silu_mul_kernel(const float *g, const float *u, float *out, long long n) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) out[i] = silu_times(g[i], u[i]);
}

__global__ void rope_kernel(float *x, int head_dim, int rope_dim, const float *c, const float *s) {
  const int h = blockIdx.x, i = threadIdx.x, half = rope_dim / 2;
  if (i >= half) return;
  float *a = x + static_cast<size_t>(h) * head_dim;
  const float x0 = a[i], x1 = a[i + half];
  a[i] = x0 * c[i] - x1 * s[i];
  a[i + half] = x1 * c[i] + x0 * s[i];
}

__global__ void store_f16_kernel(const float *x, uint16_t *y, long long n) {
  const long long i = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float v = x[i];
  // NaN stores the quiet pattern like attention_float_to_half (full_attention.cpp:22-25)
  y[i] = isnan(v) ? static_cast<uint16_t>((__float_as_uint(v) >> 16 & 0x8000u) | 0x7e00u)
                  : float_to_half_bits(v);
}

}  // namespace

hipError_t launch_embed(const q35_q4_0_block_x8 *embed, int nb, const int32_t *tokens, int batch,
                        float *x, int hidden, int32_t *counts, long long counts_stride,
                        const int32_t *slots, const uint8_t *count_input, hipStream_t stream, bool g16) {
  if (batch <= 0) return hipSuccess;
  Q35_LAUNCH((embed_kernel), batch, 256, 0, stream, embed, nb, tokens, x, hidden, counts, counts_stride,
                                          slots, count_input, g16);
  return hipGetLastError();
}

hipError_t launch_rms_norm(const float *x, const float *w, float *y, int rows, int width,
                           float eps, float offset, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  Q35_LAUNCH((rms_norm_kernel), rows, 256, 0, stream, x, w, y, width, eps, offset);
  return hipGetLastError();
}

hipError_t launch_l2_normalize(float *x, int rows, int width, float eps, float scale,
                               hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  Q35_LAUNCH((l2_normalize_kernel), rows, 256, 0, stream, x, width, eps, scale);
  return hipGetLastError();
}

hipError_t launch_conv1d_silu(float *state, int ring, const float *input, long long stride, const float *w,
                              float *out, int batch, int channels, int kernel, int begin, int end, hipStream_t stream) {
  if (batch <= 0 || begin >= end) return hipSuccess;
  const uintptr_t in0 = reinterpret_cast<uintptr_t>(input), out0 = reinterpret_cast<uintptr_t>(out);
  const uintptr_t in1 = in0 + ((batch - 1) * stride + end) * sizeof(float);
  const uintptr_t out1 = out0 + (static_cast<size_t>(batch - 1) * channels + end) * sizeof(float);
  const bool overlap = in0 < out1 && out0 < in1;
  const int runs = (batch + kConvRun - 1) / kConvRun;
  if (overlap || kernel - 1 > kConvRun || runs > 65535 || (kernel != 4 && batch < kConvGeneralMin)) {
    Q35_LAUNCH((conv1d_silu_kernel), (end - begin + 255) / 256, 256, 0, stream, state, ring, input, stride, w, out,
               batch, channels, kernel, begin, end);
    return hipGetLastError();
  }
  // four channels per thread where every row is 16-byte aligned there
  const bool vec = ((in0 | out0 | reinterpret_cast<uintptr_t>(state) | reinterpret_cast<uintptr_t>(w)) & 15) == 0 &&
                   (stride & 3) == 0 && (channels & 3) == 0 && (begin & 3) == 0 && (end & 3) == 0;
  const int threads = ((end - begin) + (vec ? 3 : 0)) / (vec ? 4 : 1);
  // wavefront-sized workgroups spread a small launch over the compute units
  const int block = static_cast<long long>(threads) * runs < 256 * 512 ? 64 : 256;
  const dim3 grid((threads + block - 1) / block, runs);
#define Q35_CONV(V, K)                                                                                              \
  Q35_LAUNCH((conv1d_silu_runs_kernel<V, K>), grid, dim3(block), 0, stream, state, ring, input, stride, w, out, batch, \
             channels, kernel, begin, end)
  if (kernel == 4) {
    if (vec) Q35_CONV(4, 4); else Q35_CONV(1, 4);
  } else {
    if (vec) Q35_CONV(4, 0); else Q35_CONV(1, 0);
  }
#undef Q35_CONV
  return hipGetLastError();
}

hipError_t launch_silu_mul(const float *g, const float *u, float *out, long long n,
                           hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  Q35_LAUNCH((silu_mul_kernel), static_cast<unsigned>((n + 255) / 256), 256, 0, stream, g, u, out, n);
  return hipGetLastError();
}

hipError_t launch_rope(float *x, int heads, int head_dim, int rope_dim, const float *c,
                       const float *s, hipStream_t stream) {
  if (heads <= 0) return hipSuccess;
  Q35_LAUNCH((rope_kernel), heads, 256, 0, stream, x, head_dim, rope_dim, c, s);
  return hipGetLastError();
}

hipError_t launch_store_f16(const float *x, uint16_t *y, long long n, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  Q35_LAUNCH((store_f16_kernel), static_cast<unsigned>((n + 255) / 256), 256, 0, stream, x, y, n);
  return hipGetLastError();
}

}  // namespace q35

// Q4-G32-DOT4 GEMV for one to four vectors in a single launch: the
// activation blocks are read in their Q8_0 X1 / X4 layout (no layout kernel),
// the int8 block dots run on the VALU dot4 unit, and each output row is the
// reference's single fma chain over the blocks in order, so the results are
// bit-exact (no split-K, no reduce kernel).
#include <algorithm>

#include "q35_device.h"
#include "q35_internal.h"

namespace q35 {

namespace {
constexpr int kMvThreads = 256;
constexpr int kMvStep = 32;  // blocks per step of a workgroup: 4 wavefronts x 8

struct MvArgs {
  const uint8_t *w;    // Q4_0BlockX8 tiles [rows / 8][nb]
  const uint8_t *act;  // X1 blocks [count][nb] (40 B) or X4 blocks [nb] (152 B)
  int nb;
  int count;
  float *out;
  long long stride;  // output row stride (floats) between vectors
};

// One workgroup per 8-row tile group, STEPS steps of kMvStep blocks per pass.
// Lane (j, h, t) = (lane / 8, lane / 4 % 2, lane % 4) of wavefront w takes block
// j + 8w of a step: 16 bytes of its tile (the words of rows 4h .. 4h+3, columns
// 8t .. 8t+7), so a wavefront reads eight tiles whole, and the eight codes of
// those columns. Per vector it forms its part of the four rows' dots
//   sum_k (u_k - 8) a_k   (sdot4 of the nibbles against the codes, on top of
//                         -8 times their sum, all in int32);
// two exchanges over t leave lane (h, t) with the whole dot of row 4h + t. The
// dot and scale = half(d_r) * s_a (q4_dot4.cpp:52-54) land in LDS, and the
// first 8 * count lanes run the row chains
// result = fma(float(dot), scale, result) block by block (q4_dot4.cpp:43-56,
// restated by q35o_dot4_matvec) while the next pass's loads are in flight.
// Bound by latency: one round trip, the dots and the chain. With each lane
// loading one row's four words (4 bytes each) and all 32 codes, 18432 x 2560
// took 13.6 us a call and four X4 vectors 21.3, this form 6.8 and 10.7.
template <int NV, bool X4, int STEPS>
__global__ __launch_bounds__(kMvThreads) void dot4_matvec_kernel(MvArgs a) {
  constexpr int kPass = kMvStep * STEPS;
  __shared__ q35_f32x2 fs[NV][8][kPass + 1];  // +1: the chain lanes' reads hit distinct banks
  const int g = blockIdx.x;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int t = lane & 3, h = (lane >> 2) & 1, j = lane >> 3, r = 4 * h + t;
  const uint8_t *tiles = a.w + static_cast<size_t>(g) * a.nb * 144;
  float res = 0.0F;
  q35_u32x4 wq[STEPS];
  uint16_t dh[STEPS];
  uint32_t c[STEPS][NV][X4 ? 2 : 3];
  float sa[STEPS][NV];
  // every load of a pass (slots past it read its last block and are not stored)
  auto load = [&](int b0) {
    const int n = min(kPass, a.nb - b0);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int b = b0 + min(j + 8 * wave + kMvStep * i, n - 1);
      const uint8_t *tile = tiles + static_cast<size_t>(b) * 144;
      wq[i] = Q35_LOAD_NT(reinterpret_cast<const q35_u32x4 *>(tile + 16 + 32 * t + 16 * h));
      dh[i] = reinterpret_cast<const uint16_t *>(tile)[r];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        if constexpr (X4) {
          // scales[4], sums[4], qs[4][32]: vector v's codes at byte 24 + 32 v
          const uint8_t *blk = a.act + static_cast<size_t>(b) * 152;
          sa[i][v] = reinterpret_cast<const float *>(blk)[v];
          const q35_u32x2 x = *reinterpret_cast<const q35_u32x2 *>(blk + 24 + 32 * v + 8 * t);
          c[i][v][0] = x[0];
          c[i][v][1] = x[1];
        } else {
          // scale, sum, qs[32] from byte 6: the word before the eight codes, then two
          const uint8_t *blk = a.act + (static_cast<size_t>(v) * a.nb + b) * 40;
          sa[i][v] = *reinterpret_cast<const float *>(blk);
          const q35_u32x2 x = *reinterpret_cast<const q35_u32x2 *>(blk + 8 + 8 * t);
          c[i][v][0] = *reinterpret_cast<const uint32_t *>(blk + 4 + 8 * t);
          c[i][v][1] = x[0];
          c[i][v][2] = x[1];
        }
      }
    }
  };
  load(0);
  for (int b0 = 0; b0 < a.nb; b0 += kPass) {
    const int n = min(kPass, a.nb - b0);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int bl = j + 8 * wave + kMvStep * i;
      const float dw = half_bits_to_float(dh[i]);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        uint32_t lo = c[i][v][0], hi = c[i][v][1];
        if constexpr (!X4) {
          lo = (lo >> 16) | (hi << 16);
          hi = (hi >> 16) | (c[i][v][2] << 16);
        }
        const int corr = Q35_SDOT4(0xF8F8F8F8u, hi, Q35_SDOT4(0xF8F8F8F8u, lo, 0));
        int p[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          p[k] = Q35_SDOT4((wq[i][k] >> 4) & 0x0f0f0f0fu, hi, Q35_SDOT4(wq[i][k] & 0x0f0f0f0fu, lo, corr));
        // lane t keeps row 4h + t: the odd lanes of a pair take rows 1 and 3,
        // then the upper lanes of a pair of pairs rows 2 and 3
        const bool t0 = (t & 1) != 0, t1 = (t & 2) != 0;
        const int a0 = (t0 ? p[1] : p[0]) + q35_row_xor_i(t0 ? p[0] : p[1], 1);
        const int a1 = (t0 ? p[3] : p[2]) + q35_row_xor_i(t0 ? p[2] : p[3], 1);
        const int dot = (t1 ? a1 : a0) + q35_row_xor_i(t1 ? a0 : a1, 2);
        if (bl < n) fs[v][r][bl] = q35_f32x2{static_cast<float>(dot), dw * sa[i][v]};
      }
    }
    lds_barrier();
    if (b0 + kPass < a.nb) load(b0 + kPass);
    if (tid < 8 * NV) {
      const int rr = tid & 7, v = tid >> 3;
      int bl = 0;
      for (; bl + 8 <= n; bl += 8) {
        // eight reads, then their terms (without the fence the compiler reads
        // and waits for one pair at a time: 1024 x 4096 4.65 against 3.7 us)
        q35_f32x2 p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] = fs[v][rr][bl + e];
        q35_compiler_fence();
#pragma unroll
        for (int e = 0; e < 8; ++e) res = fmaf(p[e][0], p[e][1], res);
      }
      for (; bl < n; ++bl) {
        const q35_f32x2 p = fs[v][rr][bl];
        res = fmaf(p[0], p[1], res);
      }
    }
    lds_barrier();
  }
  if (tid < 8 * a.count) a.out[(tid >> 3) * a.stride + g * 8 + (tid & 7)] = res;
}
}  // namespace

hipError_t launch_dot4_matvec(const q35_q4_0_block_x8 *w, const void *act, bool x4, int count, int rows, int nb,
                              float *out, long long stride, hipStream_t stream) {
  if (count < 1 || count > kMatvecMaxVectors || (x4 && count != 4) || rows <= 0 || rows % 8 != 0 || nb <= 0)
    return hipErrorInvalidValue;
  MvArgs a;
  a.w = reinterpret_cast<const uint8_t *>(w);
  a.act = static_cast<const uint8_t *>(act);
  a.nb = nb;
  a.count = count;
  a.out = out;
  a.stride = stride;
  const dim3 grid(rows / 8), block(kMvThreads);
  // As many steps per pass as the row has blocks, up to four. Longer rows are
  // passes of four: one pass of nine steps for one vector has 140 registers
  // and repeats its last block where the row is shorter (18432 rows: 160 blocks
  // 17.2 against 13.5 us, 288 blocks 23.1 against 22.6, 320 blocks 32.5 against
  // 24.2; it is ahead only for 257 to 288 blocks of few rows, 1024: 6.3 against 6.6).
#define Q35_MV(NV, X)                                                                                          \
  switch (std::min(4, (nb + kMvStep - 1) / kMvStep)) {                                                         \
    case 1: Q35_LAUNCH((dot4_matvec_kernel<NV, X, 1>), grid, block, 0, stream, a); break;                      \
    case 2: Q35_LAUNCH((dot4_matvec_kernel<NV, X, 2>), grid, block, 0, stream, a); break;                      \
    case 3: Q35_LAUNCH((dot4_matvec_kernel<NV, X, 3>), grid, block, 0, stream, a); break;                      \
    default: Q35_LAUNCH((dot4_matvec_kernel<NV, X, 4>), grid, block, 0, stream, a); break;                     \
  }
  if (x4) {
    Q35_MV(4, true)
  } else {
    switch (count) {
      case 1: Q35_MV(1, false) break;
      case 2: Q35_MV(2, false) break;
      case 3: Q35_MV(3, false) break;
      default: Q35_MV(4, false) break;
    }
  }
#undef Q35_MV
  return hipGetLastError();
}

}  // namespace q35

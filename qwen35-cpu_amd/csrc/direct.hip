// Q4-G32-DOT4 GEMM over X4 / X1 activations in one launch, for batches that do
// not fill the GPU with the dense GEMM's tiles: the activations are read in
// place (no layout kernel) and a workgroup owns all K splits of its rows (no
// partial rows in memory, no reduce kernel).
//
// One workgroup per (16 rows, 16·NT tokens), a wavefront per K split (two
// where there are more than 16). The splits, the chains within them and the
// order in which they are added are gemm_plan's, so every output has the bits
// of the split launches and of the dense GEMM.
//
// The weights are the A operand here and the activations the B operand of
// v_mfma_i32_16x16x32_i8: lane l = (G = l/16, c = l%16) supplies row c's body
// word of k-group G (columns 8G .. 8G+7) and token c's codes of the same
// columns, and receives the block dots of rows 4G .. 4G+3 with token c. So a
// lane needs one activation scale, which sits beside its codes in either
// layout, and its four row scales are eight contiguous bytes of a tile.
//
// These launches are bound by latency. KS blocks are unrolled together; how
// many of their loads are in flight is the compiler's choice (one tile keeps
// within 42 registers, about half a chunk of eight), and forcing all of them
// cost more in occupancy than it gave. Per call, against layout + split GEMM +
// reduce: 3584 x 1024, 16 vectors 11.6 -> 4.2 us; 8224 x 1024, 7 vectors 11.6 ->
// 6.2 us; 4096 x 2560, 64 vectors 18.7 -> 8.1 us.
#include <algorithm>

#include "q35_device.h"
#include "q35_internal.h"

namespace q35 {
namespace {

typedef Q35_V4I v4i;

struct DirectArgs {
  const uint8_t *w;    // Q4_0BlockX8 tiles [rows / 8][nb]
  const uint8_t *act;  // X4 blocks [tokens / 4][nb] (152 B) or X1 blocks [tokens][nb] (40 B)
  int rows, nb, tokens, splits;
  float *out;
  long long stride;
  bool vec_out;  // rows of `out` start on 16-byte boundaries
};

// The codes of a lane's k-group of one block, and its token's scale.
template <bool X4>
struct Act {
  uint32_t c[X4 ? 2 : 3];
  float s;
};

template <bool X4, int NT, int KS>
__global__ __launch_bounds__(1024) void gemm_direct_kernel(DirectArgs a) {
  Q35_DYNAMIC_SHARED(q35_f32x4, part);  // [split][NT][token][4]: rows 4i .. 4i+3 of a token
  const int waves = static_cast<int>(blockDim.x) >> 6;
  const int wave = q35_uniform(static_cast<int>(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int G = lane >> 4, c = lane & 15;
  const int nb = a.nb, ntiles = a.rows >> 3, S = a.splits;
  const int row0 = static_cast<int>(blockIdx.x) * 16, tok0 = static_cast<int>(blockIdx.y) * 16 * NT;
  // rows past the matrix read its last tile, tokens past the batch its last
  // token; neither is stored
  const int rt = row0 >> 3;
  const uint8_t *wp = a.w + static_cast<size_t>(min(rt + (c >> 3), ntiles - 1)) * nb * 144 + 16 + 32 * G + 4 * (c & 7);
  const uint8_t *dp = a.w + static_cast<size_t>(min(rt + (G >> 1), ntiles - 1)) * nb * 144 + 8 * (G & 1);
  const uint8_t *ap[NT];
  constexpr int kBlock = X4 ? 152 : 40;
  int code_off = 0, scale_off = 0;  // of the token within its block
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int tok = min(tok0 + 16 * t + c, a.tokens - 1);
    if (X4) {
      ap[t] = a.act + static_cast<size_t>(tok >> 2) * nb * kBlock;
      // tokens % 4 == 0: a clamped lane's last token has another place in its
      // group of four, whose values it may read as well
      code_off = 24 + 32 * (c & 3) + 8 * G;
      scale_off = 4 * (c & 3);
    } else {
      ap[t] = a.act + static_cast<size_t>(tok) * nb * kBlock;
      code_off = 4 + 8 * G;  // codes 8G .. 8G+7 start at byte 6 + 8G: the word before them, then two
    }
  }
  const v4i zero = {0, 0, 0, 0};
  for (int s = wave; s < S; s += waves) {
    const int b0 = (s * nb) / S, b1 = ((s + 1) * nb) / S;
    q35_f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = q35_f32x4{0.0F, 0.0F, 0.0F, 0.0F};
    for (int cb = b0; cb < b1; cb += KS) {
      uint32_t w[KS];
      q35_u32x2 d[KS];
      Act<X4> x[KS][NT];
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const size_t b = static_cast<size_t>(min(cb + i, b1 - 1));
        w[i] = *reinterpret_cast<const uint32_t *>(wp + b * 144);
        d[i] = *reinterpret_cast<const q35_u32x2 *>(dp + b * 144);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const uint8_t *p = ap[t] + b * kBlock;
          if constexpr (X4) {
            const q35_u32x2 q = *reinterpret_cast<const q35_u32x2 *>(p + code_off);
            x[i][t].c[0] = q[0];
            x[i][t].c[1] = q[1];
          } else {
            const q35_u32x2 q = *reinterpret_cast<const q35_u32x2 *>(p + code_off + 4);
            x[i][t].c[0] = *reinterpret_cast<const uint32_t *>(p + code_off);
            x[i][t].c[1] = q[0];
            x[i][t].c[2] = q[1];
          }
          x[i][t].s = *reinterpret_cast<const float *>(p + scale_off);
        }
      }
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        if (cb + i >= b1) break;  // uniform
        const long wq = unpack_word(w[i]);
        float dw[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) dw[j] = half_bits_to_float(static_cast<uint16_t>(d[i][j >> 1] >> (16 * (j & 1))));
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          uint32_t lo = x[i][t].c[0], hi = x[i][t].c[1];
          if constexpr (!X4) {
            lo = (lo >> 16) | (hi << 16);
            hi = (hi >> 16) | (x[i][t].c[2] << 16);
          }
          const long codes = static_cast<long>((static_cast<uint64_t>(hi) << 32) | lo);
          const v4i corr = Q35_MFMA_I32_16X16X32_I8(kMinus8, codes, zero, 0, 0, 0);
          const v4i D = Q35_MFMA_I32_16X16X32_I8(wq, codes, corr, 0, 0, 0);
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[t][j] = fmaf(static_cast<float>(D[j]), dw[j] * x[i][t].s, acc[t][j]);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) part[((s * NT + t) * 16 + c) * 4 + G] = acc[t];
  }
  __syncthreads();
  // the splits of four rows of a token added in split order
  constexpr int kItems = NT * 16 * 4;
  for (int e = threadIdx.x; e < kItems; e += blockDim.x) {
    const int tok = tok0 + (e >> 2), row = row0 + 4 * (e & 3);
    if (tok >= a.tokens || row >= a.rows) continue;
    q35_f32x4 v = part[e];
    for (int s = 1; s < S; ++s) v += part[s * kItems + e];
    store_row4(a.out + tok * a.stride + row, a.vec_out, v[0], v[1], v[2], v[3]);
  }
}

}  // namespace

// LDS bytes of a workgroup's split sums (at most 32 splits); launches keep
// within one 64 KiB window.
constexpr size_t kDirectMaxLds = 64 * 1024;
static size_t direct_lds(int splits, int nt) { return static_cast<size_t>(splits) * nt * 1024; }

struct DirectShape {
  int splits, nt, groups, tiles;  // token tiles per workgroup; workgroups over rows and tokens
};
static DirectShape direct_shape(int rows, int nb, int tokens, int cus) {
  DirectShape d;
  d.splits = gemm_dense_splits(rows, nb, cus, 0);
  d.groups = (rows + 15) / 16;
  // token tiles per workgroup: as few as keep the launch within 14 wavefronts
  // per compute unit, where a workgroup's own latency sets the time (1024 x
  // 3584, 64 vectors: 5.4 us with one tile, 10.2 with four); beyond that more
  // tiles share each weight load and unpack (18432 x 2560, 64 vectors: 44.0 us
  // with one tile, 32.1 with four)
  const int waves = std::min(d.splits, 16);
  d.nt = 1;
  while (d.nt < 4 && 16 * d.nt < tokens &&
         static_cast<long long>(d.groups) * ((tokens + 16 * d.nt - 1) / (16 * d.nt)) * waves > 14LL * cus)
    d.nt <<= 1;
  while (d.nt > 1 && direct_lds(d.splits, d.nt) > kDirectMaxLds) d.nt >>= 1;
  d.tiles = (tokens + 16 * d.nt - 1) / (16 * d.nt);
  return d;
}

// The lines between this kernel, the split launches (up to 64 vectors) and the
// dense GEMM (more), measured over 8 to 65536 rows and 8 to 512 blocks. Counted
// in `per_cu`, the token rows that the busiest compute unit takes in all, and
// the blocks of each.
//
// X4, up to 64 vectors: direct, 1.1 to 2.8 times as fast (18432 x 2560: 20
// vectors 18.9 against 20.8 us, 64 vectors 32.2 against 38.4), except for work
// above 20480 blocks per unit where
//   - 33 to 48 vectors leave a quarter or more of four-tile workgroups empty
//     (8224 x 128 blocks, 40 vectors: 27.5 against 24.2 us; 18432 x 160: 57.3
//     against 52.3; below, 8224 x 96: 19.6 against 20.6). From 257 to 288 blocks
//     the split launch's 32 partial rows cost as much (18432 x 288: 96.9
//     against 105.3);
//   - more than 352 blocks meet the two tiles that 32 splits leave room for
//     (8224 x 512, 20 vectors: 57.3 against 44.9; 8224 x 352: 40.3 against 42.3).
// X4, more vectors: direct where the dense tiles would leave compute units idle
// (4096 x 80 blocks, 200 vectors: 24.6 against 29.0 us), up to 256 token rows
// per unit, beyond for at most 64 blocks (320 rows: 8224 x 64, 96 vectors 22.9
// against 24.1, 8224 x 112 42.6 against 38.4).
// X1: a token's blocks lie 40 bytes apart in rows of their own, so a lane's
// loads share no cache line with its neighbours' and each block of a token
// costs a compute unit about 3.8 ns. Up to 64 vectors that has to stay below
// the two launches saved: 2000 blocks per unit, a workgroup counted as 64 more
// (8224 x 32 blocks, 7 vectors, 864: 6.3 against 11.2 us; 8224 x 64, 8 vectors,
// 1728: 10.9 against 11.6; 18432 x 80, 5 vectors, 2320: 19.4 against 16.0; 32768
// x 80, 64 vectors: 168 against 62). More vectors, against the dense GEMM's walk
// of all blocks in one wavefront: 80 token rows per unit (1024 x 80 blocks, 67
// vectors, 32 rows: 9.9 against 28.4; 2560 x 80, 96 vectors, 128 rows: 32.0
// against 28.5).
bool gemm_direct_fits(int rows, int nb, size_t tokens, int cu_count, bool x4) {
  if (tokens == 0 || tokens > size_t{65535} * 16) return false;  // grid.y
  const int n = static_cast<int>(tokens), cus = cu_count > 0 ? cu_count : 256;
  const bool few = n <= kMaxTokens;
  if (!few && gemm_dense_fits(rows, n, cus)) return false;
  const DirectShape d = direct_shape(rows, nb, n, cus);
  const long long rounds = (static_cast<long long>(d.groups) * d.tiles + cus - 1) / cus;
  if (x4) {
    const long long per_cu = rounds * 16 * d.nt;
    if (!few) return per_cu <= 256 || nb <= 64;
    const bool padded = n > 32 && n <= 48;
    return per_cu * nb <= 20480 || n <= 16 || (padded ? nb > 256 && nb <= 288 : nb <= 352);
  }
  const long long per_wg = std::min(16 * d.nt, n);
  return few ? rounds * (per_wg * nb + 64) <= 2000 : rounds * per_wg <= 80;
}

hipError_t launch_gemm_direct(const q35_q4_0_block_x8 *w, const void *act, bool x4, int rows, int nb, int tokens,
                              float *out, long long stride, int cu_count, hipStream_t stream) {
  if (!gemm_direct_fits(rows, nb, tokens, cu_count, x4) || (x4 && tokens % 4 != 0) || stride < rows)
    return hipErrorInvalidValue;
  const DirectShape d = direct_shape(rows, nb, tokens, cu_count > 0 ? cu_count : 256);
  DirectArgs a;
  a.w = reinterpret_cast<const uint8_t *>(w);
  a.act = static_cast<const uint8_t *>(act);
  a.rows = rows;
  a.nb = nb;
  a.tokens = tokens;
  a.splits = d.splits;
  a.out = out;
  a.stride = stride;
  a.vec_out = stride % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  const int nt = d.nt;
  const dim3 grid(d.groups, d.tiles), block(64 * std::min(d.splits, 16));
  const size_t lds = direct_lds(d.splits, nt);
#define Q35_DIRECT(NT, KS)                                                                             \
  if (x4)                                                                                              \
    Q35_LAUNCH((gemm_direct_kernel<true, NT, KS>), grid, block, lds, stream, a);                    \
  else                                                                                                 \
    Q35_LAUNCH((gemm_direct_kernel<false, NT, KS>), grid, block, lds, stream, a);
  if (nt == 1) {
    Q35_DIRECT(1, 8)
  } else if (nt == 2) {
    Q35_DIRECT(2, 8)
  } else {
    Q35_DIRECT(4, 4)
  }
#undef Q35_DIRECT
  return hipGetLastError();
}

}  // namespace q35

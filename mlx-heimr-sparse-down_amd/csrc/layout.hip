// The neuron-major permutation of the 4-bit down projections, on the device.
//
// hsd/layout.py:34-50 expands every nibble to a uint32, swaps axes and repacks (an 8x
// transient, done 16 experts at a time). Here a permutation is a pure 8x8 nibble-block
// transpose: the 8 words w[8*wo + n, cw] (n = 0..7) hold exactly the nibbles that the 8
// words out[8*cw + j, wo] (j = 0..7) hold, transposed. One thread transposes such a
// block in registers with three block-swap stages (4x4, 2x2, 1x1 nibble blocks); a
// workgroup stages a 32x32 tile of blocks through LDS so that both the reads (rows of
// the input) and the writes (rows of the output) are 128-byte coalesced. No transient
// memory at all; out-of-place; self-inverse.
#include "hsd_common.h"

namespace hsd {

namespace {

constexpr int kTile = 32;      // blocks per tile side: 32 input words x 32 output words
constexpr int kThreads = 256;

// In-register transpose of the 8x8 nibble matrix M[n][j] = nibble j of v[n].
__device__ __forceinline__ void transpose8x8_nibbles(uint32_t v[8]) {
#pragma unroll
  for (int n = 0; n < 4; ++n) {  // swap the off-diagonal 4x4 blocks
    const uint32_t a = v[n], b = v[n + 4];
    v[n] = (a & 0x0000FFFFu) | (b << 16);
    v[n + 4] = (a >> 16) | (b & 0xFFFF0000u);
  }
#pragma unroll
  for (int base = 0; base < 8; base += 4) {  // 2x2 blocks inside each 4x4 half
#pragma unroll
    for (int n = base; n < base + 2; ++n) {
      const uint32_t a = v[n], b = v[n + 2];
      v[n] = (a & 0x00FF00FFu) | ((b << 8) & 0xFF00FF00u);
      v[n + 2] = ((a >> 8) & 0x00FF00FFu) | (b & 0xFF00FF00u);
    }
  }
#pragma unroll
  for (int n = 0; n < 8; n += 2) {  // single nibbles inside each 2x2
    const uint32_t a = v[n], b = v[n + 1];
    v[n] = (a & 0x0F0F0F0Fu) | ((b << 4) & 0xF0F0F0F0u);
    v[n + 1] = ((a >> 4) & 0x0F0F0F0Fu) | (b & 0xF0F0F0F0u);
  }
}

// Tile (cw0, wo0) of w [R, CW] -> out [8*CW, R/8]. Every load of the tile is issued before the
// first is used (positions past the edges re-read the last one: a load under a branch would
// end in a wait per iteration).
__device__ __forceinline__ void permute_tile(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, int64_t R,
                                             int64_t CW, int64_t cw0, int64_t wo0, uint32_t* tileT, int tid) {
  const int64_t RW = R / 8;
  constexpr int kIt = (kTile * kTile) / kThreads;
  uint32_t v[kIt][8];
  const int cw_l = tid & (kTile - 1);
  const int64_t cw = min(cw0 + cw_l, CW - 1);
#pragma unroll
  for (int i = 0; i < kIt; ++i) {
    const int64_t wo = min(wo0 + (tid + kThreads * i) / kTile, RW - 1);
#pragma unroll
    for (int n = 0; n < 8; ++n) v[i][n] = src[(8 * wo + n) * CW + cw];
  }
#pragma unroll
  for (int i = 0; i < kIt; ++i) {
    const int wo_l = (tid + kThreads * i) / kTile;
    transpose8x8_nibbles(v[i]);
#pragma unroll
    for (int j = 0; j < 8; ++j) tileT[(8 * cw_l + j) * kTile + (wo_l ^ cw_l)] = v[i][j];
  }
  __syncthreads();
  const int wo_l = tid & (kTile - 1);
#pragma unroll 4
  for (int row = tid / kTile; row < 8 * kTile; row += kThreads / kTile) {
    const int cl = row >> 3;
    const int64_t orow = 8 * cw0 + row, wo = wo0 + wo_l;
    if (cw0 + cl < CW && wo < RW) dst[orow * RW + wo] = tileT[row * kTile + (wo_l ^ cl)];
  }
}

// w [batch, R, CW] -> out [batch, 8*CW, R/8]
__global__ __launch_bounds__(kThreads) void k_permute_nibbles(const uint32_t* __restrict__ w,
                                                              uint32_t* __restrict__ out,
                                                              int64_t R, int64_t CW,
                                                              int tiles_cw) {
  __shared__ uint32_t tileT[8 * kTile * kTile];  // [8*cw_l + j][wo_l ^ cw_l]
  const int64_t b = blockIdx.y;
  permute_tile(w + b * R * CW, out + b * R * CW, R, CW, (int64_t)(blockIdx.x % tiles_cw) * kTile,
               (int64_t)(blockIdx.x / tiles_cw) * kTile, tileT, (int)threadIdx.x);
}

constexpr int kT16 = 64;
// in [batch, R, C] -> out [batch, C, R], 16-bit elements.
__global__ __launch_bounds__(kThreads) void k_transpose_u16(const uint16_t* __restrict__ in,
                                                            uint16_t* __restrict__ out, int64_t R,
                                                            int64_t C, int tiles_c) {
  __shared__ uint32_t tile[kT16][kT16 + 1];
  const int tid = threadIdx.x;
  const int64_t b = blockIdx.y;
  const int64_t c0 = (int64_t)(blockIdx.x % tiles_c) * kT16;
  const int64_t r0 = (int64_t)(blockIdx.x / tiles_c) * kT16;
  const uint16_t* src = in + b * R * C;
  uint16_t* dst = out + b * R * C;
  const int lc = tid & (kT16 - 1);
  for (int lr = tid / kT16; lr < kT16; lr += kThreads / kT16) {
    const int64_t r = r0 + lr, c = c0 + lc;
    if (r < R && c < C) tile[lr][lc] = src[r * C + c];
  }
  __syncthreads();
  for (int lr = tid / kT16; lr < kT16; lr += kThreads / kT16) {
    const int64_t c = c0 + lr, r = r0 + lc;  // output row c, column r
    if (r < R && c < C) dst[c * R + r] = (uint16_t)tile[lc][lr];
  }
}

// A whole weight in one launch: the nibble tiles of every matrix, then kTR-row pieces of its
// scales and its biases [batch, R, G] -> [batch, G, R] with G <= 64. A piece's kTR rows are
// contiguous (16-byte loads) and its columns become G runs of 2 kTR bytes: 128 experts' scales
// 35 -> 12 us against 64 x 64 tiles of which G = 29 columns fill less than half. Consecutive
// nibble tiles run on one XCD, whose L2 joins the tiles' shares of a 128-byte line (rows of
// 928 and 1344 bytes are not multiples of it).
constexpr int kTR = 128;
constexpr int kGMaxT = 64;
__global__ __launch_bounds__(kThreads) void k_neuron_major(
    const uint32_t* __restrict__ w, const uint16_t* __restrict__ s, const uint16_t* __restrict__ b,
    uint32_t* __restrict__ pw, uint16_t* __restrict__ ps, uint16_t* __restrict__ pb, int64_t R, int64_t CW, int G,
    int tiles_cw, int tiles, int nperm, int pieces) {
  __shared__ __attribute__((aligned(16))) uint32_t lds[8 * kTile * kTile];
  static_assert(sizeof(uint32_t) * 8 * kTile * kTile >= sizeof(uint16_t) * kGMaxT * (kTR + 2), "the piece fits the tile");
  const int tid = threadIdx.x;
  if ((int)blockIdx.x < nperm) {
    const int id = xcd_remap((int)blockIdx.x, nperm), m = id / tiles, t = id - m * tiles;
    permute_tile(w + (int64_t)m * R * CW, pw + (int64_t)m * R * CW, R, CW, (int64_t)(t % tiles_cw) * kTile,
                 (int64_t)(t / tiles_cw) * kTile, lds, tid);
    return;
  }
  const int id = (int)blockIdx.x - nperm, half = (int)(gridDim.x - nperm) / 2;
  const bool bias = id >= half;
  const int u = bias ? id - half : id, m = u / pieces;
  const int64_t r0 = (int64_t)(u - m * pieces) * kTR;
  const int rows = (int)min((int64_t)kTR, R - r0);
  const uint16_t* src = (bias ? b : s) + ((int64_t)m * R + r0) * G;
  uint16_t* dst = (bias ? pb : ps) + (int64_t)m * R * G;
  uint16_t* tile = reinterpret_cast<uint16_t*>(lds);   // [G][kTR + 2]
  const int nv = rows * G / 8;                         // R and so rows are multiples of 8
  for (int i = tid; i < nv; i += kThreads) {
    const uint4 v = reinterpret_cast<const uint4*>(src)[i];
    const uint32_t x[4] = {v.x, v.y, v.z, v.w};
    int r = 8 * i / G, c = 8 * i - r * G;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      tile[c * (kTR + 2) + r] = (uint16_t)((k & 1) ? x[k >> 1] >> 16 : x[k >> 1]);
      if (++c == G) {
        c = 0;
        ++r;
      }
    }
  }
  __syncthreads();
  for (int i = tid; i < G * (kTR / 2); i += kThreads) {
    const int c = i / (kTR / 2), r = 2 * (i - c * (kTR / 2));
    if (r < rows)
      *reinterpret_cast<uint32_t*>(dst + (int64_t)c * R + r0 + r) = *reinterpret_cast<const uint32_t*>(&tile[c * (kTR + 2) + r]);
  }
}

}  // namespace
}  // namespace hsd

using namespace hsd;

extern "C" int hsd_permute_nibbles(const uint32_t* w, uint32_t* out, int64_t batch, int64_t rows,
                                   int64_t words, void* stream) {
  if (!w || !out) return set_error(HSD_ERR_ARG, "hsd_permute_nibbles: null pointer");
  if (batch < 0 || rows < 0 || words < 0 || rows % 8)
    return set_error(HSD_ERR_SHAPE, "hsd_permute_nibbles: rows (%lld) must be a multiple of 8",
                     (long long)rows);
  if (batch > 65535) return set_error(HSD_ERR_SHAPE, "hsd_permute_nibbles: batch > 65535");
  if (batch == 0 || rows == 0 || words == 0) return HSD_OK;
  const int64_t tcw = (words + kTile - 1) / kTile, two = (rows / 8 + kTile - 1) / kTile;
  if (tcw * two > 0x7FFFFFFF) return set_error(HSD_ERR_SHAPE, "hsd_permute_nibbles: too large");
  dim3 grid((unsigned)(tcw * two), (unsigned)batch);
  hipLaunchKernelGGL(k_permute_nibbles, grid, dim3(kThreads), 0, as_stream(stream), w, out, rows,
                     words, (int)tcw);
  return check_launch("hsd_permute_nibbles");
}

extern "C" int hsd_transpose_u16(const uint16_t* in, uint16_t* out, int64_t batch, int64_t rows,
                                 int64_t cols, void* stream) {
  if (!in || !out) return set_error(HSD_ERR_ARG, "hsd_transpose_u16: null pointer");
  if (batch < 0 || rows < 0 || cols < 0) return set_error(HSD_ERR_SHAPE, "hsd_transpose_u16: negative size");
  if (batch > 65535) return set_error(HSD_ERR_SHAPE, "hsd_transpose_u16: batch > 65535");
  if (batch == 0 || rows == 0 || cols == 0) return HSD_OK;
  const int64_t tc = (cols + kT16 - 1) / kT16, tr = (rows + kT16 - 1) / kT16;
  if (tc * tr > 0x7FFFFFFF) return set_error(HSD_ERR_SHAPE, "hsd_transpose_u16: too large");
  dim3 grid((unsigned)(tc * tr), (unsigned)batch);
  hipLaunchKernelGGL(k_transpose_u16, grid, dim3(kThreads), 0, as_stream(stream), in, out, rows,
                     cols, (int)tc);
  return check_launch("hsd_transpose_u16");
}

extern "C" int hsd_neuron_major(const uint32_t* w, const uint16_t* s, const uint16_t* b, uint32_t* pw, uint16_t* ps,
                                uint16_t* pb, int64_t batch, int64_t rows, int64_t words, int64_t groups, void* stream) {
  const char* fn = "hsd_neuron_major";
  if (!w || !s || !b || !pw || !ps || !pb) return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  if (batch < 0 || rows < 0 || rows % 8 || words < 0 || groups < 1 || groups > kGMaxT || batch > 65535)
    return set_error(HSD_ERR_SHAPE, "%s: need rows %% 8 == 0 and 1 <= groups <= %d", fn, kGMaxT);
  if (((uintptr_t)s | (uintptr_t)b) & 15u || ((uintptr_t)ps | (uintptr_t)pb) & 3u)
    return set_error(HSD_ERR_ALIGN, "%s: scales and biases must be 16-byte aligned", fn);
  if (batch == 0 || rows == 0 || words == 0) return HSD_OK;
  const int64_t tcw = (words + kTile - 1) / kTile, tiles = tcw * ((rows / 8 + kTile - 1) / kTile);
  const int64_t pieces = (rows + kTR - 1) / kTR, grid = batch * (tiles + 2 * pieces);
  if (grid > 0x7FFFFFFF || rows * groups > 0x7FFFFFFF) return set_error(HSD_ERR_SHAPE, "%s: too large", fn);
  hipLaunchKernelGGL(k_neuron_major, dim3((unsigned)grid), dim3(kThreads), 0, as_stream(stream), w, s, b, pw, ps, pb, rows,
                     words, (int)groups, (int)tcw, (int)tiles, (int)(batch * tiles), (int)pieces);
  return check_launch(fn);
}

// The projections of a prompt chunk: many token rows at once on the matrix cores.
//
//   k_rows_prep   one workgroup per token row: the input (bf16 rows, with the RMS norm, or
//                 the Mamba-2 gated norm of the SSM kernel's z) normalised and rounded as
//                 hsd_linear's prologue does it (the same instruction sequence, so the same
//                 bits), stored with every 8 inputs in the order of a weight word's nibble
//                 pairs (0 4 1 5 2 6 3 7), and the sum of every 64-input group as three bf16
//                 values (all 24 bits of the fp32 sum).
//   k_gemm_q4     y = x W^T, W affine 4-bit group 64 in the stock layout [O, I/8], and, with
//                 tiles of (token, slot) pairs sorted by expert, every expert's up projection
//                 with ReLU^2 (a grouped product over gathered rows).
//   k_gemm_bf16   y = x W^T with a bf16 weight (the router gate, the MTP head's eh_proj).
#include "hsd_common.h"

#include "gemm.h"

namespace hsd {
namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

constexpr uint32_t kBfOne2 = 0x3F803F80u;   // bf16 pair (1, 1)
constexpr uint32_t kBf16Two = 0x41804180u;  // bf16 pair (16, 16): | nibble << 3 is 16 + q
constexpr uint32_t kNibHi = 0x00780078u;

__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  const __bf16 a = (__bf16)lo, b = (__bf16)hi;
  return (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
}
__device__ __forceinline__ float lo_f(uint32_t v) { return __uint_as_float(v << 16); }
__device__ __forceinline__ float hi_f(uint32_t v) { return __uint_as_float(v & 0xFFFF0000u); }

// Offsets past any buffer of the epilogues (the host bounds those to 1 GiB), also added up
constexpr uint32_t kNoRow = 0x80000000u, kNoCol = 0x40000000u;

// -16 times both values of a bf16 pair (exact: a power of two)
__device__ __forceinline__ uint32_t neg16(uint32_t v) {
  return __builtin_amdgcn_perm(__float_as_uint(hi_f(v) * -16.0f), __float_as_uint(lo_f(v) * -16.0f), 0x07060302u);
}

// 16 bytes at a multiple of 4
struct __attribute__((packed, aligned(4))) Piece {
  u32x4 v;
};

// v as the sum of three bf16 values: all 24 bits
__device__ __forceinline__ void split3(float v, uint16_t (&p)[3]) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    p[k] = f32_to_bf16_bits(v);
    v -= bf16_bits_to_f32(p[k]);
  }
}

// ------------------------------------------------------------------ rows
constexpr int kPT = 256;   // threads per row
constexpr int kPI = 3;     // 8-input words per thread (I <= 6144)

// KIND: HSD_X_BF16 (as they are), HSD_X_RMS, HSD_X_GATED_Z. PERM: 4-bit weights' order (and
// the group sums); else the natural order. Bound by its reads and writes (a chunk of 2048
// rows of 2688: 11 MB in, 11 MB out).
template <int KIND, bool PERM>
__global__ __launch_bounds__(kPT) void k_rows_prep(const void* __restrict__ x_, int64_t x_ld,
                                                   const uint16_t* __restrict__ nw, float eps,
                                                   uint16_t* __restrict__ xp, uint16_t* __restrict__ hs, int I,
                                                   int GP) {
  __shared__ float wsum[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, NW = I / 8;
  const size_t row = blockIdx.x;
  uint32_t xo[kPI][4];
  if constexpr (KIND == HSD_X_GATED_Z) {
    const float* xr = reinterpret_cast<const float*>(x_) + row * x_ld;
    float4 y0[kPI], y1[kPI];
    float zp[kPI];
    uint4 nv[kPI];
#pragma unroll
    for (int i = 0; i < kPI; ++i) {
      const int tc = min(tid + kPT * i, NW - 1);
      y0[i] = reinterpret_cast<const float4*>(xr)[2 * tc];
      y1[i] = reinterpret_cast<const float4*>(xr)[2 * tc + 1];
      zp[i] = xr[I + 32 * (tc >> 6) + (tid & 31)];
      nv[i] = reinterpret_cast<const uint4*>(nw)[tc];
    }
#pragma unroll
    for (int i = 0; i < kPI; ++i) {
      float g = zp[i];
      g += dpp_f32<0xB1>(g);
      g += dpp_f32<0x4E>(g);
      g += dpp_f32<0x141>(g);
      g += dpp_f32<0x140>(g);
      const uint32_t gb = __float_as_uint(g);
      const auto pg = __builtin_amdgcn_permlane16_swap(gb, gb, false, false);
      g = __uint_as_float(pg[0]) + __uint_as_float(pg[1]);
      const float inv = __builtin_amdgcn_rsqf(g / 512.0f + eps);
      const float z[8] = {y0[i].x, y0[i].y, y0[i].z, y0[i].w, y1[i].x, y1[i].y, y1[i].z, y1[i].w};
      const uint32_t n4[4] = {nv[i].x, nv[i].y, nv[i].z, nv[i].w};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint32_t t = pack_bf16x2(z[2 * c] * inv, z[2 * c + 1] * inv);
        xo[i][c] = pack_bf16x2(lo_f(t) * lo_f(n4[c]), hi_f(t) * hi_f(n4[c]));
      }
    }
  } else {
    const uint4* xr = reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(x_) + row * x_ld);
#pragma unroll
    for (int i = 0; i < kPI; ++i) {
      const uint4 v = xr[min(tid + kPT * i, NW - 1)];
      xo[i][0] = v.x; xo[i][1] = v.y; xo[i][2] = v.z; xo[i][3] = v.w;
    }
    if constexpr (KIND == HSD_X_RMS) {
      uint4 nv[kPI];
#pragma unroll
      for (int i = 0; i < kPI; ++i) nv[i] = reinterpret_cast<const uint4*>(nw)[min(tid + kPT * i, NW - 1)];
      float ss = 0.0f;
#pragma unroll
      for (int i = 0; i < kPI; ++i) {
        const bool tv = tid + kPT * i < NW;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint32_t v = tv ? xo[i][c] : 0u;
          ss = dot2_bf16(v, v, ss);
        }
      }
      ss = wave_sum_dpp(ss);
      if (lane == 0) wsum[wave] = ss;
      lds_barrier();
      const float tot = ((wsum[0] + wsum[1]) + wsum[2]) + wsum[3];
      const float inv = __builtin_amdgcn_rsqf(tot / (float)I + eps);
#pragma unroll
      for (int i = 0; i < kPI; ++i) {
        const uint32_t n4[4] = {nv[i].x, nv[i].y, nv[i].z, nv[i].w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint32_t t = pack_bf16x2(lo_f(xo[i][c]) * inv, hi_f(xo[i][c]) * inv);
          xo[i][c] = pack_bf16x2(lo_f(t) * lo_f(n4[c]), hi_f(t) * hi_f(n4[c]));
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kPI; ++i) {
    const int t = tid + kPT * i;
    const uint32_t* w = xo[i];
    if (t < NW) {
      uint4 o;
      if constexpr (PERM)
        o = make_uint4((w[0] & 0xFFFFu) | (w[2] << 16), (w[0] >> 16) | (w[2] & 0xFFFF0000u),
                       (w[1] & 0xFFFFu) | (w[3] << 16), (w[1] >> 16) | (w[3] & 0xFFFF0000u));
      else
        o = make_uint4(w[0], w[1], w[2], w[3]);
      reinterpret_cast<uint4*>(xp + row * I)[t] = o;
    }
    if constexpr (PERM) {
      float s8 = 0.0f;
#pragma unroll
      for (int c = 0; c < 4; ++c) s8 = dot2_bf16(w[c], kBfOne2, s8);
      s8 += dpp_f32<0xB1>(s8);   // the 8 words of a group: quad_perm xor 1, xor 2, half mirror
      s8 += dpp_f32<0x4E>(s8);
      s8 += dpp_f32<0x141>(s8);
      const int g = t >> 3;
      if ((t & 7) == 0 && g < GP) {
        const float v = t < NW ? s8 : 0.0f;   // groups past the row (up to GP) are zero
        uint16_t p[3];
        split3(v, p);
#pragma unroll
        for (int k = 0; k < 3; ++k) hs[(row * 3 + k) * GP + g] = p[k];
      }
    }
  }
}

// ------------------------------------------------------------------ 4-bit product
// One workgroup: MT token rows x 256 outputs, 4 wavefronts of 64 outputs each, v_mfma
// 32x32x16. A stage is 128 inputs: the rows' 256 bytes (shared by the wavefronts), every
// output's 64 bytes of nibbles and its two scales, all brought to LDS by direct loads into a
// ring of two stages (one stage in flight while the other is multiplied; one barrier per
// stage). The rows' 16-byte pieces are swapped in their 128-byte group by (row % 8), the
// outputs' in their 64 bytes by (output / 4 % 4): the swap is in the load's source address,
// so the LDS side stays linear and the 16-byte fragment reads are free of bank conflicts.
// A weight word is one lane's B operand of one MFMA: 8 consecutive inputs as bf16 16 + q (a
// shift and an and-or per pair), so lane half h takes words 4h .. 4h+3 of a group and the
// rows' pieces in the same order. Per group acc = sum x (16 + q) starts from zero and
// y += s acc in fp32; sum_g (b - 16 s) sum(x) starts y: the group sums' first and second parts
// (in the two lane halves) times b and times -16 s and their third parts times both, 8 groups
// per three MFMAs, so that no bit of the fp32 sums is lost (a third part costs 3 % of the kernel).
// The matrix cores need 8 instructions per group and 32 x 64 outputs, the vector unit about
// 100 for the nibbles, the scales' products and the addresses: a wavefront of 64 rows shares
// the nibbles' part between two row blocks.
template <int MT, int MODE>
__global__ __launch_bounds__(256, MT == 32 ? 3 : 2) void k_gemm_q4(GemmArgs a) {
  constexpr int MI = MT / 32;
  constexpr int kA = MT * 256, kB = 256 * 64, kS = 256 * 4, kStage = kA + kB + kS;
  __shared__ __attribute__((aligned(1024))) char lds[2 * kStage];
  // a tile row's byte offset in y (and in res; expert products: in hsum); kNoRow: none
  __shared__ __attribute__((aligned(16))) uint32_t drow[MT], erow[MODE == kStore ? 1 : MT];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, kh = lane >> 5;
  const int I = a.I, G = I / 64, NS = I / 128;

  // ---- this workgroup's rows and outputs
  int n0, O;
  const uint32_t* w = a.w;
  const uint16_t* sp = a.s;
  const uint16_t* bp = a.b;
  int trow[MI];                    // token rows 32 mi + j (the group sums)
  int arow[MI];                    // token rows this lane loads: 8 (MI wave + i) + lane / 8
  if constexpr (MODE == kUpRelu2) {
    const int nbF = (a.F + 255) / 256, nbS = (a.FS + 255) / 256;
    const int nr = min(max(*a.ntiles, 0), a.nt_routed);
    const int total = nr * nbF + a.nt_shared * nbS;
    if ((int)blockIdx.x >= total) return;
    const int id = xcd_remap((int)blockIdx.x, total);
    // the shared expert's tiles first: consecutive tiles of an expert stay on an XCD
    const bool sh = id < a.nt_shared * nbS;
    const int u = sh ? id : id - a.nt_shared * nbS, nb = sh ? nbS : nbF;
    const int t = u / nb, tile = sh ? a.nt_routed + t : t;
    n0 = (u - t * nb) * 256;
    O = sh ? a.FS : a.F;
    const int e = a.tile_e[tile];
    if (sh) {
      w = a.sw; sp = a.ss; bp = a.sb;
    } else {
      if ((unsigned)e >= (unsigned)a.E) return;
      w += (size_t)e * O * (I / 8);
      sp += (size_t)e * O * G;
      bp += (size_t)e * O * G;
    }
    const int32_t* ts = a.tile_slot + (size_t)tile * MT;
    auto token = [&](int s) { return s < 0 ? 0 : sh ? s : s / a.topk; };
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      trow[i] = token(ts[32 * i + j]);
      arow[i] = token(ts[8 * (MI * wave + i) + (lane >> 3)]);
    }
    if (tid < MT) {
      const int s = ts[tid], NR = a.topk * a.F + a.FS, k = sh ? a.topk : max(s, 0) % a.topk, tok = token(s);
      drow[tid] = s < 0 ? kNoRow : 2u * (uint32_t)(tok * NR + k * a.F);
      erow[tid] = s < 0 ? kNoRow : 6u * (uint32_t)((tok * (a.topk + 1) + k) * a.GPH);
    }
  } else {
    const int nbm = (a.T + MT - 1) / MT, nbn = (a.O + 255) / 256;
    const int id = xcd_remap((int)blockIdx.x, nbm * nbn);
    const int nb = id / nbm, m0 = (id - nb * nbm) * MT;
    n0 = nb * 256;
    O = a.O;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      trow[i] = min(m0 + 32 * i + j, a.T - 1);
      arow[i] = min(m0 + 8 * (MI * wave + i) + (lane >> 3), a.T - 1);
    }
    if (tid < MT) {
      const bool in = m0 + tid < a.T;
      drow[tid] = in ? (uint32_t)(m0 + tid) * (uint32_t)a.y_ld * 2u : kNoRow;
      if constexpr (MODE == kResid) erow[tid] = in ? (uint32_t)(m0 + tid) * (uint32_t)a.res_ld * 2u : kNoRow;
    }
  }

  // ---- the ring's loads of one stage by this wavefront: 2 MI KB of rows, 4 KB of nibbles,
  // 256 bytes of scales (rows past the tile's end re-read row 0, outputs past the last one
  // re-read it)
  const char* asrc[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
    asrc[i] = reinterpret_cast<const char*>(a.xp + (size_t)arow[i] * I) + 16 * ((lane & 7) ^ (lane >> 3));
  const char* bsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int col = min(n0 + 64 * wave + 16 * i + (lane >> 2), O - 1);
    bsrc[i] = reinterpret_cast<const char*>(w) + (size_t)col * (I / 2) + 16 * ((lane & 3) ^ ((lane >> 4) & 3));
  }
  const char* ssrc = reinterpret_cast<const char*>(sp + (size_t)min(n0 + 64 * wave + lane, O - 1) * G);
  const uint32_t lbase = (uint32_t)(uintptr_t)(lds_void_t*)lds;
  // The direct loads are issued by inline assembly so that the ring's reads wait only on the
  // explicit counts below (M0 = the LDS address of the wavefront's 64 pieces).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  auto load16 = [&](uint32_t dst, const char* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src)
                 : "memory", "m0");
  };
  auto load4 = [&](uint32_t dst, const char* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(dst), "v"(src)
                 : "memory", "m0");
  };
#pragma clang diagnostic pop
  auto issue = [&](int st) {
    const uint32_t base = lbase + (uint32_t)(st & 1) * kStage;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int gi = 0; gi < 2; ++gi)
        load16(base + (uint32_t)(gi * MT * 128 + 1024 * (MI * wave + i)), asrc[i] + 256 * (size_t)st + 128 * gi);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      load16(base + kA + (uint32_t)(4096 * wave + 1024 * i), bsrc[i] + 64 * (size_t)st);
    load4(base + kA + kB + 256u * (uint32_t)wave, ssrc + 4 * (size_t)st);
  };
  issue(0);

  // ---- y = sum_g (b - 16 s) sum(x), while the first stage is on its way: 8 groups at a time,
  // the next ones' loads in flight. The last 8 end at the row's last group, with zero for the
  // sums that the 8 before have covered, so that every load is 16 bytes and none leaves the
  // row (with 4-byte loads clamped to the row 2048 rows of 4096 inputs took 107 us against 89);
  // rows of fewer than 8 groups take 4 bytes each, pairs past the row its last pair, where
  // the sums are zero.
  f32x16 y[MI][2];
  {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int v = 0; v < 16; ++v) y[mi][nt][v] = 0.0f;
    uint32_t coff[2];
    const char* hrow[MI];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) coff[nt] = (uint32_t)min(n0 + 64 * wave + 32 * nt + j, O - 1) * (uint32_t)(2 * G);
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
      hrow[mi] = reinterpret_cast<const char*>(a.hs + (size_t)trow[mi] * 3 * a.GP);
    const int nc = (G + 7) / 8, o1 = kh * 2 * a.GP, o2 = 4 * a.GP;   // first or second parts by half; third parts
    u32x4 hv[2][MI], h3[2][MI], bv[2][2], sv[2][2];
    auto load = [&](int c, int u) {
      c = min(c, nc - 1);
      const int g = max(min(8 * c, G - 8), 0), over = (8 * c - g) / 2;   // uniform; pairs already covered
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        hv[u][mi] = reinterpret_cast<const Piece*>(hrow[mi] + o1 + 2 * g)->v;
        h3[u][mi] = reinterpret_cast<const Piece*>(hrow[mi] + o2 + 2 * g)->v;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          hv[u][mi][q] = q < over ? 0u : hv[u][mi][q];
          h3[u][mi][q] = q < over ? 0u : h3[u][mi][q];
        }
      }
      if (G >= 8) {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          bv[u][nt] = reinterpret_cast<const Piece*>(reinterpret_cast<const char*>(bp) + 2 * g + coff[nt])->v;
          sv[u][nt] = reinterpret_cast<const Piece*>(reinterpret_cast<const char*>(sp) + 2 * g + coff[nt])->v;
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int o = 4 * min(q, G / 2 - 1);       // uniform
#pragma unroll
          for (int nt = 0; nt < 2; ++nt) {
            bv[u][nt][q] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(bp) + o + coff[nt]);
            sv[u][nt][q] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(sp) + o + coff[nt]);
          }
        }
      }
    };
    auto apply = [&](int u) {
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        u32x4 sw;
#pragma unroll
        for (int q = 0; q < 4; ++q) sw[q] = neg16(sv[u][nt][q]);
        // the third parts: b in lane half 0, -16 s in half 1
        const u32x4 bs = kh ? sw : bv[u][nt];
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
          const bf16x8 h8 = __builtin_bit_cast(bf16x8, hv[u][mi]);
          y[mi][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, h3[u][mi]), __builtin_bit_cast(bf16x8, bs), y[mi][nt], 0, 0, 0);
          y[mi][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h8, __builtin_bit_cast(bf16x8, bv[u][nt]), y[mi][nt], 0, 0, 0);
          y[mi][nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h8, __builtin_bit_cast(bf16x8, sw), y[mi][nt], 0, 0, 0);
        }
      }
    };
    load(0, 0);
    for (int c = 0; c < nc; c += 2) {
      load(c + 1, 1);
      apply(0);
      if (c + 1 >= nc) break;
      load(c + 2, 0);
      apply(1);
    }
  }

  const uint32_t nibm = opaque_vgpr(kNibHi);
  for (int st = 0; st < NS; ++st) {
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wavefront's part of stage st is in
    lds_barrier();                        // everyone's, and the other slot has been read
    if (st + 1 < NS) issue(st + 1);
    const char* base = lds + (st & 1) * kStage;
    uint32_t s2[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
      s2[nt] = *reinterpret_cast<const uint32_t*>(base + kA + kB + 256 * wave + 4 * (32 * nt + j));
#pragma unroll
    for (int gi = 0; gi < 2; ++gi) {
      uint4 bw[2];
      float sc[2];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const int n = 32 * nt + j;
        bw[nt] = *reinterpret_cast<const uint4*>(base + kA + 4096 * wave + 64 * n + 16 * ((2 * gi + kh) ^ ((n >> 2) & 3)));
        sc[nt] = gi ? hi_f(s2[nt]) : lo_f(s2[nt]);
      }
      bf16x8 bf[2][4];
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        const uint32_t q4[4] = {bw[nt].x, bw[nt].y, bw[nt].z, bw[nt].w};
#pragma unroll
        for (int q = 0; q < 4; ++q)
          bf[nt][q] = __builtin_bit_cast(bf16x8, make_uint4(((q4[q] << 3) & nibm) | kBf16Two, ((q4[q] >> 1) & nibm) | kBf16Two,
                                                            ((q4[q] >> 5) & nibm) | kBf16Two, ((q4[q] >> 9) & nibm) | kBf16Two));
      }
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        f32x16 acc[2] = {};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = 32 * mi + j;
          const bf16x8 av = __builtin_bit_cast(
              bf16x8, *reinterpret_cast<const uint4*>(base + gi * MT * 128 + 128 * r + 16 * ((4 * kh + q) ^ (r & 7))));
#pragma unroll
          for (int nt = 0; nt < 2; ++nt)
            acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bf[nt][q], acc[nt], 0, 0, 0);
        }
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
#pragma unroll
          for (int v = 0; v < 16; ++v) y[mi][nt][v] = fmaf(sc[nt], acc[nt][v], y[mi][nt][v]);
      }
    }
  }

  // ---- outputs: lane column n, rows 32 mi + 8 (v / 4) + 4 kh + v % 4. Buffer stores at 32-bit
  // offsets, which drop what lies past the buffer: rows and columns that are none have offsets
  // there, so there is no branch and no 64-bit address per row.
  const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(a.y, (short)0, (int)a.y_bytes, 0x00020000);
  uint32_t col[2];
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int n = n0 + 64 * wave + 32 * nt + j;
    col[nt] = n < O ? 2u * (uint32_t)n : kNoCol;
  }
  auto put = [&](uint32_t row, const uint32_t (&u)[2]) {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) __builtin_amdgcn_raw_buffer_store_b16((short)u[nt], yr, row + col[nt], 0, 0);
  };
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    u32x4 ro[4], eo[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ro[q] = *reinterpret_cast<const u32x4*>(&drow[32 * mi + 8 * q + 4 * kh]);
      if constexpr (MODE != kStore) eo[q] = *reinterpret_cast<const u32x4*>(&erow[32 * mi + 8 * q + 4 * kh]);
    }
    uint32_t rv[MODE == kResid ? 16 : 1][2];
    if constexpr (MODE == kResid) {
      const __amdgpu_buffer_rsrc_t rr =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.res), (short)0, (int)a.res_bytes, 0x00020000);
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          rv[v][nt] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rr, eo[v >> 2][v & 3] + col[nt], 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const uint32_t p = pack_bf16x2(y[mi][0][v], y[mi][1][v]);
      if constexpr (MODE == kStore) {
        put(ro[v >> 2][v & 3], {p & 0xFFFFu, p >> 16});
      } else if constexpr (MODE == kResid) {
        const uint32_t r = pack_bf16x2(lo_f(rv[v][0]) + lo_f(p), lo_f(rv[v][1]) + hi_f(p));
        put(ro[v >> 2][v & 3], {r & 0xFFFFu, r >> 16});
      } else {
        // h = square(relu(bf16(u))), NaN kept. F and FS are multiples of 64, so a wavefront's 64
        // outputs are one group (or past the end): its sum over the half-wavefront's lanes in
        // a fixed order, written by lanes 0 and 32 for the down projection
        float r0 = lo_f(p), r1 = hi_f(p);
        r0 = r0 < 0.0f ? 0.0f : r0;
        r1 = r1 < 0.0f ? 0.0f : r1;
        const uint32_t h = pack_bf16x2(r0 * r0, r1 * r1);
        put(ro[v >> 2][v & 3], {h & 0xFFFFu, h >> 16});
        if (a.hsum) {   // uniform
          float t = lo_f(h) + hi_f(h);
          t += dpp_f32<0xB1>(t);
          t += dpp_f32<0x4E>(t);
          t += dpp_f32<0x141>(t);
          t += dpp_f32<0x140>(t);
          const uint32_t tb = __float_as_uint(t);
          const auto pt = __builtin_amdgcn_permlane16_swap(tb, tb, false, false);
          t = __uint_as_float(pt[0]) + __uint_as_float(pt[1]);
          const __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc(a.hsum, (short)0, (int)a.hsum_bytes, 0x00020000);
          uint16_t p3[3];
          split3(t, p3);
          const uint32_t off = eo[v >> 2][v & 3] + (j == 0 && col[0] != kNoCol ? 2u * (uint32_t)(n0 / 64 + wave) : kNoCol);
#pragma unroll
          for (int k = 0; k < 3; ++k)
            __builtin_amdgcn_raw_buffer_store_b16((short)p3[k], hr, off + 2u * (uint32_t)(k * a.GPH), 0, 0);
        }
      }
    }
  }
}

// ------------------------------------------------------------------ expert down products
// part[(t, slot)] = gain * h W over the tiles of k_tiles, W neuron-major (rows = inputs f,
// words of 8 consecutive outputs), and k_sum_resid adds a token's parts in slot order to its
// residual. Workgroup: MT slots x 512 outputs, 4 wavefronts of 128 outputs. A stage is one
// 64-neuron group: the slots' 128 bytes of h, 64 weight rows of 256 bytes and the group's
// scales, by direct loads into a ring. A lane's 8 words (8 consecutive neurons, one word
// column) are a block of 8 neurons x 8 outputs; the two lanes that share it take 4 outputs
// each: a v_perm pairs two neurons' halves and a shift and an and-or make the bf16 pair, so
// the lane's outputs are 4 consecutive columns, one per MFMA. The weight rows' 64-byte
// quarters are swapped in neighbouring pairs for the upper 8 rows of every 16, so the two lane
// halves read different banks. Every neuron of the layer is multiplied: a tile of 24 tokens has
// a live token in nearly every row (90 % zeros: 1 - 0.9^24 = 92 %), where the union lists (k_gemm
// in prefill.hip) save nothing for their passes over h. Tiles of few tokens read mostly dead rows
// (2.8 tokens: 74 %): up to 12 rows a block takes the union lists (hsd/model.py).
struct DownArgs {
  const uint16_t* h;       // [T, topk*F + FS]
  const uint16_t* hsum;    // [T * (topk + 1), 3 GPH]
  const float* gains;      // [T, topk + 1]
  const uint32_t* w;       // [E, F, D/8]
  const uint16_t* s;       // [E, F/64, D]
  const uint16_t* b;
  const uint32_t* sw;      // [FS, D/8]
  const uint16_t* ss;
  const uint16_t* sb;
  const int32_t* tile_e;
  const int32_t* tile_slot;
  const int32_t* ntiles;
  float* part;             // [T * (topk + 1), D]
  uint32_t part_bytes;     // below 1 GiB
  int nt_routed, nt_shared, T, D, F, FS, topk, E, GPH;
};

template <int MT>
__global__ __launch_bounds__(256, 2) void k_gemm_down(DownArgs a) {
  constexpr int MI = MT / 32, kRing = 3;
  constexpr int kA = MT * 128, kB = 64 * 256, kS = 1024, kStage = kA + kB + kS;
  __shared__ __attribute__((aligned(1024))) char lds[kRing * kStage];
  __shared__ __attribute__((aligned(16))) uint32_t srow[MT];   // a slot's byte offset in part
  __shared__ __attribute__((aligned(16))) float grow[MT];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, kh = lane >> 5, D = a.D;
  const int nb = (D + 511) / 512;
  const int nr = min(max(*a.ntiles, 0), a.nt_routed);
  // the shared expert's tiles first (they are the longest), spread over the XCDs by
  // themselves: one remap over both kinds gives two XCDs most of the long ones (512 rows 169
  // against 137 us, 2048 rows 411 against 293 us)
  const int ns = a.nt_shared * nb, bid = (int)blockIdx.x;
  const bool sh = bid < ns;
  if (bid >= ns + nr * nb) return;
  const int id = sh ? xcd_remap(bid, ns) : xcd_remap(bid - ns, nr * nb);
  const int t = id / nb, n0 = (id - t * nb) * 512 + 128 * wave;
  const int tile = sh ? a.nt_routed + t : t;
  const int e = a.tile_e[tile];
  const int FF = sh ? a.FS : a.F, G = FF / 64, NR = a.topk * a.F + a.FS;
  if (!sh && (unsigned)e >= (unsigned)a.E) return;
  const uint32_t* w = sh ? a.sw : a.w + (size_t)e * FF * (D / 8);
  const uint16_t* sp = sh ? a.ss : a.s + (size_t)e * G * D;
  const uint16_t* bp = sh ? a.sb : a.b + (size_t)e * G * D;
  const int32_t* ts = a.tile_slot + (size_t)tile * MT;
  auto hoff = [&](int s) { return s < 0 ? 0 : sh ? (size_t)s * NR + a.topk * a.F : (size_t)(s / a.topk) * NR + (s % a.topk) * a.F; };
  auto sidx = [&](int s) { return s < 0 ? 0 : sh ? s * (a.topk + 1) + a.topk : (s / a.topk) * (a.topk + 1) + s % a.topk; };
  int hrow[MI];
  const char* asrc[MI];
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    hrow[i] = sidx(ts[32 * i + j]);
    asrc[i] = reinterpret_cast<const char*>(a.h + hoff(ts[8 * (MI * wave + i) + (lane >> 3)])) + 16 * ((lane & 7) ^ (lane >> 3));
  }
  if (tid < MT) {
    const int s = ts[tid];
    srow[tid] = s < 0 ? kNoRow : 4u * (uint32_t)sidx(s) * (uint32_t)D;
    grow[tid] = a.gains[sidx(s)];
  }
  // weight rows: 4 per load, 16 lanes each; wavefront w loads rows 16 w .. 16 w + 15 of a
  // group (columns past D re-read the last piece)
  const char* bsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 16 * wave + 4 * i + (lane >> 4), pc = (lane & 15) ^ (4 * ((row >> 3) & 1));
    const int byte = min((n0 - 128 * wave) / 2 + 16 * pc, D / 2 - 16);
    bsrc[i] = reinterpret_cast<const char*>(w) + (size_t)row * (D / 2) + byte;
  }
  const char* ssrc = reinterpret_cast<const char*>(sp) + 2 * min(n0 + 2 * lane, D - 2);
  const uint32_t lbase = (uint32_t)(uintptr_t)(lds_void_t*)lds;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  auto load16 = [&](uint32_t dst, const char* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src)
                 : "memory", "m0");
  };
  auto load4 = [&](uint32_t dst, const char* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(dst), "v"(src)
                 : "memory", "m0");
  };
#pragma clang diagnostic pop
  constexpr int kLoads = MI + 5;   // per wavefront and stage
  auto issue = [&](int g, int slot) {
    const uint32_t base = lbase + (uint32_t)slot * kStage;
#pragma unroll
    for (int i = 0; i < MI; ++i) load16(base + 1024u * (uint32_t)(MI * wave + i), asrc[i] + 128 * (size_t)g);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      load16(base + kA + 1024u * (uint32_t)(4 * wave + i), bsrc[i] + (size_t)g * 32 * D);
    load4(base + kA + kB + 256u * (uint32_t)wave, ssrc + (size_t)g * 2 * D);
  };
  issue(0, 0);
  issue(min(1, G - 1), 1);

  // ---- y = sum_g (b - 16 s) sum(h): the group sums (in three parts, as above) times b and
  // -16 s, 8 groups at a time with the next ones' loads in flight; groups past the last are
  // zeroed on both sides (their sums are not written)
  f32x16 y[MI][4];
  {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) y[mi][i][v] = 0.0f;
    const int col = min(n0 + 4 * j, D - 4), nc = (G + 7) / 8;
    const char* hr[MI];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
      hr[mi] = reinterpret_cast<const char*>(a.hsum + (size_t)hrow[mi] * 3 * a.GPH);
    const int o1 = kh * 2 * a.GPH, o2 = 4 * a.GPH;   // first or second parts by half; third parts
    u32x4 hv[2][MI], h3[2][MI];
    u32x2 r[2][2][8];
    auto load = [&](int c, int u) {
      c = min(c, nc - 1);
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        hv[u][mi] = *reinterpret_cast<const u32x4*>(hr[mi] + o1 + 16 * c);
        h3[u][mi] = *reinterpret_cast<const u32x4*>(hr[mi] + o2 + 16 * c);
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const size_t o = (size_t)min(8 * c + q, G - 1) * D + col;
        r[u][0][q] = *reinterpret_cast<const u32x2*>(bp + o);
        r[u][1][q] = *reinterpret_cast<const u32x2*>(sp + o);
      }
    };
    auto apply = [&](int c, int u) {
      const int live = G - 8 * c;                    // groups of this chunk
      auto keep = [&](uint32_t x, int p) { return 2 * p + 1 < live ? x : 2 * p < live ? x & 0xFFFFu : 0u; };
      bf16x8 h8[MI], hx[MI];
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) {
        h8[mi] = __builtin_bit_cast(
            bf16x8, u32x4{keep(hv[u][mi][0], 0), keep(hv[u][mi][1], 1), keep(hv[u][mi][2], 2), keep(hv[u][mi][3], 3)});
        hx[mi] = __builtin_bit_cast(
            bf16x8, u32x4{keep(h3[u][mi][0], 0), keep(h3[u][mi][1], 1), keep(h3[u][mi][2], 2), keep(h3[u][mi][3], 3)});
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        u32x4 f[3];                                  // b, -16 s, and by lane half for the third parts
#pragma unroll
        for (int p = 0; p < 4; ++p) {
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            uint32_t w = __builtin_amdgcn_perm(r[u][k][2 * p + 1][i >> 1], r[u][k][2 * p][i >> 1],
                                               (i & 1) ? 0x07060302u : 0x05040100u);
            if (k) w = neg16(w);
            f[k][p] = keep(w, p);
          }
          f[2][p] = kh ? f[1][p] : f[0][p];
        }
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
          for (int k = 0; k < 3; ++k)
            y[mi][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k == 2 ? hx[mi] : h8[mi], __builtin_bit_cast(bf16x8, f[k]), y[mi][i], 0, 0, 0);
      }
    };
    load(0, 0);
    for (int c = 0; c < nc; c += 2) {
      load(c + 1, 1);
      apply(c, 0);
      if (c + 1 >= nc) break;
      load(c + 2, 0);
      apply(c + 1, 1);
    }
  }

  const uint32_t nibm = opaque_vgpr(kNibHi);
  // half jq = j & 1 of two words: the low word's 16 bits, then the high word's
  const uint32_t psel = (j & 1) ? 0x07060302u : 0x05040100u;
  const int cw = 4 * (4 * wave + 0) + (j >> 1);   // word column in the 64-word row
  const bool active = n0 < D;
  int slot = 0;
  for (int g = 0; g < G; ++g) {
    // the loads of groups g and g + 1 are in flight (past the last group: of the last again)
    __builtin_amdgcn_s_waitcnt(0x0F70 | kLoads);   // vmcnt(kLoads): group g is in
    lds_barrier();
    {
      int ns = slot + 2;
      ns = ns >= kRing ? ns - kRing : ns;
      issue(min(g + 2, G - 1), ns);
    }
    if (active) {
      const char* base = lds + slot * kStage;
      const uint2 s4 = *reinterpret_cast<const uint2*>(base + kA + kB + 256 * wave + 8 * j);
      const float sc[4] = {lo_f(s4.x), hi_f(s4.x), lo_f(s4.y), hi_f(s4.y)};
      uint32_t pr[4][4];
      bf16x8 av[4][MI];
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        uint32_t wd[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int row = 16 * st + 8 * kh + q;
          wd[q] = *reinterpret_cast<const uint32_t*>(base + kA + 256 * row + 4 * (cw ^ (16 * kh)));
        }
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) {
          const int r = 32 * mi + j;
          av[st][mi] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(base + 128 * r + 16 * ((2 * st + kh) ^ (r & 7))));
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) pr[st][p] = __builtin_amdgcn_perm(wd[2 * p + 1], wd[2 * p], psel);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x16 acc[MI] = {};
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          uint32_t f[4];
#pragma unroll
          for (int p = 0; p < 4; ++p) {
            const uint32_t v = pr[st][p];
            f[p] = ((i == 0 ? v << 3 : i == 1 ? v >> 1 : i == 2 ? v >> 5 : v >> 9) & nibm) | kBf16Two;
          }
          const bf16x8 bv = __builtin_bit_cast(bf16x8, make_uint4(f[0], f[1], f[2], f[3]));
#pragma unroll
          for (int mi = 0; mi < MI; ++mi)
            acc[mi] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[st][mi], bv, acc[mi], 0, 0, 0);
        }
#pragma unroll
        for (int mi = 0; mi < MI; ++mi)
#pragma unroll
          for (int v = 0; v < 16; ++v) y[mi][i][v] = fmaf(sc[i], acc[mi][v], y[mi][i][v]);
      }
    }
    slot = slot + 1 == kRing ? 0 : slot + 1;
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);   // no ring load outlives the workgroup
  if (!active) return;
  // 16-byte buffer stores at 32-bit offsets (a pad slot's lies past the buffer: dropped)
  const __amdgpu_buffer_rsrc_t pr = __builtin_amdgcn_make_buffer_rsrc(a.part, (short)0, (int)a.part_bytes, 0x00020000);
  const uint32_t cb = 4u * (uint32_t)(n0 + 4 * j);
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u32x4 ro = *reinterpret_cast<const u32x4*>(&srow[32 * mi + 8 * q + 4 * kh]);
      const f32x4 gn = *reinterpret_cast<const f32x4*>(&grow[32 * mi + 8 * q + 4 * kh]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int v = 4 * q + i;
        const f32x4 o = {gn[i] * y[mi][0][v], gn[i] * y[mi][1][v], gn[i] * y[mi][2][v], gn[i] * y[mi][3][v]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, o), pr, ro[i] + cb, 0, 0);
      }
    }
}

// x[t] = bf16(x[t] + bf16(sum of the token's parts in slot order)); a slot whose expert id is
// out of range is dropped (its part was not written). Thread: 4 outputs.
template <int K>
__global__ __launch_bounds__(256) void k_sum_resid(const float* __restrict__ part, const int32_t* __restrict__ sel,
                                                   const uint16_t* __restrict__ res, int64_t res_ld,
                                                   uint16_t* __restrict__ y, int64_t y_ld, int T, int D, int topk, int E) {
  const int D4 = D / 4;
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (size_t)T * D4) return;
  const size_t t = idx / D4, o = (idx - t * D4) * 4;
  const int nk = K > 0 ? K : topk;
  const float4* p = reinterpret_cast<const float4*>(part + t * (nk + 1) * D + o);
  const uint2 rv = *reinterpret_cast<const uint2*>(res + t * res_ld + o);
  float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  auto add = [](float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); };
  if constexpr (K > 0) {
    int e[K];
    float4 v[K + 1];
#pragma unroll
    for (int k = 0; k < K; ++k) e[k] = sel[t * K + k];
#pragma unroll
    for (int k = 0; k <= K; ++k) v[k] = p[(size_t)k * D4];
#pragma unroll
    for (int k = 0; k < K; ++k) s = (unsigned)e[k] < (unsigned)E ? add(s, v[k]) : s;
    s = add(s, v[K]);
  } else {
    for (int k = 0; k < nk; ++k)
      if ((unsigned)sel[t * nk + k] < (unsigned)E) s = add(s, p[(size_t)k * D4]);
    s = add(s, p[(size_t)nk * D4]);
  }
  auto out = [](float v, float r) { return (uint32_t)f32_to_bf16_bits(r + bf16_bits_to_f32(f32_to_bf16_bits(v))); };
  *reinterpret_cast<uint2*>(y + t * y_ld + o) =
      make_uint2(out(s.x, lo_f(rv.x)) | (out(s.y, hi_f(rv.x)) << 16), out(s.z, lo_f(rv.y)) | (out(s.w, hi_f(rv.y)) << 16));
}

// ------------------------------------------------------------------ bf16 product
// A workgroup of 8 wavefronts: 32 token rows x 32 outputs, the inputs split over the
// wavefronts in contiguous runs of 16 and the partial sums added in wavefront order through
// LDS. Fragments come straight from global memory (16 bytes per lane; the rows and the
// weight stay in L2). PERM: the rows are in k_rows_prep's order (the weight's pairs are
// brought to it with v_perm). The router gate (128 outputs) has few tiles: small ones and the
// inputs over 8 wavefronts keep its chain of loads short.
constexpr int kGW = 8;
template <bool PERM>
__global__ __launch_bounds__(64 * kGW) void k_gemm_bf16(const uint16_t* __restrict__ x, int64_t x_ld,
                                                        const uint16_t* __restrict__ w, uint16_t* __restrict__ y,
                                                        int64_t y_ld, int T, int O, int I) {
  __shared__ float red[kGW - 1][16][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = lane & 31, kh = lane >> 5;
  const int nbm = (T + 31) / 32, nbn = (O + 31) / 32;
  const int id = xcd_remap((int)blockIdx.x, nbm * nbn);
  const int nb = id / nbm, m0 = (id - nb * nbm) * 32, n0 = nb * 32;
  const int nk = (I + 15) / 16, per = (nk + kGW - 1) / kGW, k0 = wave * per, k1 = min(k0 + per, nk);
  const uint16_t* xr = x + (size_t)min(m0 + j, T - 1) * x_ld;
  const uint16_t* wr = w + (size_t)min(n0 + j, O - 1) * I;
  f32x16 acc = {};
  // steps in flight; the loop has no branch around a load or its use (the compiler would
  // wait for every load in flight where the paths merge): a step past the run re-reads the
  // last one and is multiplied as zeros
  constexpr int U = 8;
  uint4 av[U], bv[U];
  auto load = [&](int u, int k) {
    const int o = min(16 * k + 8 * kh, I - 8);
    av[u] = *reinterpret_cast<const uint4*>(xr + o);
    bv[u] = *reinterpret_cast<const uint4*>(wr + o);
  };
#pragma unroll
  for (int u = 0; u < U; ++u) load(u, k0 + u);
  for (int k = k0; k < k1; k += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // I % 16 == 8: the upper half of the last step is past the row
      const bool live = k + u < k1 && 16 * (k + u) + 8 * kh < I;
      const uint4 a = make_uint4(live ? av[u].x : 0u, live ? av[u].y : 0u, live ? av[u].z : 0u, live ? av[u].w : 0u);
      uint4 b = bv[u];
      if constexpr (PERM)
        b = make_uint4((b.x & 0xFFFFu) | (b.z << 16), (b.x >> 16) | (b.z & 0xFFFF0000u),
                       (b.y & 0xFFFFu) | (b.w << 16), (b.y >> 16) | (b.w & 0xFFFF0000u));
      b = make_uint4(live ? b.x : 0u, live ? b.y : 0u, live ? b.z : 0u, live ? b.w : 0u);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
      load(u, k + U + u);
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int v = 0; v < 16; ++v) red[wave - 1][v][lane] = acc[v];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int s = 0; s < kGW - 1; ++s)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] += red[s][v][lane];
  const int n = n0 + j;
  if (n >= O) return;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int r = m0 + 8 * (v >> 2) + 4 * kh + (v & 3);
    if (r < T) y[(size_t)r * y_ld + n] = f32_to_bf16_bits(acc[v]);
  }
}

// Many rows of many outputs (the MTP head's eh_proj on a long prompt): 128 token rows x 128
// outputs per workgroup, 64 x 64 per wavefront. 64 inputs of both sides are brought to LDS by
// direct loads into a ring of two stages, the rows' 16-byte pieces swapped by (row % 8) in the
// source address: half of what 64 x 64 tiles took from L2, and no wavefront waits on fragments
// of its own. 2048 rows, 5376 -> 2688: 237 -> 79 us (750 TFLOP/s); the rest is a last wave of 80
// workgroups beside 256 CUs and the loop's serial stages (54 us however few the tiles).
constexpr int kTileM = 128;
template <bool PERM>
__global__ __launch_bounds__(256, 2) void k_gemm_bf16_tiles(const uint16_t* __restrict__ x, int64_t x_ld,
                                                            const uint16_t* __restrict__ w, uint16_t* __restrict__ y,
                                                            int64_t y_ld, int T, int O, int I) {
  constexpr int kA = kTileM * 128, kStage = 2 * kA;   // 64 inputs of the rows, then of the outputs
  __shared__ __attribute__((aligned(1024))) char lds[2 * kStage];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, kh = lane >> 5, NS = I / 64;
  const int nbm = (T + kTileM - 1) / kTileM, nbn = (O + kTileM - 1) / kTileM;
  const int id = xcd_remap((int)blockIdx.x, nbm * nbn);
  const int nb = id / nbm, m0 = (id - nb * nbm) * kTileM, n0 = nb * kTileM;
  // this wavefront's loads: 4 of 8 rows and 4 of 8 outputs (past the end: the last one again)
  const char *asrc[4], *bsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 8 * (4 * wave + i) + (lane >> 3), pc = 16 * ((lane & 7) ^ (lane >> 3));
    asrc[i] = reinterpret_cast<const char*>(x + (size_t)min(m0 + r, T - 1) * x_ld) + pc;
    bsrc[i] = reinterpret_cast<const char*>(w + (size_t)min(n0 + r, O - 1) * I) + pc;
  }
  const uint32_t lbase = (uint32_t)(uintptr_t)(lds_void_t*)lds;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  auto load16 = [&](uint32_t dst, const char* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src)
                 : "memory", "m0");
  };
#pragma clang diagnostic pop
  auto issue = [&](int st) {
    const uint32_t base = lbase + (uint32_t)(st & 1) * kStage + 4096u * (uint32_t)wave;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      load16(base + 1024u * i, asrc[i] + 128 * (size_t)st);
      load16(base + kA + 1024u * i, bsrc[i] + 128 * (size_t)st);
    }
  };
  issue(0);
  const int wm = 64 * (wave & 1), wn = 64 * (wave >> 1);
  f32x16 acc[2][2] = {};
  for (int st = 0; st < NS; ++st) {
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wavefront's part of stage st is in
    lds_barrier();                        // everyone's, and the other slot has been read
    if (st + 1 < NS) issue(st + 1);
    const char* base = lds + (st & 1) * kStage;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      bf16x8 av[2], bv[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int off = 128 * (32 * i + j) + 16 * ((2 * s + kh) ^ (j & 7));
        av[i] = *reinterpret_cast<const bf16x8*>(base + 128 * wm + off);
        u32x4 b = *reinterpret_cast<const u32x4*>(base + kA + 128 * wn + off);
        if constexpr (PERM)
          b = u32x4{(b.x & 0xFFFFu) | (b.z << 16), (b.x >> 16) | (b.z & 0xFFFF0000u),
                    (b.y & 0xFFFFu) | (b.w << 16), (b.y >> 16) | (b.w & 0xFFFF0000u)};
        bv[i] = __builtin_bit_cast(bf16x8, b);
      }
#pragma unroll
      for (int mi = 0; mi < 2; ++mi)
#pragma unroll
        for (int ni = 0; ni < 2; ++ni)
          acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[mi], bv[ni], acc[mi][ni], 0, 0, 0);
    }
  }
#pragma unroll
  for (int ni = 0; ni < 2; ++ni) {
    const int n = n0 + wn + 32 * ni + j;
    if (n >= O) continue;
#pragma unroll
    for (int mi = 0; mi < 2; ++mi)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = m0 + wm + 32 * mi + 8 * (v >> 2) + 4 * kh + (v & 3);
        if (r < T) y[(size_t)r * y_ld + n] = f32_to_bf16_bits(acc[mi][ni][v]);
      }
  }
}

}  // namespace
}  // namespace hsd

using namespace hsd;

namespace {
inline int64_t group_pitch(int64_t I) { return (I / 64 + 7) / 8 * 8; }
}  // namespace

extern "C" int hsd_rows_prep(const void* x, int64_t x_ld, int x_kind, const uint16_t* norm_w, float eps,
                             uint16_t* xp, uint16_t* hs, int64_t T, int64_t I, void* stream) {
  const char* fn = "hsd_rows_prep";
  if (!x || !xp || (x_kind != HSD_X_BF16 && !norm_w)) return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  if (x_kind != HSD_X_BF16 && x_kind != HSD_X_RMS && x_kind != HSD_X_GATED_Z)
    return set_error(HSD_ERR_ARG, "%s: x_kind %d", fn, x_kind);
  if (T < 0 || T > 0x7FFFFFFF || I <= 0 || I > 8 * kPT * kPI || I % (hs ? 64 : 8) ||
      (x_kind == HSD_X_GATED_Z && (I % 512 || x_ld < I + I / 16)) || x_ld < I)
    return set_error(HSD_ERR_SHAPE, "%s: bad sizes", fn);
  const int64_t esz = x_kind == HSD_X_GATED_Z ? 4 : 2;
  if (((uintptr_t)x | (uintptr_t)xp | (uintptr_t)norm_w) & 15u || x_ld * esz % 16)
    return set_error(HSD_ERR_ALIGN, "%s: x, xp and norm_w must be 16-byte aligned", fn);
  if (T == 0) return HSD_OK;
  const dim3 grid((unsigned)T), blk(kPT);
  hipStream_t st = as_stream(stream);
  const int GP = (int)group_pitch(I);
#define HSD_PREP(K, P) \
  hipLaunchKernelGGL((k_rows_prep<K, P>), grid, blk, 0, st, x, x_ld, norm_w, eps, xp, hs, (int)I, GP)
  if (x_kind == HSD_X_BF16) {
    if (hs) HSD_PREP(HSD_X_BF16, true); else HSD_PREP(HSD_X_BF16, false);
  } else if (x_kind == HSD_X_RMS) {
    if (hs) HSD_PREP(HSD_X_RMS, true); else HSD_PREP(HSD_X_RMS, false);
  } else {
    if (hs) HSD_PREP(HSD_X_GATED_Z, true); else HSD_PREP(HSD_X_GATED_Z, false);
  }
#undef HSD_PREP
  return check_launch(fn);
}

namespace {
int gemm_q4_checks(const char* fn, const void* xp, const void* hs, const void* w, const void* s, const void* b,
                   int64_t T, int64_t O, int64_t I) {
  if (!xp || !hs || !w || !s || !b) return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  if (T < 0 || T > (1 << 20) || O <= 0 || O > (1 << 24) || I < 128 || I % 128 || I > 8 * kPT * kPI)
    return set_error(HSD_ERR_SHAPE, "%s: need I %% 128 == 0, I <= %d", fn, 8 * kPT * kPI);
  if (((uintptr_t)xp | (uintptr_t)hs | (uintptr_t)w) & 15u || ((uintptr_t)s | (uintptr_t)b) & 3u)
    return set_error(HSD_ERR_ALIGN, "%s: rows and weights must be 16-byte, scales 4-byte aligned", fn);
  return HSD_OK;
}
}  // namespace

extern "C" int hsd_gemm_q4(const uint16_t* xp, const uint16_t* hs, const uint32_t* w, const uint16_t* s,
                           const uint16_t* b, uint16_t* y, int64_t y_ld, const uint16_t* res, int64_t res_ld,
                           int64_t T, int64_t O, int64_t I, void* stream) {
  const char* fn = "hsd_gemm_q4";
  const int rc = gemm_q4_checks(fn, xp, hs, w, s, b, T, O, I);
  if (rc) return rc;
  if (!y) return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  if (y_ld < O || (res && res_ld < O)) return set_error(HSD_ERR_SHAPE, "%s: bad row strides", fn);
  if (T == 0) return HSD_OK;
  GemmArgs a{};
  a.xp = xp; a.hs = hs; a.w = w; a.s = s; a.b = b; a.y = y; a.y_ld = y_ld; a.res = res; a.res_ld = res_ld;
  a.T = (int)T; a.O = (int)O; a.I = (int)I; a.GP = (int)group_pitch(I);
  const int64_t yb = ((T - 1) * y_ld + O) * 2, rb = res ? ((T - 1) * res_ld + O) * 2 : 0;
  if (yb >= kNoCol || rb >= kNoCol) return set_error(HSD_ERR_SHAPE, "%s: y and res must be below 1 GiB", fn);
  a.y_bytes = (uint32_t)yb;
  a.res_bytes = (uint32_t)rb;
  const int64_t nbn = (O + 255) / 256;
  hipStream_t st = as_stream(stream);
  {
    const int rr = launch_gemm_rows(fn, a, res ? kResid : kStore, st);   // few rows
    if (rr != 1) return rr;
  }
  const bool wide = nbn * ((T + 63) / 64) >= 256;
#define HSD_GEMM(MT, MODE) \
  hipLaunchKernelGGL((k_gemm_q4<MT, MODE>), dim3((unsigned)(nbn * ((T + MT - 1) / MT))), dim3(256), 0, st, a)
  if (res) {
    if (wide) HSD_GEMM(64, kResid); else HSD_GEMM(32, kResid);
  } else {
    if (wide) HSD_GEMM(64, kStore); else HSD_GEMM(32, kStore);
  }
#undef HSD_GEMM
  return check_launch(fn);
}

extern "C" int hsd_moe_up_gemm(const uint16_t* xp, const uint16_t* hs, const int32_t* tile_e,
                               const int32_t* tile_slot, const int32_t* ntiles, const uint32_t* w1,
                               const uint16_t* s1, const uint16_t* b1, const uint32_t* sw1, const uint16_t* ss1,
                               const uint16_t* sb1, uint16_t* hcat, uint16_t* hsum, int64_t T, int64_t D, int64_t F,
                               int64_t FS, int64_t topk, int64_t E, int64_t tt, void* stream) {
  const char* fn = "hsd_moe_up_gemm";
  int rc = gemm_q4_checks(fn, xp, hs, w1, s1, b1, T, F, D);
  if (!rc) rc = gemm_q4_checks(fn, xp, hs, sw1, ss1, sb1, T, FS, D);
  if (rc) return rc;
  if (!tile_e || !tile_slot || !ntiles || !hcat) return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  if ((tt != 32 && tt != 64) || topk <= 0 || E <= 0) return set_error(HSD_ERR_SHAPE, "%s: tt must be 32 or 64", fn);
  if (F % 64 || FS % 64 || T * (topk * F + FS) > 0x7FFFFFFF)
    return set_error(HSD_ERR_SHAPE, "%s: need F %% 64 == 0 and FS %% 64 == 0, and sizes that fit 31 bits", fn);
  if (T == 0) return HSD_OK;
  GemmArgs a{};
  a.hsum = hsum;
  a.GPH = (int)group_pitch(F > FS ? F : FS);
  const int64_t yb = T * (topk * F + FS) * 2, hb = T * (topk + 1) * 6 * a.GPH;
  if (yb >= kNoCol || hb >= kNoCol) return set_error(HSD_ERR_SHAPE, "%s: hcat and hsum must be below 1 GiB", fn);
  a.y_bytes = (uint32_t)yb;
  a.hsum_bytes = hsum ? (uint32_t)hb : 0;
  a.xp = xp; a.hs = hs; a.w = w1; a.s = s1; a.b = b1; a.y = hcat;
  a.sw = sw1; a.ss = ss1; a.sb = sb1; a.tile_e = tile_e; a.tile_slot = tile_slot; a.ntiles = ntiles;
  a.nt_routed = (int)(T * topk / tt + E);
  a.nt_shared = (int)((T + tt - 1) / tt);
  a.T = (int)T; a.I = (int)D; a.GP = (int)group_pitch(D);
  a.F = (int)F; a.FS = (int)FS; a.topk = (int)topk; a.E = (int)E;
  // at most one tile per expert holds fewer than tt slots, and no more than T * topk experts occur
  const int64_t most = T * topk / tt + (E < T * topk ? E : T * topk);
  const int64_t grid = most * ((F + 255) / 256) + a.nt_shared * ((FS + 255) / 256);
  if (grid > 0x7FFFFFFF) return set_error(HSD_ERR_SHAPE, "%s: sizes too large", fn);
  if (tt == 32) {
    const int rr = launch_gemm_rows(fn, a, kUpRelu2, as_stream(stream));
    if (rr != 1) return rr;
  }
  if (tt == 32)
    hipLaunchKernelGGL((k_gemm_q4<32, kUpRelu2>), dim3((unsigned)grid), dim3(256), 0, as_stream(stream), a);
  else
    hipLaunchKernelGGL((k_gemm_q4<64, kUpRelu2>), dim3((unsigned)grid), dim3(256), 0, as_stream(stream), a);
  return check_launch(fn);
}

extern "C" int hsd_gemm_bf16(const uint16_t* x, int64_t x_ld, int permuted, const uint16_t* w, uint16_t* y,
                             int64_t y_ld, int64_t T, int64_t O, int64_t I, void* stream) {
  const char* fn = "hsd_gemm_bf16";
  if (!x || !w || !y) return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  if (T < 0 || T > (1 << 20) || O <= 0 || O > (1 << 24) || I <= 0 || I % 8 || x_ld < I || y_ld < O || x_ld % 8)
    return set_error(HSD_ERR_SHAPE, "%s: need I and x_ld multiples of 8", fn);
  if (((uintptr_t)x | (uintptr_t)w) & 15u) return set_error(HSD_ERR_ALIGN, "%s: x and w must be 16-byte aligned", fn);
  if (T == 0) return HSD_OK;
  hipStream_t st = as_stream(stream);
#define HSD_GB(K, GRID, BLOCK)                                                                               \
  hipLaunchKernelGGL((K), dim3((unsigned)(GRID)), dim3(BLOCK), 0, st, x, x_ld, w, y, y_ld, (int)T, (int)O, (int)I)
  // the tiled kernel from 32 tiles on (5376 -> 2688: 128 rows, 21 tiles, 54 us against 48; 256
  // rows, 42 tiles, 54 against 69; 512 rows 54 against 133); it steps by 64 inputs
  const int64_t tiles = ((T + kTileM - 1) / kTileM) * ((O + kTileM - 1) / kTileM);
  if (tiles >= 32 && I % 64 == 0) {
    if (permuted) HSD_GB(k_gemm_bf16_tiles<true>, tiles, 256); else HSD_GB(k_gemm_bf16_tiles<false>, tiles, 256);
  } else {
    const int64_t small = ((T + 31) / 32) * ((O + 31) / 32);
    if (permuted) HSD_GB(k_gemm_bf16<true>, small, 512); else HSD_GB(k_gemm_bf16<false>, small, 512);
  }
#undef HSD_GB
  return check_launch(fn);
}

extern "C" size_t hsd_moe_down_workspace_bytes(int64_t T, int64_t D, int64_t topk) {
  if (T <= 0 || D <= 0 || topk <= 0) return 0;
  return (size_t)T * (topk + 1) * D * sizeof(float);
}

extern "C" int hsd_moe_down_gemm(const uint16_t* hcat, const uint16_t* hsum, const int32_t* sel, const float* gains,
                                 const int32_t* tile_e, const int32_t* tile_slot, const int32_t* ntiles,
                                 const uint32_t* pw, const uint16_t* ps, const uint16_t* pb, const uint32_t* spw,
                                 const uint16_t* sps, const uint16_t* spb, const uint16_t* res, int64_t res_ld,
                                 uint16_t* y, int64_t y_ld, int64_t T, int64_t D, int64_t F, int64_t FS, int64_t topk,
                                 int64_t E, int64_t tt, void* workspace, size_t workspace_bytes, void* stream) {
  const char* fn = "hsd_moe_down_gemm";
  if (!hcat || !hsum || !sel || !gains || !tile_e || !tile_slot || !ntiles || !pw || !ps || !pb || !spw || !sps || !spb ||
      !res || !y)
    return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  if ((tt != 32 && tt != 64) || T < 0 || D < 128 || D % 128 || F <= 0 || F % 64 || FS <= 0 || FS % 64 || topk <= 0 || E <= 0 ||
      res_ld < D || y_ld < D || res_ld % 4 || y_ld % 4)
    return set_error(HSD_ERR_SHAPE, "%s: need tt 32 or 64, D %% 128 == 0, F %% 64 == 0, FS %% 64 == 0", fn);
  if (T * (topk * F + FS) > 0x7FFFFFFF || T * (topk + 1) > 0x7FFFFFFF || D > (1 << 20) || F > (1 << 20) || FS > (1 << 20))
    return set_error(HSD_ERR_SHAPE, "%s: sizes too large", fn);
  if (((uintptr_t)hcat | (uintptr_t)hsum | (uintptr_t)pw | (uintptr_t)spw | (uintptr_t)workspace) & 15u ||
      ((uintptr_t)ps | (uintptr_t)pb | (uintptr_t)sps | (uintptr_t)spb | (uintptr_t)res | (uintptr_t)y) & 7u)
    return set_error(HSD_ERR_ALIGN, "%s: h, sums and weights must be 16-byte, the rest 8-byte aligned", fn);
  if (T == 0) return HSD_OK;
  if (!workspace || workspace_bytes < hsd_moe_down_workspace_bytes(T, D, topk))
    return set_error(HSD_ERR_WORKSPACE, "%s: workspace too small", fn);
  if (T * (topk + 1) * D * 4 >= kNoCol) return set_error(HSD_ERR_SHAPE, "%s: the workspace must be below 1 GiB", fn);
  DownArgs a{};
  a.part_bytes = (uint32_t)(T * (topk + 1) * D * 4);
  a.h = hcat; a.hsum = hsum; a.gains = gains; a.w = pw; a.s = ps; a.b = pb; a.sw = spw; a.ss = sps; a.sb = spb;
  a.tile_e = tile_e; a.tile_slot = tile_slot; a.ntiles = ntiles; a.part = reinterpret_cast<float*>(workspace);
  a.nt_routed = (int)(T * topk / tt + E);
  a.nt_shared = (int)((T + tt - 1) / tt);
  a.T = (int)T; a.D = (int)D; a.F = (int)F; a.FS = (int)FS; a.topk = (int)topk; a.E = (int)E;
  a.GPH = (int)group_pitch(F > FS ? F : FS);
  const int64_t most = T * topk / tt + (E < T * topk ? E : T * topk);
  const int64_t grid = (most + a.nt_shared) * ((D + 511) / 512), sg = (T * (D / 4) + 255) / 256;
  if (grid > 0x7FFFFFFF || sg > 0x7FFFFFFF) return set_error(HSD_ERR_SHAPE, "%s: sizes too large", fn);
  hipStream_t st = as_stream(stream);
  if (tt == 32) hipLaunchKernelGGL(k_gemm_down<32>, dim3((unsigned)grid), dim3(256), 0, st, a);
  else hipLaunchKernelGGL(k_gemm_down<64>, dim3((unsigned)grid), dim3(256), 0, st, a);
  const int rc = check_launch(fn);
  if (rc) return rc;
  if (topk == 6)
    hipLaunchKernelGGL(k_sum_resid<6>, dim3((unsigned)sg), dim3(256), 0, st, a.part, sel, res, res_ld, y, y_ld, (int)T,
                       (int)D, (int)topk, (int)E);
  else
    hipLaunchKernelGGL(k_sum_resid<0>, dim3((unsigned)sg), dim3(256), 0, st, a.part, sel, res, res_ld, y, y_ld, (int)T,
                       (int)D, (int)topk, (int)E);
  return check_launch(fn);
}

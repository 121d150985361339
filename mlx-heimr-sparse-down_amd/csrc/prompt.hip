// A prompt chunk's recurrent and attention mixers, and its sequence bookkeeping: many
// consecutive positions P .. P+T-1 (P a device int) of one sequence at once.
//
//   k_conv_rows   the depthwise causal conv + silu of every channel and row (fp32), and dt
//                 and exp(A dt) of every head and row.
//   k_scan        the state-space recurrence over the rows, one workgroup per (head, 16
//                 state rows): the state stays in registers for the whole chunk.
//   k_kv_append   the chunk's keys and values into the cache.
//   k_attn_prompt causal GQA attention of the chunk's rows over the cache on the matrix cores.
//   k_prompt_*    token gather and state advance.
// The prompt has Ttot tokens, of which rows P .. Ttot-1 are new: a row past them (P > 0) is
// computed but leaves nothing behind.
#include <type_traits>

#include "hsd_common.h"

namespace hsd {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
// staging registers that go from global memory to LDS unread (an array of the HIP vector
// structs copied like that stays in scratch memory)
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kK = 4;       // conv kernel
constexpr int kN = 128;     // state size
constexpr int kPB = 16;     // state rows per workgroup

// the chunk's rows that belong to the prompt
__device__ __forceinline__ int valid_rows(int P, int Ttot, int T) { return min(max(Ttot - P, 0), T); }

// ------------------------------------------------------------------ conv, dt
// Thread: 8 channels x kCR rows with a sliding window (each input row read once per thread,
// kCR + 3 rows for kCR outputs). Bound by the fp32 writes (2048 rows: 50 MB).
constexpr int kCR = 8;
__global__ __launch_bounds__(256) void k_conv_rows(const uint16_t* __restrict__ cin, int64_t ld,
                                                   const uint16_t* __restrict__ dt_raw, int64_t dt_ld,
                                                   const uint16_t* __restrict__ conv_w,
                                                   const uint16_t* __restrict__ conv_b,
                                                   const float* __restrict__ A_log, const float* __restrict__ dt_bias,
                                                   const uint16_t* __restrict__ convs, const int32_t* __restrict__ cur,
                                                   int nslab, float* __restrict__ co, float* __restrict__ dtA, int T,
                                                   int CD, int H, float dt_lo, float dt_hi) {
  const int r0 = blockIdx.y * kCR, CB = (CD / 8 + 255) / 256;
  if ((int)blockIdx.x == CB) {   // dt and exp(A dt) of rows r0 .. r0 + 7, [row][2][H]
    for (int i = threadIdx.x; i < kCR * H; i += 256) {
      const int r = r0 + i / H, h = i % H;
      if (r >= T) break;
      const float A = -expf(A_log[h]);
      const float v = softplus_f32(bf16_bits_to_f32(dt_raw[(size_t)r * dt_ld + h]) + dt_bias[h]);
      const float d = fminf(fmaxf(v, dt_lo), dt_hi);
      dtA[(size_t)r * 2 * H + h] = d;
      dtA[(size_t)r * 2 * H + H + h] = expf(A * d);
    }
    return;
  }
  const int c8 = blockIdx.x * 256 + threadIdx.x;
  if (c8 >= CD / 8) return;
  const int c = *cur;
  const uint16_t* cs = convs + (size_t)((unsigned)c < (unsigned)nslab ? c : 0) * (kK - 1) * CD + 8 * c8;
  uint4 win[kCR + kK - 1];
#pragma unroll
  for (int i = 0; i < kCR + kK - 1; ++i) {   // rows r0 - 3 ..: before row 0 the cached window
    const int r = r0 + i - (kK - 1);
    const uint16_t* src = r < 0 ? cs + (size_t)(r + kK - 1) * CD : cin + (size_t)min(r, T - 1) * ld + 8 * c8;
    win[i] = *reinterpret_cast<const uint4*>(src);
  }
  uint4 wv[4];   // [8 channels][4 taps]
#pragma unroll
  for (int i = 0; i < 4; ++i) wv[i] = reinterpret_cast<const uint4*>(conv_w + (size_t)32 * c8)[i];
  const uint4 bv = *reinterpret_cast<const uint4*>(conv_b + 8 * c8);
  auto elem = [](const uint4& v, int i) {
    const uint32_t w = i < 2 ? v.x : i < 4 ? v.y : i < 6 ? v.z : v.w;
    return (i & 1) ? __uint_as_float(w & 0xFFFF0000u) : __uint_as_float(w << 16);
  };
#pragma unroll
  for (int r = 0; r < kCR; ++r) {
    if (r0 + r < T) {
      float o[8];
#pragma unroll
      for (int ch = 0; ch < 8; ++ch) {
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < kK; ++j) acc = fmaf(elem(wv[ch >> 1], 4 * (ch & 1) + j), elem(win[r + j], ch), acc);
        o[ch] = silu_f32(acc + elem(bv, ch));
      }
      float4* dst = reinterpret_cast<float4*>(co + (size_t)(r0 + r) * CD + 8 * c8);
      dst[0] = make_float4(o[0], o[1], o[2], o[3]);
      dst[1] = make_float4(o[4], o[5], o[6], o[7]);
    }
  }
}

// ------------------------------------------------------------------ scan
// The state after every row is k_mamba_ssm's, bit for bit (the same product and fma per
// element); y = sum_n S C adds in another order. Workgroup = (head, 16 state rows), 8
// wavefronts; wavefront w owns state rows 2w and 2w + 1, lane l their elements 2l and 2l + 1,
// for all rows of the chunk: a row's B and C are read from LDS once for both state rows, and
// two wavefronts per SIMD issue twice as fast as one (an instruction per 2.5 cycles against 5).
// kTS rows' inputs are staged in LDS at a time, the next ones' in registers meanwhile; after
// them the 2 x kTS lane sums are added over the lanes by halving: v_permlane32_swap and
// v_permlane16_swap bring two values' lane halves together, then DPP steps between lanes that
// keep one value each (70 instructions for 32 sums over 64 lanes).
// Bound by the serial chain over the rows: vector instructions (a stage is about 500 per
// wavefront) and LDS reads alternate with one barrier per stage. 2048 rows, 64 heads of 64 x
// 128: 323 us with 4 wavefronts of 8 elements per lane, one per SIMD; 279 with 8; 221 with the
// inputs read two stages ahead, a stage's outputs written under the next one's rows and B and C
// in one LDS read.
constexpr int kTS = 16;
constexpr int kSW = 8;      // wavefronts

// a + b of two values summed over one lane bit: lanes with the bit clear keep a's sum, the
// others b's (CTRL: a DPP control that pairs the lanes)
template <int CTRL>
__device__ __forceinline__ float halve(float a, float b, bool bit) {
  const float keep = bit ? b : a, give = bit ? a : b;
  return keep + dpp_f32<CTRL>(give);
}

__global__ __launch_bounds__(64 * kSW, 2) void k_scan(
    const float* __restrict__ co, const float* __restrict__ dtA, const uint16_t* __restrict__ cin, int64_t cin_ld,
    const uint16_t* __restrict__ gate, int64_t gate_ld, const float* __restrict__ Dp, float* __restrict__ ssm,
    uint16_t* __restrict__ convs, const int32_t* __restrict__ cur_ptr, const int32_t* __restrict__ pos, int nslab,
    float* __restrict__ z, int64_t z_ld, int T, int Ttot, int H, int P, int G, int32_t* __restrict__ status) {
  constexpr int kT = 64 * kSW;
  __shared__ __attribute__((aligned(16))) f32x4 bc[2][kTS][kN / 2];                  // B and C of elements 2 l, 2 l + 1
  __shared__ __attribute__((aligned(16))) float xs[2][kTS][kPB], xd[2][kPB / 2][kTS][2];   // x; x dt by state row pair
  __shared__ __attribute__((aligned(16))) float ds[2][kTS];                          // exp(A dt)
  __shared__ float ys[2][kTS][kPB + 1];
  const int npb = P / kPB, lb = xcd_remap((int)blockIdx.x, H * npb);
  const int hh = lb / npb, pblk = lb - hh * npb, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int DI = H * P, GN = G * kN, CD = DI + 2 * GN, hpg = H / G, g = hh / hpg;
  const int cur = *cur_ptr, V = valid_rows(*pos, Ttot, T);
  const float Dh = bf16_bits_to_f32(f32_to_bf16_bits(Dp[hh]));
  if ((unsigned)cur >= (unsigned)nslab) {
    for (int i = tid; i < T * kPB; i += kT)
      z[(size_t)(i / kPB) * z_ld + (size_t)hh * P + pblk * kPB + i % kPB] = __int_as_float(0x7FC00000);
    for (int i = tid; i < T; i += kT) z[(size_t)i * z_ld + DI + (size_t)hh * npb + pblk] = __int_as_float(0x7FC00000);
    if (tid == 0 && status) atomicOr(status, (int32_t)HSD_STATUS_BAD_STATE);
    return;
  }
  const int dst_slab = (cur + V) % nslab;
  // the conv window after row V - 1: this workgroup's 16 channels, and its group's B and C
  // channels in one workgroup per group; every read of the old window precedes the writes
  const bool owner = (hh % hpg == 0) && pblk == 0;
  if (V > 0) {
    const int nch = owner ? kPB + 2 * kN : kPB, t = min(tid, nch - 1);
    static_assert(kPB + 2 * kN <= kT, "a channel per thread");
    const int ch = t < kPB ? hh * P + pblk * kPB + t
                           : t < kPB + kN ? DI + g * kN + (t - kPB) : DI + GN + g * kN + (t - kPB - kN);
    uint16_t wv[kK - 1];
#pragma unroll
    for (int i = 0; i < kK - 1; ++i) {
      const int r = V - (kK - 1) + i;
      wv[i] = r < 0 ? convs[((size_t)cur * (kK - 1) + r + kK - 1) * CD + ch] : cin[(size_t)r * cin_ld + ch];
    }
    __syncthreads();
    if (tid < nch) {
#pragma unroll
      for (int i = 0; i < kK - 1; ++i) convs[((size_t)dst_slab * (kK - 1) + i) * CD + ch] = wv[i];
    }
  }
  const int pl = 2 * wave;                             // this wavefront's first state row of the 16
  const size_t slab = (size_t)H * P * kN, soff = ((size_t)hh * P + pblk * kPB + pl) * kN + 2 * lane;
  f32x2 S[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) S[i] = *reinterpret_cast<const f32x2*>(ssm + (size_t)cur * slab + soff + i * kN);

  // staging, two stages ahead: 16 rows x (32 + 32 float4 of B and C, 16 of x) and (dt, exp(A dt))
  struct Regs {
    f32x4 rb[2];
    float rx, rdt, rda;
    uint16_t gv;
  };
  auto load = [&](Regs& u, int t0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + kT * i, r = min(t0 + (idx >> 6), T - 1), q = idx & 63;
      u.rb[i] = *reinterpret_cast<const f32x4*>(co + (size_t)r * CD + DI + (q < 32 ? 0 : GN) + g * kN + 4 * (q & 31));
    }
    const int r = min(t0 + (tid >> 4 & 15), T - 1);
    u.rx = co[(size_t)r * CD + (size_t)hh * P + pblk * kPB + (tid & 15)];
    u.rdt = dtA[(size_t)r * 2 * H + hh];
    u.rda = dtA[(size_t)r * 2 * H + H + hh];
    u.gv = gate[(size_t)r * gate_ld + (size_t)hh * P + pblk * kPB + (tid & 15)];
  };
  auto store = [&](const Regs& u, int b) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + kT * i, r = idx >> 6, q = idx & 63;
      f32x2* dst = reinterpret_cast<f32x2*>(&bc[b][r][2 * (q & 31)]) + (q >> 5);
      dst[0] = f32x2{u.rb[i].x, u.rb[i].y};
      dst[2] = f32x2{u.rb[i].z, u.rb[i].w};
    }
    if (tid < 256) {
      const int r = tid >> 4, c = tid & 15;
      xs[b][r][c] = u.rx;
      xd[b][c >> 1][r][c & 1] = u.rx * u.rdt;
      if (c == 0) ds[b][r] = u.rda;
    }
  };
  // z and the 16 channels' sums of z^2 of the stage at t0, from ys[b] (whole wavefronts)
  auto finish = [&](int t0, int b, uint16_t gv) {
    if (tid < 256) {
      const int r = tid >> 4, c = tid & 15;
      float o = ys[b][r][c] * silu_f32(bf16_bits_to_f32(gv));
      if (t0 + r < T) z[(size_t)(t0 + r) * z_ld + (size_t)hh * P + pblk * kPB + c] = o;
      o = o * o;
      o += dpp_f32<0xB1>(o);
      o += dpp_f32<0x4E>(o);
      o += dpp_f32<0x141>(o);
      o += dpp_f32<0x140>(o);
      if (c == 0 && t0 + r < T) z[(size_t)(t0 + r) * z_ld + DI + (size_t)hh * npb + pblk] = o;
    }
  };
  // the stage at t0, in buffer kB: its gate values gv[kB], the next stage's inputs in nx (to
  // the other buffer at the end), the one's after that on their way to fill
  uint16_t gv[2];
  auto stage = [&](int t0, auto B, const Regs& nx, Regs& fill) {
    constexpr int b = decltype(B)::value;
    __syncthreads();                               // stage t0 in LDS; the last one's ys complete, its buffer read
    load(fill, t0 + 2 * kTS);                      // past the chunk: its last row again, unused
    if (t0) finish(t0 - kTS, b ^ 1, gv[b ^ 1]);
    const int n = min(kTS, T - t0);
    float y[2][kTS];
    auto row = [&](int r) {
      const f32x4 v = bc[b][r][lane];
      const f32x2 x = *reinterpret_cast<const f32x2*>(&xd[b][wave][r][0]);
      const float a = ds[b][r];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        S[i].x = fmaf(a, S[i].x, x[i] * v.x);
        S[i].y = fmaf(a, S[i].y, x[i] * v.y);
        y[i][r] = fmaf(S[i].y, v.w, S[i].x * v.z);
      }
    };
    auto save = [&]() {
#pragma unroll
      for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x2*>(ssm + (size_t)dst_slab * slab + soff + i * kN) = S[i];
    };
    if (n == kTS && (V - 1 < t0 || V - 1 >= t0 + kTS - 1)) {
#pragma unroll
      for (int r = 0; r < kTS; ++r) row(r);
      if (V - 1 == t0 + kTS - 1) save();
    } else {
#pragma unroll
      for (int r = 0; r < kTS; ++r) {
        y[0][r] = y[1][r] = 0.0f;
        if (r < n) {                               // uniform
          row(r);
          if (t0 + r == V - 1) save();
        }
      }
    }
    // lane sums: after the swaps lanes 32 .. 63 hold state row 1's values and lane bit 4 the
    // upper 8 rows of the stage, then lane bits 3, 2, 1 a row each of what is left; lane bit 0
    // holds both halves of one sum
    float v[kTS], w[8], u[4], q2[2];
#pragma unroll
    for (int r = 0; r < kTS; ++r) {
      const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[0][r]), __float_as_uint(y[1][r]), false, false);
      v[r] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    }
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[r]), __float_as_uint(v[r + 8]), false, false);
      w[r] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = halve<0x140>(w[r], w[r + 4], lane & 8);    // row_mirror
#pragma unroll
    for (int r = 0; r < 2; ++r) q2[r] = halve<0x141>(u[r], u[r + 2], lane & 4);   // row_half_mirror
    float s1 = halve<0x4E>(q2[0], q2[1], lane & 2);                                // quad_perm [2, 3, 0, 1]
    s1 += dpp_f32<0xB1>(s1);                                                       // quad_perm [1, 0, 3, 2]
    {
      const int r = 8 * (lane >> 4 & 1) + 4 * (lane >> 3 & 1) + 2 * (lane >> 2 & 1) + (lane >> 1 & 1);
      const int c = pl + (lane >> 5);
      ys[b][r][c] = s1 + xs[b][r][c] * Dh;         // (two lanes write one value)
    }
    store(nx, b ^ 1);
    gv[b ^ 1] = nx.gv;
  };
  Regs r0, r1;
  load(r0, 0);
  load(r1, kTS);
  store(r0, 0);
  gv[0] = r0.gv;
  int t0 = 0;
  for (;;) {
    stage(t0, std::integral_constant<int, 0>{}, r1, r0);
    if (t0 + kTS >= T) break;
    t0 += kTS;
    stage(t0, std::integral_constant<int, 1>{}, r0, r1);
    if (t0 + kTS >= T) break;
    t0 += kTS;
  }
  __syncthreads();
  if ((t0 / kTS) & 1)
    finish(t0, 1, gv[1]);
  else
    finish(t0, 0, gv[0]);
}

// ------------------------------------------------------------------ attention
constexpr int kHD = 128;

// A bf16 pair with zeros in place of infinities and NaNs.
__device__ __forceinline__ uint32_t finite2(uint32_t v) {
  return ((v & 0x7F80u) == 0x7F80u ? 0u : v & 0xFFFFu) | ((v & 0x7F800000u) == 0x7F800000u ? 0u : v & 0xFFFF0000u);
}

__device__ __forceinline__ bool bad_pos(int P, int V, int64_t smax) { return P < 0 || P + (int64_t)V > smax; }

__global__ __launch_bounds__(256) void k_kv_append(const uint16_t* __restrict__ kv, int64_t ld,
                                                   uint16_t* __restrict__ kc, uint16_t* __restrict__ vc, int64_t smax,
                                                   const int32_t* __restrict__ pos, int T, int Ttot, int HKV,
                                                   int32_t* __restrict__ status) {
  const int P = *pos, V = valid_rows(P, Ttot, T);
  if (bad_pos(P, V, smax)) {
    if (blockIdx.x == 0 && threadIdx.x == 0 && status) atomicOr(status, (int32_t)HSD_STATUS_BAD_STATE);
    return;
  }
  // 16-byte pieces: [row][k heads | v heads][16]
  const int per = 2 * HKV * 16;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int r = (int)(i / per), rem = (int)(i - (int64_t)r * per);
  if (r >= V) return;
  const int h = rem >> 4, pc = rem & 15;
  const uint4 v = reinterpret_cast<const uint4*>(kv + (size_t)r * ld + h * kHD)[pc];
  uint16_t* dst = h < HKV ? kc + ((size_t)h * smax + P + r) * kHD : vc + ((size_t)(h - HKV) * smax + P + r) * kHD;
  reinterpret_cast<uint4*>(dst)[pc] = v;
}

// Workgroup: 32 query rows x 4 query heads of one kv head, a wavefront per head, so a
// 64-key tile of K and V is staged in LDS once for four heads. S^T = K Q^T (a lane then holds
// 32 keys of one query, so the softmax is per lane plus one half-wavefront exchange, and the
// probabilities are already a B operand), O^T = V^T P^T. The probabilities enter the second
// product as three bf16 parts (all 24 bits of the fp32 value), three MFMAs per fragment. K rows are stored with their 16-byte pieces
// swapped by (key % 16), V transposed with 8-byte pieces swapped by (dim / 2 % 16): no bank
// conflicts. The last query tiles have the most keys and are launched first. A masked key's
// probability is zero, which the product turns into NaN where its V is not finite: a tile that
// holds keys some row does not see (one or two per workgroup) is looked through for such values,
// and they are left out of the product and added to the rows that do see them.
__global__ __launch_bounds__(256, 2) void k_attn_prompt(const uint16_t* __restrict__ qkv, int64_t ld,
                                                        const uint16_t* __restrict__ kc,
                                                        const uint16_t* __restrict__ vc, int64_t smax,
                                                        const int32_t* __restrict__ pos, uint16_t* __restrict__ out,
                                                        int64_t out_ld, int T, int Ttot, int HQ, int HKV, float scale) {
  __shared__ __attribute__((aligned(16))) char ks[64 * 256];
  __shared__ __attribute__((aligned(16))) char vt[kHD * 128];
  const int P = *pos, V = valid_rows(P, Ttot, T);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = lane & 31, kh = lane >> 5;
  const int nq = (T + 31) / 32, nh = HQ / 4;
  const int qt = nq - 1 - (int)blockIdx.x / nh, hb = (int)blockIdx.x % nh;
  const int hq = 4 * hb + wave, hk = hq / (HQ / HKV), q0 = 32 * qt;
  if (bad_pos(P, V, smax)) {   // flagged by k_kv_append; the rows' outputs are zero
    for (int i = tid; i < 32 * 64; i += 256) {
      const int r = q0 + (i >> 6);
      if (r < T) reinterpret_cast<uint4*>(out + (size_t)r * out_ld + hb * 4 * kHD)[i & 63] = make_uint4(0, 0, 0, 0);
    }
    return;
  }
  // keys 0 .. last are visible to some row of this tile; nothing past the prompt is read
  const int last = min(P + min(q0 + 31, max(V, 1) - 1), (int)smax - 1);
  const int ntile = last / 64 + 1;
  bf16x8 qf[8];
  {
    const uint16_t* qr = qkv + (size_t)min(q0 + j, T - 1) * ld + hq * kHD + 8 * kh;
#pragma unroll
    for (int s = 0; s < 8; ++s) qf[s] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(qr + 16 * s));
  }
  const uint16_t* kb = kc + (size_t)hk * smax * kHD;
  const uint16_t* vb = vc + (size_t)hk * smax * kHD;
  u32x4 kr[4], vr[2][2];
  auto load = [&](int t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {   // K: 16 keys per pass, 16 pieces each
      const int key = min(64 * t + 16 * i + (tid >> 4), last);
      kr[i] = reinterpret_cast<const u32x4*>(kb + (size_t)key * kHD)[tid & 15];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)     // V: key pair tid % 32, dims 8 (tid / 32 + 8 i) ..
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int key = min(64 * t + 2 * (tid & 31) + u, last);
        vr[i][u] = reinterpret_cast<const u32x4*>(vb + (size_t)key * kHD)[(tid >> 5) + 8 * i];
      }
  };
  f32x16 o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[d][v] = 0.0f;
  float m = -INFINITY, l = 0.0f;
  const int qpos = P + q0 + j;
  load(0);
  for (int t = 0; t < ntile; ++t) {
    __syncthreads();                                 // the previous tile has been read
    const bool diag = 64 * t + 63 > P + q0;          // uniform: a key that row q0 does not see
    bool odd = false;                                // a value of this thread's that is not finite
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = 16 * i + (tid >> 4);
      *reinterpret_cast<u32x4*>(ks + 256 * key + 16 * ((tid & 15) ^ (key & 15))) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int kp = tid & 31, d0 = 8 * ((tid >> 5) + 8 * i);
      const bool l0 = 64 * t + 2 * kp <= last, l1 = 64 * t + 2 * kp + 1 <= last;
      const uint32_t w0[4] = {vr[i][0].x, vr[i][0].y, vr[i][0].z, vr[i][0].w};
      const uint32_t w1[4] = {vr[i][1].x, vr[i][1].y, vr[i][1].z, vr[i][1].w};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        uint32_t a0 = l0 ? w0[c] : 0u, a1 = l1 ? w1[c] : 0u;
        if (diag) {
          const uint32_t f0 = finite2(a0), f1 = finite2(a1);
          odd = odd || f0 != a0 || f1 != a1;
          a0 = f0;
          a1 = f1;
        }
        const int d = d0 + 2 * c;                     // dims d, d + 1 share (d / 2)
        const int pc = (kp >> 1) ^ ((d >> 1) & 15);
        *reinterpret_cast<uint32_t*>(vt + 128 * d + 8 * pc + 4 * (kp & 1)) = (a0 & 0xFFFFu) | (a1 << 16);
        *reinterpret_cast<uint32_t*>(vt + 128 * (d + 1) + 8 * pc + 4 * (kp & 1)) = (a0 >> 16) | (a1 & 0xFFFF0000u);
      }
    }
    bool repair = false;                             // uniform
    if (diag)
      repair = __syncthreads_or(odd);
    else
      __syncthreads();
    load(t + 1);                                     // past the last tile: its last key, unused
    f32x16 s[2] = {};
#pragma unroll
    for (int st = 0; st < 8; ++st)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int key = 32 * b + j;
        const bf16x8 kf = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const uint4*>(ks + 256 * key + 16 * ((2 * st + kh) ^ (key & 15))));
        s[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[st], s[b], 0, 0, 0);
      }
    float mx = -INFINITY;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int key = 64 * t + 32 * b + 8 * (v >> 2) + 4 * kh + (v & 3);
        s[b][v] = key <= qpos ? s[b][v] * scale : -INFINITY;
        mx = fmaxf(mx, s[b][v]);
      }
    {
      const uint32_t c = __float_as_uint(mx);
      const auto pp = __builtin_amdgcn_permlane32_swap(c, c, false, false);
      mx = fmaxf(__uint_as_float(pp[0]), __uint_as_float(pp[1]));
    }
    const float mn = fmaxf(m, mx);                   // finite from the first tile on: key 0 is visible
    const float corr = __expf(m - mn);
    m = mn;
    l *= corr;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[d][v] *= corr;
    bf16x8 ph[4], pm[4], pl[4];                      // 16-key steps: registers 8 (st % 2) .. of block st / 2
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        const float pv = __expf(s[st >> 1][8 * (st & 1) + v] - mn);
        l += pv;
        const __bf16 hi = (__bf16)pv;
        ph[st][v] = hi;
        const float rest = pv - (float)hi;
        const __bf16 mid = (__bf16)rest;
        pm[st][v] = mid;
        pl[st][v] = (__bf16)(rest - (float)mid);
      }
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const int dim = 32 * d + j, sw = (dim >> 1) & 15;
        const uint2 v0 = *reinterpret_cast<const uint2*>(vt + 128 * dim + 8 * ((4 * st + kh) ^ sw));
        const uint2 v1 = *reinterpret_cast<const uint2*>(vt + 128 * dim + 8 * ((4 * st + 2 + kh) ^ sw));
        const bf16x8 vf = __builtin_bit_cast(bf16x8, make_uint4(v0.x, v0.y, v1.x, v1.y));
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, ph[st], o[d], 0, 0, 0);
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pm[st], o[d], 0, 0, 0);
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pl[st], o[d], 0, 0, 0);
      }
    if (repair) {
#pragma unroll 1
      for (int key = 64 * t; key <= min(64 * t + 63, last); ++key)
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const uint2 w = *reinterpret_cast<const uint2*>(vb + (size_t)key * kHD + 32 * d + 8 * b + 4 * kh);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const uint32_t x = ((u < 2 ? w.x : w.y) >> (16 * (u & 1))) & 0xFFFFu;
              if ((x & 0x7F80u) == 0x7F80u && key <= qpos) o[d][4 * b + u] += bf16_bits_to_f32(x);
            }
          }
    }
  }
  {
    const uint32_t c = __float_as_uint(l);
    const auto pp = __builtin_amdgcn_permlane32_swap(c, c, false, false);
    l = __uint_as_float(pp[0]) + __uint_as_float(pp[1]);
  }
  if (q0 + j < T) {
    const float inv = 1.0f / l;
    uint16_t* orow = out + (size_t)(q0 + j) * out_ld + hq * kHD;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        uint32_t w[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
          w[u] = (uint32_t)f32_to_bf16_bits(o[d][4 * b + 2 * u] * inv) |
                 ((uint32_t)f32_to_bf16_bits(o[d][4 * b + 2 * u + 1] * inv) << 16);
        *reinterpret_cast<uint2*>(orow + 32 * d + 8 * b + 4 * kh) = make_uint2(w[0], w[1]);
      }
  }
}

// ------------------------------------------------------------------ sequence
// dst[i] = prompt[clamp(POS + offset + i)]
__global__ void k_prompt_tokens(const int32_t* __restrict__ src, int n, const int32_t* __restrict__ seq, int offset,
                                int count, int32_t* __restrict__ dst) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < count) dst[i] = src[min(max(seq[HSD_SEQ_POS] + offset + i, 0), n - 1)];
}

__global__ void k_prompt_advance(int32_t* seq, int T, int B, int nslab) {
  if (threadIdx.x == 0) {
    const int p = seq[HSD_SEQ_POS], valid = valid_rows(p, T, B);
    seq[HSD_SEQ_POS] = p + valid;
    if (nslab > 0) seq[HSD_SEQ_CUR] = (seq[HSD_SEQ_CUR] + valid) % nslab;
    seq[HSD_SEQ_HEAD_POS] += valid_rows(p, T - 1, B);
  }
}

}  // namespace
}  // namespace hsd

using namespace hsd;

extern "C" size_t hsd_mamba_scan_workspace_bytes(int64_t T, int64_t H, int64_t P, int64_t N, int64_t G) {
  if (T <= 0 || H <= 0 || P <= 0 || N <= 0 || G <= 0) return 0;
  return (size_t)T * (H * P + 2 * G * N + 2 * H) * sizeof(float);
}

extern "C" int hsd_mamba_scan(const uint16_t* conv_in, int64_t conv_in_ld, const uint16_t* dt_raw, int64_t dt_ld,
                              const uint16_t* gate, int64_t gate_ld, const uint16_t* conv_w, const uint16_t* conv_b,
                              const float* A_log, const float* dt_bias, const float* Dp, float* ssm_slabs,
                              uint16_t* conv_slabs, const int32_t* cur, int64_t nslab, const int32_t* pos, float* z,
                              int64_t z_ld, int64_t T, int64_t Ttot, int64_t H, int64_t P, int64_t N, int64_t G,
                              float dt_lo, float dt_hi, int32_t* dev_status, void* workspace, size_t workspace_bytes,
                              void* stream) {
  const char* fn = "hsd_mamba_scan";
  if (!conv_in || !dt_raw || !gate || !conv_w || !conv_b || !A_log || !dt_bias || !Dp || !ssm_slabs || !conv_slabs ||
      !cur || !pos || !z)
    return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  const int64_t DI = H * P, CD = DI + 2 * G * N;
  // k_conv_rows has T / kCR in grid.y
  if (T < 1 || T > 65535 * kCR || Ttot < 0 || Ttot > 0x7FFFFFFF || H <= 0 || G <= 0 || H % G || H > 65535 || P <= 0 ||
      P % kPB || N != kN || nslab < 1 || nslab > 64 || CD % 8)
    return set_error(HSD_ERR_SHAPE, "%s: need T <= %d, N == %d, P %% %d == 0, H %% G == 0", fn, 65535 * kCR, kN, kPB);
  if (conv_in_ld < CD || dt_ld < H || gate_ld < DI || z_ld < DI + DI / 16)
    return set_error(HSD_ERR_SHAPE, "%s: bad row strides", fn);
  if (((uintptr_t)conv_in | (uintptr_t)conv_w | (uintptr_t)conv_b | (uintptr_t)conv_slabs | (uintptr_t)ssm_slabs |
       (uintptr_t)workspace) & 15u || conv_in_ld % 8)
    return set_error(HSD_ERR_ALIGN, "%s: 16-byte aligned pointers and row strides", fn);
  if (!workspace || workspace_bytes < hsd_mamba_scan_workspace_bytes(T, H, P, N, G))
    return set_error(HSD_ERR_WORKSPACE, "%s: workspace too small", fn);
  float* co = reinterpret_cast<float*>(workspace);
  float* dtA = co + (size_t)T * CD;
  hipStream_t st = as_stream(stream);
  const unsigned cb = (unsigned)((CD / 8 + 255) / 256);
  hipLaunchKernelGGL(k_conv_rows, dim3(cb + 1, (unsigned)((T + kCR - 1) / kCR)), dim3(256), 0, st, conv_in, conv_in_ld,
                     dt_raw, dt_ld, conv_w, conv_b, A_log, dt_bias, conv_slabs, cur, (int)nslab, co, dtA, (int)T, (int)CD,
                     (int)H, dt_lo, dt_hi);
  int rc = check_launch(fn);
  if (rc) return rc;
  hipLaunchKernelGGL(k_scan, dim3((unsigned)(H * (P / kPB))), dim3(64 * kSW), 0, st, co, dtA, conv_in, conv_in_ld, gate, gate_ld,
                     Dp, ssm_slabs, conv_slabs, cur, pos, (int)nslab, z, z_ld, (int)T, (int)Ttot, (int)H, (int)P, (int)G,
                     dev_status);
  return check_launch(fn);
}

extern "C" int hsd_kv_append(const uint16_t* kv, int64_t kv_ld, int64_t T, int64_t Ttot, uint16_t* k_cache,
                             uint16_t* v_cache, int64_t smax, const int32_t* pos, int64_t HKV, int64_t HD,
                             int32_t* dev_status, void* stream) {
  const char* fn = "hsd_kv_append";
  if (!kv || !k_cache || !v_cache || !pos) return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  if (T < 1 || T > (1 << 20) || Ttot < 0 || Ttot > 0x7FFFFFFF || HD != kHD || HKV <= 0 || HKV > 4096 || smax < 1 ||
      smax > (1 << 24) || kv_ld < 2 * HKV * HD || kv_ld % 8)
    return set_error(HSD_ERR_SHAPE, "%s: bad sizes", fn);
  if (((uintptr_t)kv | (uintptr_t)k_cache | (uintptr_t)v_cache) & 15u)
    return set_error(HSD_ERR_ALIGN, "%s: 16-byte aligned pointers", fn);
  const int64_t pieces = T * 2 * HKV * 16;
  hipLaunchKernelGGL(k_kv_append, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, as_stream(stream), kv, kv_ld, k_cache,
                     v_cache, smax, pos, (int)T, (int)Ttot, (int)HKV, dev_status);
  return check_launch(fn);
}

extern "C" int hsd_attn_prompt(const uint16_t* qkv, int64_t qkv_ld, int64_t T, int64_t Ttot, uint16_t* k_cache,
                               uint16_t* v_cache, int64_t smax, const int32_t* pos, uint16_t* out, int64_t out_ld,
                               int64_t HQ, int64_t HKV, int64_t HD, float scale, int32_t* dev_status, void* stream) {
  const char* fn = "hsd_attn_prompt";
  if (!qkv || !k_cache || !v_cache || !pos || !out) return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  if (T < 1 || T > (1 << 20) || Ttot < 0 || Ttot > 0x7FFFFFFF || HD != kHD || HKV <= 0 || HQ <= 0 || HQ % HKV ||
      (HQ / HKV) % 4 || smax < 1 || smax > (1 << 24))
    return set_error(HSD_ERR_SHAPE, "%s: need head dim %d and a multiple of 4 query heads per kv head", fn, kHD);
  if (qkv_ld < (HQ + 2 * HKV) * HD || qkv_ld % 8 || out_ld < HQ * HD || out_ld % 8)
    return set_error(HSD_ERR_SHAPE, "%s: bad row strides", fn);
  if (((uintptr_t)qkv | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) & 15u)
    return set_error(HSD_ERR_ALIGN, "%s: 16-byte aligned pointers", fn);
  hipStream_t st = as_stream(stream);
  const int rc = hsd_kv_append(qkv + HQ * HD, qkv_ld, T, Ttot, k_cache, v_cache, smax, pos, HKV, HD, dev_status, stream);
  if (rc) return rc;
  hipLaunchKernelGGL(k_attn_prompt, dim3((unsigned)((T + 31) / 32 * (HQ / 4))), dim3(256), 0, st, qkv, qkv_ld, k_cache,
                     v_cache, smax, pos, out, out_ld, (int)T, (int)Ttot, (int)HQ, (int)HKV, scale);
  return check_launch(fn);
}

extern "C" int hsd_prompt_tokens(const int32_t* src, int64_t n, const int32_t* seq, int64_t offset, int64_t count,
                                 int32_t* dst, void* stream) {
  if (!src || !seq || !dst) return set_error(HSD_ERR_ARG, "hsd_prompt_tokens: null pointer");
  if (n < 1 || n > 0x7FFFFFFF || count < 1 || count > (1 << 24) || offset < -(1 << 30) || offset > (1 << 30))
    return set_error(HSD_ERR_SHAPE, "hsd_prompt_tokens: bad sizes");
  hipLaunchKernelGGL(k_prompt_tokens, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, as_stream(stream), src, (int)n,
                     seq, (int)offset, (int)count, dst);
  return check_launch("hsd_prompt_tokens");
}

extern "C" int hsd_prompt_advance(int32_t* seq, int64_t T, int64_t B, int64_t nslab, void* stream) {
  if (!seq) return set_error(HSD_ERR_ARG, "hsd_prompt_advance: null pointer");
  if (T < 0 || T > 0x7FFFFFFF || B < 1 || B > (1 << 24) || nslab < 0 || nslab > 64)
    return set_error(HSD_ERR_SHAPE, "hsd_prompt_advance: bad sizes");
  hipLaunchKernelGGL(k_prompt_advance, dim3(1), dim3(64), 0, as_stream(stream), seq, (int)T, (int)B, (int)nslab);
  return check_launch("hsd_prompt_advance");
}

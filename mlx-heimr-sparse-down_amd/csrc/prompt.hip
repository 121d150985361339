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
#include "hsd_common.h"

namespace hsd {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
// staging registers that go from global memory to LDS unread (an array of the HIP vector
// structs copied like that stays in scratch memory)
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
// The arithmetic of a row is k_mamba_ssm's (the same fma, product and lane order), so the
// states and z equal a row-by-row run's. Workgroup = (head, 16 state rows); wavefront w owns
// state rows 4w .. 4w+3, 16 lanes per row with 8 state elements each, for all rows of the
// chunk. kTS rows' inputs are staged in LDS at a time, the next ones in registers meanwhile.
// Bound by the vector unit's issue (about 30 instructions per row and wavefront, one
// wavefront per SIMD): rows are a serial chain of one fma.
constexpr int kTS = 16;
__global__ __launch_bounds__(256, 1) void k_scan(
    const float* __restrict__ co, const float* __restrict__ dtA, const uint16_t* __restrict__ cin, int64_t cin_ld,
    const uint16_t* __restrict__ gate, int64_t gate_ld, const float* __restrict__ Dp, float* __restrict__ ssm,
    uint16_t* __restrict__ convs, const int32_t* __restrict__ cur_ptr, const int32_t* __restrict__ pos, int nslab,
    float* __restrict__ z, int64_t z_ld, int T, int Ttot, int H, int P, int G, int32_t* __restrict__ status) {
  // a lane's 8 B (C) elements as two float4, the 16 lanes' first ones, then their second
  // ones: consecutive lanes read consecutive 16 bytes (no bank conflicts)
  __shared__ __attribute__((aligned(16))) f32x4 Bs[2][kTS][2][kN / 8], Cs[2][kTS][2][kN / 8];
  __shared__ __attribute__((aligned(16))) float xs[2][kTS][kPB];
  __shared__ float ds[2][kTS][2];
  __shared__ float ys[kTS][kPB + 1];
  const int npb = P / kPB, lb = xcd_remap((int)blockIdx.x, H * npb);
  const int hh = lb / npb, pblk = lb - hh * npb, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int DI = H * P, GN = G * kN, CD = DI + 2 * GN, hpg = H / G, g = hh / hpg;
  const int cur = *cur_ptr, V = valid_rows(*pos, Ttot, T);
  const float Dh = bf16_bits_to_f32(f32_to_bf16_bits(Dp[hh]));
  if ((unsigned)cur >= (unsigned)nslab) {
    for (int i = tid; i < T * kPB; i += 256)
      z[(size_t)(i / kPB) * z_ld + (size_t)hh * P + pblk * kPB + i % kPB] = __int_as_float(0x7FC00000);
    for (int i = tid; i < T; i += 256) z[(size_t)i * z_ld + DI + (size_t)hh * npb + pblk] = __int_as_float(0x7FC00000);
    if (tid == 0 && status) atomicOr(status, (int32_t)HSD_STATUS_BAD_STATE);
    return;
  }
  const int dst_slab = (cur + V) % nslab;
  // the conv window after row V - 1: this workgroup's 16 channels, and its group's B and C
  // channels in one workgroup per group; every read of the old window precedes the writes
  const bool owner = (hh % hpg == 0) && pblk == 0;
  if (V > 0) {
    const int nch = owner ? kPB + 2 * kN : kPB;
    uint16_t wv[2][kK - 1];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = min(tid + 256 * u, nch - 1);
      const int ch = t < kPB ? hh * P + pblk * kPB + t
                             : t < kPB + kN ? DI + g * kN + (t - kPB) : DI + GN + g * kN + (t - kPB - kN);
#pragma unroll
      for (int i = 0; i < kK - 1; ++i) {
        const int r = V - (kK - 1) + i;
        wv[u][i] = r < 0 ? convs[((size_t)cur * (kK - 1) + r + kK - 1) * CD + ch] : cin[(size_t)r * cin_ld + ch];
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = tid + 256 * u;
      if (t < nch) {
        const int ch = t < kPB ? hh * P + pblk * kPB + t
                               : t < kPB + kN ? DI + g * kN + (t - kPB) : DI + GN + g * kN + (t - kPB - kN);
#pragma unroll
        for (int i = 0; i < kK - 1; ++i) convs[((size_t)dst_slab * (kK - 1) + i) * CD + ch] = wv[u][i];
      }
    }
  }
  const int ri = lane >> 4, c8 = lane & 15, pl = 4 * wave + ri, p = pblk * kPB + pl;
  const size_t slab = (size_t)H * P * kN, soff = ((size_t)hh * P + p) * kN + 8 * c8;
  float4 S0 = *reinterpret_cast<const float4*>(ssm + (size_t)cur * slab + soff);
  float4 S1 = *reinterpret_cast<const float4*>(ssm + (size_t)cur * slab + soff + 4);

  // staging: 16 rows x (32 + 32 float4 of B and C, 4 of x) and (dt, exp(A dt))
  f32x4 rb[4], rx;
  float rd;
  uint16_t gv;
  auto load = [&](int t0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + 256 * i, r = min(t0 + (idx >> 6), T - 1), q = idx & 63;
      rb[i] = *reinterpret_cast<const f32x4*>(co + (size_t)r * CD + DI + (q < 32 ? 0 : GN) + g * kN + 4 * (q & 31));
    }
    rx = *reinterpret_cast<const f32x4*>(co + (size_t)min(t0 + (tid >> 2 & 15), T - 1) * CD + (size_t)hh * P + pblk * kPB +
                                          4 * (tid & 3));
    rd = dtA[(size_t)min(t0 + (tid >> 1 & 15), T - 1) * 2 * H + (tid & 1) * H + hh];
    gv = gate[(size_t)min(t0 + (tid >> 4), T - 1) * gate_ld + (size_t)hh * P + pblk * kPB + (tid & 15)];
  };
  auto store = [&](int b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = tid + 256 * i, r = idx >> 6, q = idx & 63;
      (q < 32 ? Bs[b][r][q & 1] : Cs[b][r][q & 1])[(q & 31) >> 1] = rb[i];
    }
    if (tid < 64) *reinterpret_cast<f32x4*>(&xs[b][tid >> 2][4 * (tid & 3)]) = rx;
    if (tid < 32) ds[b][tid >> 1][tid & 1] = rd;
  };
  load(0);
  store(0);
  int b = 0;
  for (int t0 = 0; t0 < T; t0 += kTS, b ^= 1) {
    const uint16_t gcur = gv;
    __syncthreads();                               // stage b in LDS, ys read
    load(t0 + kTS);                                // past the chunk: its last row again, unused
    const int n = min(kTS, T - t0);
    float yk = 0.0f;
    // a row's inputs; the next kPF rows' are read while kPF rows are computed (one wavefront
    // per SIMD: nothing else hides the LDS latency)
    struct In {
      f32x4 B0, B1, C0, C1;
      float x, dt, a;
    };
    auto fetch = [&](In& v, int r) {
      v.B0 = Bs[b][r][0][c8];
      v.B1 = Bs[b][r][1][c8];
      v.C0 = Cs[b][r][0][c8];
      v.C1 = Cs[b][r][1][c8];
      v.x = xs[b][r][pl];
      v.dt = ds[b][r][0];
      v.a = ds[b][r][1];
    };
    auto row = [&](const In& v, int r) {
      const f32x4 B0 = v.B0, B1 = v.B1, C0 = v.C0, C1 = v.C1;
      const float xdt = v.x * v.dt, a = v.a;
      S0.x = fmaf(a, S0.x, xdt * B0.x);
      S0.y = fmaf(a, S0.y, xdt * B0.y);
      S0.z = fmaf(a, S0.z, xdt * B0.z);
      S0.w = fmaf(a, S0.w, xdt * B0.w);
      S1.x = fmaf(a, S1.x, xdt * B1.x);
      S1.y = fmaf(a, S1.y, xdt * B1.y);
      S1.z = fmaf(a, S1.z, xdt * B1.z);
      S1.w = fmaf(a, S1.w, xdt * B1.w);
      float y = S0.x * C0.x;
      y = fmaf(S0.y, C0.y, y);
      y = fmaf(S0.z, C0.z, y);
      y = fmaf(S0.w, C0.w, y);
      y = fmaf(S1.x, C1.x, y);
      y = fmaf(S1.y, C1.y, y);
      y = fmaf(S1.z, C1.z, y);
      y = fmaf(S1.w, C1.w, y);
      y += dpp_f32<0xB1>(y);
      y += dpp_f32<0x4E>(y);
      y += dpp_f32<0x141>(y);
      y += dpp_f32<0x140>(y);
      yk = c8 == r ? y : yk;                       // lane c8 keeps row c8's (a select, no branch per row)
    };
    auto save = [&]() {
      float* dst = ssm + (size_t)dst_slab * slab + soff;
      *reinterpret_cast<float4*>(dst) = S0;
      *reinterpret_cast<float4*>(dst + 4) = S1;
    };
    if (n == kTS && (V - 1 < t0 || V - 1 >= t0 + kTS - 1)) {
      constexpr int kPF = 4;
      In in[2][kPF];
#pragma unroll
      for (int u = 0; u < kPF; ++u) fetch(in[0][u], u);
#pragma unroll
      for (int r0 = 0; r0 < kTS; r0 += kPF) {
#pragma unroll
        for (int u = 0; u < kPF; ++u)
          if (r0 + kPF < kTS) fetch(in[(r0 / kPF + 1) & 1][u], r0 + kPF + u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kPF; ++u) row(in[(r0 / kPF) & 1][u], r0 + u);
      }
      if (V - 1 == t0 + kTS - 1) save();
    } else {
      for (int r = 0; r < n; ++r) {
        In v;
        fetch(v, r);
        row(v, r);
        if (t0 + r == V - 1) save();
      }
    }
    ys[c8][pl] = yk + xs[b][c8][pl] * Dh;
    __syncthreads();                               // ys complete
    {
      const int r = tid >> 4, c = tid & 15;
      float v = ys[r][c] * silu_f32(bf16_bits_to_f32(gcur));
      if (r < n) z[(size_t)(t0 + r) * z_ld + (size_t)hh * P + pblk * kPB + c] = v;
      // the 16 channels' sum of z^2 in channel order, lane 15 of each row
      v = v * v;
      float s = __shfl(v, lane & 48, 64);
#pragma unroll
      for (int i = 1; i < kPB; ++i) s += __shfl(v, (lane & 48) + i, 64);
      if (c == 0 && r < n) z[(size_t)(t0 + r) * z_ld + DI + (size_t)hh * npb + pblk] = s;
    }
    store(b ^ 1);
  }
}

// ------------------------------------------------------------------ attention
constexpr int kHD = 128;

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
// conflicts. The last query tiles have the most keys and are launched first.
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
        const uint32_t a0 = l0 ? w0[c] : 0u, a1 = l1 ? w1[c] : 0u;
        const int d = d0 + 2 * c;                     // dims d, d + 1 share (d / 2)
        const int pc = (kp >> 1) ^ ((d >> 1) & 15);
        *reinterpret_cast<uint32_t*>(vt + 128 * d + 8 * pc + 4 * (kp & 1)) = (a0 & 0xFFFFu) | (a1 << 16);
        *reinterpret_cast<uint32_t*>(vt + 128 * (d + 1) + 8 * pc + 4 * (kp & 1)) = (a0 >> 16) | (a1 & 0xFFFF0000u);
      }
    }
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
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pl[st], o[d], 0, 0, 0);
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
        o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pm[st], o[d], 0, 0, 0);
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
  if (T < 1 || T > (1 << 20) || Ttot < 0 || Ttot > 0x7FFFFFFF || H <= 0 || G <= 0 || H % G || H > 65535 || P <= 0 ||
      P % kPB || N != kN || nslab < 1 || nslab > 64 || CD % 8)
    return set_error(HSD_ERR_SHAPE, "%s: need N == %d, P %% %d == 0, H %% G == 0", fn, kN, kPB);
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
  hipLaunchKernelGGL(k_scan, dim3((unsigned)(H * (P / kPB))), dim3(256), 0, st, co, dtA, conv_in, conv_in_ld, gate, gate_ld,
                     Dp, ssm_slabs, conv_slabs, cur, pos, (int)nslab, z, z_ld, (int)T, (int)Ttot, (int)H, (int)P, (int)G,
                     dev_status);
  return check_launch(fn);
}

extern "C" int hsd_attn_prompt(const uint16_t* qkv, int64_t qkv_ld, int64_t T, int64_t Ttot, uint16_t* k_cache,
                               uint16_t* v_cache, int64_t smax, const int32_t* pos, uint16_t* out, int64_t out_ld,
                               int64_t HQ, int64_t HKV, int64_t HD, float scale, int32_t* dev_status, void* stream) {
  const char* fn = "hsd_attn_prompt";
  if (!qkv || !k_cache || !v_cache || !pos) return set_error(HSD_ERR_ARG, "%s: null pointer", fn);
  if (T < 1 || T > (1 << 20) || Ttot < 0 || Ttot > 0x7FFFFFFF || HD != kHD || HKV <= 0 || HQ <= 0 || HQ % HKV ||
      (HQ / HKV) % 4 || smax < 1 || smax > (1 << 24))
    return set_error(HSD_ERR_SHAPE, "%s: need head dim %d and a multiple of 4 query heads per kv head", fn, kHD);
  if (qkv_ld < (HQ + 2 * HKV) * HD || qkv_ld % 8 || (out && (out_ld < HQ * HD || out_ld % 8)))
    return set_error(HSD_ERR_SHAPE, "%s: bad row strides", fn);
  if (((uintptr_t)qkv | (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)out) & 15u)
    return set_error(HSD_ERR_ALIGN, "%s: 16-byte aligned pointers", fn);
  hipStream_t st = as_stream(stream);
  const int64_t pieces = T * 2 * HKV * 16;
  hipLaunchKernelGGL(k_kv_append, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, st, qkv + HQ * HD, qkv_ld, k_cache,
                     v_cache, smax, pos, (int)T, (int)Ttot, (int)HKV, dev_status);
  const int rc = check_launch(fn);
  if (rc || !out) return rc;
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

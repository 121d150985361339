// 4-bit products of a prompt chunk with the rows held in registers: y = x W^T for tiles of 32
// token rows, W streamed once past each tile (hsd_gemm_q4 and hsd_moe_up_gemm; the ring kernel
// of gemm.hip takes what this one does not).
#include "hsd_common.h"

#include "gemm.h"

namespace hsd {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void_t;

constexpr uint32_t kBf16Two = 0x41804180u;  // bf16 pair (16, 16): | nibble << 3 is 16 + q
constexpr uint32_t kNibHi = 0x00780078u;
constexpr int kWv = 8;                      // wavefronts per workgroup

__device__ __forceinline__ bf16x8 unpack(uint32_t x, uint32_t nibm) {
  return __builtin_bit_cast(bf16x8, u32x4{((x << 3) & nibm) | kBf16Two, ((x >> 1) & nibm) | kBf16Two,
                                          ((x >> 5) & nibm) | kBf16Two, ((x >> 9) & nibm) | kBf16Two});
}

// Eight bf16 values (in the low halves) as an MFMA operand.
__device__ __forceinline__ bf16x8 pack8(const uint32_t (&v)[8]) {
  return __builtin_bit_cast(bf16x8, u32x4{v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16});
}

// One workgroup per CU walks a contiguous run of (tile, output block) units, tile by tile. Its
// 8 wavefronts split the inputs: wavefront w holds its eighth of the tile's 32 rows as MFMA A
// fragments in registers (up to kNG groups of 64 inputs x 16 registers) for the whole tile, and
// per 32-output block reads its eighth of the block's nibbles straight into registers: each
// group's next ones as soon as the group has left them, so nearly a whole block ahead. A weight
// byte is read once per 32 rows, in runs whose eight readers share the DRAM page, nothing of
// it passes LDS, and a block costs one barrier, for the sum of the eight partial products. (Four
// wavefronts of twice the inputs do not fit: the rows' registers went to the accumulator file
// and back before every MFMA.) The arithmetic is k_gemm_q4's (gemm.hip): per group acc = sum x
// (16 + q), y += s acc in fp32, and the group sums times b - 16 s; the eighths are added in
// order. 128 experts' up projections: 64 rows 117 -> 98 us, 512 rows 161 -> 139 us against the
// ring kernel, whose waits on 64-byte pieces of 256 rows they replace.
constexpr int kNG = 6;
template <int MODE>
__global__ __launch_bounds__(64 * kWv, 2) void k_gemm_rows(GemmArgs a) {
  constexpr int UB = MODE == kUpRelu2 ? 2 : 1;       // blocks of 32 outputs per unit
  __shared__ __attribute__((aligned(16))) f32x2 red[2][kWv][64][8];
  __shared__ __attribute__((aligned(16))) uint16_t sbuf[2][2][32 * 64];   // scales, biases of a block
  __shared__ int drow[32], srow[32];
  __shared__ float hpart[32];       // kUpRelu2: the group sums of a unit's first block
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, kh = lane >> 5;
  const int I = a.I, G = I / 64;
  // this wavefront's groups
  const int base = G / kWv, rem = G % kWv, cnt = base + (wave < rem ? 1 : 0), g0 = wave * base + min(wave, rem);

  // ---- this workgroup's units
  const int unF = MODE == kUpRelu2 ? a.F / 64 : (a.O + 31) / 32, unS = MODE == kUpRelu2 ? a.FS / 64 : 0;
  int nr, ns = 0;
  if constexpr (MODE == kUpRelu2) {
    nr = min(max(*a.ntiles, 0), a.nt_routed);
    ns = a.nt_shared;
  } else {
    nr = (a.T + 31) / 32;
  }
  const int64_t total = (int64_t)nr * unF + (int64_t)ns * unS;
  const int wg = xcd_remap((int)blockIdx.x, a.grid);
  const int64_t u1 = total * (wg + 1) / a.grid;
  int64_t u = total * wg / a.grid;
  const uint32_t nibm = opaque_vgpr(kNibHi);

  while (u < u1) {
    // ---- the run's next tile: units u .. of it
    const bool sh = MODE == kUpRelu2 && u < (int64_t)ns * unS;
    const int64_t v = MODE == kUpRelu2 && !sh ? u - (int64_t)ns * unS : u;
    const int un = sh ? unS : unF;
    const int t = (int)(v / un), f0 = (int)(v - (int64_t)t * un);
    const int f1 = (int)min((int64_t)un, f0 + (u1 - u));
    u += f1 - f0;
    const uint32_t* w = a.w;
    const uint16_t* sp = a.s;
    const uint16_t* bp = a.b;
    int O = a.O;
    const int32_t* ts = nullptr;
    int slot;                       // this lane's tile row: token (or slot) index, -1 past the end
    if constexpr (MODE == kUpRelu2) {
      const int tile = sh ? a.nt_routed + t : t, e = __builtin_amdgcn_readfirstlane(a.tile_e[tile]);
      O = sh ? a.FS : a.F;
      if (sh) {
        w = a.sw; sp = a.ss; bp = a.sb;
      } else {
        if ((unsigned)e >= (unsigned)a.E) continue;
        w += (size_t)e * O * (I / 8);
        sp += (size_t)e * O * G;
        bp += (size_t)e * O * G;
      }
      ts = a.tile_slot + (size_t)tile * 32;
      slot = ts[j];
    } else {
      slot = 32 * t + j < a.T ? 32 * t + j : -1;
    }
    const int row = slot < 0 ? 0 : MODE == kUpRelu2 && !sh ? slot / a.topk : slot;
    __syncthreads();                // the previous tile's epilogue has read drow and the buffers
    if (tid < 32) {
      if constexpr (MODE == kUpRelu2) {
        const int NR = a.topk * a.F + a.FS, k = sh ? a.topk : max(slot, 0) % a.topk;
        drow[tid] = slot < 0 ? -1 : row * NR + k * a.F;
        srow[tid] = row * (a.topk + 1) + k;
      } else {
        drow[tid] = slot;
      }
    }

    // ---- a block's loads: its scales and biases (4 G pieces of 16 bytes each, one per
    // thread), then this wavefront's nibbles (outputs past the last one re-read it, groups past
    // the wavefront's last re-read one and are multiplied as zeros)
    u32x4 sv, bv, bw[kNG];
    const int b1 = f1 * UB;
    auto load_scales = [&](int blk) {
      const int n0 = 32 * blk, np = min(32, O - n0) * G / 8;
      const int p = min(tid, np - 1);
      sv = reinterpret_cast<const u32x4*>(sp + (size_t)n0 * G)[p];
      bv = reinterpret_cast<const u32x4*>(bp + (size_t)n0 * G)[p];
    };
    auto store_scales = [&](int buf) {
      if (tid < 4 * G) {
        reinterpret_cast<u32x4*>(sbuf[buf][0])[tid] = sv;
        reinterpret_cast<u32x4*>(sbuf[buf][1])[tid] = bv;
      }
    };
    auto words = [&](int blk) { return w + (size_t)min(32 * blk + j, O - 1) * (I / 8) + 4 * kh; };
    auto load_word = [&](const uint32_t* src, int g) {
      bw[g] = *reinterpret_cast<const u32x4*>(src + 8 * min(g0 + g, G - 1));
    };
    load_scales(f0 * UB);
    // the tile's rows and group sums
    bf16x8 av[kNG][4], hf, h3;
    {
      const uint16_t* xr = a.xp + (size_t)row * I + 32 * kh;
#pragma unroll
      for (int g = 0; g < kNG; ++g)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          av[g][q] = *reinterpret_cast<const bf16x8*>(xr + 64 * min(g0 + g, G - 1) + 8 * q);
      // lane half 0: the sums' first parts, half 1: their second parts; and their third parts
      const uint16_t* hr = a.hs + (size_t)row * 3 * a.GP;
      uint32_t hv[8], hw[8];
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        hv[g] = hr[kh * a.GP + min(g0 + g, G - 1)];
        hw[g] = hr[2 * a.GP + min(g0 + g, G - 1)];
        hv[g] = g < cnt ? hv[g] : 0u;
        hw[g] = g < cnt ? hw[g] : 0u;
      }
      hf = pack8(hv);
      h3 = pack8(hw);
    }
    {
      const uint32_t* src = words(f0 * UB);
#pragma unroll
      for (int g = 0; g < kNG; ++g) load_word(src, g);
    }
    store_scales(0);
    __syncthreads();

    // block blk (its scales in sbuf[B]); the next block's scales first, then each group's
    // nibbles into the registers that the group has just left: nearly a whole block ahead
    auto step = [&](int blk, auto B) {
      constexpr int kB = decltype(B)::value;
      const int nx = min(blk + 1, b1 - 1);
      load_scales(nx);
      const uint32_t* src = words(nx);
      const uint16_t* sl = &sbuf[kB][0][j * G];
      const uint16_t* bl = &sbuf[kB][1][j * G];
      // this wavefront's scales and biases (a missing group's are zero: it adds nothing), and
      // the group sums' part: sums x b, then sums x -16 s
      float sc[kNG];
      uint32_t sn[8], bn[8];
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        sn[g] = bn[g] = 0u;
        if (g < kNG) {
          const int gc = min(g0 + g, G - 1);
          const uint32_t su = g < cnt ? sl[gc] : 0u;
          sc[g] = bf16_bits_to_f32(su);
          sn[g] = __float_as_uint(sc[g] * -16.0f) >> 16;   // exact
          bn[g] = g < cnt ? bl[gc] : 0u;
        }
      }
      const bf16x8 sf = pack8(sn);
      const bf16x8 bf = pack8(bn);
      f32x16 y = {};
      y = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hf, bf, y, 0, 0, 0);
      y = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hf, sf, y, 0, 0, 0);
      y = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h3, kh ? sf : bf, y, 0, 0, 0);
#pragma unroll
      for (int g = 0; g < kNG; ++g) {
        bf16x8 wf[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) wf[q] = unpack(bw[g][q], nibm);
        load_word(src, g);
        f32x16 acc = {};
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[g][q], wf[q], acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) y[i] = fmaf(sc[g], acc[i], y[i]);
      }
      // the eight parts: registers 2 p, 2 p + 1 of every wavefront to wavefront p (pieces
      // swapped by the lane against bank conflicts)
#pragma unroll
      for (int p = 0; p < 8; ++p) red[kB][wave][lane][p ^ ((lane >> 2) & 7)] = f32x2{y[2 * p], y[2 * p + 1]};
      store_scales(kB ^ 1);
      __syncthreads();
      const int ps = wave ^ ((lane >> 2) & 7);
      f32x2 o = red[kB][0][lane][ps];
#pragma unroll
      for (int s = 1; s < kWv; ++s) o += red[kB][s][lane][ps];
      // rows 8 (wave / 2) + 4 kh + 2 (wave % 2) + i, output 32 blk + j
      const int n = 32 * blk + j;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 8 * (wave >> 1) + 4 * kh + 2 * (wave & 1) + i, d = drow[r];
        const uint16_t uo = f32_to_bf16_bits(o[i]);
        if constexpr (MODE == kStore) {
          if (d >= 0 && n < O) a.y[(size_t)d * a.y_ld + n] = uo;
        } else if constexpr (MODE == kResid) {
          if (d >= 0 && n < O)
            a.y[(size_t)d * a.y_ld + n] =
                f32_to_bf16_bits(bf16_bits_to_f32(a.res[(size_t)d * a.res_ld + n]) + bf16_bits_to_f32(uo));
        } else {
          const float ub = bf16_bits_to_f32(uo), rl = ub != ub ? ub : fmaxf(ub, 0.0f);
          const uint16_t h = f32_to_bf16_bits(rl * rl);
          if (d >= 0) a.y[(size_t)d + n] = h;
          float tsum = bf16_bits_to_f32(h);
          tsum += dpp_f32<0xB1>(tsum);
          tsum += dpp_f32<0x4E>(tsum);
          tsum += dpp_f32<0x141>(tsum);
          tsum += dpp_f32<0x140>(tsum);
          const uint32_t tb = __float_as_uint(tsum);
          const auto pt = __builtin_amdgcn_permlane16_swap(tb, tb, false, false);
          tsum = __uint_as_float(pt[0]) + __uint_as_float(pt[1]);
          if constexpr (kB == 0) {
            if (j == 0) hpart[r] = tsum;              // read by this lane, in the unit's second block
          } else if (j == 0 && d >= 0 && a.hsum) {
            float hv = hpart[r] + tsum;               // as three bf16 values
            uint16_t* hp = a.hsum + (size_t)srow[r] * 3 * a.GPH + (blk >> 1);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
              const uint16_t p = f32_to_bf16_bits(hv);
              hp[k * a.GPH] = p;
              hv -= bf16_bits_to_f32(p);
            }
          }
        }
      }
    };
    for (int blk = f0 * UB; blk < b1; blk += 2) {
      step(blk, std::integral_constant<int, 0>{});
      if (blk + 1 >= b1) break;
      step(blk + 1, std::integral_constant<int, 1>{});
    }
  }
}

// Rows of 4096 inputs (the projections out of the Mamba-2 and attention mixers): an eighth is 8
// groups, 128 registers of rows, which leaves none for nibbles in flight. Here the block's
// weights come to LDS in two stages of half a row (32 runs of 1 KB, one direct load each), the
// next stage while one is multiplied, with a block's scales and biases in its first stage; a
// stage costs one barrier. A row's 16-byte pieces are swapped in their 128 bytes by the row, in
// the load's source address, so that the fragment reads of 8 rows fall in different banks. The
// next group's nibbles are unpacked beside a group's MFMAs (scheduling barriers: a sum moved
// past the stage's barrier would hold 64 registers). 64 rows 31 -> 14 us (out_proj).
template <int MODE>
__global__ __launch_bounds__(64 * kWv, 2) void k_gemm_rows_4096(GemmArgs a) {
  constexpr int I = 4096, G = I / 64, NS = 4, NG = 2 * NS;   // groups per wavefront: stage, all
  constexpr int kStage = 32 * 1024, kScale = 8 * 1024;       // a stage's nibbles, a block's scales and biases
  // two stages | two blocks' scales and biases | the eighths' exchange
  __shared__ __attribute__((aligned(1024))) char lds[2 * kStage + 2 * kScale + kWv * 64 * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, kh = lane >> 5, O = a.O;
  char* redp = lds + 2 * kStage + 2 * kScale;
  const uint32_t lbase = (uint32_t)(uintptr_t)(lds_void_t*)lds;
  const uint32_t nibm = opaque_vgpr(kNibHi);

  // ---- this workgroup's units: (tile of 32 rows, 32 outputs)
  const int un = (O + 31) / 32;
  const int64_t total = (int64_t)((a.T + 31) / 32) * un;
  const int wg = xcd_remap((int)blockIdx.x, a.grid);
  const int64_t u1 = total * (wg + 1) / a.grid;
  int64_t u = total * wg / a.grid;

  // chunk wave + 8 i of a stage is row wave + 8 i's 1 KB: one lane offset and a scalar step
  const uint32_t voff = (uint32_t)(wave * (I / 2) + 16 * (lane ^ wave));
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  // 1 KB to LDS by direct load: M0 = its LDS address. In inline assembly so that the LDS reads
  // wait on the explicit counts below only.
  auto load_lds = [&](uint32_t dst, const void* src, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(src)
                 : "memory", "m0");
  };
#pragma clang diagnostic pop
  // a block's first output: the last block ends at O (its outputs that the block before has are
  // not written)
  auto out0 = [&](int blk) { return min(32 * blk, O - 32); };
  auto issue = [&](int blk, int half, int buf) {
    const int n0 = out0(blk);
    const char* src = reinterpret_cast<const char*>(a.w) + (size_t)n0 * (I / 2) + 1024 * half;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      load_lds(lbase + (uint32_t)(buf * kStage + 1024 * (wave + kWv * i)), src + i * kWv * (I / 2), voff);
    if (half == 0) {   // 4 KB of scales, 4 KB of biases: 1 KB per wavefront
      const char* sb = reinterpret_cast<const char*>((wave < 4 ? a.s : a.b) + (size_t)n0 * G) + 1024 * (wave & 3);
      load_lds(lbase + (uint32_t)(2 * kStage + (blk & 1) * kScale + 1024 * wave), sb, 16u * (uint32_t)lane);
    }
  };

  while (u < u1) {
    const int t = (int)(u / un), b0 = (int)(u - (int64_t)t * un), b1 = (int)min((int64_t)un, b0 + (u1 - u));
    u += b1 - b0;
    __syncthreads();                // the previous tile's last stage has been read
    issue(b0, 0, 0);
    // the tile's rows and group sums (lane half 0: the sums' first parts, half 1: the second)
    const int row = min(32 * t + j, a.T - 1);
    bf16x8 av[NG][4], hf, h3;
    {
      const uint16_t* xr = a.xp + (size_t)row * I + 256 * wave + 32 * kh;
      const uint16_t* hr = a.hs + (size_t)row * 3 * a.GP + NS * wave;
      uint32_t hv[8], hw[8];
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int gg = (g / NS) * (G / 2) + g % NS;
#pragma unroll
        for (int q = 0; q < 4; ++q) av[g][q] = *reinterpret_cast<const bf16x8*>(xr + 64 * gg + 8 * q);
        hv[g] = hr[kh * a.GP + gg];
        hw[g] = hr[2 * a.GP + gg];
      }
      hf = pack8(hv);
      h3 = pack8(hw);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();

    int buf = 0;
    for (int blk = b0; blk < b1; ++blk) {
      f32x16 y = {};
      const uint16_t* sl = reinterpret_cast<const uint16_t*>(lds + 2 * kStage + (blk & 1) * kScale) + j * G + NS * wave;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        // the next stage's loads (past the last block: of the last again)
        issue(half ? min(blk + 1, b1 - 1) : blk, half ^ 1, buf ^ 1);
        if (half == 0) {            // the group sums' part: sums x b, then sums x -16 s
          uint32_t sn[8], bn[8];
#pragma unroll
          for (int g = 0; g < NG; ++g) {
            const int gg = (g / NS) * (G / 2) + g % NS;
            sn[g] = __float_as_uint(bf16_bits_to_f32(sl[gg]) * -16.0f) >> 16;   // exact
            bn[g] = sl[2048 + gg];
          }
          const bf16x8 bf = pack8(bn), sf = pack8(sn);
          y = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hf, bf, y, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f32_32x32x16_bf16(hf, sf, y, 0, 0, 0);
          y = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h3, kh ? sf : bf, y, 0, 0, 0);
        }
        const char* wl = lds + buf * kStage + 1024 * j + 128 * wave;
        u32x4 xw[NS];
        float sc[NS];
#pragma unroll
        for (int g = 0; g < NS; ++g) {
          xw[g] = *reinterpret_cast<const u32x4*>(wl + 16 * ((2 * g + kh) ^ (j & 7)));
          sc[g] = bf16_bits_to_f32(sl[half * (G / 2) + g]);
        }
        bf16x8 cur[4], nxt[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) cur[q] = unpack(xw[0][q], nibm);
        f32x16 acc[2];
#pragma unroll
        for (int g = 0; g < NS; ++g) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x16 zero = {};
            acc[g & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[half * NS + g][q], cur[q], q ? acc[g & 1] : zero, 0, 0, 0);
            if (g + 1 < NS) nxt[q] = unpack(xw[g + 1][q], nibm);
            if (g > 0) {
#pragma unroll
              for (int i = 4 * q; i < 4 * q + 4; ++i) y[i] = fmaf(sc[g - 1], acc[(g - 1) & 1][i], y[i]);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) cur[q] = nxt[q];
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) y[i] = fmaf(sc[NS - 1], acc[(NS - 1) & 1][i], y[i]);
        if (half == 0) asm volatile("" : "+v"(y));
        if (half == 1) {
          // the eight parts: registers 2 p, 2 p + 1 of every wavefront to wavefront p (pieces
          // swapped by the lane against bank conflicts); read again after the next block's first
          // barrier at the earliest
          f32x2* rw = reinterpret_cast<f32x2*>(redp) + (wave * 64 + lane) * 8;
#pragma unroll
          for (int p = 0; p < 8; ++p) rw[p ^ ((lane >> 2) & 7)] = f32x2{y[2 * p], y[2 * p + 1]};
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);          // this wavefront's part of the next stage is in
        lds_barrier();                               // everyone's, and this stage has been read
        buf ^= 1;
      }
      const f32x2* rr = reinterpret_cast<const f32x2*>(redp) + lane * 8 + (wave ^ ((lane >> 2) & 7));
      f32x2 o = rr[0];
#pragma unroll
      for (int s = 1; s < kWv; ++s) o += rr[s * 64 * 8];
      // rows 8 (wave / 2) + 4 kh + 2 (wave % 2) + i, output out0(blk) + j
      const int n = out0(blk) + j;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int d = 32 * t + 8 * (wave >> 1) + 4 * kh + 2 * (wave & 1) + i;
        if (d < a.T && n >= 32 * blk) {
          const uint16_t uo = f32_to_bf16_bits(o[i]);
          if constexpr (MODE == kStore)
            a.y[(size_t)d * a.y_ld + n] = uo;
          else
            a.y[(size_t)d * a.y_ld + n] =
                f32_to_bf16_bits(bf16_bits_to_f32(a.res[(size_t)d * a.res_ld + n]) + bf16_bits_to_f32(uo));
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);              // no direct load outlives its tile
  }
}

}  // namespace

// The rules: the expert products in 32-row tiles always; a dense product with rows of up to 3072
// inputs for up to 64 token rows (10304 outputs: 16 rows 20.5 -> 13.3 us, 32 rows 19.9 -> 16.9,
// 64 rows 20.7 -> 20.5; 96 rows 21.3 in the ring kernel against 32.2 here: its 64-row tiles
// share the unpacking); with rows of 4096 inputs for up to 256 (2688 outputs and a residual:
// 64 rows 31 -> 14 us, 256 rows 32.4 -> 23.9; 384 rows 33.2 there against 35.7 here).
int launch_gemm_rows(const char* fn, GemmArgs a, int mode, hipStream_t st) {
  const bool wide = a.I == 4096 && mode != kUpRelu2;
  if (!wide && a.I > 64 * kNG * kWv) return 1;
  if (mode != kUpRelu2 && (a.O < 32 || a.O % 8 || a.T > (wide ? 256 : 64))) return 1;
  const uintptr_t al = (uintptr_t)a.s | (uintptr_t)a.b | (uintptr_t)a.ss | (uintptr_t)a.sb;
  if (al & 15u) return 1;           // scales and biases are read in 16-byte pieces
#define HSD_ROWS(K)                                                                                  \
  do {                                                                                               \
    a.grid = resident_workgroups(reinterpret_cast<const void*>(&K), 64 * kWv, 0, 256);               \
    hipLaunchKernelGGL((K), dim3((unsigned)a.grid), dim3(64 * kWv), 0, st, a);                       \
  } while (0)
  if (wide) {
    if (mode == kStore) HSD_ROWS(k_gemm_rows_4096<kStore>); else HSD_ROWS(k_gemm_rows_4096<kResid>);
  } else if (mode == kStore) {
    HSD_ROWS(k_gemm_rows<kStore>);
  } else if (mode == kResid) {
    HSD_ROWS(k_gemm_rows<kResid>);
  } else {
    HSD_ROWS(k_gemm_rows<kUpRelu2>);
  }
#undef HSD_ROWS
  return check_launch(fn);
}

}  // namespace hsd

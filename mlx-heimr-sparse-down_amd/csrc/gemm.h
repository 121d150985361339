// The arguments of the 4-bit products of a prompt chunk (gemm.hip, gemm_rows.hip).
#pragma once

#include "hsd_common.h"

namespace hsd {

struct GemmArgs {
  const uint16_t* xp;      // [T, I] prepared rows
  const uint16_t* hs;      // [T, 3 GP] group sums, as the sum of three bf16 values
  const uint32_t* w;       // [O, I/8] (expert products: [E, F, I/8])
  const uint16_t* s;       // [O, I/64]
  const uint16_t* b;
  uint16_t* y;
  int64_t y_ld;
  const uint16_t* res;
  int64_t res_ld;
  // expert products
  const uint32_t* sw;
  const uint16_t* ss;
  const uint16_t* sb;
  const int32_t* tile_e;
  const int32_t* tile_slot;
  const int32_t* ntiles;   // [0]: routed tiles in use
  uint16_t* hsum;          // nullable, [T * (topk + 1), 3 GPH]: the outputs' group sums
  int GPH;
  int nt_routed;           // first shared tile
  int nt_shared;
  int T, O, I, GP;
  int F, FS, topk, E;
  uint32_t y_bytes, res_bytes, hsum_bytes;   // the buffers' sizes, below 1 GiB
  int grid;                // k_gemm_rows: its workgroups
};

enum GemmMode : int { kStore = 0, kResid = 1, kUpRelu2 = 2 };

// gemm_rows.hip: launches k_gemm_rows (32-row tiles) for `mode`; 1 when it does not take the
// sizes, else the launch's status.
int launch_gemm_rows(const char* fn, GemmArgs a, int mode, hipStream_t st);

}  // namespace hsd

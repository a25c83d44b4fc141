// A small layer's down projection and combine (moe_small.hip).
#pragma once
#include "moe_common.h"

struct SmallDown {
  const uint8_t *hq, *wd;    // (M k, I) codes in flat order, (E, D, I) codes, and their scales
  const float *sh, *swd;
  const uint8_t *hsq, *ws;   // the shared expert's (SI 0: none)
  const float *shs, *sws;
  const int32_t* ids;        // (M, k)
  const float* w;
  const float* shared_gate;
  const void* residual;
  int io_f32;                // of residual and out
  void* out;
  int M, D, E, k, I, SI;
};
// Selections that a lane of it holds, 1 or 2, where a batch that reads its selections itself (moe_gemm_scan_rows) takes this launch,
// or 0
int moe_small_down_lanes(int M, int D, int E, int k, int I, int SI);
int moe_small_down(const SmallDown& a, int lanes, moe_stream_t stream);

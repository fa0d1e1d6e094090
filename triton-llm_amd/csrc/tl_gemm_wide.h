// The 16-bit prompt products (tl_gemm_wide.hip), as tl_gemm.hip launches them.
#pragma once

#include "tl_gemm.h"

namespace tlg {

// A tile of C, and the microseconds one costs a busy device: a fixed part
// (first loads, stores) and a part per 32 k.
struct WidePlan {
  int tm, tn;
  double tile_us, stage_us;
  int ksplit, kt_per;  // K-slices, and 32-k stages of one
};

// The tile and K split (min_split to max_split slices) of the least modelled time:
// rounds of one tile a CU, plus the reduce pass over the fp32 partials of a split.
WidePlan gemm_wide_plan(int m, int k, const GemmGroups& G, int min_split, int max_split);

// p's tiles, split and items are w's; p.vec_store marks the groups whose rows
// take 16-byte stores (the reduce's own runs when K is split).
int launch_gemm_wide(const GemmParams& p, const WidePlan& w, int dtype, hipStream_t st);

}  // namespace tlg

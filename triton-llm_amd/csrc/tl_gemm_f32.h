// The fp32 prompt products (tl_gemm_f32.hip), as tl_gemm.hip launches them.
#pragma once

#include "tl_gemm.h"

namespace tlg {

// A tile height (128 columns), K-slices, 32-k stages of one, and the modelled time.
struct F32Plan {
  int tm, ksplit, kt_per;
  double us;
};

// The plan of the least modelled time with min_split to max_split K-slices.
F32Plan gemm_f32_plan(int m, int k, const GemmGroups& G, int min_split, int max_split);

// p's tiles are tm x 128 (tm 128 or 64), its stages 32 k.
int launch_gemm_f32(const GemmParams& p, int tm, hipStream_t st);

}  // namespace tlg

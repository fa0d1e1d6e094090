// The plan of a product of more than eight rows on the matrix cores, as
// tl_gemm.hip launches it and sizes its workspace by.
#pragma once

#include "tl_gemm_f32.h"
#include "tl_gemm_wide.h"

namespace tlg {

struct PromptPlan {
  WidePlan wide;  // 16-bit
  int tm, tn, ksplit, kt_per;
};

// For a C that overlaps A or B (in_place) K is cut in two at least, where
// the workspace query has room for it; without a workspace, whole K only.
PromptPlan gemm_prompt_plan(int m, int k, const GemmGroups& G, int esize, bool in_place, bool workspace = true);

// Bytes of the partials of ksplit K-slices.
size_t gemm_split_bytes(int m, const GemmGroups& G, int ksplit);

}  // namespace tlg

"""The plans of the matrix-core products (csrc/tl_gemm_plan.h), on the CPU: what
the workspace query answers holds the plan that launches, and the GPU tests'
shapes reach every tile, whole and with K split.  A small host program calls the
built library's plan functions; they need no device (256 CUs, or the cap)."""

import os
import re
import shutil
import subprocess

import numpy as np
import pytest

from tests import test_gpu_gemm as tg

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "triton-llm_amd", "csrc")
LIB = os.path.join(ROOT, "triton-llm_amd", "triton_llm", "_lib")

MAIN = r"""
#include "tl_gemm_plan.h"
#include <cstdio>
#include "triton_llm_hip.h"
int main() {  // lines: m k esize cus count n...; per line, plain and in place: tm tn ksplit bytes; the query
  int m, k, esize, count;
  while (scanf("%d %d %d %d %d", &m, &k, &esize, &tl_overrides.max_cus, &count) == 5) {
    tlg::GemmGroups G{};
    G.count = count;
    for (int g = 0; g < count; ++g)
      if (scanf("%d", &G.n[g]) != 1) return 1;
    for (int in_place = 0; in_place < 2; ++in_place) {
      const tlg::PromptPlan P = tlg::gemm_prompt_plan(m, k, G, esize, in_place);
      printf("%d %d %d %zu ", P.tm, P.tn, P.ksplit, tlg::gemm_split_bytes(m, G, P.ksplit));
    }
    printf("%zu\n", tl_gemm_grouped_workspace_bytes(m, k, count, G.n, esize == 4 ? TL_DTYPE_F32 : TL_DTYPE_BF16));
  }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc) or not os.path.exists(os.path.join(LIB, "libtriton_llm_hip.so")):
        pytest.skip("hipcc or the built library not available")
    d = tmp_path_factory.mktemp("plans")
    (d / "main.hip").write_text(MAIN)
    res = subprocess.run([hipcc, "--offload-host-only", "-std=c++17", "-I", CSRC, "-I", os.path.join(ROOT, "include"),
                          str(d / "main.hip"), "-L", LIB, "-l:libtriton_llm_hip.so", f"-Wl,-rpath,{LIB}",
                          "-o", str(d / "main")], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr

    def run(cases):  # (m, k, ns, esize, cus) -> rows of tm tn ksplit bytes (plain, in place), query
        text = "".join(f"{m} {k} {e} {c} {len(ns)} {' '.join(map(str, ns))}\n" for m, k, ns, e, c in cases)
        out = subprocess.run([str(d / "main")], input=text, capture_output=True, text=True, check=True).stdout
        got = [[int(x) for x in line.split()] for line in out.splitlines()]
        assert len(got) == len(cases)
        return got

    return run


def _shapes(test):  # (M, K, Ns, cus) of the test's parameters; no cap where it sets none
    (mark,) = [m for m in test.pytestmark if m.name == "parametrize" and m.args[0].startswith("M,K,Ns")]
    return [tuple(p) + (0,) * (4 - len(p)) for p in mark.args[1]]


@pytest.mark.parametrize("esize", [2, 4])
def test_query_holds_the_plan(plans, esize):
    rng = np.random.default_rng(esize)
    size = lambda hi: int(np.exp(rng.uniform(0, np.log(hi))))  # noqa: E731
    cases = [(8 + size(2000), 1 + size(8200), tuple(8 * size(1000) for _ in range(rng.integers(1, 5))), esize, cus)
             for cus in (0, 0, 0, 4) for _ in range(3000)]
    for case, (_, _, s, b, _, _, s_in, b_in, query) in zip(cases, plans(cases)):
        assert b <= query, case
        if s > 1:
            assert query == b, case
        if query > 0:  # then a C that overlaps A or B is cut, within that room
            assert s_in > 1 and b_in <= query, case


def test_gpu_shapes_reach_every_wide_tile(plans):
    cases = [(m, k, ns, 2, cus) for m, k, ns, cus in _shapes(tg.test_gemm_wide_tiles)]
    got = {(tm, tn, s > 1) for tm, tn, s, *_ in plans(cases)}
    with open(os.path.join(CSRC, "tl_gemm_wide.hip")) as f:  # the tiles of its table
        table = re.search(r"kWidePlans\[\] = \{(.*?)\};", f.read(), re.S).group(1)
    tiles = {(int(tm), int(tn)) for tm, tn in re.findall(r"\{(\d+), (\d+),", table)}
    assert len(tiles) == 6 and got == {(*t, split) for t in tiles for split in (False, True)}


@pytest.mark.parametrize("test", [tg.test_gemm_prompt_fp32_plans, tg.test_gemm_fp32_parts_tiles,
                                  tg.test_gemm_fp32_outliers])
def test_gpu_shapes_reach_both_fp32_tiles(plans, test):
    got = {(tm, s > 1) for tm, _, s, *_ in plans([(m, k, ns, 4, cus) for m, k, ns, cus in _shapes(test)])}
    assert got == {(tm, split) for tm in (64, 128) for split in (False, True)}

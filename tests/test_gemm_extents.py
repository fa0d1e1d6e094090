"""The extent the GEMM kernels give a buffer resource (csrc/tl_gemm.h
view_bytes), on the CPU: for operands that are columns of wider rows no chunk
that a tile loads, and that the hardware's range check lets through, may lie
past the allocation the view ends in.  The function is compiled for the host
from the header the kernels include."""

import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "triton-llm_amd", "csrc")

# (rows, parent width, view columns, tile columns): the view is the parent's last columns
CASES = [(3072, 5120, 1024, 192), (960, 1600, 320, 256), (40, 136, 8, 128), (1, 264, 200, 128), (7, 72, 72, 64)]


@pytest.fixture(scope="module")
def extents(tmp_path_factory):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    d = tmp_path_factory.mktemp("extents")
    src = d / "main.hip"
    src.write_text('#include "tl_gemm.h"\n#include <cstdio>\n#include <cstdlib>\n'
                   "int main(int c, char** v) {\n"
                   "  for (int i = 1; i + 3 < c; i += 4)\n"
                   "    printf(\"%u\\n\", tlg::view_bytes(atoll(v[i]), atoll(v[i + 1]), atoll(v[i + 2]), atoi(v[i + 3])));\n"
                   "}\n")
    res = subprocess.run([hipcc, "--offload-host-only", "-std=c++17", "-I", CSRC, str(src), "-o", str(d / "main")],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr

    def run(args):
        flat = [str(x) for a in args for x in a]
        out = subprocess.run([str(d / "main"), *flat], capture_output=True, text=True, check=True)
        return [int(x) for x in out.stdout.split()]

    return run


@pytest.mark.parametrize("esize", [2, 4])
def test_loads_in_range_stay_in_the_parent(extents, esize):
    got = extents([(r, w, n, esize) for r, w, n, _ in CASES])
    for (rows, width, n, tile), size in zip(CASES, got):
        parent = np.empty((rows, width), np.uint16 if esize == 2 else np.float32)
        view = parent[:, width - n:]
        base = view.ctypes.data - parent.ctypes.data
        assert size == np.lib.array_utils.byte_bounds(view)[1] - view.ctypes.data
        # 16-byte chunks of the last row from the last tile's first column to its end
        chunk = 16 // esize
        first = (n - 1) // tile * tile
        at = [((rows - 1) * width + c) * esize for c in range(first, first + tile, chunk)]
        assert all(base + a + 16 <= parent.nbytes for a in at if a < size)
        if n % tile and width > n:  # a resource of rows * ld bytes lets chunks past the parent through
            assert any(base + a + 16 > parent.nbytes for a in at if a < rows * width * esize)
    assert extents([(0, 8, 8, esize)]) == [0]

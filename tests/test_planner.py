"""The GEMM planner over the operand layouts, compiled for the host (no GPU, no HIP)."""
import ctypes
import os
import random
import subprocess

import pytest

from tests.test_capi import OK, ROOT, Plan

CSRC = os.path.join(ROOT, "wmma_ops_amd", "csrc")
NN, TN, NT = 0, 1, 2  # wmma_amd::GemmLayout
SHIM = """
#include "plan.hpp"
extern "C" int layout_plan(int layout, int M, int N, int K, size_t max_ws, wmma_gemm_plan* out) {
    *out = wmma_gemm_plan{};
    return wmma_amd::make_layout_plan(static_cast<wmma_amd::GemmLayout>(layout), M, N, K,
                                      WMMA_TILE_AUTO, 256, max_ws, out);
}
"""


@pytest.fixture(scope="module")
def layout_plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("planner")
    (d / "shim.cpp").write_text(SHIM)
    so = str(d / "planner.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-I", CSRC, str(d / "shim.cpp"),
                    os.path.join(CSRC, "plan.cpp"), "-o", so], check=True)
    f = ctypes.CDLL(so).layout_plan
    f.argtypes = [ctypes.c_int] * 4 + [ctypes.c_size_t, ctypes.POINTER(Plan)]
    return f


# The row counts around each whole number of rounds of 256 x 256 tiles, where plans are cut in
# two, of common layer sizes; then shapes of any kind.
LAYERS = [(4096, 4096), (11008, 4096), (4096, 11008), (12288, 4096), (14336, 4096), (22016, 4096),
          (24576, 4096), (18944, 3584), (5120, 5120), (13824, 5120), (8192, 8192), (4100, 4099)]


def _shapes():
    for n, k in LAYERS:
        yield from ((m, n, k) for m in range(257, 8193, 3))
    rng = random.Random(1)
    for _ in range(20000):
        yield rng.randint(257, 8192), rng.randint(64, 16384), rng.randint(64, 16384)


@pytest.mark.parametrize("layout", [NN, TN, NT])
@pytest.mark.parametrize("max_ws", [2 ** 64 - 1, 32 << 20])
def test_two_part_edges_fit_their_plan(layout_plan, layout, max_ws):
    # The launch plans the edge again, in the layout it runs in, and refuses a plan that does
    # not hold the edge's workspace.
    p, e, parts = Plan(), Plan(), 0
    for m, n, k in _shapes():
        assert layout_plan(layout, m, n, k, max_ws, ctypes.byref(p)) == OK
        assert p.workspace_bytes <= max_ws
        if p.edge_dim == 0:
            continue
        parts += 1
        em, en = (m - p.edge_at, n) if p.edge_dim == 1 else (m, n - p.edge_at)
        assert layout_plan(layout, em, en, k, max_ws, ctypes.byref(e)) == OK
        assert e.edge_dim == 0, (m, n, k)
        assert e.workspace_bytes == p.workspace_bytes, (m, n, k, em, en)
    assert parts > 1000

"""The order in which varlen attention workgroups take their blocks (flash_sched.hpp), without a
GPU: the rule that chooses it, and that every block of every sequence is one workgroup's.  The
host functions are the header's own; the search of a wave and the ids are modelled here."""
import ctypes
import os
import random
import subprocess

import pytest

from tests.test_capi import ROOT

CSRC = os.path.join(ROOT, "wmma_ops_amd", "csrc")
SHIM = """
#include "flash_sched.hpp"
using namespace wmma_amd;
extern "C" int ordered(long B, long heads, long blocks, long parts, int causal) {
    return varlen_ordered(B, heads, blocks, parts, causal != 0);
}
extern "C" int grid_y(long B, long total, long longest, long block) {
    return varlen_grid_y(B, total, longest, block);
}
extern "C" int at_least(int kv, int causal, int owned, int other, int t) {
    return kv ? (causal ? varlen_at_least<true, true, 128>(owned, other, t)
                        : varlen_at_least<true, false, 128>(owned, other, t))
              : (causal ? varlen_at_least<false, true, 128>(owned, other, t)
                        : varlen_at_least<false, false, 128>(owned, other, t));
}
"""
BLOCK = 128


@pytest.fixture(scope="module")
def sched(tmp_path_factory):
    d = tmp_path_factory.mktemp("sched")
    (d / "shim.hip").write_text(SHIM)
    so = str(d / "sched.so")
    subprocess.run([os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc"), "-O1",
                    "-std=c++17", "--offload-host-only", "-fPIC", "-shared", "-I", CSRC,
                    str(d / "shim.hip"), "-o", so], check=True)
    L = ctypes.CDLL(so)
    L.ordered.argtypes = [ctypes.c_long] * 4 + [ctypes.c_int]
    L.grid_y.argtypes = [ctypes.c_long] * 4
    return L


# (sequences, heads, blocks of the longest, parts, causal) on both sides of each line.
@pytest.mark.parametrize("args,ordered", [
    ((8, 8, 4, 1, 1), 0), ((8, 8, 5, 1, 1), 1),        # a CU for every workgroup (256)
    ((4, 2, 16, 2, 1), 0), ((4, 2, 16, 3, 1), 1),      # ... the parts of a block counted
    ((64, 8, 2, 1, 1), 0), ((64, 8, 3, 1, 1), 1),      # blocks enough for the search
    ((65, 8, 3, 1, 1), 0), ((65, 8, 4, 1, 1), 1),      # ... which takes 64 sequences a pass
    ((300, 40, 9, 1, 0), 0), ((300, 40, 10, 1, 0), 1),
    ((1002, 8, 4, 1, 1), 0),
    ((6, 32, 16, 1, 1), 0), ((6, 8, 16, 1, 1), 1),     # whole rows of 32 heads: not causal
    ((6, 64, 16, 1, 1), 0), ((6, 40, 16, 1, 1), 1),
    ((3, 32, 16, 1, 0), 0), ((4, 32, 16, 1, 0), 1),    # ... and no mask from four sequences on
    ((3, 40, 16, 1, 0), 1),
])
def test_order_rule(sched, args, ordered):
    assert sched.ordered(*args) == ordered


def _lengths(cu, total, longest):
    out = []
    for a, b in zip(cu, cu[1:]):
        lo = min(max(a, 0), total)
        out.append(min(min(max(b, lo), total) - lo, longest))
    return out


def _search(sched, kv, causal, owned, other, longest_other, idx):
    """varlen_item: the sequence and block of item idx, heaviest first; None past the last."""
    def at_least(t):
        return [sched.at_least(kv, causal, o, x, t) for o, x in zip(owned, other)]
    if idx >= sum(at_least(0)):
        return None
    lo, hi, above = 0, (longest_other + BLOCK - 1) // BLOCK + 1, 0
    while hi - lo > 1:
        mid = (lo + hi) // 2
        n = sum(at_least(mid))
        if n > idx:
            lo = mid
        else:
            hi, above = mid, n
    rank = idx - above
    for b, (all_, more) in enumerate(zip(at_least(lo), at_least(hi))):
        if rank < all_ - more:
            nb = -(-owned[b] // BLOCK)
            return b, (more + rank if kv else nb - 1 - more - rank)
        rank -= all_ - more
    raise AssertionError(idx)


def _batches():
    yield [0, 700], 700, 700
    yield [0, 128, 128, 255, 512, 640, 641], 641, 257          # edges, an empty one
    yield [40, 90, 90, 300], 400, 210                          # gaps in front and behind
    yield [0, 100, 400, 401], 401, 64                          # past the longest length
    yield [400, 400], 400, 8
    yield [17 * i for i in range(71)], 17 * 70, 17             # more sequences than lanes
    rng = random.Random(4)
    for _ in range(12):
        lens = [rng.choice([0, 1, 127, 128, 129, 256, 300, 513, 1000]) for _ in range(rng.randint(1, 90))]
        cu = [rng.randint(0, 300)]
        for n in lens:
            cu.append(cu[-1] + n)
        yield cu, cu[-1] + rng.randint(0, 500), max(max(lens), 1) + rng.choice([0, 0, 77, -1])


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("kv", [0, 1])
def test_every_block_is_one_item(sched, kv, causal):
    for cu, total, longest in _batches():
        lens = _lengths(cu, total, longest)
        B, rows = len(lens), sched.grid_y(len(lens), total, longest, BLOCK)
        items = [_search(sched, kv, causal, lens, lens, longest, i) for i in range(B * rows)]
        found = [x for x in items if x is not None]
        want = [(b, k) for b, n in enumerate(lens) for k in range(-(-n // BLOCK))]
        assert sorted(found) == want, (cu, total, longest)
        assert items[:len(found)] == found  # none behind the last
        if causal:  # heaviest first: blocks of the other side that a block walks
            weight = [-(-lens[b] // BLOCK) - k if kv else k + 1 for b, k in found]
            assert weight == sorted(weight, reverse=True)


@pytest.mark.parametrize("x", [1, 3, 8, 24, 31, 32, 40, 64, 96])
@pytest.mark.parametrize("y,z", [(1, 1), (7, 1), (5, 3), (64, 2)])
def test_linear_ids_are_a_permutation(x, y, z):
    n = x * y * z  # flash_linear_id: the engines of every other whole row of 32 ids mirrored
    ids = [i ^ 24 if (x & 31) and (i & 32) and (i | 31) < n else i for i in range(n)]
    assert sorted(ids) == list(range(n))
    assert all(i % 8 == j % 8 for i, j in enumerate(ids))

"""Launch sizes against the dispatch limit of 2^32 work items per dimension:
the slicing helpers of the engine's host code, compiled by themselves, at the
sizes of plans whose quartet list passes the limit and at small limits that
cut everywhere."""
import ctypes
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "gradscf_amd" / "csrc"

SHIM = r"""
#include "launch_limits.h"
extern "C" {
long long blocks(int threads) { return gscf::grid_blocks(threads); }
long long items(int lanes) { return gscf::grid_items(lanes); }
int slices(long long total, long long limit, long long* out, int cap) {
  int n = 0;
  gscf::for_slices(total, limit, [&](int64_t b, int64_t c) {
    if (n < cap) { out[2 * n] = b; out[2 * n + 1] = c; }
    ++n;
  });
  return n;
}
// pieces of `nr` ranges packed one after another: (range, first block, count, launch, blocks before it)
int cuts(const long long* blocks, int nr, long long limit, long long* out, int cap) {
  int n = 0;
  int64_t used = 0, launch = 0;
  for (int r = 0; r < nr; ++r)
    gscf::cut_blocks(blocks[r], limit, used, [&](int64_t first, int64_t count, bool fresh) {
      launch += fresh;
      if (n < cap) {
        const long long row[5] = {r, first, count, launch, used};
        for (int k = 0; k < 5; ++k) out[5 * n + k] = row[k];
      }
      ++n;
    });
  return n;
}
}
"""


@pytest.fixture(scope="module")
def limits(tmp_path_factory):
    d = tmp_path_factory.mktemp("limits")
    (d / "shim.cc").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", "-o", str(d / "shim.so"),
                    str(d / "shim.cc")], check=True)
    lib = ctypes.CDLL(str(d / "shim.so"))
    lib.blocks.restype = lib.items.restype = ctypes.c_longlong
    lib.slices.argtypes = [ctypes.c_longlong, ctypes.c_longlong, ctypes.c_void_p, ctypes.c_int]
    lib.cuts.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_longlong, ctypes.c_void_p, ctypes.c_int]
    return lib


def _slices(lib, total, limit):
    out = (ctypes.c_longlong * 4096)()
    n = lib.slices(total, limit, out, 2048)
    assert n <= 2048
    return [(out[2 * i], out[2 * i + 1]) for i in range(n)]


@pytest.mark.parametrize("threads", [64, 128, 256, 512, 1024])
def test_grid_stays_below_the_work_item_limit(limits, threads):
    n = limits.blocks(threads)
    assert n * threads < 2 ** 32 <= (n + 1) * threads


@pytest.mark.parametrize("lanes", [1, 3, 9, 18, 36])
def test_items_of_several_lanes_stay_below_the_limit(limits, lanes):
    n = limits.items(lanes)
    assert -(-n * lanes // 256) * 256 < 2 ** 32 <= (n + 1) * lanes + 512


@pytest.mark.parametrize("total,limit", [(0, 7), (1, 7), (6, 7), (7, 7), (8, 7), (100, 7), (100, 1),
                                         # quartets of 36 cc-pVDZ waters without screening (93528 pairs)
                                         (93528 * 93529 // 2, (2 ** 32 - 1) // 256 * 256)])
def test_slices_cover_every_entry_once(limits, total, limit):
    got = _slices(limits, total, limit)
    at = 0
    for begin, count in got:
        assert begin == at and 0 < count <= limit
        at += count
    assert at == total and len(got) == -(-total // limit)


@pytest.mark.parametrize("blocks,limit", [([5], 10), ([10], 10), ([11], 10), ([3, 4, 3], 10), ([3, 4, 4], 10),
                                          ([0, 25, 0, 1], 10), ([7, 30, 2], 1), ([], 10),
                                          # contracted s pairs of 181 hydrogens, 8 tasks a block
                                          ([16471 * 16472 // 2 // 8 + 1, 40], (2 ** 32 - 1) // 256)])
def test_cuts_fill_launches_in_order(limits, blocks, limit):
    """Every block of every range lies in one launch, at the next free place
    of it, and only the last launch is not full."""
    arr = (ctypes.c_longlong * max(1, len(blocks)))(*blocks)
    out = (ctypes.c_longlong * (5 * 256))()
    n = limits.cuts(arr, len(blocks), limit, out, 256)
    assert n <= 256
    place, done = 0, [0] * len(blocks)
    for i in range(n):
        r, first, count, launch, used = out[5 * i:5 * i + 5]
        assert first == done[r] and count > 0 and used + count <= limit
        assert launch * limit + used == place
        done[r] += count
        place += count
    assert done == list(blocks)

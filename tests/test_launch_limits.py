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
int slices(long long total, long long limit, long long* out, int cap) {
  int n = 0;
  gscf::for_slices(total, limit, [&](int64_t b, int64_t c) {
    if (n < cap) { out[2 * n] = b; out[2 * n + 1] = c; }
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
    lib.blocks.restype = ctypes.c_longlong
    lib.slices.argtypes = [ctypes.c_longlong, ctypes.c_longlong, ctypes.c_void_p, ctypes.c_int]
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

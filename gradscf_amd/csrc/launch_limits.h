// Sizes of one launch (host code, no HIP headers).
//
// A dispatch counts its work items per dimension in 32 bits.  A launch with
// gridDim.x * blockDim.x of 2^32 or more reports no error and runs only part of
// its workgroups (seen with packed integrals of 220 hydrogens, 1.2e10 lanes:
// most of the result was never written).  Launches whose size grows with the
// molecule are cut into slices below that.
#pragma once
#include <algorithm>
#include <cstdint>

namespace gscf {

constexpr int64_t kGridThreads = (int64_t(1) << 32) - 1;

// Workgroups of `threads` lanes one launch may have along x.
constexpr int64_t grid_blocks(int threads) { return kGridThreads / threads; }

// Items of `lanes` lanes each that one launch of 256-lane workgroups may have.
constexpr int64_t grid_items(int lanes) { return grid_blocks(256) * 256 / lanes; }

// launch(begin, count) over consecutive slices of [0, total), at most `limit`
// entries each.
template <class F>
void for_slices(int64_t total, int64_t limit, F&& launch) {
  for (int64_t begin = 0; begin < total; begin += limit) launch(begin, std::min(limit, total - begin));
}

// Cuts a range of `blocks` blocks into pieces of consecutive launches of at
// most `limit` blocks.  used: blocks the open launch holds already, updated;
// piece(first block, count, fresh) with fresh where the piece opens a new
// launch (whose used is then zero).
template <class F>
void cut_blocks(int64_t blocks, int64_t limit, int64_t& used, F&& piece) {
  for (int64_t first = 0; first < blocks;) {
    const bool fresh = used == limit;
    if (fresh) used = 0;
    const int64_t count = std::min(blocks - first, limit - used);
    piece(first, count, fresh);
    used += count;
    first += count;
  }
}

}  // namespace gscf

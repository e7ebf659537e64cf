// Inverse of dense blocks over many workgroups each (rs_inv.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "rs_device.hpp"

namespace iegpu {

constexpr int kInvMax = 1024 + 192;  // the largest root with 64 holes' border
// Panel flags at the end of a block's piv row, the last one its counter of
// started panels.
constexpr int kInvFlags = 80;
static_assert((kInvMax + 15) / 16 < kInvFlags, "a flag per panel and the counter");

// Blocks b = 0 .. n_blocks - 1 of size n = act_cnt[b] + extra, column-major
// (ld n) at a + stride b, destroyed; the inverse goes to out + stride b, or
// behind the block (a + stride b + n^2) when out is null.  piv + piv_stride
// b: the pivot rows (n ints) and, in its last kInvFlags ints, the panel
// flags and counter, zeroed before the launch.
template <typename R>
struct InvBlocks {
  R* a;
  R* out;
  int64_t stride;
  int* piv;
  int piv_stride;
  int extra;
};

// Inverts the blocks with nmin < n <= nmax (<= kInvMax) on st.  An exact
// zero pivot raises kErrSingular in s.err, a wait that did not end kErrWait.
template <typename R>
void launch_block_inverse(const DevState& s, const InvBlocks<R>& blk, int n_blocks, int nmin,
                          int nmax, hipStream_t st);

}  // namespace iegpu

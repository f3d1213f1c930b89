// The order in which column dots are summed, shared by the kernels that form
// them: blocks of consecutive rows (dotBlocks); within a block lane v of
// DOT_LANES adds rows r0 + v, r0 + v + DOT_LANES, ... in order, and the lanes
// are folded in halves (v += v + 32, 16, .. 1).  A thread may stand for several
// lanes, ty + R u, so the order, and with it every bit of a column's dot,
// depends on the rows alone and not on how many columns share a launch.
#pragma once
#include "common.hpp"

#include <algorithm>

namespace dfx
{
  namespace k
  {
    constexpr int DOT_LANES = 64;

    // row blocks of the column dots: 64 rows or more (enough workgroups for
    // the GPU from small vectors on), at most 1024 blocks
    inline u32 dotBlocks(u32 N) { return std::max(1u, std::min(1024u, (u32)(((u64)N + 63) / 64))); }
    inline u32 dotRows(u32 N, u32 nBlocks) { return (u32)(((u64)N + nBlocks - 1) / nBlocks); }

    // the folds between the U lanes of one thread
    template <int U, class V>
    __device__ inline V foldLanes(V (&acc)[U])
    {
#pragma unroll
      for (int h = U / 2; h > 0; h >>= 1)
#pragma unroll
        for (int u = 0; u < h; ++u)
          acc[u] += acc[u + h];
      return acc[0];
    }
  } // namespace k
} // namespace dfx

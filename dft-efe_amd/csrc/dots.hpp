// The order in which column dots are summed, shared by the kernels that form
// them.  Rows come in groups of DOT_LANES; block b takes groups b, b + nBlocks,
// ...; in it, lane v adds row v of each of its groups in order, and the lanes are
// folded in halves (v += v + 32, 16, .. 1).  A thread may stand for several
// lanes and a workgroup for several blocks or some of the columns, so the order,
// and with it every bit of a column's dot, depends on the rows alone and not on
// how many columns share a launch.
#pragma once
#include "common.hpp"

#include <algorithm>

namespace dfx
{
  namespace k
  {
    constexpr int DOT_LANES = 64;
    inline u32 dotGroups(u32 N) { return (u32)(((u64)N + DOT_LANES - 1) / DOT_LANES); }
    // one block a group up to half of DOT_BLOCKS (enough workgroups for the GPU
    // from small vectors on), then as many as share the groups evenly
    inline u32 dotBlocks(u32 N)
    {
      const u32 groups = dotGroups(N), turns = std::max(1u, groups / (DOT_BLOCKS / 2));
      return std::max(1u, (groups + turns - 1) / turns);
    }

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

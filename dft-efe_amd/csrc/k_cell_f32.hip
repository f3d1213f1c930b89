// The FP32 cell kernels (k_cell.hpp), a translation unit of their own so that
// both precisions compile side by side.
#include "k_cell.hpp"

namespace dfx
{
  namespace k
  {
    DFX_INST_CELL(float)
  } // namespace k
} // namespace dfx

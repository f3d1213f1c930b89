// The fixed-order sum of an enriched dof's partial rows, one workgroup of 256
// threads per (enriched dof, 16 columns): 16 slot lanes take every 16th slot
// and keep 16 loads in flight; the lane sums are combined in lane order, so
// the result does not depend on timing.  Shared by the reduction of the
// colour-by-colour apply and the row sums of the slot apply (the same bits).
#pragma once
#include "common.hpp"

namespace dfx
{
  namespace k
  {
    // slot indices are staged in LDS per chunk of IDX (one coalesced load
    // instead of a dependent index load per value); lane sl adds slots sl,
    // sl + SL, ... in ascending order (IDX is a multiple of SL)
    template <class T>
    struct EnrReduce
    {
      static constexpr int CB = 16, SL = 16, U = 16, IDX = 2048;
      T   part[SL][CB];
      u32 sIdx[IDX];

      // the sum of rows slots[e0 .. e1) of yE (leading dimension B) at column
      // j, valid in the threads with threadIdx.x < CB (and j < B)
      __device__ T sum(const u32 *__restrict__ slots, u32 e0, u32 e1, const T *__restrict__ yE,
                       u32 B, u32 j)
      {
        const int cj = threadIdx.x % CB, sl = threadIdx.x / CB;
        T         acc = 0;
        for (u32 c0 = e0; c0 < e1; c0 += IDX)
          {
            const u32 cn = min((u32)IDX, e1 - c0);
            __syncthreads(); // the previous chunk's indices are no longer read
            for (u32 t = threadIdx.x; t < cn; t += blockDim.x)
              sIdx[t] = slots[c0 + t];
            __syncthreads();
            if (j < B)
              for (u32 e = sl; e < cn; e += SL * U)
                {
                  T v[U];
#pragma unroll
                  for (int u = 0; u < U; ++u)
                    {
                      const u32 ee = e + u * SL;
                      v[u]         = ee < cn ? yE[(u64)sIdx[ee] * B + j] : (T)0;
                    }
#pragma unroll
                  for (int u = 0; u < U; ++u)
                    acc += v[u];
                }
          }
        part[sl][cj] = acc;
        __syncthreads();
        T s = 0;
        if (sl == 0)
#pragma unroll
          for (int q = 0; q < SL; ++q)
            s += part[q][cj];
        return s;
      }
    };
  } // namespace k
} // namespace dfx

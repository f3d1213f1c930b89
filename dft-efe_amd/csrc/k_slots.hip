// The row sums of the slot apply: every cell's product lies in its map slots'
// rows (cellSlots), and each dof's row is the sum of its slots' rows in a
// fixed order, with the step that follows the apply formed in the same launch.
#include "dots.hpp"
#include "enr_reduce.hpp"
#include "kernels.hpp"
#include "res_update.hpp"

#include <algorithm>

namespace dfx
{
  namespace k
  {
    namespace
    {
      template <class T, int V>
      struct Vec
      {
        typedef T type __attribute__((ext_vector_type(V)));
      };
      template <class T>
      struct Vec<T, 1>
      {
        typedef T type;
      };
      __device__ inline double at(double v, int) { return v; }
      __device__ inline float  at(float v, int) { return v; }
      template <class VT>
      __device__ inline auto at(VT v, int e)
      {
        return v[e];
      }
      template <class T>
      __device__ inline void put(T &v, int, T s)
      {
        v = s;
      }
      template <class VT, class T>
      __device__ inline void put(VT &v, int e, T s)
      {
        v[e] = s;
      }

      // The sum of a row's slots in order, V columns from j on.  The first slot
      // sits in the row's head, so that its load does not wait for the list of
      // the others
      template <class T, int V>
      __device__ inline typename Vec<T, V>::type rowSum(RowHead h, const u32 *__restrict__ rest,
                                                        const T *__restrict__ slots, u32 B, u32 j)
      {
        using vt      = typename Vec<T, V>::type;
        const u32 cnt = h.rest >> ROW_COUNT_SHIFT;
        vt        s{};
        if (cnt)
          s += *reinterpret_cast<const vt *>(slots + (u64)h.slot0 * B + j);
        if (cnt > 1)
          {
            const u32 *q = rest + (h.rest & ((1u << ROW_COUNT_SHIFT) - 1));
            for (u32 e = 0; e + 1 < cnt; e += 4)
              {
                vt v[4];
#pragma unroll
                for (u32 k = 0; k < 4; ++k)
                  if (e + k + 1 < cnt)
                    v[k] = *reinterpret_cast<const vt *>(slots + (u64)q[e + k] * B + j);
#pragma unroll
                for (u32 k = 0; k < 4; ++k)
                  if (e + k + 1 < cnt)
                    s += v[k];
              }
          }
        return s;
      }

      // Blocks below nE * ceil(B / 16): one enriched dof and 16 columns each
      // (EnrReduce; first, as they run longest).  The others: one thread per
      // classical row and V columns (V: one 16-byte vector where widths and
      // addresses allow); most rows (a cell's interior) have one slot.  Bound by
      // memory: B values read per slot, written per row (p = 3, 16^3 cells, 40
      // columns: FP32 63 MB in 14.8 us, FP64 with the residual step 239 MB in 35.6)
      template <class T, int V, bool RES>
      __global__ __launch_bounds__(256) void slotSumK(
        const RowHead *__restrict__ heads, const u32 *__restrict__ rest,
        const u32 *__restrict__ enrOff, const u32 *__restrict__ enrSlots, u32 nC, u32 nE,
        const T *__restrict__ slots, u32 B, T *x, u32 ldx, T *y, u32 ldy, int zeroX,
        ResFuse<T> rf)
      {
        using vt = typename Vec<T, V>::type;
        __shared__ EnrReduce<T> red;
        const u32 nb = (B + EnrReduce<T>::CB - 1) / EnrReduce<T>::CB;
        if (blockIdx.x < nE * nb)
          {
            const u32 g = blockIdx.x / nb;
            const u32 j = (blockIdx.x % nb) * EnrReduce<T>::CB + threadIdx.x % EnrReduce<T>::CB;
            const T   s = red.sum(enrSlots, enrOff[g], enrOff[g + 1], slots, B, j);
            if (threadIdx.x < EnrReduce<T>::CB && j < B)
              {
                if constexpr (RES)
                  {
                    const u64 o = (u64)(nC + g) * ldx + j;
                    rf.res[o]   = resUpdate<T>(s, x[o], rf.res[o], rf.r0[o], rf.mu[j],
                                               (T)rf.coef[0], (T)rf.coef[1], (T)rf.coef[2]);
                  }
                else
                  y[(u64)(nC + g) * ldy + j] = s;
              }
            return;
          }
        const u32 nv = B / V;
        const u64 t  = (u64)(blockIdx.x - nE * nb) * 256 + threadIdx.x;
        if (t >= (u64)nC * nv)
          return;
        u32 row, j;
        if ((t >> 32) == 0)
          row = (u32)t / nv, j = ((u32)t - row * nv) * V;
        else
          row = (u32)(t / nv), j = (u32)(t - (u64)row * nv) * V;
        const RowHead h   = heads[row];
        const u32     cnt = h.rest >> ROW_COUNT_SHIFT;
        if (cnt == ROW_ZERO)
          {
            if constexpr (!RES)
              {
                *reinterpret_cast<vt *>(y + (u64)row * ldy + j) = vt{};
                if (zeroX)
                  *reinterpret_cast<vt *>(x + (u64)row * ldx + j) = vt{};
              }
            return;
          }
        const u64 o = (u64)row * ldx + j;
        vt        xv{}, rv{}, zv{};
        if constexpr (RES)
          {
            xv = *reinterpret_cast<const vt *>(x + o);
            rv = *reinterpret_cast<const vt *>(rf.res + o);
            zv = *reinterpret_cast<const vt *>(rf.r0 + o);
          }
        const vt s = rowSum<T, V>(h, rest, slots, B, j);
        if constexpr (RES)
          {
            const T a1 = (T)rf.coef[0], a2 = (T)rf.coef[1], c = (T)rf.coef[2];
            vt      out{};
#pragma unroll
            for (int e = 0; e < V; ++e)
              put(out, e, resUpdate<T>(at(s, e), at(xv, e), at(rv, e), at(zv, e), rf.mu[j + e],
                                       a1, a2, c));
            *reinterpret_cast<vt *>(rf.res + o) = out;
          }
        else
          *reinterpret_cast<vt *>(y + (u64)row * ldy + j) = s;
      }
      // The row sums with the column dots x.y of the same rows (PCG's p.w, FP64,
      // two columns a thread, B even), in the order of dots.hpp: a workgroup
      // takes P column pairs of G blocks, 64 / U row threads of U lanes each; an
      // enriched dof's product is a partial sum of its own, after the blocks'.
      // Saves the separate dot a read of x and y and a launch (16^3 cells,
      // p = 3, 8 columns: 7.9 + 6.3 us for the two)
      template <int U>
      __global__ __launch_bounds__(256) void slotSumDotK(
        const RowHead *__restrict__ heads, const u32 *__restrict__ rest,
        const u32 *__restrict__ enrOff, const u32 *__restrict__ enrSlots, u32 nC, u32 nE,
        const double *__restrict__ slots, u32 B, double *x, double *y, u32 nBlocks, u32 P, u32 G,
        double *__restrict__ partials)
      {
        using T         = double;
        using vt        = Vec<double, 2>::type;
        constexpr u32 R = DOT_LANES / U;
        __shared__ EnrReduce<T> red;
        __shared__ vt           sum[256];
        const u32 nb = (B + EnrReduce<T>::CB - 1) / EnrReduce<T>::CB, nParts = nBlocks + nE;
        if (blockIdx.x < nE * nb)
          {
            const u32 g = blockIdx.x / nb;
            const u32 j = (blockIdx.x % nb) * EnrReduce<T>::CB + threadIdx.x % EnrReduce<T>::CB;
            const T   s = red.sum(enrSlots, enrOff[g], enrOff[g + 1], slots, B, j);
            if (threadIdx.x < EnrReduce<T>::CB && j < B)
              {
                const u64 o                               = (u64)(nC + g) * B + j;
                y[o]                                      = s;
                partials[(u64)j * nParts + nBlocks + g] = x[o] * s;
              }
            return;
          }
        const u32  nCh = (B / 2 + P - 1) / P, wg = blockIdx.x - nE * nb;
        const u32  sub = threadIdx.x / (R * P), q = threadIdx.x - sub * R * P, r = q / P;
        const u32  blk = wg / nCh * G + sub, j = (wg % nCh * P + (q - r * P)) * 2;
        const bool on  = sub < G && blk < nBlocks && j < B;
        const u32  nGroups = (nC + DOT_LANES - 1) / DOT_LANES;
        vt         acc[U]{};
        if (on)
          for (u32 g = blk; g < nGroups; g += nBlocks)
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (const u32 row = g * DOT_LANES + r + u * R; row < nC)
                {
                  const RowHead h = heads[row];
                  const u64     o = (u64)row * B + j;
                  if (h.rest >> ROW_COUNT_SHIFT == ROW_ZERO)
                    {
                      *reinterpret_cast<vt *>(y + o) = vt{};
                      *reinterpret_cast<vt *>(x + o) = vt{};
                      continue;
                    }
                  const vt xv = *reinterpret_cast<const vt *>(x + o);
                  const vt s  = rowSum<T, 2>(h, rest, slots, B, j);
                  *reinterpret_cast<vt *>(y + o) = s;
                  acc[u][0] = fma(xv[0], s[0], acc[u][0]);
                  acc[u][1] = fma(xv[1], s[1], acc[u][1]);
                }
        sum[threadIdx.x] = foldLanes(acc);
        __syncthreads();
        // the folds between the row threads, two at a time
#pragma unroll
        for (u32 h = R / 2; h > 0; h /= 4)
          {
            const u32 hh = h / 2;
            vt       *v  = sum + threadIdx.x;
            if (r < (hh ? hh : 1u) && sub < G)
              v[0] = hh ? (v[0] + v[h * P]) + (v[hh * P] + v[(hh + h) * P]) : v[0] + v[h * P];
            __syncthreads();
          }
        if (on && r == 0)
          {
            partials[(u64)j * nParts + blk]       = sum[threadIdx.x][0];
            partials[(u64)(j + 1) * nParts + blk] = sum[threadIdx.x][1];
          }
      }
    } // namespace

    bool slotSumDot(hipStream_t s, const dfx_op *op, const double *slots, View<double> x,
                    View<double> y, double *partials, double *out)
    {
      const u32 nC = op->nClassical, nE = op->nDofs - nC, B = y.B;
      auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
      if (B < 2 || B % 2 || B > 128 || x.ld != B || y.ld != B || !aligned(slots) ||
          !aligned(x.p) || !aligned(y.p) || !nC || nE > DOT_BLOCKS ||
          nC > 0xffffff00u)
        return false;
      const u32 nBlocks = dotBlocks(nC), nv = B / 2;
      const u32 nb      = (B + EnrReduce<double>::CB - 1) / EnrReduce<double>::CB;
      // 4 U column pairs fit beside 64 / U row threads.  A thread's rows wait for
      // each other's lists, so U stays at 4 or less (40 columns, 117 649 rows: U = 8
      // took the solve 3 % longer) and lower where workgroups are few (20 columns,
      // 35 937 rows: 9 %); the pairs spread evenly over the chunks; with one or
      // two pairs a workgroup holds several blocks
      u32 U = nv <= 4 ? 1 : nv <= 8 ? 2 : 4;
      while (U > 1 && (u64)nBlocks * ((nv + 4 * U - 1) / (4 * U)) < 640)
        U /= 2;
      const u32 nCh = (nv + 4 * U - 1) / (4 * U), P = (nv + nCh - 1) / nCh;
      const u32 G    = std::max(1u, 256 / (DOT_LANES / U * P));
      const u32 grid = nE * nb + (nBlocks + G - 1) / G * nCh;
      auto go = [&](auto kern) {
        kern<<<grid, 256, 0, s>>>(op->rowHeads.as<RowHead>(), op->slotRest.as<u32>(),
                                  op->enrSlotOffsets.as<u32>(), op->enrMapSlots.as<u32>(), nC, nE,
                                  slots, B, x.p, y.p, nBlocks, P, G, partials);
      };
      switch (U)
        {
          case 1: go(slotSumDotK<1>); break;
          case 2: go(slotSumDotK<2>); break;
          default: go(slotSumDotK<4>); break;
        }
      checkLaunch("slotSumDot");
      colDotsFinal(s, partials, nBlocks + nE, B, out);
      return true;
    }

    template <class T>
    void slotSum(hipStream_t s, const dfx_op *op, const T *slots, View<T> x, View<T> y,
                 bool zeroX, const ResFuse<T> *rf)
    {
      const u32 nC = op->nClassical, nE = op->nDofs - nC, B = y.B;
      if (!B || !op->nDofs)
        return;
      constexpr u32 V = 16 / sizeof(T);
      auto aligned    = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
      const bool vec  = B % V == 0 && x.ld % V == 0 && y.ld % V == 0 && aligned(slots) &&
                       aligned(x.p) && aligned(y.p) &&
                       (!rf || (aligned(rf->res) && aligned(rf->r0)));
      const u64 grid = (u64)nE * ((B + EnrReduce<T>::CB - 1) / EnrReduce<T>::CB) +
                       ((u64)nC * (vec ? B / V : B) + 255) / 256;
      DFX_REQUIRE(grid < (1ull << 31), "too many columns for the row sums");
      auto go = [&](auto kern) {
        kern<<<(unsigned)grid, 256, 0, s>>>(
          op->rowHeads.as<RowHead>(), op->slotRest.as<u32>(), op->enrSlotOffsets.as<u32>(),
          op->enrMapSlots.as<u32>(), nC, nE, slots, B, x.p, x.ld, y.p, y.ld, zeroX ? 1 : 0,
          rf ? *rf : ResFuse<T>{});
      };
      if (rf)
        vec ? go(slotSumK<T, (int)V, true>) : go(slotSumK<T, 1, true>);
      else
        vec ? go(slotSumK<T, (int)V, false>) : go(slotSumK<T, 1, false>);
      checkLaunch("slotSum");
    }
    template void slotSum<double>(hipStream_t, const dfx_op *, const double *, View<double>,
                                  View<double>, bool, const ResFuse<double> *);
    template void slotSum<float>(hipStream_t, const dfx_op *, const float *, View<float>,
                                 View<float>, bool, const ResFuse<float> *);
  } // namespace k
} // namespace dfx

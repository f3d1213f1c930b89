// The FP64 cell kernels (k_cell.hpp) and the small kernels around the cell
// apply: enriched-row reduction, folded diagonal, cell diagonals, repacking.
#include "k_cell.hpp"
#include "enr_reduce.hpp"

namespace dfx
{
  namespace k
  {
    namespace
    {
      // y[nC + g, j] = sum over the cells of g of yE[slot, j]
      template <class T>
      __global__ __launch_bounds__(256) void enrReduceK(const u32 *__restrict__ off,
                                                        const u32 *__restrict__ slots,
                                                        u32 nC, const T *__restrict__ yE,
                                                        u32 B, T *__restrict__ y, u32 ldy)
      {
        __shared__ EnrReduce<T> red;
        const u32 g = blockIdx.x, j = blockIdx.y * EnrReduce<T>::CB + threadIdx.x % EnrReduce<T>::CB;
        const T   s = red.sum(slots, off[g], off[g + 1], yE, B, j);
        if (threadIdx.x < EnrReduce<T>::CB && j < B)
          y[(u64)(nC + g) * ldy + j] = s;
      }

      template <class T>
      __global__ void repackK(const CellMeta *meta, const u32 *pos, const u32 *order,
                              const double *raw, const u64 *rawOff, T *frag)
      {
        constexpr int G  = Mfma<T>::G;
        constexpr int KB = 4 * G;
        const CellMeta cm = meta[pos[blockIdx.x]];
        const u32      e  = order[pos[blockIdx.x]];
        const int      n  = (int)cm.n;
        const int      mt = (n + 15) >> 4;
        const int      nkb  = (n + KB - 1) / KB;
        const u64      tot  = (u64)mt * nkb * 64 * G;
        const double  *A    = raw + rawOff[e];
        T             *F    = frag + (sizeof(T) == 8 ? cm.fragOff64 : cm.fragOff32);
        for (u64 idx = threadIdx.x; idx < tot; idx += blockDim.x)
          {
            const int s    = (int)(idx % G);
            const u64 q    = idx / G;
            const int lane = (int)(q % 64);
            const u64 blk  = q / 64;
            const int kb   = (int)(blk % nkb);
            const int mtile = (int)(blk / nkb);
            const int j    = mtile * 16 + (lane & 15);
            const int kk   = kb * KB + G * (lane >> 4) + s;
            F[idx] = (j < n && kk < n) ? (T)A[(u64)kk + (u64)n * j] : (T)0;
          }
      }


      // content hash of every cell's matrix (words mixed with their place), one
      // workgroup per cell
      __global__ __launch_bounds__(256) void cellHashK(const u64 *__restrict__ raw,
                                                       const u64 *__restrict__ off,
                                                       u64 *__restrict__ out)
      {
        __shared__ u64 sm[256];
        const u64      o = off[blockIdx.x], n = off[blockIdx.x + 1] - o;
        u64            acc = 0;
        for (u64 i = threadIdx.x; i < n; i += 256)
          {
            u64 z = raw[o + i] + (i + 1) * 0x9e3779b97f4a7c15ull; // splitmix64 finalizer
            z     = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
            z     = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
            acc += z ^ (z >> 31);
          }
        sm[threadIdx.x] = acc;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1)
          {
            if ((int)threadIdx.x < w)
              sm[threadIdx.x] += sm[threadIdx.x + w];
            __syncthreads();
          }
        if (threadIdx.x == 0)
          out[blockIdx.x] = sm[0];
      }

      // differs[b] = 1 when cells a[b] and c[b] (of one size) differ in any bit
      __global__ __launch_bounds__(256) void cellDiffersK(const u64 *__restrict__ raw,
                                                          const u64 *__restrict__ off,
                                                          const u32 *__restrict__ a,
                                                          const u32 *__restrict__ c,
                                                          u32 *__restrict__ differs)
      {
        const u64 oa = off[a[blockIdx.x]], oc = off[c[blockIdx.x]],
                  n  = off[a[blockIdx.x] + 1] - oa;
        int diff = 0;
        for (u64 i = threadIdx.x; i < n; i += 256)
          diff |= raw[oa + i] != raw[oc + i];
        diff = __syncthreads_or(diff);
        if (threadIdx.x == 0)
          differs[blockIdx.x] = diff ? 1u : 0u;
      }

    } // namespace

    namespace
    {
      __global__ void gatherDiagK(const double *d, const u32 *map, u64 n, u32 nC, double *out)
      {
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            const u32 m = map[t];
            out[t]      = m < nC ? d[m] : 1.0;
          }
      }
    } // namespace

    void gatherDiag(hipStream_t s, const double *d, const u32 *map, u64 n, u32 nC,
                    double *out)
    {
      if (!n)
        return;
      const u64 g = (n + 255) / 256;
      gatherDiagK<<<(unsigned)(g > 65536 ? 65536 : g), 256, 0, s>>>(d, map, n, nC, out);
      checkLaunch("gatherDiag");
    }

    template <class T>
    void enrichedReduce(hipStream_t s, const dfx_op *op, const T *yE, View<T> y)
    {
      const u32 nE = op->nDofs - op->nClassical;
      if (!nE || !y.B)
        return;
      DFX_REQUIRE((y.B + 15) / 16 <= 65535, "too many columns for the enriched reduction");
      enrReduceK<T><<<dim3(nE, (y.B + 15) / 16), 256, 0, s>>>(
        op->enrSlotOffsets.as<u32>(), op->enrSlots.as<u32>(), op->nClassical, yE, y.B,
        y.p, y.ld);
      checkLaunch("enrichedReduce");
    }

    namespace
    {
      // one block per cell (launch order): diagonal entry i of the cell's
      // FP64 fragment-ordered matrix.  Entry (lane l, value v) of block
      // (mt, kb) holds A_e^T[mt 16 + l % 16][kb 8 + 2 (l / 16) + v], so A_e(i, i)
      // sits at mt = i / 16, kb = i / 8, l = 16 ((i % 8) / 2) + i % 16, v = i % 2
      __global__ void cellDiagK(const CellMeta *__restrict__ meta,
                                const double *__restrict__ frag, double *__restrict__ out)
      {
        const CellMeta cm  = meta[blockIdx.x];
        const u32      nkb = (cm.n + 7) / 8;
        for (u32 i = threadIdx.x; i < cm.n; i += blockDim.x)
          {
            const u32 mt = i / 16, kb = i / 8, l = 16 * ((i % 8) / 2) + i % 16, v = i % 2;
            out[cm.mapOff + i] = frag[cm.fragOff64 + ((u64)(mt * nkb + kb) * 64 + l) * 2 + v];
          }
      }
    } // namespace

    void cellDiag(hipStream_t s, const dfx_op *op, double *out)
    {
      if (!op->nCells)
        return;
      cellDiagK<<<op->nCells, 256, 0, s>>>(op->meta.as<CellMeta>(), op->frag64.as<double>(),
                                           out);
      checkLaunch("cellDiag");
    }

    template <class T>
    void repackCells(hipStream_t s, const dfx_op *op, u32 nPos, const u32 *pos, const u32 *order,
                     const double *raw, const u64 *rawOffsets, T *frag)
    {
      if (!nPos)
        return;
      repackK<T><<<nPos, 256, 0, s>>>(op->meta.as<CellMeta>(), pos, order, raw, rawOffsets, frag);
      checkLaunch("repackCells");
    }

    void cellHashes(hipStream_t s, u32 nCells, const double *raw, const u64 *rawOffsets,
                    u64 *out)
    {
      cellHashK<<<nCells, 256, 0, s>>>(reinterpret_cast<const u64 *>(raw), rawOffsets, out);
      checkLaunch("cellHashes");
    }

    void cellsDiffer(hipStream_t s, u32 n, const double *raw, const u64 *rawOffsets, const u32 *a,
                     const u32 *b, u32 *differs)
    {
      cellDiffersK<<<n, 256, 0, s>>>(reinterpret_cast<const u64 *>(raw), rawOffsets, a, b,
                                     differs);
      checkLaunch("cellsDiffer");
    }

    template void enrichedReduce<double>(hipStream_t, const dfx_op *, const double *,
                                         View<double>);
    template void enrichedReduce<float>(hipStream_t, const dfx_op *, const float *,
                                        View<float>);
    template void repackCells<double>(hipStream_t, const dfx_op *, u32, const u32 *, const u32 *,
                                      const double *, const u64 *, double *);
    template void repackCells<float>(hipStream_t, const dfx_op *, u32, const u32 *, const u32 *,
                                     const double *, const u64 *, float *);
    DFX_INST_CELL(double)
  } // namespace k
} // namespace dfx

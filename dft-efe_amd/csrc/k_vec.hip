// Streaming kernels of libdfx: vector updates of the Chebyshev recurrences,
// column reductions, constraint distribution and the stand-alone cell
// gather / scatter.  All HBM-bound; written as grid-stride loops over
// N x B views with a leading dimension (column blocks of a wider multivector
// are addressed in place, without the reference's per-dof copy loops,
// src/linearAlgebra/ChebyshevFilteredEigenSolver.t.cpp:246-333).
#include <algorithm>
#include <type_traits>
#include <vector>

#include "dots.hpp"
#include "kernels.hpp"
#include "res_update.hpp"

namespace dfx
{
  namespace k
  {
    namespace
    {
      constexpr int TPB = 256;

      inline unsigned gridFor(u64 n)
      {
        u64 g = (n + TPB - 1) / TPB;
        if (g > 65536ull * 8)
          g = 65536ull * 8;
        return (unsigned)(g ? g : 1);
      }

      // flat index -> (row, col) of an N x B view
      struct RC
      {
        u32 i, j;
      };
      __device__ inline RC rc(u64 t, u32 B)
      {
        if ((t >> 32) == 0) // 32-bit division while the flat index fits
          {
            const u32 tt = (u32)t, i = tt / B;
            return {i, tt - i * B};
          }
        u32 i = (u32)(t / B);
        return {i, (u32)(t - (u64)i * B)};
      }

      template <class T>
      __global__ void fillK(T *x, u32 N, u32 B, u32 ld, T v)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC r = rc(t, B);
            x[(u64)r.i * ld + r.j] = v;
          }
      }

      // SplitMix64 (Steele, Lea, Flood 2014): output t is the mix of
      // seed + (t + 1) * golden gamma, so every element is independent
      template <class T>
      __global__ void fillRandomK(T *x, u32 N, u32 B, u32 ld, u64 seed, double a, double b)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            u64 z = seed + (t + 1) * 0x9E3779B97F4A7C15ULL;
            z     = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
            z     = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
            z     = z ^ (z >> 31);
            const double u = (double)(z >> 11) * (1.0 / 9007199254740992.0);
            RC r = rc(t, B);
            x[(u64)r.i * ld + r.j] = (T)(a + (b - a) * u);
          }
      }

      template <class To, class Ti>
      __global__ void convertK(To *y, u32 ldy, const Ti *x, u32 ldx, u32 N, u32 B)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC r = rc(t, B);
            y[(u64)r.i * ldy + r.j] = (To)x[(u64)r.i * ldx + r.j];
          }
      }

      template <class T>
      __global__ void axpbyK(T *z, u32 ldz, T a, const T *x, u32 ldx, T b,
                             const T *y, u32 ldy, u32 N, u32 B)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC r  = rc(t, B);
            T  xv = x[(u64)r.i * ldx + r.j], yv = y[(u64)r.i * ldy + r.j];
            z[(u64)r.i * ldz + r.j] = a * xv + b * yv;
          }
      }

      // one element of the blocked axpby (shared with the residual filter's
      // result and the fused CG update): the multiply-add written out, so
      // that the rounding does not depend on which operands the compiler
      // sees as constants
      template <class T>
      __device__ inline T axpbyOne(T a1, double a, T xv, T b1, double b, T yv)
      {
        return fma(b1 * (T)b, yv, a1 * (T)a * xv);
      }

      template <class T>
      __global__ void axpbyBlockedK(T *z, u32 ldz, T a1, const double *a,
                                    const T *x, u32 ldx, T b1, const double *b,
                                    const T *y, u32 ldy, u32 N, u32 B)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC r  = rc(t, B);
            T  xv = x[(u64)r.i * ldx + r.j], yv = y[(u64)r.i * ldy + r.j];
            z[(u64)r.i * ldz + r.j] = axpbyOne<T>(a1, a[r.j], xv, b1, b[r.j], yv);
          }
      }

      // PCG search direction p = d o r + beta p with beta = zrNew / zr per
      // column (the division of the separate beta launch, the diagonal
      // scaling's product, then the blocked axpby's element with unit
      // coefficients); V columns per thread
      template <int V>
      __global__ void cgDirectionK(double *p, const double *r, const double *d,
                                   const double *zrNew, const double *zr, u32 N, u32 B)
      {
        typedef double vt __attribute__((ext_vector_type(2)));
        const u64 n = (u64)N * B / V;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC        c = rc(t, B / V);
            const u64 o = (u64)c.i * B + c.j * V;
            double    rv[V], pv[V];
            if constexpr (V == 2)
              {
                const vt a = *reinterpret_cast<const vt *>(r + o);
                const vt b = *reinterpret_cast<const vt *>(p + o);
                rv[0] = a[0], rv[1] = a[1], pv[0] = b[0], pv[1] = b[1];
              }
            else
              rv[0] = r[o], pv[0] = p[o];
#pragma unroll
            for (int e = 0; e < V; ++e)
              {
                const u32    j    = c.j * V + e;
                const double beta = zrNew[j] / zr[j];
                pv[e]             = axpbyOne<double>(1.0, 1.0, d[c.i] * rv[e], 1.0, beta, pv[e]);
              }
            if constexpr (V == 2)
              *reinterpret_cast<vt *>(p + o) = vt{pv[0], pv[1]};
            else
              p[o] = pv[0];
          }
      }

      template <class T>
      __global__ void diagScaleK(T *y, u32 ldy, const double *d, const T *x,
                                 u32 ldx, u32 N, u32 B)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC r = rc(t, B);
            y[(u64)r.i * ldy + r.j] = (T)d[r.i] * x[(u64)r.i * ldx + r.j];
          }
      }

      // y_E[i, j] = sum_k E[i + nE k] x_E[k, j]: one workgroup per row i and
      // 64 columns; four k lanes per column each add k = lane, lane + 4, ...
      // in ascending order, combined in lane order (fixed, deterministic)
      template <class T>
      __global__ __launch_bounds__(256) void enrBlockK(T *y, u32 ldy, const double *E,
                                                       const T *x, u32 ldx, u32 nC, u32 nE,
                                                       u32 B)
      {
        __shared__ T part[4][64];
        const u32 i = blockIdx.x, cj = threadIdx.x % 64, kl = threadIdx.x / 64;
        const u32 j = blockIdx.y * 64 + cj;
        T         acc = 0;
        if (j < B)
          {
            // eight k of a lane loaded before they are added (in the same
            // ascending order), so that the loads are in flight together
            u32 kk = kl;
            for (; kk + 28 < nE; kk += 32)
              {
                T ev[8], xv[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                  {
                    const u32 k = kk + 4u * u;
                    ev[u]       = (T)E[i + (u64)nE * k];
                    xv[u]       = x[(u64)(nC + k) * ldx + j];
                  }
#pragma unroll
                for (int u = 0; u < 8; ++u)
                  acc += ev[u] * xv[u];
              }
            for (; kk < nE; kk += 4)
              acc += (T)E[i + (u64)nE * kk] * x[(u64)(nC + kk) * ldx + j];
          }
        part[kl][cj] = acc;
        __syncthreads();
        if (kl == 0 && j < B)
          y[(u64)(nC + i) * ldy + j] = ((part[0][cj] + part[1][cj]) + part[2][cj]) + part[3][cj];
      }

      // pass 1 of the column dots in the order of dots.hpp.  A workgroup takes C
      // columns of NB blocks: C columns x R row threads, each of U lanes of every
      // block.  Two blocks for 8 columns, so that four rows of a thread are in
      // flight together (117 649 rows, 1 column: update 9.1 -> 6.9 us)
      template <int C>
      struct DotShape
      {
        static constexpr int R = TPB / C, U = DOT_LANES / R, NB = U < 4 ? 4 / U : 1;
        static_assert(R <= DOT_LANES && NB * U % 4 == 0, "whole lanes, batches of four rows");
      };
      template <int C>
      struct DotPlace
      {
        using S = DotShape<C>;
        u32 blk, j, nBlocks, nGroups, N; // the first block, this thread's column
        int ty;
        __device__ DotPlace(u32 N_, u32 B, u32 nBlocks_)
          : nBlocks(nBlocks_), nGroups((u32)(((u64)N_ + DOT_LANES - 1) / DOT_LANES)), N(N_),
            ty(threadIdx.x / C)
        {
          const u32 nCh = (B + C - 1) / C, w = blockIdx.x / nCh;
          blk           = w * S::NB;
          j             = (blockIdx.x - w * nCh) * C + threadIdx.x % C;
        }
        // calls load(t, row) for four rows, then use(t, block, lane, row).  In
        // place of a row that is not there the first one is loaded again, and not
        // used: with a branch per load each waited for the one before
        template <class Load, class Use>
        __device__ inline void rows(Load load, Use use) const
        {
          for (u32 g = blk; g < nGroups; g += nBlocks)
#pragma unroll
            for (int f = 0; f < S::NB * S::U; f += 4)
              {
                u32  row[4];
                bool ok[4];
#pragma unroll
                for (int t = 0; t < 4; ++t)
                  {
                    const u32 nb = (f + t) / S::U, u = (f + t) % S::U;
                    row[t]       = (g + nb) * DOT_LANES + ty + u * S::R;
                    ok[t]        = blk + nb < nBlocks && g + nb < nGroups && row[t] < N;
                    row[t]       = ok[t] ? row[t] : t ? row[0] : N - 1;
                  }
#pragma unroll
                for (int t = 0; t < 4; ++t)
                  load(t, row[t]);
#pragma unroll
                for (int t = 0; t < 4; ++t)
                  if (ok[t])
                    use(t, (f + t) / S::U, (f + t) % S::U, row[t]);
              }
        }
        // the columns' sums over the blocks, M of them per column: every thread
        // leaves its lanes' folds in LDS, the i-th set of C threads folds those of
        // sum i / NB and block i % NB and calls put(sum, block, value)
        template <int M, class Put>
        __device__ inline void sums(double (&acc)[M][S::NB][S::U], u32 B, Put put) const
        {
          __shared__ double red[M][S::NB][TPB];
#pragma unroll
          for (int m = 0; m < M; ++m)
#pragma unroll
            for (int nb = 0; nb < S::NB; ++nb)
              red[m][nb][threadIdx.x] = foldLanes(acc[m][nb]);
          __syncthreads();
          const int m = ty / S::NB, nb = ty % S::NB;
          if (m >= M || j >= B || blk + nb >= nBlocks)
            return;
          double v[S::R];
#pragma unroll
          for (int q = 0; q < S::R; ++q)
            v[q] = red[m][nb][q * C + threadIdx.x % C];
          put(m, blk + nb, foldLanes(v));
        }
      };
      // calls go(columns, workgroups) with the widest shape that leaves the GPU
      // a workgroup per CU: wide ones read a row's lines whole, but a small vector
      // has few blocks (N = 1331: 21).  16 columns at least: with 8 the update of
      // 29 791 x 10 values took 8.4 us instead of 5.4
      template <class Go>
      void dotShape(u32 N, u32 B, Go go)
      {
        const u32 nBlocks = dotBlocks(N);
        u32       C       = B <= 8 ? 8 : B <= 16 ? 16 : B <= 32 ? 32 : 64;
        while (C > 16 && (u64)nBlocks * ((B + C - 1) / C) < 256)
          C /= 2;
        auto launch = [&](auto c) {
          constexpr u32 W = decltype(c)::value, NB = DotShape<W>::NB;
          const u64     grid = (u64)((nBlocks + NB - 1) / NB) * ((B + W - 1) / W);
          DFX_REQUIRE(grid < (1ull << 31), "too many columns for the dots");
          go(c, (unsigned)grid);
        };
        switch (C)
          {
            case 8: return launch(std::integral_constant<int, 8>{});
            case 16: return launch(std::integral_constant<int, 16>{});
            case 32: return launch(std::integral_constant<int, 32>{});
            default: return launch(std::integral_constant<int, 64>{});
          }
      }

      // partials: column-major, nParts of them per column
      template <class T, int C>
      __global__ __launch_bounds__(TPB) void colDotsK(const T *x, u32 ldx, const T *y, u32 ldy,
                                                      u32 N, u32 B, u32 nBlocks, u32 nParts,
                                                      double *partials)
      {
        using S = DotShape<C>;
        const DotPlace<C> at(N, B, nBlocks);
        const u32         j = at.j;
        double            acc[1][S::NB][S::U]{};
        if (j < B)
          {
            T xv[4], yv[4];
            at.rows([&](int t, u32 i) { xv[t] = x[(u64)i * ldx + j], yv[t] = y[(u64)i * ldy + j]; },
                    [&](int t, int nb, int u, u32) {
                      acc[0][nb][u] = fma((double)xv[t], (double)yv[t], acc[0][nb][u]);
                    });
          }
        at.sums(acc, B,
                [&](int, u32 blk, double s) { partials[(u64)j * nParts + blk] = s; });
      }

      // rows whose dot is a partial sum of its own, after `first` others
      __global__ void rowProductsK(const double *x, u32 ldx, const double *y, u32 ldy, u32 N,
                                   u32 B, u32 first, u32 nParts, double *partials)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            const RC r = rc(t, B);
            partials[(u64)r.j * nParts + first + r.i] =
              x[(u64)r.i * ldx + r.j] * y[(u64)r.i * ldy + r.j];
          }
      }

      // The PCG update of one iteration with a Jacobi preconditioner, fused:
      //   xn = x + alpha p, r -= alpha w, and the partial sums of z.r and r.r
      // with z = d o r (alpha = zr / pw per column, formed here as cgAlphaK
      // does; z itself is formed again where it is used).
      // Rows, lanes and sums follow colDotsK exactly, and each element is the
      // blocked axpby's / the diagonal scaling's expression, so every value is the
      // separate launches' bit for bit.  partials: those of z.r in columns
      // [0, B), of r.r in [B, 2B); N x B arrays with leading dimension B.
      // Bound by memory: 4 reads and 2 writes per value (with z, a copy of x and
      // 16 lanes for 8 columns it took 15.5 us at 117 649 x 8, now 9.1)
      template <int C>
      __global__ __launch_bounds__(TPB) void cgUpdateK(const double *x, double *xn, double *r,
                                                       const double *p, const double *w,
                                                       const double *d, const double *zr,
                                                       const double *pw, u32 N, u32 B,
                                                       u32 nBlocks, double *partials)
      {
        using S = DotShape<C>;
        const DotPlace<C> at(N, B, nBlocks);
        const u32         j = at.j;
        double            acc[2][S::NB][S::U]{}; // z.r, r.r
        if (j < B)
          {
            const double alpha = zr[j] / pw[j], nalpha = -zr[j] / pw[j];
            double       xv[4], pv[4], rv[4], wv[4], dv[4];
            at.rows(
              [&](int t, u32 i) {
                const u64 o = (u64)i * B + j;
                xv[t] = x[o], pv[t] = p[o], rv[t] = r[o], wv[t] = w[o], dv[t] = d[i];
              },
              [&](int t, int nb, int u, u32 i) {
                const u64    o  = (u64)i * B + j;
                const double rn = axpbyOne<double>(1.0, 1.0, rv[t], 1.0, nalpha, wv[t]);
                const double zn = dv[t] * rn;
                xn[o]         = axpbyOne<double>(1.0, 1.0, xv[t], 1.0, alpha, pv[t]);
                r[o]          = rn;
                acc[0][nb][u] = fma(zn, rn, acc[0][nb][u]);
                acc[1][nb][u] = fma(rn, rn, acc[1][nb][u]);
              });
          }
        at.sums(acc, B, [&](int m, u32 blk, double s) {
          partials[((u64)m * B + j) * nBlocks + blk] = s;
        });
      }

      // partial sums of |a1 a_j x_ij + b1 b_j y_ij|^2 per column without
      // writing the combination: colDotsK's rows, lanes and folds and the
      // blocked axpby's element, so the norms are those of the separate
      // launches bit for bit (N x B arrays with leading dimension B)
      template <int C>
      __global__ __launch_bounds__(TPB) void combNormsK(double a1, const double *a,
                                                        const double *x, double b1,
                                                        const double *b, const double *y, u32 N,
                                                        u32 B, u32 nBlocks, double *partials)
      {
        using S = DotShape<C>;
        const DotPlace<C> at(N, B, nBlocks);
        const u32         j = at.j;
        double            acc[1][S::NB][S::U]{};
        if (j < B)
          {
            const double aj = a[j], bj = b[j];
            double       xv[4], yv[4];
            at.rows([&](int t, u32 i) { xv[t] = x[(u64)i * B + j], yv[t] = y[(u64)i * B + j]; },
                    [&](int t, int nb, int u, u32) {
                      const double v = axpbyOne<double>(a1, aj, xv[t], b1, bj, yv[t]);
                      acc[0][nb][u]  = fma(v, v, acc[0][nb][u]);
                    });
          }
        at.sums(acc, B,
                [&](int, u32 blk, double s) { partials[(u64)j * nBlocks + blk] = s; });
      }

      // one workgroup per column: thread t adds partials t, t + 256, ... in
      // order, then a fixed-shape tree over the 256 sums (deterministic; the
      // partial count depends on the rows only, so a column's result does not
      // depend on how many columns share the call).  Columns from hostFrom on
      // also go to host (pinned memory).  All latency: eight loads are in
      // flight together, the tree's last six levels stay in one wave, and a
      // column's partials lie side by side (117 649 rows, 8 columns: the solve
      // 5 % shorter than with a row of columns per block)
      __global__ __launch_bounds__(256) void colDotsFinalK(const double *partials, u32 nBlocks,
                                                           double *out, double *host,
                                                           u32 hostFrom)
      {
        __shared__ double red[256];
        const u32 j = blockIdx.x;
        double    s = 0.0;
        for (u32 b = threadIdx.x; b < nBlocks; b += 8 * 256)
          {
            double v[8];
#pragma unroll
            for (u32 k = 0; k < 8; ++k)
              if (b + k * 256 < nBlocks)
                v[k] = partials[(u64)j * nBlocks + b + k * 256];
#pragma unroll
            for (u32 k = 0; k < 8; ++k)
              if (b + k * 256 < nBlocks)
                s += v[k];
          }
        red[threadIdx.x] = s;
        __syncthreads();
        if (threadIdx.x >= 64)
          return;
        // the tree's levels 128 and 64, then within the wave
        s = (red[threadIdx.x] + red[threadIdx.x + 128]) +
            (red[threadIdx.x + 64] + red[threadIdx.x + 192]);
#pragma unroll
        for (int w = 32; w > 0; w >>= 1)
          s += __shfl_down(s, w);
        if (threadIdx.x == 0)
          {
            out[j] = s;
            if (host && j >= hostFrom)
              __hip_atomic_store(host + (j - hostFrom), s, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_SYSTEM);
          }
      }

      template <class T>
      __global__ void chebStepK(T *xp, u32 ldp, const T *hx, u32 ldh,
                                const double *dinv, const T *tE, u32 ldt, u32 nC,
                                const T *xk, u32 ldk, T alpha, T beta, T gamma,
                                u32 N, u32 B)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC r = rc(t, B);
            T  tv;
            if (r.i < nC)
              tv = (T)dinv[r.i] * hx[(u64)r.i * ldh + r.j];
            else
              tv = tE[(u64)r.i * ldt + r.j];
            const T s1 = alpha * tv + beta * xk[(u64)r.i * ldk + r.j];
            T      &o  = xp[(u64)r.i * ldp + r.j];
            o          = (T)1 * s1 + gamma * o;
          }
      }

      template <class T>
      __global__ void resStepK(T *res, u32 ldr, const T *s2, u32 lds, const T *rn,
                               u32 ldn, const T *r0, u32 ld0, const double *mu,
                               const double *coef, u32 N, u32 B)
      {
        const u64 n      = (u64)N * B;
        const T   alpha1 = (T)coef[0], alpha2 = (T)coef[1], c = (T)coef[2];
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC r = rc(t, B);
            T &o = res[(u64)r.i * ldr + r.j];
            o    = resUpdate<T>(s2[(u64)r.i * lds + r.j], rn[(u64)r.i * ldn + r.j], o,
                                r0[(u64)r.i * ld0 + r.j], mu[r.j], alpha1, alpha2, c);
          }
      }

      // resStepK on contiguous N x B arrays (every leading dimension B) with
      // B a multiple of the 16-byte vector: one vector of V columns per
      // thread, the same arithmetic per element
      template <class T>
      __global__ void resStepVecK(T *__restrict__ res, const T *__restrict__ s2,
                                  const T *__restrict__ rn, const T *__restrict__ r0,
                                  const double *__restrict__ mu,
                                  const double *__restrict__ coef, u32 nVec, u32 B)
      {
        constexpr int V = 16 / sizeof(T);
        typedef T vt __attribute__((ext_vector_type(V)));
        const T alpha1 = (T)coef[0], alpha2 = (T)coef[1], c = (T)coef[2];
        for (u32 t = blockIdx.x * blockDim.x + threadIdx.x; t < nVec;
             t += gridDim.x * blockDim.x)
          {
            const u32 j0 = (t * V) % B;
            const vt  a  = reinterpret_cast<const vt *>(s2)[t];
            const vt  b  = reinterpret_cast<const vt *>(rn)[t];
            const vt  z  = reinterpret_cast<const vt *>(r0)[t];
            vt        o  = reinterpret_cast<const vt *>(res)[t];
#pragma unroll
            for (int e = 0; e < V; ++e)
              o[e] = resUpdate<T>(a[e], b[e], o[e], z[e], mu[j0 + e], alpha1, alpha2, c);
            reinterpret_cast<vt *>(res)[t] = o;
          }
      }

      // content hash of n 64-bit words: the wrapping sum over i of
      // mix(x[i] + (i + 1) golden), mix the splitmix64 finalizer; a sum, so
      // the value does not depend on the order the blocks add up in
      __device__ inline u64 mix64(u64 z)
      {
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        return z ^ (z >> 31);
      }
      __global__ __launch_bounds__(256) void hashWordsK(const u64 *__restrict__ x, u64 n,
                                                        u64 *__restrict__ partials)
      {
        __shared__ u64 sm[256];
        u64            acc = 0;
        for (u64 i = blockIdx.x * 256ull + threadIdx.x; i < n; i += (u64)gridDim.x * 256)
          acc += mix64(x[i] + (i + 1) * 0x9e3779b97f4a7c15ull);
        sm[threadIdx.x] = acc;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1)
          {
            if ((int)threadIdx.x < w)
              sm[threadIdx.x] += sm[threadIdx.x + w];
            __syncthreads();
          }
        if (threadIdx.x == 0)
          partials[blockIdx.x] = sm[0];
      }

      // the residual step on the rows a fused cell apply leaves to it (listed
      // in `rows`: constrained, enriched and cell-less rows), after the
      // enriched reduction and the child->parent step have finished y there
      template <class T>
      __global__ void resFixK(T *res, const T *s2, u32 lds, const T *rn, const T *r0, u32 ld,
                              const u32 *__restrict__ rows, u32 nRows,
                              const double *mu, const double *coef, u32 B)
      {
        const u64 n      = (u64)nRows * B;
        const T   alpha1 = (T)coef[0], alpha2 = (T)coef[1], c = (T)coef[2];
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            const RC  r = rc(t, B);
            const u32 i = rows[r.i];
            const u64 o = (u64)i * ld + r.j;
            res[o]      = resUpdate<T>(s2[(u64)i * lds + r.j], rn[o], res[o], r0[o], mu[r.j],
                                       alpha1, alpha2, c);
          }
      }

      // residual filter set-up from the FP64 seed Y (ChebyshevFilter.t.cpp:
      // 330-359): r0 = Y, rn = a Y + b Y (a = alpha1, b = 0, the reference's
      // axpby), res = 0, in T; the same arithmetic as the separate
      // convert / axpby / convert / fill launches
      template <class T>
      __device__ inline void resSeedOne(double y, double a, double b, T &r0, T &rn, T &res)
      {
        r0  = (T)y;
        rn  = (T)fma(a, y, b * y);
        res = (T)0.0;
      }

      template <class T>
      __global__ void resSeedK(T *r0, T *rn, T *res, u32 ld, const double *Y, u32 ldy,
                               double a, double b, u32 N, u32 B)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC        r = rc(t, B);
            const u64 o = (u64)r.i * ld + r.j;
            resSeedOne<T>(Y[(u64)r.i * ldy + r.j], a, b, r0[o], rn[o], res[o]);
          }
      }

      // the seed from kept products: Y = AX - lambda o BX (the blocked
      // axpby's element) is formed in registers and converted as resSeedK
      // does, without being written
      template <class T>
      __global__ void resSeedFromK(T *r0, T *rn, T *res, u32 ld, const double *AX,
                                   const double *BX, u32 ldp, const double *ones,
                                   const double *lam, double a, double b, u32 N, u32 B)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC           r = rc(t, B);
            const u64    p = (u64)r.i * ldp + r.j, o = (u64)r.i * ld + r.j;
            const double y = axpbyOne<double>(1.0, ones[r.j], AX[p], -1.0, lam[r.j], BX[p]);
            resSeedOne<T>(y, a, b, r0[o], rn[o], res[o]);
          }
      }

      // residual filter result (ChebyshevFilter.t.cpp:424-441): z = a1 a[j]
      // (double) x + b1 b[j] y with x the last residual in T; the arithmetic of
      // a conversion followed by the FP64 blocked axpby
      template <class T>
      __global__ void resFinalK(double *z, u32 ldz, double a1, const double *a, const T *x,
                                u32 ldx, double b1, const double *b, const double *y, u32 ldy,
                                u32 N, u32 B)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC           r  = rc(t, B);
            const double xv = (double)x[(u64)r.i * ldx + r.j], yv = y[(u64)r.i * ldy + r.j];
            z[(u64)r.i * ldz + r.j] = axpbyOne<double>(a1, a[r.j], xv, b1, b[r.j], yv);
          }
      }

      // resFinalK with the diagonal apply folded in: x[i, j] = (T)(d[i] r[i, j])
      // on the first nC rows (diagScaleK's product), xE[i, j] below them
      template <class T>
      __global__ void resFinalDiagK(double *z, u32 ldz, double a1, const double *a,
                                    const T *r, const double *d, u32 nC, const T *xE, u32 ldx,
                                    double b1, const double *b, const double *y, u32 ldy,
                                    u32 N, u32 B)
      {
        const u64 n = (u64)N * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC        rr = rc(t, B);
            const u64 o  = (u64)rr.i * ldx + rr.j;
            const T   xt = rr.i < nC ? (T)d[rr.i] * r[o] : xE[o];
            const double xv = (double)xt, yv = y[(u64)rr.i * ldy + rr.j];
            z[(u64)rr.i * ldz + rr.j] = axpbyOne<double>(a1, a[rr.j], xv, b1, b[rr.j], yv);
          }
      }

      // ------------------------------------------------ constraints
      // ConstraintsInternal.cpp:38-107 restated per (row, column): the row's
      // value is inhom + sum_j w_j x[col_j] accumulated with fma in entry order.
      template <class T>
      __global__ void p2cK(T *x, u32 ld, const u32 *rows, const u32 *rowOff,
                           const u32 *cols, const double *w, const double *inhom,
                           u32 nRows, u32 B)
      {
        const u64 n = (u64)nRows * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC  r  = rc(t, B);
            T   v  = (T)inhom[r.i];
            u32 e0 = rowOff[r.i], e1 = rowOff[r.i + 1];
            for (u32 e = e0; e < e1; ++e)
              v = fma((T)w[e], x[(u64)cols[e] * ld + r.j], v);
            x[(u64)rows[r.i] * ld + r.j] = v;
          }
      }

      // ConstraintsInternal.cpp:113-170 without atomics: each parent gathers
      // w * x[row] from its children in the rows' order, which is the order
      // of the reference's sequential loop, so the result is identical.
      template <class T>
      __global__ void c2pParentsK(T *y, u32 ld, const u32 *par, const u32 *parOff,
                                  const u32 *parRowDof, const double *parW,
                                  u32 nPar, u32 B)
      {
        const u64 n = (u64)nPar * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC  r   = rc(t, B);
            T  &dst = y[(u64)par[r.i] * ld + r.j];
            T   acc = dst;
            u32 e0 = parOff[r.i], e1 = parOff[r.i + 1];
            for (u32 e = e0; e < e1; ++e)
              acc = fma((T)parW[e], y[(u64)parRowDof[e] * ld + r.j], acc);
            dst = acc;
          }
      }

      template <class T>
      __global__ void setRowsK(T *x, u32 ld, const u32 *rows, u32 nRows, u32 B, T v)
      {
        const u64 n = (u64)nRows * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC r = rc(t, B);
            x[(u64)rows[r.i] * ld + r.j] = v;
          }
      }

      // ------------------------------------------------ gather / scatter
      template <class T>
      __global__ void gatherK(const u32 *map, u64 nSlots, const T *x, u32 ldx,
                              T *xc, u32 ldc, u32 B)
      {
        const u64 n = nSlots * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            const u64 s = t / B, j = t - s * B;
            xc[s * ldc + j] = x[(u64)map[s] * ldx + j];
          }
      }

      template <class T>
      __global__ void scatterAddK(const u32 *off, const u32 *slots, u32 nDofs,
                                  const T *yc, u32 ldc, T *y, u32 ldy, u32 B)
      {
        const u64 n = (u64)nDofs * B;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < n;
             t += (u64)gridDim.x * blockDim.x)
          {
            RC r   = rc(t, B);
            T &dst = y[(u64)r.i * ldy + r.j];
            T  acc = dst;
            for (u32 e = off[r.i]; e < off[r.i + 1]; ++e)
              acc += yc[(u64)slots[e] * ldc + r.j];
            dst = acc;
          }
      }
    } // namespace

    // ==================================================== launchers
    template <class T>
    void fill(hipStream_t s, View<T> x, double v)
    {
      const u64 n = (u64)x.N * x.B;
      if (!n)
        return;
      fillK<T><<<gridFor(n), TPB, 0, s>>>(x.p, x.N, x.B, x.ld, (T)v);
      checkLaunch("fill");
    }

    template <class T>
    void fillRandom(hipStream_t s, View<T> x, u64 seed, double a, double b)
    {
      const u64 n = (u64)x.N * x.B;
      if (!n)
        return;
      fillRandomK<T><<<gridFor(n), TPB, 0, s>>>(x.p, x.N, x.B, x.ld, seed, a, b);
      checkLaunch("fillRandom");
    }

    template <class To, class Ti>
    void convert(hipStream_t s, View<To> d, View<const Ti> x)
    {
      const u64 n = (u64)x.N * x.B;
      if (!n)
        return;
      convertK<To, Ti><<<gridFor(n), TPB, 0, s>>>(d.p, d.ld, x.p, x.ld, x.N, x.B);
      checkLaunch("convert");
    }

    template <class T>
    void axpby(hipStream_t s, View<T> z, double a, View<const T> x, double b,
               View<const T> y)
    {
      const u64 n = (u64)z.N * z.B;
      if (!n)
        return;
      axpbyK<T><<<gridFor(n), TPB, 0, s>>>(z.p, z.ld, (T)a, x.p, x.ld, (T)b, y.p,
                                           y.ld, z.N, z.B);
      checkLaunch("axpby");
    }

    template <class T>
    void axpbyBlocked(hipStream_t s, View<T> z, double a1, const double *a,
                      View<const T> x, double b1, const double *b, View<const T> y)
    {
      const u64 n = (u64)z.N * z.B;
      if (!n)
        return;
      axpbyBlockedK<T><<<gridFor(n), TPB, 0, s>>>(z.p, z.ld, (T)a1, a, x.p, x.ld,
                                                  (T)b1, b, y.p, y.ld, z.N, z.B);
      checkLaunch("axpbyBlocked");
    }

    template <class T>
    void diagScale(hipStream_t s, View<T> y, const double *d, View<const T> x,
                   u32 nRowsDiag)
    {
      const u64 n = (u64)nRowsDiag * x.B;
      if (!n)
        return;
      diagScaleK<T><<<gridFor(n), TPB, 0, s>>>(y.p, y.ld, d, x.p, x.ld, nRowsDiag, x.B);
      checkLaunch("diagScale");
    }

    template <class T>
    void enrichedBlock(hipStream_t s, View<T> y, const double *E, View<const T> x,
                       u32 nC, u32 nE)
    {
      const u64 n = (u64)nE * x.B;
      if (!n)
        return;
      enrBlockK<T><<<dim3(nE, (x.B + 63) / 64), 256, 0, s>>>(y.p, y.ld, E, x.p, x.ld, nC, nE,
                                                             x.B);
      checkLaunch("enrichedBlock");
    }

    void colDotsFinal(hipStream_t s, const double *partials, u32 nBlocks, u32 B, double *out,
                      double *host, u32 hostFrom)
    {
      colDotsFinalK<<<B, 256, 0, s>>>(partials, nBlocks, out, host, hostFrom);
      checkLaunch("colDotsFinal");
    }

    namespace
    {
      // pass 1 over the first N rows of x, the first of nParts partial sums
      template <class T>
      void colDotsPartials(hipStream_t s, View<const T> x, View<const T> y, u32 N, u32 nParts,
                           double *partials)
      {
        dotShape(N, x.B, [&](auto c, unsigned grid) {
          colDotsK<T, decltype(c)::value><<<grid, TPB, 0, s>>>(x.p, x.ld, y.p, y.ld, N, x.B,
                                                               dotBlocks(N), nParts, partials);
        });
        checkLaunch("colDots");
      }
    } // namespace

    template <class T>
    void colDots(hipStream_t s, View<const T> x, View<const T> y, double *partials,
                 double *out)
    {
      if (!x.B)
        return;
      const u32 nBlocks = dotBlocks(x.N);
      colDotsPartials<T>(s, x, y, x.N, nBlocks, partials);
      colDotsFinal(s, partials, nBlocks, x.B, out);
    }

    void colDotsApart(hipStream_t s, View<const double> x, View<const double> y, u32 nC,
                      double *partials, double *out)
    {
      const u32 B = x.B, nE = x.N - nC, nBlocks = dotBlocks(nC);
      if (!B)
        return;
      colDotsPartials<double>(s, x, y, nC, nBlocks + nE, partials);
      if (nE)
        {
          rowProductsK<<<gridFor((u64)nE * B), TPB, 0, s>>>(
            x.p + (u64)nC * x.ld, x.ld, y.p + (u64)nC * y.ld, y.ld, nE, B, nBlocks, nBlocks + nE,
            partials);
          checkLaunch("rowProducts");
        }
      colDotsFinal(s, partials, nBlocks + nE, B, out);
    }

    void combinationNorms(hipStream_t s, double a1, const double *a, View<const double> x,
                          double b1, const double *b, View<const double> y, double *partials,
                          double *out)
    {
      const u32 B = x.B, N = x.N;
      if (!B)
        return;
      DFX_REQUIRE(x.ld == B && y.ld == B && y.N == N && y.B == B,
                  "combination norms: contiguous multivectors of one shape expected");
      const u32 nBlocks = dotBlocks(N);
      dotShape(N, B, [&](auto c, unsigned grid) {
        combNormsK<decltype(c)::value><<<grid, TPB, 0, s>>>(a1, a, x.p, b1, b, y.p, N, B, nBlocks,
                                                            partials);
      });
      checkLaunch("combNorms");
      colDotsFinal(s, partials, nBlocks, B, out);
    }

    void cgUpdate(hipStream_t s, View<double> x, View<double> xn, View<double> r,
                  View<const double> p, View<const double> w, const double *d,
                  const double *zr, const double *pw, double *partials, double *zrrr,
                  double *rrHost)
    {
      const u32 B = x.B, N = x.N;
      if (!B)
        return;
      DFX_REQUIRE(x.ld == B && xn.ld == B && r.ld == B && p.ld == B && w.ld == B,
                  "CG update: contiguous multivectors expected");
      const u32 nBlocks = dotBlocks(N);
      dotShape(N, B, [&](auto c, unsigned grid) {
        cgUpdateK<decltype(c)::value><<<grid, TPB, 0, s>>>(x.p, xn.p, r.p, p.p, w.p, d, zr, pw, N,
                                                           B, nBlocks, partials);
      });
      checkLaunch("cgUpdate");
      colDotsFinal(s, partials, nBlocks, 2 * B, zrrr, rrHost, B);
    }

    void cgDirection(hipStream_t s, View<double> p, View<const double> r, const double *d,
                     const double *zrNew, const double *zr)
    {
      const u64 n = (u64)p.N * p.B;
      if (!n)
        return;
      DFX_REQUIRE(p.ld == p.B && r.ld == r.B && r.N == p.N && r.B == p.B,
                  "CG direction: contiguous multivectors of one shape expected");
      if (p.B % 2 == 0) // scratch vectors: 256-byte aligned
        cgDirectionK<2><<<gridFor(n / 2), TPB, 0, s>>>(p.p, r.p, d, zrNew, zr, p.N, p.B);
      else
        cgDirectionK<1><<<gridFor(n), TPB, 0, s>>>(p.p, r.p, d, zrNew, zr, p.N, p.B);
      checkLaunch("cgDirection");
    }

    template <class T>
    void chebStep(hipStream_t s, View<T> xp, View<const T> hx, const double *dinv,
                  View<const T> tE, u32 nC, View<const T> xk, double alpha,
                  double beta, double gamma)
    {
      const u64 n = (u64)xp.N * xp.B;
      if (!n)
        return;
      chebStepK<T><<<gridFor(n), TPB, 0, s>>>(xp.p, xp.ld, hx.p, hx.ld, dinv, tE.p,
                                              tE.ld, nC, xk.p, xk.ld, (T)alpha,
                                              (T)beta, (T)gamma, xp.N, xp.B);
      checkLaunch("chebStep");
    }

    template <class T>
    void resStep(hipStream_t s, View<T> res, View<const T> s2, View<const T> rn,
                 View<const T> r0, const double *mu, const double *coef)
    {
      const u64 n = (u64)res.N * res.B;
      if (!n)
        return;
      constexpr u32 V       = 16 / sizeof(T);
      auto          aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
      if (res.ld == res.B && s2.ld == res.B && rn.ld == res.B && r0.ld == res.B &&
          res.B % V == 0 && n / V < (1ull << 32) && aligned(res.p) && aligned(s2.p) &&
          aligned(rn.p) && aligned(r0.p))
        {
          const u64 nv = n / V;
          resStepVecK<T><<<gridFor(nv), TPB, 0, s>>>(res.p, s2.p, rn.p, r0.p, mu, coef,
                                                     (u32)nv, res.B);
          checkLaunch("resStepVec");
          return;
        }
      resStepK<T><<<gridFor(n), TPB, 0, s>>>(res.p, res.ld, s2.p, s2.ld, rn.p, rn.ld,
                                             r0.p, r0.ld, mu, coef, res.N, res.B);
      checkLaunch("resStep");
    }

    u64 hashWords(hipStream_t s, const void *x, u64 nWords, u64 *partials)
    {
      if (!nWords)
        return 0;
      u64 blocks = (nWords + 255) / 256;
      if (blocks > HASH_BLOCKS)
        blocks = HASH_BLOCKS;
      hashWordsK<<<(unsigned)blocks, 256, 0, s>>>(static_cast<const u64 *>(x), nWords,
                                                  partials);
      checkLaunch("hashWords");
      std::vector<u64> h(blocks);
      DFX_HIP(hipMemcpyAsync(h.data(), partials, blocks * sizeof(u64), hipMemcpyDeviceToHost,
                             s));
      DFX_HIP(hipStreamSynchronize(s));
      u64 sum = 0;
      for (u64 v : h)
        sum += v;
      return sum;
    }

    template <class T>
    void resFix(hipStream_t s, View<T> res, View<const T> s2, View<const T> rn,
                View<const T> r0, const u32 *rows, u32 nRows, const double *mu,
                const double *coef)
    {
      const u64 n = (u64)nRows * res.B;
      if (!n)
        return;
      DFX_REQUIRE(res.ld == rn.ld && rn.ld == r0.ld, "residual fix-up: one leading dimension");
      resFixK<T><<<gridFor(n), TPB, 0, s>>>(res.p, s2.p, s2.ld, rn.p, r0.p, res.ld, rows, nRows,
                                            mu, coef, res.B);
      checkLaunch("resFix");
    }

    template <class T>
    void resSeed(hipStream_t s, View<T> r0, View<T> rn, View<T> res, View<const double> Y,
                 double alpha1)
    {
      const u64 n = (u64)Y.N * Y.B;
      if (!n)
        return;
      DFX_REQUIRE(r0.ld == rn.ld && rn.ld == res.ld, "residual seed: one leading dimension");
      resSeedK<T><<<gridFor(n), TPB, 0, s>>>(r0.p, rn.p, res.p, r0.ld, Y.p, Y.ld, alpha1, 0.0,
                                             Y.N, Y.B);
      checkLaunch("resSeed");
    }

    template <class T>
    void resSeedFrom(hipStream_t s, View<T> r0, View<T> rn, View<T> res, View<const double> AX,
                     View<const double> BX, const double *ones, const double *lam,
                     double alpha1)
    {
      const u64 n = (u64)AX.N * AX.B;
      if (!n)
        return;
      DFX_REQUIRE(r0.ld == rn.ld && rn.ld == res.ld && AX.ld == BX.ld,
                  "residual seed: one leading dimension");
      resSeedFromK<T><<<gridFor(n), TPB, 0, s>>>(r0.p, rn.p, res.p, r0.ld, AX.p, BX.p, AX.ld,
                                                 ones, lam, alpha1, 0.0, AX.N, AX.B);
      checkLaunch("resSeedFrom");
    }

    template <class T>
    void resFinal(hipStream_t s, View<double> z, double a1, const double *a, View<const T> x,
                  double b1, const double *b, View<const double> y)
    {
      const u64 n = (u64)z.N * z.B;
      if (!n)
        return;
      resFinalK<T><<<gridFor(n), TPB, 0, s>>>(z.p, z.ld, a1, a, x.p, x.ld, b1, b, y.p, y.ld,
                                              z.N, z.B);
      checkLaunch("resFinal");
    }

    template <class T>
    void resFinalDiag(hipStream_t s, View<double> z, double a1, const double *a,
                      View<const T> r, const double *d, u32 nC, View<const T> xE, double b1,
                      const double *b, View<const double> y)
    {
      const u64 n = (u64)z.N * z.B;
      if (!n)
        return;
      DFX_REQUIRE(r.ld == xE.ld && r.N == z.N && xE.N == z.N && nC <= z.N,
                  "residual result: shapes do not match");
      resFinalDiagK<T><<<gridFor(n), TPB, 0, s>>>(z.p, z.ld, a1, a, r.p, d, nC, xE.p, r.ld, b1,
                                                  b, y.p, y.ld, z.N, z.B);
      checkLaunch("resFinalDiag");
    }

    template <class T>
    void p2c(hipStream_t s, const dfx_constraints *c, View<T> x)
    {
      if (!c || !c->nRows || !x.B)
        return;
      const u64 n = (u64)c->nRows * x.B;
      p2cK<T><<<gridFor(n), TPB, 0, s>>>(x.p, x.ld, c->rows.as<u32>(),
                                         c->rowOffsets.as<u32>(), c->cols.as<u32>(),
                                         c->weights.as<double>(), c->inhom.as<double>(),
                                         c->nRows, x.B);
      checkLaunch("p2c");
    }

    template <class T>
    void c2p(hipStream_t s, const dfx_constraints *c, View<T> y)
    {
      if (!c || !c->nRows || !y.B)
        return;
      if (c->nParents)
        {
          const u64 n = (u64)c->nParents * y.B;
          c2pParentsK<T><<<gridFor(n), TPB, 0, s>>>(
            y.p, y.ld, c->parents.as<u32>(), c->parentOffsets.as<u32>(),
            c->parentRowDofs.as<u32>(), c->parentWeights.as<double>(), c->nParents,
            y.B);
          checkLaunch("c2pParents");
        }
      const u64 n = (u64)c->nRows * y.B;
      setRowsK<T><<<gridFor(n), TPB, 0, s>>>(y.p, y.ld, c->rows.as<u32>(), c->nRows,
                                             y.B, (T)0);
      checkLaunch("c2pZero");
    }

    template <class T>
    void setRows(hipStream_t s, const dfx_constraints *c, View<T> x, double v)
    {
      if (!c || !c->nRows || !x.B)
        return;
      const u64 n = (u64)c->nRows * x.B;
      setRowsK<T><<<gridFor(n), TPB, 0, s>>>(x.p, x.ld, c->rows.as<u32>(), c->nRows,
                                             x.B, (T)v);
      checkLaunch("setRows");
    }

    template <class T>
    void gather(hipStream_t s, const u32 *map, u64 nSlots, View<const T> x, View<T> xc)
    {
      const u64 n = nSlots * x.B;
      if (!n)
        return;
      gatherK<T><<<gridFor(n), TPB, 0, s>>>(map, nSlots, x.p, x.ld, xc.p, xc.ld, x.B);
      checkLaunch("gather");
    }

    template <class T>
    void scatterAdd(hipStream_t s, const u32 *off, const u32 *slots, u32 nDofs,
                    View<const T> yc, View<T> y)
    {
      const u64 n = (u64)nDofs * y.B;
      if (!n)
        return;
      scatterAddK<T><<<gridFor(n), TPB, 0, s>>>(off, slots, nDofs, yc.p, yc.ld, y.p,
                                                y.ld, y.B);
      checkLaunch("scatterAdd");
    }

#define DFX_INST_T(T)                                                              \
  template void fill<T>(hipStream_t, View<T>, double);                             \
  template void fillRandom<T>(hipStream_t, View<T>, u64, double, double);          \
  template void axpby<T>(hipStream_t, View<T>, double, View<const T>, double,      \
                         View<const T>);                                           \
  template void axpbyBlocked<T>(hipStream_t, View<T>, double, const double *,      \
                                View<const T>, double, const double *,             \
                                View<const T>);                                    \
  template void diagScale<T>(hipStream_t, View<T>, const double *, View<const T>,  \
                             u32);                                                 \
  template void enrichedBlock<T>(hipStream_t, View<T>, const double *,             \
                                 View<const T>, u32, u32);                         \
  template void colDots<T>(hipStream_t, View<const T>, View<const T>, double *,    \
                           double *);                                              \
  template void chebStep<T>(hipStream_t, View<T>, View<const T>, const double *,   \
                            View<const T>, u32, View<const T>, double, double,     \
                            double);                                               \
  template void resStep<T>(hipStream_t, View<T>, View<const T>, View<const T>,     \
                           View<const T>, const double *, const double *);         \
  template void resFix<T>(hipStream_t, View<T>, View<const T>, View<const T>,      \
                          View<const T>, const u32 *, u32, const double *,         \
                          const double *);                                         \
  template void resSeedFrom<T>(hipStream_t, View<T>, View<T>, View<T>,             \
                               View<const double>, View<const double>,             \
                               const double *, const double *, double);            \
  template void resSeed<T>(hipStream_t, View<T>, View<T>, View<T>,                 \
                           View<const double>, double);                            \
  template void resFinal<T>(hipStream_t, View<double>, double, const double *,     \
                            View<const T>, double, const double *,                 \
                            View<const double>);                                   \
  template void resFinalDiag<T>(hipStream_t, View<double>, double, const double *, \
                                View<const T>, const double *, u32, View<const T>, \
                                double, const double *, View<const double>);       \
  template void p2c<T>(hipStream_t, const dfx_constraints *, View<T>);             \
  template void c2p<T>(hipStream_t, const dfx_constraints *, View<T>);             \
  template void setRows<T>(hipStream_t, const dfx_constraints *, View<T>, double); \
  template void gather<T>(hipStream_t, const u32 *, u64, View<const T>, View<T>);  \
  template void scatterAdd<T>(hipStream_t, const u32 *, const u32 *, u32,          \
                              View<const T>, View<T>);

    DFX_INST_T(double)
    DFX_INST_T(float)
    template void convert<double, float>(hipStream_t, View<double>, View<const float>);
    template void convert<float, double>(hipStream_t, View<float>, View<const double>);
    template void convert<double, double>(hipStream_t, View<double>, View<const double>);
    template void convert<float, float>(hipStream_t, View<float>, View<const float>);
  } // namespace k
} // namespace dfx

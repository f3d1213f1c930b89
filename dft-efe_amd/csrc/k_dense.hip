// Tall-skinny dense kernels of the orthonormalization and Rayleigh-Ritz
// steps, FP64 MFMA (v_mfma_f64_16x16x4f64):
//   gram:   S = X^T Y      (computeXTransOpX, src/linearAlgebra/
//                           OrthonormalizationFunctions.t.cpp:1178-1380 and
//                           RayleighRitzEigenSolver.t.cpp:488-844; only the
//                           lower block triangle is formed, as there)
//   rotate: Xo = X Q       (the subspace rotations, OrthonormalizationFunctions.t.cpp:
//                           380-394 and RayleighRitzEigenSolver.t.cpp:272-286)
// The N-long reduction of gram is split over row chunks whose partial n x n
// blocks are summed in chunk order by a second kernel: deterministic, no
// atomics.
#include "kernels.hpp"

#include <algorithm>

namespace dfx
{
  namespace k
  {
    namespace
    {
      typedef double d4_t __attribute__((ext_vector_type(4)));
      constexpr int GB  = 64; // S block edge handled by one workgroup
      constexpr int KS  = 32; // rows per LDS slab
      constexpr int MAXCHUNKS = 192;

      __device__ inline d4_t mfma64(double a, double b, d4_t c)
      {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
      }

      // grid.x: lower-triangular block pair index, grid.y: row chunk
      __global__ __launch_bounds__(256) void gramK(const double *__restrict__ X, u32 ldx,
                                                   const double *__restrict__ Y, u32 ldy,
                                                   u32 N, u32 n, u32 rowsPerChunk,
                                                   double *__restrict__ partials)
      {
        __shared__ double sX[KS][GB];
        __shared__ double sY[KS][GB];
        // decode block pair (ab >= bb)
        u32 p = blockIdx.x, ab = 0;
        while (p > ab)
          {
            p -= ab + 1;
            ++ab;
          }
        const u32 bb = p;
        const u32 a0 = ab * GB, b0 = bb * GB;
        const u32 r0 = blockIdx.y * rowsPerChunk;
        const u32 r1 = min(N, r0 + rowsPerChunk);
        const int w = threadIdx.x >> 6, l = threadIdx.x & 63;

        d4_t acc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc[t] = d4_t{0, 0, 0, 0};

        for (u32 i0 = r0; i0 < r1; i0 += KS)
          {
            for (int t = threadIdx.x; t < KS * GB; t += 256)
              {
                const int kk = t / GB, c = t % GB;
                const u32 i  = i0 + kk;
                double    xv = 0.0, yv = 0.0;
                if (i < r1)
                  {
                    if (a0 + c < n)
                      xv = X[(u64)i * ldx + a0 + c];
                    if (b0 + c < n)
                      yv = Y[(u64)i * ldy + b0 + c];
                  }
                sX[kk][c] = xv;
                sY[kk][c] = yv;
              }
            __syncthreads();
#pragma unroll
            for (int kk = 0; kk < KS; kk += 4)
              {
                const double a = sX[kk + (l >> 4)][w * 16 + (l & 15)];
#pragma unroll
                for (int t = 0; t < 4; ++t)
                  acc[t] = mfma64(a, sY[kk + (l >> 4)][t * 16 + (l & 15)], acc[t]);
              }
            __syncthreads();
          }
        // partial block -> partials[chunk][a + n b] (column-major n x n)
        double *P = partials + (u64)blockIdx.y * n * n;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            {
              const u32 a = a0 + w * 16 + (l >> 4) + 4 * v;
              const u32 b = b0 + t * 16 + (l & 15);
              if (a < n && b < n)
                P[a + (u64)n * b] = acc[t][v];
            }
      }

      // S[a + n b] = sum over chunks (in order); lower triangle mirrored up
      __global__ void gramReduceK(const double *partials, u32 nChunks, u32 n,
                                  double *S)
      {
        const u64 tot = (u64)n * n;
        for (u64 t = blockIdx.x * (u64)blockDim.x + threadIdx.x; t < tot;
             t += (u64)gridDim.x * blockDim.x)
          {
            const u32 a = (u32)(t % n), b = (u32)(t / n);
            const u32 lo = a >= b ? a : b, hi = a >= b ? b : a; // element (lo, hi), lo >= hi
            // blocks with ab >= bb were computed; (lo, hi) lies in such a block
            double s = 0.0;
            for (u32 c = 0; c < nChunks; ++c)
              s += partials[(u64)c * n * n + lo + (u64)n * hi];
            S[t] = s;
          }
      }

      // ---- rows of X through raw buffers: offsets past `bytes` read 0, and
      // a pair of columns may start at any multiple of 8 bytes
      typedef double   d2_t __attribute__((ext_vector_type(2)));
      typedef unsigned u4_t __attribute__((ext_vector_type(4)));
      typedef unsigned u2_t __attribute__((ext_vector_type(2)));
      typedef __amdgpu_buffer_rsrc_t rsrc_t;
      constexpr u32 OFF_NONE = 0x80000000u;
      __device__ inline rsrc_t rows(const double *p, u64 bytes)
      {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(p), (short)0,
                                                 (int)(bytes < 0x7fffffffull ? bytes : 0x7fffffffull),
                                                 0x00020000);
      }
      // columns k and k + 1 (k even; 0 from column n on) of the row at byte
      // offset off, in two steps so that nothing waits between a load and its
      // use: the last column of an odd count arrives as the second half of a
      // load that starts one column earlier (a lone column comes by itself)
      __device__ inline d2_t loadPair(rsrc_t r, u32 off, int k, int n)
      {
        if (n == 1) // uniform
          return d2_t{__builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(
                                                   r, k == 0 ? off : OFF_NONE, 0, 0)),
                      0.0};
        return __builtin_bit_cast(
          d2_t, __builtin_amdgcn_raw_buffer_load_b128(
                  r, k < n ? off + 8u * (k + 1 == n ? k - 1 : k) : OFF_NONE, 0, 0));
      }
      __device__ inline d2_t pairOf(d2_t v, int k, int n)
      {
        return n > 1 && k + 1 == n ? d2_t{v[1], 0.0} : v;
      }

      // S = X^T Y, every lower-triangular 16 x 16 tile of S for one row chunk
      // in one workgroup (8 waves, a run of TPW tiles each; a wave past the last
      // tile repeats it), so X and Y are read once.  Rows run in slabs of KR staged in LDS as row pairs
      // ([pair][column][2]: a lane's operand for two MFMA steps is one 16-byte
      // read without bank conflicts), two slabs deep: before a slab's MFMAs the
      // next slab's rows, requested a slab ago, go to the other half and those
      // of the one after it are requested; one barrier a slab.  Up to seven
      // tiles a wave (n <= 160) two workgroups share a CU (64 KiB of LDS and at
      // most 128 VGPRs each), above that one with slabs twice as long.  Bound
      // by FP64 MFMA and memory alike at n = 200.  One 16-row slab at a time
      // and operands read right before their use measured, before -> now:
      // N = 531 k, n = 200: 800 -> 620 us (40 TFLOP/s); N = 184 k, n = 101:
      // 417 -> 78 us (3.8 TB/s); N = 30 k, n = 20: 109 -> 13 us (chunks of
      // 1024 rows left most CUs idle)
      template <int NBP, int TPW>
      __global__ __launch_bounds__(512, TPW <= 7 ? 4 : 2) void gramAllK(const double *__restrict__ X, u32 ldx,
                                                         const double *__restrict__ Y, u32 ldy,
                                                         u32 N, u32 n, u32 nTiles,
                                                         u32 rowsPerChunk,
                                                         double *__restrict__ partials)
      {
        constexpr int KR = (TPW <= 7 ? 2048 : 4096) / NBP; // 8 to 32 rows
        constexpr int UT = (KR / 2) * (NBP / 2); // row pair x column pair units per matrix
        constexpr int MAT = KR * NBP;            // doubles per matrix and slab
        extern __shared__ __align__(16) unsigned char smemG[];
        double   *sm = reinterpret_cast<double *>(smemG); // [2 slabs][X, Y][KR / 2][NBP][2]
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
        const int q = l >> 4, c = l & 15;
        // tile p (lower triangle, row-major over ta >= tb) -> (ta, tb)
        int ta[TPW], tb[TPW];
        {
          const u32 p0 = min((u32)w * TPW, nTiles - 1);
          u32       p = p0, a = 0;
          while (p > a)
            p -= ++a;
#pragma unroll
          for (int j = 0; j < TPW; ++j)
            {
              ta[j] = (int)a;
              tb[j] = (int)p;
              if (p0 + j + 1 >= nTiles) // the last tile again
                continue;
              if (p == a)
                p = 0, ++a;
              else
                ++p;
            }
        }
        const u32    r0 = blockIdx.x * rowsPerChunk, r1 = min(N, r0 + rowsPerChunk);
        const rsrc_t rX = rows(X + (u64)r0 * ldx, (u64)(r1 - r0) * ldx * 8);
        const rsrc_t rY = rows(Y + (u64)r0 * ldy, (u64)(r1 - r0) * ldy * 8);
        const u32    nRows = r1 - r0;
        // units t, t + 512 of X and of Y: row pair t / (NBP / 2), column pair
        constexpr int UPT = (UT + 511) / 512;
        d2_t          v[2][UPT][2];
        auto          request = [&](u32 i0) {
#pragma unroll
          for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int u = 0; u < UPT; ++u)
              {
                const int t = threadIdx.x + 512 * u, col = 2 * (t % (NBP / 2));
                const u32 i = i0 + 2 * (t / (NBP / 2)), ld = m ? ldy : ldx;
#pragma unroll
                for (int h = 0; h < 2; ++h)
                  v[m][u][h] = loadPair(m ? rY : rX, (i + h) * ld * 8, i + h < nRows ? col : (int)n,
                                        (int)n);
              }
        };
        auto store = [&](int buf) {
#pragma unroll
          for (int m = 0; m < 2; ++m)
#pragma unroll
            for (int u = 0; u < UPT; ++u)
              {
                const int  t = threadIdx.x + 512 * u, col = 2 * (t % (NBP / 2));
                double    *d = sm + (buf * 2 + m) * MAT + (t / (NBP / 2)) * NBP * 2 + 2 * col;
                const d2_t p = pairOf(v[m][u][0], col, (int)n), r = pairOf(v[m][u][1], col, (int)n);
                *reinterpret_cast<d2_t *>(d)     = d2_t{p[0], r[0]};
                *reinterpret_cast<d2_t *>(d + 2) = d2_t{p[1], r[1]};
              }
        };
        static_assert(UT % 512 == 0, "whole units per thread");
        d4_t acc[TPW];
#pragma unroll
        for (int j = 0; j < TPW; ++j)
          acc[j] = d4_t{0, 0, 0, 0};
        request(0);
        store(0);
        request(KR); // rows past the chunk read 0
        __syncthreads();
        int buf = 0;
        for (u32 i0 = 0; i0 < nRows; i0 += KR, buf ^= 1)
          {
            if (i0 + KR < nRows) // uniform
              {
                store(buf ^ 1);
                request(i0 + 2 * KR);
              }
            const double *sX = sm + buf * 2 * MAT, *sY = sX + MAT;
#pragma unroll 2
            for (int kb = 0; kb < KR / 8; ++kb)
              {
                const int at = ((kb * 4 + q) * NBP + c) * 2;
                // a tile's operands are read before the previous tile's MFMAs;
                // X's only where the next row of tiles begins
                d2_t a = *reinterpret_cast<const d2_t *>(sX + at + ta[0] * 32), an = a;
                d2_t bn = *reinterpret_cast<const d2_t *>(sY + at + tb[0] * 32);
#pragma unroll
                for (int j = 0; j < TPW; ++j)
                  {
                    const d2_t b = bn;
                    a            = an;
                    if (j + 1 < TPW)
                      {
                        bn = *reinterpret_cast<const d2_t *>(sY + at + tb[j + 1] * 32);
                        if (tb[j + 1] == 0)
                          an = *reinterpret_cast<const d2_t *>(sX + at + ta[j + 1] * 32);
                      }
                    acc[j] = mfma64(a[0], b[0], acc[j]);
                    acc[j] = mfma64(a[1], b[1], acc[j]);
                  }
              }
            __syncthreads();
          }
        // fragment order: lane l of tile p, row (l / 16) + 4 v, column l % 16
        double *P = partials + ((u64)blockIdx.x * nTiles + w * TPW) * 256;
#pragma unroll
        for (int j = 0; j < TPW; ++j)
          if ((u32)(w * TPW + j) < nTiles)
            *reinterpret_cast<d4_t *>(P + j * 256 + 4 * l) = acc[j];
      }

      // S from the chunks' tiles: 16 elements x 16 chunk lanes per workgroup,
      // lane k adds chunks k, k + 16, ... in order, the lane sums in lane
      // order; the lower triangle mirrored up.  Bound by memory (n = 200, 512
      // chunks: 95 MB in 19 us; one thread per element took 217)
      __global__ __launch_bounds__(256) void gramTilesK(const double *__restrict__ partials,
                                                        u32 nChunks, u32 nTiles, u32 n, double *S)
      {
        __shared__ double red[16][17];
        const u32 e = blockIdx.x * 16 + threadIdx.x % 16, k = threadIdx.x / 16;
        double    s = 0.0;
#pragma unroll 8
        for (u32 ch = k; ch < nChunks; ch += 16)
          s += partials[(u64)ch * nTiles * 256 + e];
        red[k][threadIdx.x % 16] = s;
        __syncthreads();
        if (k)
          return;
        s = 0.0;
#pragma unroll
        for (int h = 0; h < 16; ++h)
          s += red[h][threadIdx.x];
        u32 p = e / 256, a = 0;
        while (p > a)
          p -= ++a;
        const u32 lane = (e % 256) / 4, ra = a * 16 + (lane >> 4) + 4 * (e % 4),
                  cb = p * 16 + (lane & 15);
        if (ra < n && cb <= ra)
          {
            S[ra + (u64)n * cb] = s;
            S[cb + (u64)n * ra] = s;
          }
      }

      // Q (column-major n x n) in operand order for rotateAllK: K block kb of
      // 8 rows, column tile t, lane l, two values: rows 8 kb + 2 (l / 16) + s,
      // column 16 t + l % 16, zero past n
      __global__ void packQK(const double *__restrict__ Q, u32 n, u32 nbt, u32 nkb,
                             double *__restrict__ Qf)
      {
        const u32 tot = nkb * nbt * 128;
        for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < tot; i += gridDim.x * blockDim.x)
          {
            const u32 l = (i / 2) % 64, t = (i / 128) % nbt, kb = i / (128 * nbt);
            const u32 k = 8 * kb + 2 * (l >> 4) + i % 2, col = 16 * t + (l & 15);
            Qf[i]       = k < n && col < n ? Q[k + (u64)n * col] : 0.0;
          }
      }

      // Xo = X Q for every column in one pass over X: a wave owns 16 rows and
      // all NBT column tiles, its rows' operand straight from
      // memory (16 bytes a lane and K block, one slab ahead); Q, in operand
      // order, runs through LDS in slabs of 16 rows, two deep, shared by the
      // four waves.  The tile count is a template parameter: with a test per
      // tile the LDS reads cannot run ahead of the MFMAs (1043 against 870 us
      // at N = 531 k, n = 200).  Bound by FP64 MFMA (N = 2.1 M, n = 200: 3.6 ms,
      // 48 TFLOP/s; the library products measured 3.2 to 7.0 ms for it,
      // depending on the library's version) or memory (n <= 100; N = 184 k,
      // n = 101: 118 us, 2.5 TB/s, library 283)
      constexpr int RW = 4;
      template <int NBT>
      __global__ __launch_bounds__(64 * RW, 2) void rotateAllK(const double *__restrict__ X,
                                                               u32 ldx, u32 N, u32 n,
                                                               const double *__restrict__ Qf,
                                                               double *__restrict__ Xo, u32 ldo)
      {
        constexpr int PF = (2 * NBT + RW - 1) / RW; // 16-byte words of a slab per thread
        __shared__ d2_t sQ[2][2 * NBT * 64];
        const int    w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
        const int    q = l >> 4, c = l & 15;
        const u64    row0 = (u64)blockIdx.x * (16 * RW) + 16 * w;
        const u32    nr   = row0 < N ? (u32)min((u64)16, N - row0) : 0u; // live rows
        const rsrc_t rX   = rows(X + (nr ? row0 : 0) * ldx, (u64)nr * ldx * 8);
        constexpr u32 words = 2 * NBT * 64, nSlabs = NBT;
        d2_t         pf[PF], aN[2];
        auto         request = [&](u32 slab) {
          const d2_t *src = reinterpret_cast<const d2_t *>(Qf) + (u64)slab * words;
#pragma unroll
          for (int u = 0; u < PF; ++u)
            {
              const u32 t = threadIdx.x + 64 * RW * u;
              pf[u]       = t < words ? src[t] : d2_t{0, 0};
            }
#pragma unroll
          for (int h = 0; h < 2; ++h)
            aN[h] = loadPair(rX, (u32)c * ldx * 8, (int)(16 * slab + 8 * h + 2 * q), (int)n);
        };
        auto store = [&](int buf) {
#pragma unroll
          for (int u = 0; u < PF; ++u)
            if (const u32 t = threadIdx.x + 64 * RW * u; t < words)
              sQ[buf][t] = pf[u];
        };
        d4_t acc[NBT];
#pragma unroll
        for (int t = 0; t < NBT; ++t)
          acc[t] = d4_t{0, 0, 0, 0};
        d2_t a[2];
        request(0);
        store(0);
        a[0] = aN[0], a[1] = aN[1];
        if (nSlabs > 1)
          request(1);
        __syncthreads();
        for (u32 slab = 0; slab < nSlabs; ++slab)
          {
            const d2_t aX[2] = {aN[0], aN[1]}; // the next slab's operand
            if (slab + 1 < nSlabs)
              store((slab & 1) ^ 1);
            if (slab + 2 < nSlabs)
              request(slab + 2);
            const d2_t *Qs = sQ[slab & 1] + l;
#pragma unroll
            for (int h = 0; h < 2; ++h)
              {
                if (slab + 1 == nSlabs) // the only slab that meets column n
                  a[h] = pairOf(a[h], 16 * slab + 8 * h + 2 * q, (int)n);
#pragma unroll
                for (int t0 = 0; t0 < NBT; t0 += 4)
                {
                  d2_t b[4];
#pragma unroll
                  for (int t = 0; t < 4; ++t)
                    if (t0 + t < NBT)
                      b[t] = Qs[(h * NBT + t0 + t) * 64];
#pragma unroll
                  for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                      if (t0 + t < NBT)
                        acc[t0 + t] = mfma64(a[h][s], b[t][s], acc[t0 + t]);
                }
              }
            a[0] = aX[0], a[1] = aX[1];
            __syncthreads();
          }
#pragma unroll
        for (int t = 0; t < NBT; ++t)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            {
              const u32 i = q + 4 * v, b = 16 * t + c;
              if (i < nr && b < n)
                Xo[(row0 + i) * ldo + b] = acc[t][v];
            }
      }

      u32 chunksFor(u32 N) { return std::max(1u, std::min<u32>(MAXCHUNKS, (N + 2047) / 2048)); }
      // the all-tile kernel (n <= 256): padded columns, rows per slab, tiles, and
      // row chunks of at least two slabs, up to two per CU and 1 GiB of rows
      struct GramPlan
      {
        u32 nbp, nTiles, tpw, sm, rows, chunks;
      };
      GramPlan gramPlan(u32 N, u32 n, u32 ld)
      {
        GramPlan  g;
        const u32 nbt = (n + 15) / 16;
        g.nbp         = nbt <= 4 ? 64 : nbt <= 8 ? 128 : 256;
        g.nTiles      = nbt * (nbt + 1) / 2;
        g.tpw         = (g.nTiles + 7) / 8;
        g.sm          = g.tpw <= 7 ? 2048 : 4096;
        const u32 kr  = g.sm / g.nbp;
        u64       r   = std::max<u64>(2 * kr, ((u64)N + 511) / 512);
        r             = std::min<u64>(r, std::max<u64>(kr, (1ull << 27) / ld));
        g.rows        = (u32)((r + kr - 1) / kr * kr);
        g.chunks      = std::max(1u, (N + g.rows - 1) / g.rows);
        return g;
      }
    } // namespace

    size_t gramPartialsNeeded(u32 N, u32 n, u32 ld)
    {
      if (n > 256)
        return (size_t)chunksFor(N) * n * n;
      const GramPlan g = gramPlan(N, n, ld);
      return (size_t)g.chunks * g.nTiles * 256;
    }

    void gram(hipStream_t s, View<const double> X, View<const double> Y, double *partials,
              size_t partialsCap, double *S)
    {
      const u32 n = X.B, N = X.N;
      DFX_REQUIRE(Y.B == n && Y.N == N, "gram: shape mismatch");
      if (!n)
        return;
      if (n <= 256) // all tiles in one workgroup per row chunk
        {
          const u32      ld = std::max(X.ld, Y.ld);
          const GramPlan g  = gramPlan(N, n, ld);
          DFX_REQUIRE(partialsCap >= (size_t)g.chunks * g.nTiles * 256, "gram: partials too small");
          DFX_REQUIRE((u64)g.rows * ld * 8 < (1ull << 31), "gram: leading dimension too large");
          const size_t lds = 2 * 2 * g.sm * sizeof(double);
          auto go = [&](auto kern) {
            if (lds > 64 * 1024)
              DFX_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            kern<<<g.chunks, 512, lds, s>>>(X.p, X.ld, Y.p, Y.ld, N, n, g.nTiles, g.rows, partials);
          };
          switch (g.tpw) // tiles per wave: ceil(nbt (nbt + 1) / 16) for nbt column tiles
            {
              case 1: go(gramAllK<64, 1>); break;                                   // nbt 1..3
              case 2: g.nbp == 64 ? go(gramAllK<64, 2>) : go(gramAllK<128, 2>); break; // 4, 5
              case 3: go(gramAllK<128, 3>); break;
              case 4: go(gramAllK<128, 4>); break;
              case 5: go(gramAllK<128, 5>); break;
              case 6: go(gramAllK<256, 6>); break; // nbt 9
              case 7: go(gramAllK<256, 7>); break;
              case 9: go(gramAllK<256, 9>); break;
              case 10: go(gramAllK<256, 10>); break;
              case 12: go(gramAllK<256, 12>); break;
              case 14: go(gramAllK<256, 14>); break;
              case 15: go(gramAllK<256, 15>); break;
              default: go(gramAllK<256, 17>); break;
            }
          checkLaunch("gramAll");
          gramTilesK<<<g.nTiles * 16, 256, 0, s>>>(partials, g.chunks, g.nTiles, n, S);
          checkLaunch("gramTiles");
          return;
        }
      const u32 nChunks = chunksFor(N);
      DFX_REQUIRE(partialsCap >= (size_t)nChunks * n * n, "gram: partials too small");
      const u32 nb     = (n + GB - 1) / GB;
      const u32 nPairs = nb * (nb + 1) / 2;
      const u32 rows   = (N + nChunks - 1) / nChunks;
      gramK<<<dim3(nPairs, nChunks), 256, 0, s>>>(X.p, X.ld, Y.p, Y.ld, N, n, rows,
                                                     partials);
      checkLaunch("gram");
      const u64 tot = (u64)n * n;
      gramReduceK<<<(unsigned)std::min<u64>(4096, (tot + 255) / 256), 256, 0, s>>>(
        partials, nChunks, n, S);
      checkLaunch("gramReduce");
    }

    void rotate(hipStream_t s, View<const double> X, const double *Q, View<double> Xo,
                double *qf, rocblas_handle blas, bool library)
    {
      // Q: n x n column-major, device
      const u32 n = X.B, N = X.N;
      DFX_REQUIRE(Xo.B == n && Xo.N == N, "rotate: shape mismatch");
      if (!n || !N)
        return;
      if (n > 256 || library)
        {
          // column-major view: Xo^T (n x N, ld Xo.ld) = Q^T (n x n) X^T
          // (n x N, ld X.ld)
          DFX_REQUIRE(N <= 0x7fffffffu, "rotate: too many rows");
          const double one = 1.0, zero = 0.0;
          CaptureLock  lk(captureMutex());
          rocblas_set_pointer_mode(blas, rocblas_pointer_mode_host);
          if (rocblas_dgemm(blas, rocblas_operation_transpose, rocblas_operation_none,
                            (rocblas_int)n, (rocblas_int)N, (rocblas_int)n, &one, Q,
                            (rocblas_int)n, X.p, (rocblas_int)X.ld, &zero, Xo.p,
                            (rocblas_int)Xo.ld) != rocblas_status_success)
            throw Error(DFX_E_HIP, "rocblas_dgemm (rotation) failed");
          return;
        }
      const u32 nbt = (n + 15) / 16;
      packQK<<<std::min<u32>(1024, (2 * nbt * nbt * 128 + 255) / 256), 256, 0, s>>>(Q, n, nbt,
                                                                                   2 * nbt, qf);
      checkLaunch("packQ");
      const u64 grid = ((u64)N + 16 * RW - 1) / (16 * RW);
      DFX_REQUIRE((u64)16 * X.ld * 8 < (1ull << 31) && grid < (1ull << 31),
                  "rotate: leading dimension too large");
      auto go = [&](auto kern) {
        kern<<<(unsigned)grid, 64 * RW, 0, s>>>(X.p, X.ld, N, n, qf, Xo.p, Xo.ld);
      };
      switch (nbt)
        {
          case 1: go(rotateAllK<1>); break;
          case 2: go(rotateAllK<2>); break;
          case 3: go(rotateAllK<3>); break;
          case 4: go(rotateAllK<4>); break;
          case 5: go(rotateAllK<5>); break;
          case 6: go(rotateAllK<6>); break;
          case 7: go(rotateAllK<7>); break;
          case 8: go(rotateAllK<8>); break;
          case 9: go(rotateAllK<9>); break;
          case 10: go(rotateAllK<10>); break;
          case 11: go(rotateAllK<11>); break;
          case 12: go(rotateAllK<12>); break;
          case 13: go(rotateAllK<13>); break;
          case 14: go(rotateAllK<14>); break;
          case 15: go(rotateAllK<15>); break;
          default: go(rotateAllK<16>); break;
        }
      checkLaunch("rotateAll");
    }
  } // namespace k
} // namespace dfx

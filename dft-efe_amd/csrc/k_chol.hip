// Cholesky factor of a small symmetric matrix and the inverse of the factor,
// transposed, in one workgroup (CholeskyGramSchmidt's dense part,
// src/linearAlgebra/OrthonormalizationFunctions.t.cpp:356-394: potrf, the
// check of the diagonal, trtri, and the transposed factor that rotates X).
// Launched as library calls with the host between them it took about 0.45 ms
// of kernels and as much of copies and waits at n = 200; here 13 panels follow
// each other without leaving the device (133 + 42 us).  Bound by the chain of
// panels: a block's 16 pivots, the product that follows, two barriers.
#include "kernels.hpp"

namespace dfx
{
  namespace k
  {
    namespace
    {
      typedef double d4_t __attribute__((ext_vector_type(4)));

      __device__ inline d4_t mfma64(double a, double b, d4_t c)
      {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
      }
      __device__ inline double lane(double v, int l)
      {
        const long long u = __builtin_bit_cast(long long, v);
        const int       lo = __builtin_amdgcn_readlane((int)u, l);
        const int       hi = __builtin_amdgcn_readlane((int)(u >> 32), l);
        return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
      }

      // Factor of a 16 x 16 block and the factor's inverse, one wave: lane r
      // (mod 16) holds row r in registers, pivots and columns pass by readlane.
      // D: the block (row-major, LDS); replaced by the inverse
      __device__ inline void factor16(double *D, int l, int *info)
      {
        const int r = l & 15;
        double    a[16], x[16];
#pragma unroll
        for (int c = 0; c < 16; ++c)
          a[c] = D[r * 16 + c];
        bool bad = false;
#pragma unroll
        for (int c = 0; c < 16; ++c)
          {
            const double d = sqrt(lane(a[c], c));
            // not positive, not a number, or a diagonal below 1e-14
            bad  = bad || !(d >= 1e-14);
            a[c] = r == c ? d : a[c] / d;
#pragma unroll
            for (int e = c + 1; e < 16; ++e)
              a[e] = fma(-a[c], lane(a[c], e), a[e]);
          }
        if (bad && l == 0)
          *info = 1;
        // column r of the inverse, top down
#pragma unroll
        for (int i = 0; i < 16; ++i)
          {
            double s = i == r ? 1.0 : 0.0;
#pragma unroll
            for (int c = 0; c < i; ++c)
              s = fma(-lane(a[c], i), x[c], s);
            x[i] = s / lane(a[i], i);
          }
        if (l < 16)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            D[i * 16 + r] = i >= r ? x[i] : 0.0;
      }

      // S (n x n column-major, lower triangle read); L: ld x ld with ld = 16
      // ceil(n / 16), the blocks below the diagonal; Dg: the inverses of the
      // diagonal blocks.  The matrix is padded with the identity.  16 waves;
      // wave w owns the w-th 16-row block of a panel.
      //
      // Products are formed transposed (rows of the result: the panel's
      // columns), so that an accumulator is the next product's operand as it
      // stands: element v of lane l holds k = l / 16 + 4 v, the operand of step v.
      __global__ __launch_bounds__(1024) void cholFactorK(const double *__restrict__ S, u32 n,
                                                          double *L, double *__restrict__ Dg,
                                                          int *info)
      {
        __shared__ double D[256]; // the diagonal block, then its factor's inverse (row-major)
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
        const int q = l >> 4, c = l & 15;
        const int nb = (int)(n + 15) / 16;
        const u32 ld = 16 * nb;
        if (threadIdx.x == 0) // wave 0, which alone sets it later
          *info = 0;
        for (int j = 0; j < nb; ++j)
          {
            const int i = j + w; // this wave's row block
            d4_t      p{};
            if (i < nb)
              {
                // P^T = S_ij^T - sum_k L_jk L_ik^T
                const double *Lj = L + 16 * j + c + (u64)q * ld, *Li = L + 16 * i + c + (u64)q * ld;
                d4_t          acc{};
                for (int k = 0; k < j; ++k)
                  {
                    double a[4], b[4];
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                      {
                        a[v] = Lj[(u64)(16 * k + 4 * v) * ld];
                        b[v] = Li[(u64)(16 * k + 4 * v) * ld];
                      }
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                      acc = mfma64(a[v], b[v], acc);
                  }
#pragma unroll
                for (int v = 0; v < 4; ++v)
                  {
                    const u32 row = 16 * i + c, col = 16 * j + q + 4 * v;
                    // the lower triangle: in the diagonal block by symmetry
                    const u32    lo = row >= col ? row : col, hi = row >= col ? col : row;
                    const double s  = lo < n ? S[lo + (u64)n * hi] : (row == col ? 1.0 : 0.0);
                    p[v]            = s - acc[v];
                  }
              }
            // (barriers between one lane's LDS writes and another's reads,
            // also within wave 0)
            if (w == 0)
#pragma unroll
              for (int v = 0; v < 4; ++v)
                D[c * 16 + q + 4 * v] = p[v];
            __syncthreads();
            if (w == 0)
              factor16(D, l, info);
            __syncthreads();
            if (w == 0)
#pragma unroll
              for (int v = 0; v < 4; ++v)
                Dg[256 * j + 64 * v + l] = D[64 * v + l];
            if (i < nb && w > 0)
              {
                // L_ij^T = D_j P^T
                d4_t r{};
#pragma unroll
                for (int v = 0; v < 4; ++v)
                  r = mfma64(D[c * 16 + 4 * v + q], p[v], r);
#pragma unroll
                for (int v = 0; v < 4; ++v)
                  L[16 * i + c + (u64)(16 * j + q + 4 * v) * ld] = r[v];
              }
            __syncthreads();
          }
      }

      // Block column w of the inverse, one wave (X_w = D_w, X_i = -D_i sum_k
      // L_ik X_k), held in registers: the columns do not wait for each other
      __global__ __launch_bounds__(64) void triInverseK(const double *__restrict__ L,
                                                        const double *__restrict__ D, u32 n,
                                                        double *__restrict__ Q)
      {
        const int l = threadIdx.x, q = l >> 4, c = l & 15, w = blockIdx.x, nb = gridDim.x;
        const u32 ld = 16 * nb;
        d4_t      X[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (i < nb)
            {
              d4_t x{};
              if (i == w)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                  x[v] = D[256 * i + (q + 4 * v) * 16 + c];
              if (i > w)
                {
                  d4_t acc{};
#pragma unroll
                  for (int k = 0; k < i; ++k)
                    if (k >= w)
#pragma unroll
                      for (int v = 0; v < 4; ++v)
                        acc = mfma64(L[16 * i + c + (u64)(16 * k + 4 * v + q) * ld], X[k][v], acc);
#pragma unroll
                  for (int v = 0; v < 4; ++v)
                    x = mfma64(-D[256 * i + c * 16 + 4 * v + q], acc[v], x);
                }
              X[i] = x;
              // Q[a, b] = L^-1[b, a]
#pragma unroll
              for (int v = 0; v < 4; ++v)
                {
                  const u32 b = 16 * i + q + 4 * v, a = 16 * w + c;
                  if (a < n && b < n)
                    Q[a + (u64)n * b] = x[v];
                }
            }
      }
    } // namespace

    void cholInverse(hipStream_t s, const double *S, u32 n, double *L, double *Q, int *info)
    {
      DFX_REQUIRE(n >= 1 && n <= 256, "cholInverse: 1..256 columns");
      const u32 nb = (n + 15) / 16;
      double   *D  = L + (size_t)256 * nb * nb; // 256 values per diagonal block
      cholFactorK<<<1, 1024, 0, s>>>(S, n, L, D, info);
      checkLaunch("cholFactor");
      triInverseK<<<nb, 64, 0, s>>>(L, D, n, Q);
      checkLaunch("triInverse");
    }
  } // namespace k
} // namespace dfx

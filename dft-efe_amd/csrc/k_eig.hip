// The parts of the projected eigenproblem (RayleighRitzEigenSolver.t.cpp:
// 233-301, LAPACK's dsyevd) around the library's divide and conquer: the
// Householder reduction to tridiagonal form and the return of the tridiagonal
// eigenvectors.  The reflectors, their order and signs are LAPACK's (dsytrd,
// lower triangle), so the results are dsyevd's up to rounding.
#include "kernels.hpp"

#include <algorithm>

namespace dfx
{
  namespace k
  {
    namespace
    {
      // v of another lane by a DPP control word (0 where it names no lane):
      // register moves of a few cycles where a shuffle goes through the LDS
      template <int CTRL, int ROWS = 0xf>
      __device__ inline double dpp(double v)
      {
        const long long u  = __builtin_bit_cast(long long, v);
        const int       lo = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, ROWS, 0xf, true);
        const int       hi = __builtin_amdgcn_update_dpp(0, (int)(u >> 32), CTRL, ROWS, 0xf, true);
        return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
      }
      // sum over the wave, in every lane: row_shr 1, 2, 4, 8 leave a row's sum
      // in its last lane, row_bcast 15 and 31 add the rows up into lane 63
      __device__ inline double waveSum(double v)
      {
        v += dpp<0x111>(v);
        v += dpp<0x112>(v);
        v += dpp<0x114>(v);
        v += dpp<0x118>(v);
        v += dpp<0x142, 0xa>(v);
        v += dpp<0x143, 0xc>(v);
        const long long u = __builtin_bit_cast(long long, v);
        return __builtin_bit_cast(double,
                                  ((long long)__builtin_amdgcn_readlane((int)(u >> 32), 63) << 32) |
                                    (unsigned)__builtin_amdgcn_readlane((int)u, 63));
      }
      // sum over 8 and 16 neighbouring lanes, in each of them (quad swaps and
      // half-row mirror; row rotations)
      __device__ inline double sum8(double v)
      {
        v += dpp<0xb1>(v);
        v += dpp<0x4e>(v);
        return v + dpp<0x141>(v);
      }
      __device__ inline double sum16(double v)
      {
        v += dpp<0x128>(v);
        v += dpp<0x124>(v);
        v += dpp<0x122>(v);
        return v + dpp<0x121>(v);
      }

      // Tridiagonal form of a symmetric matrix of up to 128 columns, one
      // workgroup with the whole matrix in LDS (both triangles, so that rows
      // are columns).  Per reflector: its norm and the dot v.p are summed by
      // every wave for itself (no barrier), the matrix-vector product and the
      // rank-2 update go eight lanes to a row; three barriers.  Bound by that
      // chain of n steps: n = 20 / 40 / 101 takes 27 / 57 / 206 us, the library's
      // kernel 52 / 140 / 645.  A (n x n column-major, global): lower
      // triangle read, reflector i left below its diagonal; ld % 32 == 8 spreads
      // four rows over all LDS banks
      __global__ __launch_bounds__(1024) void tridiagK(double *A, int n, int ld, double *d,
                                                       double *e, double *tau)
      {
        extern __shared__ __align__(16) double sm[];
        double   *M = sm, *v = sm + (size_t)n * ld, *p = v + 128;
        const int t = threadIdx.x, l = t & 63, row = t >> 3, kl = t & 7;
        for (int i = t; i < n * n; i += 1024)
          {
            const int c = i / n, r = i - c * n;
            if (r >= c)
              M[c * ld + r] = M[r * ld + c] = A[i];
          }
        __syncthreads();
        for (int i = 0; i + 1 < n; ++i)
          {
            // x = column i below the diagonal (row i of M), this lane's elements
            const double *x  = M + i * ld;
            const int     k0 = i + 1;
            const double  x0 = k0 + 1 + l < n ? x[k0 + 1 + l] : 0.0;
            const double  x1 = k0 + 65 + l < n ? x[k0 + 65 + l] : 0.0;
            const double  alpha = x[k0];
            const double  ss    = waveSum(fma(x0, x0, x1 * x1));
            double        beta = alpha, ta = 0.0, scale = 0.0;
            if (ss > 0.0)
              {
                beta  = -copysign(sqrt(fma(alpha, alpha, ss)), alpha);
                ta    = (beta - alpha) / beta;
                scale = 1.0 / (alpha - beta);
              }
            if (t < 64)
              {
                if (l == 0)
                  {
                    d[i]   = x[i];
                    e[i]   = beta;
                    tau[i] = ta;
                    v[k0]  = 1.0;
                  }
                if (k0 + 1 + l < n)
                  A[(size_t)i * n + k0 + 1 + l] = v[k0 + 1 + l] = x0 * scale;
                if (k0 + 65 + l < n)
                  A[(size_t)i * n + k0 + 65 + l] = v[k0 + 65 + l] = x1 * scale;
              }
            __syncthreads();
            // p = tau A22 v
            {
              double s = 0.0;
              if (row >= k0 && row < n)
                for (int k = k0 + kl; k < n; k += 8)
                  s = fma(M[row * ld + k], v[k], s);
              s = sum8(s);
              if (kl == 0 && row >= k0 && row < n)
                p[row] = ta * s;
            }
            __syncthreads();
            // A22 -= v w' + w v', w = p - tau / 2 (p.v) v
            const double y0 = k0 + l < n ? p[k0 + l] * v[k0 + l] : 0.0;
            const double y1 = k0 + 64 + l < n ? p[k0 + 64 + l] * v[k0 + 64 + l] : 0.0;
            const double a2 = -0.5 * ta * waveSum(y0 + y1);
            if (row >= k0 && row < n)
              {
                const double vr = v[row], wr = fma(a2, vr, p[row]);
                for (int k = k0 + kl; k < n; k += 8)
                  {
                    const double vk = v[k], wk = fma(a2, vk, p[k]);
                    M[row * ld + k] -= vr * wk + wr * vk;
                  }
              }
            __syncthreads();
          }
        if (t == 0)
          d[n - 1] = M[(n - 1) * ld + n - 1];
      }

      // V = Q C with Q = H(0) H(1) .. H(n - 2), H(i) = I - tau_i v_i v_i', v_i
      // below the diagonal of A's column i (1 on the row under it): 16 lanes own
      // a column of C (rows lane, lane + 16, ...) and apply the reflectors in
      // turn, G at a time, the next G requested meanwhile; the columns do not
      // wait for each other.  Bound by that chain (n = 40: 39 steps).  As n
      // launches of three library kernels this took about 0.3 ms at n = 20 and
      // 0.5 ms at n = 40
      template <int E, int G>
      __global__ __launch_bounds__(64) void reflectK(const double *__restrict__ A,
                                                     const double *__restrict__ tau, int n,
                                                     const double *__restrict__ C, double *V)
      {
        const int r0 = threadIdx.x & 15, col = blockIdx.x * 4 + (threadIdx.x >> 4);
        const int cc = col < n ? col : n - 1; // (a spare group repeats the last column)
        double    c[E], v[G][E], vn[G][E], ta[G], tn[G];
#pragma unroll
        for (int u = 0; u < E; ++u)
          c[u] = r0 + 16 * u < n ? C[(size_t)cc * n + r0 + 16 * u] : 0.0;
        // reflectors i, i - 1, .. (past the first: none, tau 0)
        auto load = [&](int i, double(*o)[E], double *t) {
#pragma unroll
          for (int g = 0; g < G; ++g)
            {
              const int k = i - g;
              t[g]        = k >= 0 ? tau[k] : 0.0;
#pragma unroll
              for (int u = 0; u < E; ++u)
                {
                  const int r = r0 + 16 * u;
                  o[g][u] = r == k + 1 ? 1.0
                            : (k >= 0 && r > k + 1 && r < n) ? A[(size_t)k * n + r] : 0.0;
                }
            }
        };
        load(n - 2, v, ta);
        for (int i = n - 2; i >= 0; i -= G)
          {
            load(i - G, vn, tn);
#pragma unroll
            for (int g = 0; g < G; ++g)
              {
                double s = 0.0;
#pragma unroll
                for (int u = 0; u < E; ++u)
                  s = fma(v[g][u], c[u], s);
                s = -ta[g] * sum16(s);
#pragma unroll
                for (int u = 0; u < E; ++u)
                  c[u] = fma(s, v[g][u], c[u]);
              }
#pragma unroll
            for (int g = 0; g < G; ++g)
              {
                ta[g] = tn[g];
#pragma unroll
                for (int u = 0; u < E; ++u)
                  v[g][u] = vn[g][u];
              }
          }
        if (col < n)
#pragma unroll
          for (int u = 0; u < E; ++u)
            if (r0 + 16 * u < n)
              V[(size_t)col * n + r0 + 16 * u] = c[u];
      }
    } // namespace

    void tridiagonalize(hipStream_t s, double *A, u32 n, double *d, double *e, double *tau)
    {
      DFX_REQUIRE(n >= 2 && n <= TRIDIAG_MAX, "tridiagonalize: 2..128 columns");
      const int    ld  = (int)((n + 23) / 32 * 32 + 8);
      const size_t lds = ((size_t)n * ld + 256) * sizeof(double);
      if (lds > 64 * 1024)
        DFX_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&tridiagK),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 152 * 1024));
      tridiagK<<<1, 1024, lds, s>>>(A, (int)n, ld, d, e, tau);
      checkLaunch("tridiagonalize");
    }

    void applyReflectors(hipStream_t s, const double *A, const double *tau, u32 n, const double *C,
                         double *V)
    {
      DFX_REQUIRE(n >= 2 && n <= 256, "applyReflectors: 2..256 columns");
      auto go = [&](auto kern) {
        kern<<<(n + 3) / 4, 64, 0, s>>>(A, tau, (int)n, C, V);
        checkLaunch("applyReflectors");
      };
      if (n <= 32)
        go(reflectK<2, 4>);
      else if (n <= 64)
        go(reflectK<4, 4>);
      else if (n <= 128)
        go(reflectK<8, 4>);
      else
        go(reflectK<16, 2>);
    }
  } // namespace k
} // namespace dfx

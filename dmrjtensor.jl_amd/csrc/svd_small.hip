// Batched one-sided Jacobi (Hestenes) SVD for small charge sectors.
//
// One workgroup per sector matrix M (R x C, column-major, ld R).  With
// n = min(R, C) <= 64 the working matrix X (rows x n, the columns of M or of
// M^T) and the accumulated rotation V (n x n) live in LDS.  Column pairs are
// rotated in the round-robin (circle) order, n/2 disjoint pairs per round,
// one group of G lanes per pair; sweeps repeat until no pair has
// |x_p . x_q| > eps sqrt(|x_p|^2 |x_q|^2).  Output has the layout of the LAPACK
// gesdd call it replaces for these sizes: S descending, U (R x n, ld R),
// Vt (n x C, ld n).
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "internal.h"

namespace dmrj {

constexpr int kSvdThreads = 256;

__device__ inline double group_sum(double v, int G) {
  for (int o = G / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__global__ __launch_bounds__(kSvdThreads) void k_svd_small(const SmallSvdJob* __restrict__ jobs,
                                                           int njobs) {
  extern __shared__ double lds[];
  const SmallSvdJob jb = jobs[blockIdx.x];
  const bool tr = jb.R < jb.C;             // work on M^T when M is wide
  const int rows = tr ? jb.C : jb.R;       // length of a working column
  const int n = tr ? jb.R : jb.C;          // number of working columns
  const int np = (n + 1) & ~1;             // even number of players
  double* X = lds;                          // [np][rows]
  double* V = lds + (size_t)np * rows;      // [np][n]
  __shared__ double sig[64];
  __shared__ int perm[64];
  __shared__ int rotated;
  const int tid = threadIdx.x;
  // load
  for (int e = tid; e < np * rows; e += kSvdThreads) {
    const int col = e / rows, r = e % rows;
    double v = 0.0;
    if (col < n) v = tr ? jb.M[(int64_t)col + (int64_t)r * jb.R] : jb.M[(int64_t)r + (int64_t)col * jb.R];
    X[e] = v;
  }
  for (int e = tid; e < np * n; e += kSvdThreads) V[e] = ((e / n) == (e % n)) ? 1.0 : 0.0;
  __syncthreads();
  const int P = np / 2;
  int G = 64;
  while (G > 1 && G * P > kSvdThreads) G >>= 1;
  const int grp = tid / G, gl = tid % G;
  const double eps = 2.220446049250313e-16;
  for (int sweep = 0; sweep < 60; ++sweep) {
    if (tid == 0) rotated = 0;
    __syncthreads();
    for (int rd = 0; rd < np - 1; ++rd) {
      if (grp < P) {
        auto player = [&](int k) { return k == 0 ? 0 : ((k - 1 + rd) % (np - 1)) + 1; };
        int p = player(grp), q = player(np - 1 - grp);
        if (p > q) { const int t = p; p = q; q = t; }
        if (q < n) {
          double* xp = X + (size_t)p * rows;
          double* xq = X + (size_t)q * rows;
          double a = 0.0, b = 0.0, g = 0.0;
          for (int r = gl; r < rows; r += G) {
            const double u = xp[r], w = xq[r];
            a += u * u;
            b += w * w;
            g += u * w;
          }
          a = group_sum(a, G);
          b = group_sum(b, G);
          g = group_sum(g, G);
          if (fabs(g) > eps * sqrt(a * b) && g != 0.0) {
            const double zeta = (b - a) / (2.0 * g);
            const double t = (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
            const double c = 1.0 / sqrt(1.0 + t * t), s = c * t;
            for (int r = gl; r < rows; r += G) {
              const double u = xp[r], w = xq[r];
              xp[r] = c * u - s * w;
              xq[r] = s * u + c * w;
            }
            double* vp = V + (size_t)p * n;
            double* vq = V + (size_t)q * n;
            for (int r = gl; r < n; r += G) {
              const double u = vp[r], w = vq[r];
              vp[r] = c * u - s * w;
              vq[r] = s * u + c * w;
            }
            if (gl == 0) rotated = 1;
          }
        }
      }
      __syncthreads();
    }
    const int any = rotated;
    __syncthreads();
    if (!any) break;
  }
  // singular values = column norms
  for (int col = grp; grp < P && col < n; col += P) {
    double a = 0.0;
    const double* x = X + (size_t)col * rows;
    for (int r = gl; r < rows; r += G) a += x[r] * x[r];
    a = group_sum(a, G);
    if (gl == 0) sig[col] = sqrt(a);
  }
  __syncthreads();
  if (tid == 0) {
    for (int i = 0; i < n; ++i) perm[i] = i;
    for (int i = 1; i < n; ++i) {  // stable insertion sort, descending
      const int pi = perm[i];
      int j = i - 1;
      while (j >= 0 && sig[perm[j]] < sig[pi]) {
        perm[j + 1] = perm[j];
        --j;
      }
      perm[j + 1] = pi;
    }
  }
  __syncthreads();
  for (int i = tid; i < n; i += kSvdThreads) jb.S[i] = sig[perm[i]];
  // left vectors of the working matrix: X[:,k]/sigma_k (rows); right: V[:,k] (n)
  // M = X V^T (working) -> if !tr: U = X/sigma (R x n), Vt = V^T (n x C)
  //                       if  tr: M^T = X V^T -> M = V X^T: U = V (R x n), Vt = (X/sigma)^T (n x C)
  for (int e = tid; e < n * rows; e += kSvdThreads) {
    const int k = e / rows, r = e % rows;
    const int src = perm[k];
    const double sg = sig[src];
    const double val = sg > 0.0 ? X[(size_t)src * rows + r] / sg : 0.0;
    if (!tr)
      jb.U[(int64_t)r + (int64_t)k * jb.R] = val;      // U[r, k], ld R
    else
      jb.Vt[(int64_t)k + (int64_t)r * n] = val;        // Vt[k, r], ld n
  }
  for (int e = tid; e < n * n; e += kSvdThreads) {
    const int k = e / n, r = e % n;
    const double val = V[(size_t)perm[k] * n + r];
    if (!tr)
      jb.Vt[(int64_t)k + (int64_t)r * n] = val;        // Vt[k, r] = V[r, k]
    else
      jb.U[(int64_t)r + (int64_t)k * jb.R] = val;      // U[r, k] = V[r, k]
  }
}

// The same for sides up to 16, real or complex (interleaved planes: imaginary
// parts after the real ones), bound by the latency of its rounds: 16 lanes a
// pair, so that the inner products are summed inside a DPP row, an approximate
// tangent (any nearby rotation serves) and a Newton reciprocal root for the
// cosine, and the pair stored with the larger column first, which makes graded
// matrices converge in fewer sweeps.  Complex pairs are turned to a real inner
// product by the phase of the second column.  The accumulated factor drifts
// from unitarity by the rounding of its rotations; one Newton-Schulz step
// V (3 - V^H V) / 2 takes that out, so neither factor needs a
// re-orthonormalisation afterwards (17 launches for the kernel above).  A pair
// counts as orthogonal at 4 eps of its norms (above: eps, but without the last
// step); measured errors of factors and values are no larger.  Bond
// step at m = 16: 451 to 250 us; real-time TDVP pass of 14 sites at m = 12,
// whose complex sectors took the blocked solver: 11.4 to 10.1 ms.
constexpr int kTinyThreads = 128;

__device__ inline double row_sum(double v) {  // over the 16 lanes of a DPP row, in all of them
  auto ror = [](double x, auto ctrl) {
    constexpr int C = decltype(ctrl)::value;
    return x + __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), C, 0xf, 0xf, true),
                                __builtin_amdgcn_update_dpp(0, __double2loint(x), C, 0xf, 0xf, true));
  };
  v = ror(v, std::integral_constant<int, 0x128>());
  v = ror(v, std::integral_constant<int, 0x124>());
  v = ror(v, std::integral_constant<int, 0x122>());
  return ror(v, std::integral_constant<int, 0x121>());
}

__device__ inline double newton_rsqrt(double h) {
  double y = __builtin_amdgcn_rsq(h);
  y = fma(0.5 * y, fma(-h * y, y, 1.0), y);
  return fma(0.5 * y, fma(-h * y, y, 1.0), y);
}

template <bool Z>
__global__ __launch_bounds__(kTinyThreads) void k_svd_tiny(const SmallSvdJob* __restrict__ jobs, double scale) {
  extern __shared__ double lds[];
  __shared__ double E[Z ? 2 : 1][16 * 16];
  __shared__ double sig[16];
  __shared__ int perm[16];
  __shared__ int rotated[2];
  const SmallSvdJob jb = jobs[blockIdx.x];
  const bool tr = jb.R < jb.C;             // work on M^H when M is wide
  const int rows = tr ? jb.C : jb.R, n = tr ? jb.R : jb.C, np = (n + 1) & ~1;
  const int xs = np * rows, vs = np * n;   // planes
  double* X = lds;                         // [np][rows], imaginary plane after it
  double* V = lds + (Z ? 2 : 1) * xs;      // [np][n]
  const int tid = threadIdx.x, grp = tid >> 4, gl = tid & 15;
  const int64_t plane = (int64_t)jb.R * jb.C;
  for (int e = tid; e < xs; e += kTinyThreads) {
    const int col = e / rows, r = e - col * rows;
    const int64_t o = tr ? (int64_t)col + (int64_t)r * jb.R : (int64_t)r + (int64_t)col * jb.R;
    X[e] = col < n ? scale * jb.M[o] : 0.0;
    if constexpr (Z) X[xs + e] = col < n ? (tr ? -scale : scale) * jb.M[plane + o] : 0.0;
  }
  for (int e = tid; e < vs; e += kTinyThreads) {
    V[e] = e / n == e % n ? 1.0 : 0.0;
    if constexpr (Z) V[vs + e] = 0.0;
  }
  if (tid < 2) rotated[tid] = 0;
  __syncthreads();
  constexpr double tol2 = 16.0 * 2.220446049250313e-16 * 2.220446049250313e-16;
  // rotates columns xp, xq of an array of `len` rows: p' = c p - s q~, q' = s p
  // + c q~ with q~ = (wr + i wi) q, exchanged when swap
  auto rotate = [&](double* xp, double* xq, int len, int pl, double c, double s, double wr, double wi, bool swap) {
    for (int r = gl; r < len; r += 16) {
      const double p = xp[r], q = xq[r];
      if constexpr (Z) {
        const double pi = xp[pl + r], qi = xq[pl + r];
        const double xr = wr * q - wi * qi, xi = wr * qi + wi * q;
        const double ar = c * p - s * xr, ai = c * pi - s * xi, br = s * p + c * xr, bi = s * pi + c * xi;
        xp[r] = swap ? br : ar;
        xp[pl + r] = swap ? bi : ai;
        xq[r] = swap ? ar : br;
        xq[pl + r] = swap ? ai : bi;
      } else {
        const double a = c * p - s * q, b = s * p + c * q;
        xp[r] = swap ? b : a;
        xq[r] = swap ? a : b;
      }
    }
  };
  for (int sweep = 0; sweep < 60 && n > 1; ++sweep) {
    for (int rd = 0; rd < np - 1; ++rd) {
      if (grp < np / 2) {
        auto player = [&](int k) { return k == 0 ? 0 : (k - 1 + rd) % (np - 1) + 1; };
        const int k0 = player(grp), k1 = player(np - 1 - grp), p = min(k0, k1), q = max(k0, k1);
        if (q < n) {
          double* xp = X + p * rows;
          double* xq = X + q * rows;
          double a = 0.0, b = 0.0, g = 0.0, gi = 0.0;
#pragma unroll 4
          for (int r = gl; r < rows; r += 16) {
            const double u = xp[r], w = xq[r];
            a += u * u;
            b += w * w;
            g += u * w;
            if constexpr (Z) {
              const double ui = xp[xs + r], wi = xq[xs + r];
              a += ui * ui;
              b += wi * wi;
              g += ui * wi;
              gi += u * wi - ui * w;
            }
          }
          a = row_sum(a);
          b = row_sum(b);
          g = row_sum(g);
          double wr = 1.0, wi = 0.0, g2 = g * g;
          if constexpr (Z) {
            gi = row_sum(gi);
            g2 += gi * gi;
          }
          const bool go = g2 > tol2 * a * b && g2 > 1e-290;
          if (go || a < b) {
            double c = 1.0, s = 0.0;
            bool swap = a < b;
            if (go) {
              if constexpr (Z) {
                const double y = newton_rsqrt(g2);
                wr = g * y;
                wi = -gi * y;
                g = g2 * y;
              }
              const double d = b - a, z = d * __builtin_amdgcn_rcp(2.0 * g), h = fabs(z);
              double t;  // sign(z) / (|z| + sqrt(1 + z^2))
              if (h < 1e15) {
                const float f = (float)h;
                t = (double)__builtin_amdgcn_rcpf(f + __builtin_amdgcn_sqrtf(fmaf(f, f, 1.0f)));
                if (z < 0.0) t = -t;
              } else {
                t = g * __builtin_amdgcn_rcp(d);
              }
              c = newton_rsqrt(1.0 + t * t);
              s = c * t;
              swap = a - t * g < b + t * g;
              if (gl == 0) rotated[sweep & 1] = 1;
            }
            rotate(xp, xq, rows, xs, c, s, wr, wi, swap);
            rotate(V + p * n, V + q * n, n, vs, c, s, wr, wi, swap);
          }
        }
      }
      __syncthreads();
    }
    const int any = rotated[sweep & 1];
    if (tid == 0) rotated[(sweep + 1) & 1] = 0;
    __syncthreads();
    if (!any) break;
  }
  // singular values: column norms, descending
  for (int col = grp; col < n; col += kTinyThreads / 16) {
    double a = 0.0;
    for (int r = gl; r < rows; r += 16) {
      a += X[col * rows + r] * X[col * rows + r];
      if constexpr (Z) a += X[xs + col * rows + r] * X[xs + col * rows + r];
    }
    a = row_sum(a);
    if (gl == 0) sig[col] = sqrt(a);
  }
  // E = (3 - V^H V) / 2
  for (int e = tid; e < n * n; e += kTinyThreads) {
    const int i = e / n, j = e - i * n;
    double gr = 0.0, gi = 0.0;
    for (int r = 0; r < n; ++r) {
      const double u = V[i * n + r], w = V[j * n + r];
      gr += u * w;
      if constexpr (Z) {
        const double ui = V[vs + i * n + r], wi = V[vs + j * n + r];
        gr += ui * wi;
        gi += u * wi - ui * w;
      }
    }
    E[0][i * 16 + j] = (i == j ? 1.5 : 0.0) - 0.5 * gr;
    if constexpr (Z) E[Z ? 1 : 0][i * 16 + j] = -0.5 * gi;
  }
  __syncthreads();
  if (tid < n) {
    int rank = 0;
    for (int i = 0; i < n; ++i) rank += sig[i] > sig[tid] || (sig[i] == sig[tid] && i < tid);
    perm[rank] = tid;
    jb.S[rank] = sig[tid] / scale;
  }
  __syncthreads();
  // tall: U = X / sigma, Vt = V^H; wide: U = V, Vt = (X / sigma)^H
  const int64_t pu = (int64_t)jb.R * n, pv = (int64_t)n * jb.C;
  for (int e = tid; e < n * rows; e += kTinyThreads) {
    const int k = e / rows, r = e - k * rows, src = perm[k];
    const double sg = sig[src];
    const double x = sg > 0.0 ? X[src * rows + r] / sg : 0.0;
    const int64_t o = tr ? (int64_t)k + (int64_t)r * n : (int64_t)r + (int64_t)k * jb.R;
    (tr ? jb.Vt : jb.U)[o] = x;
    if constexpr (Z) {
      const double y = sg > 0.0 ? X[xs + src * rows + r] / sg : 0.0;
      if (tr)
        jb.Vt[pv + o] = -y;
      else
        jb.U[pu + o] = y;
    }
  }
  for (int e = tid; e < n * n; e += kTinyThreads) {
    const int k = e / n, r = e - k * n, src = perm[k];
    double x = 0.0, y = 0.0;
    for (int i = 0; i < n; ++i) {
      const double v = V[i * n + r], f = E[0][i * 16 + src];
      x += v * f;
      if constexpr (Z) {
        const double vi = V[vs + i * n + r], fi = E[Z ? 1 : 0][i * 16 + src];
        x -= vi * fi;
        y += v * fi + vi * f;
      }
    }
    const int64_t o = tr ? (int64_t)r + (int64_t)k * jb.R : (int64_t)k + (int64_t)r * n;
    (tr ? jb.U : jb.Vt)[o] = x;
    if constexpr (Z) {
      if (tr)
        jb.U[pu + o] = y;
      else
        jb.Vt[pv + o] = -y;
    }
  }
}

// Singular triplets from the eigenpairs of the augmented symmetric matrix
// [[0, M], [M^T, 0]] (size N >= R + C, zero padded): eigenvalue +sigma_i with
// eigenvector (u_i; v_i)/sqrt(2).  Eigenvalues are ascending, so sigma_i is
// column N-1-i.  Each half is normalised by its own norm.
__global__ __launch_bounds__(256) void k_aug_extract(const AugJob* __restrict__ jobs,
                                                     const int2* __restrict__ work, int nwork) {
  for (int wi = blockIdx.x; wi < nwork; wi += gridDim.x) {
    const int2 w = work[wi];
    const AugJob jb = jobs[w.x];
    const int i = w.y;
    const int col = jb.N - 1 - i;
    const double* v = jb.A + (int64_t)col * jb.N;
    double nt = 0.0, nb = 0.0;
    for (int r = threadIdx.x; r < jb.R; r += 256) nt += v[r] * v[r];
    for (int r = threadIdx.x; r < jb.C; r += 256) nb += v[jb.R + r] * v[jb.R + r];
    __shared__ double red[2][4];
    for (int o = 32; o > 0; o >>= 1) {
      nt += __shfl_down(nt, o, 64);
      nb += __shfl_down(nb, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
      red[0][threadIdx.x >> 6] = nt;
      red[1][threadIdx.x >> 6] = nb;
    }
    __syncthreads();
    const double st = sqrt(red[0][0] + red[0][1] + red[0][2] + red[0][3]);
    const double sb = sqrt(red[1][0] + red[1][1] + red[1][2] + red[1][3]);
    __syncthreads();
    const double it = st > 0.0 ? 1.0 / st : 0.0, ib = sb > 0.0 ? 1.0 / sb : 0.0;
    for (int r = threadIdx.x; r < jb.R; r += 256) jb.U[(int64_t)r + (int64_t)i * jb.R] = v[r] * it;
    for (int r = threadIdx.x; r < jb.C; r += 256) jb.Vt[(int64_t)i + (int64_t)r * jb.kmin] = v[jb.R + r] * ib;
    if (threadIdx.x == 0) jb.S[i] = fabs(jb.W[col]);
  }
}

void launch_aug_extract(Context& c, const std::vector<AugJob>& jobs) {
  if (jobs.empty()) return;
  std::vector<int2> work;
  for (size_t j = 0; j < jobs.size(); ++j)
    for (int i = 0; i < jobs[j].kmin; ++i) work.push_back(make_int2((int)j, i));
  auto* dj = (AugJob*)c.upload(jobs.data(), jobs.size() * sizeof(AugJob));
  auto* dw = (int2*)c.upload(work.data(), work.size() * sizeof(int2));
  const int grid = (int)std::min<size_t>(work.size(), (size_t)c.num_cu * 8);
  hipLaunchKernelGGL(k_aug_extract, dim3(grid), dim3(256), 0, c.stream, dj, dw, (int)work.size());
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw Error(-3, std::string("HIP: ") + hipGetErrorString(e));
}

size_t small_svd_lds(int R, int C, bool cplx) {
  const int rows = R < C ? C : R;
  const int n = R < C ? R : C;
  const int np = (n + 1) & ~1;
  return ((size_t)np * rows + (size_t)np * n) * sizeof(double) * (cplx ? 2 : 1);
}

// Launches on the context's side stream after everything queued on the main
// stream so far (inputs, the job table upload); the caller joins with
// hipStreamWaitEvent(c.stream, c.side_out) before reading the results.
// Returns whether a kernel was launched.
bool launch_svd_small(Context& c, const std::vector<SmallSvdJob>& jobs, size_t lds_bytes, bool cplx, double scale) {
  if (jobs.empty()) return false;
  auto* dj = (SmallSvdJob*)c.upload(jobs.data(), jobs.size() * sizeof(SmallSvdJob));
  auto ok = [](hipError_t e) {
    if (e != hipSuccess) throw Error(-3, std::string("HIP: ") + hipGetErrorString(e));
  };
  ok(hipEventRecord(c.side_in, c.stream));
  ok(hipStreamWaitEvent(c.side, c.side_in, 0));
  const dim3 g((unsigned)jobs.size());
  if (scale == 0.0)
    hipLaunchKernelGGL(k_svd_small, g, dim3(kSvdThreads), lds_bytes, c.side, dj, (int)jobs.size());
  else if (cplx)
    hipLaunchKernelGGL(k_svd_tiny<true>, g, dim3(kTinyThreads), lds_bytes, c.side, dj, scale);
  else
    hipLaunchKernelGGL(k_svd_tiny<false>, g, dim3(kTinyThreads), lds_bytes, c.side, dj, scale);
  ok(hipGetLastError());
  ok(hipEventRecord(c.side_out, c.side));
  return true;
}

}  // namespace dmrj

// Batched SVD of the larger charge sectors: QR-preconditioned block one-sided
// Jacobi on the FP64 matrix cores.
//
// The wanted orthonormal vectors of a sector M (R x C) are the left singular
// vectors of A0 = M (dir > 0: U) or A0 = M^T (dir < 0: V), an n x o matrix
// with K = min(n, o).  Two unpivoted Householder factorisations precede the
// Jacobi sweeps (the preconditioning of Drmac and Veselic, SIAM J. Matrix
// Anal. Appl. 29 (2008), with a column sort in place of the pivoting):
//   A0 P = Q0 R0, A1 = R0^T;  A1 = Q1 R1, A2 = R1^T
// (P orders the columns by decreasing norm).  Two-site tensors are graded on
// both sides, so every factorisation moves A_i closer to a diagonal matrix:
// on the 433 x 462 sector of an m=1024 Heisenberg state the sweeps fall from
// 20 (columns sorted, no factorisation) over 10 to 7, and the error of the
// singular values from 5e-14 to 1e-15 of the largest.  Jacobi sweeps then
// rotate the columns of A2 until they are orthogonal, A2 V = W D, so that
// R1 = V D W^T, A1 = Q1 V D W^T, R0 = W D (Q1 V)^T, and the vectors are
// Q0 [W; 0]: neither V nor Q1 nor P is needed.
//
// Storage: column panels of 16, row-major inside a panel, so that a 16 x 16
// tile is 256 consecutive doubles and register r of lane l of a wave's tile
// (row 4r + l/16, column l%16: the accumulator layout of
// v_mfma_f64_16x16x4f64) is element 64 r + l.  That same layout is both the
// A operand (transposed) and the B operand of the Gram products.
//
// Launches: one per panel of a factorisation (every slab of 16 columns is a
// work-group that keeps its columns in registers, applies the block
// reflector of the panel and writes its finished rows of R transposed into
// the next matrix; the group of the next panel goes on to factorise it, so
// panel and update are one launch), one per Jacobi round (every block pair a
// work-group: Gram matrix, one inner sweep, product), one for the vectors.
// All sectors of a bond are in the same launches.
//
// What bounds it is latency, not bytes or flops: a bond is about 2 K/16 panel
// launches of 20 to 45 us (K the largest sector; 16 dependent columns each)
// and 7 to 8 sweeps of K/16 rounds of 15 to 45 us.  Bond step at the middle of
// an m=1024 Heisenberg chain (sectors to 508): 31.0 ms with the batched
// eigensolve of the augmented matrices, five launches per column of R + C,
// 7.1 ms with this; m=2048 Hubbard (sectors to 1164): 134 and 31 ms.  A third
// factorisation (of A2) saves a sweep and costs its panels: 7.3 and 30.7 ms, and
// 1.06 against 0.98 ms at a single 100 x 100 sector.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "dmrj.h"
#include "internal.h"

#define HIP_OK(x)                                                                        \
  do {                                                                                   \
    hipError_t e_ = (x);                                                                 \
    if (e_ != hipSuccess) throw dmrj::Error(-3, std::string("HIP: ") + hipGetErrorString(e_)); \
  } while (0)

namespace dmrj {

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef double double2_t __attribute__((ext_vector_type(2)));

namespace {

__device__ __forceinline__ double4_t mfma(double a, double b, double4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// The value of lane J of every row of 16 lanes (DPP row_newbcast).
template <int J>
__device__ __forceinline__ double row_bcast(double x) {
  const int2 v = __builtin_bit_cast(int2, x);
  int2 r;
  r.x = __builtin_amdgcn_update_dpp(0, v.x, 0x150 + J, 0xf, 0xf, true);
  r.y = __builtin_amdgcn_update_dpp(0, v.y, 0x150 + J, 0xf, 0xf, true);
  return __builtin_bit_cast(double, r);
}

// Sum over the four rows of 16 lanes, in every lane (lane swaps of VALU
// registers instead of LDS permutes).
__device__ __forceinline__ double sum_rows(double x) {
  int2 v = __builtin_bit_cast(int2, x);
  auto lo = __builtin_amdgcn_permlane32_swap(v.x, v.x, false, false);
  auto hi = __builtin_amdgcn_permlane32_swap(v.y, v.y, false, false);
  x = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
  v = __builtin_bit_cast(int2, x);
  lo = __builtin_amdgcn_permlane16_swap(v.x, v.x, false, false);
  hi = __builtin_amdgcn_permlane16_swap(v.y, v.y, false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}

// 1 / sqrt(x) and 1 / x for normal x: the hardware's approximation (relative
// error below 2^-20) and one step of third order, which leaves rounding
// errors only.  A fifth of the instructions of the IEEE forms, which carry the
// latency of every reflector and rotation.
__device__ __forceinline__ double fast_rsqrt(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}
__device__ __forceinline__ double fast_rcp(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);
  return fma(y * e, 1.0 + e, y);
}

// Tangent of the Jacobi rotation from its cotangent of the double angle
// f >= 0 (1e-38 for the pairs of columns furthest apart: no overflow in f^2).
__device__ __forceinline__ float jacobi_tangent(float f) {
  return __builtin_amdgcn_rcpf(f + (f < 1e15f ? __builtin_amdgcn_sqrtf(fmaf(f, f, 1.0f)) : f));
}

// The wave's number in its work-group, in a scalar register.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

__device__ __forceinline__ int blocks16(int n) { return (n + 15) >> 4; }

constexpr int kGroup = 2;  // register tiles whose loads are in flight together

struct QrShared {
  double* red;   // NW x 256 partial tiles
  double* w;     // 256
  double* dots;  // 2 x NW x 16
  double* piv;   // 2 x 16
  double* s;     // 256: V^T V above the diagonal
  double* tau;   // 16
};

// W = V^T A over the register tiles of the work-group's slab (tiles of
// row blocks base + w + NW i), summed over the waves; every lane returns its
// elements in the B operand layout.
template <int NW, int TPW>
__device__ __forceinline__ double4_t slab_vta(const double* V, int base, int rb, const double4_t (&a)[TPW],
                                              const QrShared& sh) {
  const int w = wave_id(), lane = threadIdx.x & 63;
  double4_t acc = {0.0, 0.0, 0.0, 0.0};
  // groups of tiles: the loads of a group are in flight together; tiles past
  // the end are zero, so any tile of V will do for them
#pragma unroll
  for (int i0 = 0; i0 < TPW; i0 += kGroup)
    if (base + w + NW * i0 < rb) {
#pragma unroll
      for (int i = i0; i < i0 + kGroup; ++i) {
        const double* v = V + (int64_t)min(base + w + NW * i, rb - 1) * 256 + lane;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc = mfma(v[64 * r], a[i][r], acc);
      }
    }
#pragma unroll
  for (int r = 0; r < 4; ++r) sh.red[w * 256 + 64 * r + lane] = acc[r];
  __syncthreads();
  if (threadIdx.x < 256) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < NW; ++k) t += sh.red[k * 256 + threadIdx.x];
    sh.w[threadIdx.x] = t;
  }
  __syncthreads();
  double4_t r;
#pragma unroll
  for (int k = 0; k < 4; ++k) r[k] = sh.w[64 * k + lane];
  return r;
}

// A -= V Y on the register tiles; Y's register s holds row 4 (l/16) + s of
// column l%16, the reduction index order of V's four consecutive elements.
template <int NW, int TPW>
__device__ __forceinline__ void slab_sub(const double* V, int base, int rb, double4_t (&a)[TPW], double4_t Y) {
  const int w = wave_id(), lane = threadIdx.x & 63;
#pragma unroll
  for (int i0 = 0; i0 < TPW; i0 += kGroup)
    if (base + w + NW * i0 < rb) {
#pragma unroll
      for (int i = i0; i < i0 + kGroup; ++i) {
        const int b = base + w + NW * i;
        const double z = b < rb ? -1.0 : 0.0;  // tiles past the end stay zero
        const double2_t* v =
            (const double2_t*)(V + (int64_t)min(b, rb - 1) * 256 + (lane & 15) * 16 + 4 * (lane >> 4));
        const double2_t v0 = v[0], v1 = v[1];
        a[i] = mfma(z * v0[0], Y[0], a[i]);
        a[i] = mfma(z * v0[1], Y[1], a[i]);
        a[i] = mfma(z * v1[0], Y[2], a[i]);
        a[i] = mfma(z * v1[1], Y[3], a[i]);
      }
    }
}

// One column of a panel: Householder reflector of column J (pivot in row J of
// the pivot tile, tile 0 of wave pw) and its application to the columns
// right of it.  One reduction gives the products of column J with all 16
// columns: the norm, the update coefficients and the inner products of the
// reflectors that the triangular factor needs.
template <int J, int NW, int TPW>
__device__ __forceinline__ void panel_column(double4_t (&a)[TPW], int nt, bool top, const QrShared& sh) {
  const int w = wave_id(), lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  double4_t dots = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < TPW; ++i)
    if (i < nt) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double x = row_bcast<J>(a[i][r]);
        const double y = (i == 0 && top && 4 * r + g <= J) ? 0.0 : a[i][r];
        dots[r] = fma(x, y, dots[r]);
      }
    }
  const double dot = sum_rows((dots[0] + dots[1]) + (dots[2] + dots[3]));
  double* d = sh.dots + (J & 1) * NW * 16;
  double* pv = sh.piv + (J & 1) * 16;
  if (g == 0) d[w * 16 + c] = dot;
  if (top && g == (J & 3)) pv[c] = a[0][J >> 2];
  __syncthreads();
  double part[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < NW; ++k) part[k & 3] += d[k * 16 + c];
  const double tot = (part[0] + part[1]) + (part[2] + part[3]);
  const double pr = pv[c];
  const double xn = row_bcast<J>(tot), alpha = row_bcast<J>(pr);
  double tau = 0.0, beta = alpha, scale = 0.0;
  if (xn > 0.0) {
    const double h = fma(alpha, alpha, xn);
    const double ri = copysign(fast_rsqrt(h), -alpha);  // 1 / beta
    beta = h * ri;
    tau = fma(-alpha, ri, 1.0);
    scale = fast_rcp(alpha - beta);
  }
  const double vc = fma(scale, tot, pr);   // v_J . column c (c < J: the column is v_c)
  const double wc = c > J ? tau * vc : 0.0;
  if (w == 0 && g == 0) {
    if (c < J) sh.s[c * 16 + J] = vc;
    if (c == J) sh.tau[J] = tau;
  }
  // column J becomes the reflector, x + (scale - 1) x, the columns right of it
  // lose w_c scale x: one multiply-add with a coefficient per column.  The
  // broadcasts of the first pass are made again: held across the barrier they
  // would take as many registers as the tiles.
  const double coef = c == J ? scale - 1.0 : -wc * scale;
#pragma unroll
  for (int i = 0; i < TPW; ++i)
    if (i < nt) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        double x = a[i][r];
        asm volatile("" : "+v"(x));
        const double y = fma(coef, row_bcast<J>(x), x);
        if (i == 0 && top) {
          const int row = 4 * r + g;
          a[i][r] = row > J ? y : row == J ? (c == J ? beta : x - wc) : x;
        } else {
          a[i][r] = y;
        }
      }
    }
}

template <int J, int NW, int TPW>
__device__ __forceinline__ void panel_columns(double4_t (&a)[TPW], int nt, bool top, const QrShared& sh) {
  if constexpr (J < 16) {
    panel_column<J, NW, TPW>(a, nt, top, sh);
    panel_columns<J + 1, NW, TPW>(a, nt, top, sh);
  }
}

}  // namespace

// One step of factorisation `which` (A[which] = Q R, A[which + 1] = R^T): the
// block reflector of panel s applied to the slabs right of it, and panel
// s + 1 factorised by its slab's group.  s = -1 factorises panel 0.
//
// A slab of 16 columns per work-group, its rows in registers (NW x TPW tiles
// of 16): read once, written once, V read from L2 twice (once per operand
// layout).  The step's length is that of the group that goes on to the
// panel: 16 columns of one reduction and one barrier each.
template <int NW, int TPW>
__global__ __launch_bounds__(NW * 64) void k_qj_qr(const QjJob* __restrict__ jobs, int which, int s) {
  __shared__ double red[NW * 256], wl[256], dots[2 * NW * 16], piv[32], sm[256], taul[16];
  const QrShared sh{red, wl, dots, piv, sm, taul};
  const QjJob& jb = jobs[blockIdx.y];
  const int rows = which == 0 ? jb.n : jb.o, cols = which == 0 ? jb.o : jb.K;
  const int rb = blocks16(rows), nb = blocks16(cols), np = min(rb, nb);
  const int t = s + 1 + blockIdx.x;
  if (s >= np || t >= nb) return;
  const int w = wave_id(), lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int base = max(s, 0);
  double* P = jb.A[which] + (int64_t)t * rb * 256;
  double4_t a[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int b = base + w + NW * i;
#pragma unroll
    for (int r = 0; r < 4; ++r) a[i][r] = b < rb ? P[(int64_t)b * 256 + 64 * r + lane] : 0.0;
  }
  double* An = jb.A[which + 1];
  const int rbn = nb;  // row blocks of the next matrix
  if (s >= 0) {
    const double* V = jb.A[which] + (int64_t)s * rb * 256;
    const double* T = jb.T[which] + (int64_t)s * 256;
    const double4_t W = slab_vta<NW, TPW>(V, base, rb, a, sh);
    // Y = T^T W, its rows ordered for slab_sub: row i = 4r + g of the product is row 4g + r of Y
    const int m = 4 * (c & 3) + (c >> 2);
    double4_t Y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 4; ++k) Y = mfma(T[(4 * k + g) * 16 + m], W[k], Y);
    slab_sub<NW, TPW>(V, base, rb, a, Y);
    if (w == 0) {  // rows 16 s .. of R are final: transposed into the next matrix
      double* q = An + (int64_t)s * rbn * 256 + (int64_t)t * 256 + c * 16 + g;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        q[4 * r] = a[0][r];
        a[0][r] = 0.0;
      }
    }
  }
  const bool factor = t == s + 1 && t < np;
  const int pw = s >= 0 ? 1 : 0;  // wave of the pivot tile
  if (factor) {
    const bool top = w == pw;
    panel_columns<0, NW, TPW>(a, (rb - base - w + NW - 1) / NW, top, sh);
    if (top) {
      double* q = An + (int64_t)t * rbn * 256 + (int64_t)t * 256 + c * 16 + g;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * r + g;
        q[4 * r] = row <= c ? a[0][r] : 0.0;
        a[0][r] = row > c ? a[0][r] : row == c ? 1.0 : 0.0;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int b = base + w + NW * i;
    if (b < rb && !(s >= 0 && b == s)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) P[(int64_t)b * 256 + 64 * r + lane] = a[i][r];
    }
  }
  if (!factor) return;
  __syncthreads();
  // T = (diag(1/tau) + strictly upper V^T V)^-1, one column per lane
  if (w == 0 && g == 0) {
    double x[16];
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      double acc0 = 0.0, acc1 = 0.0;
#pragma unroll
      for (int k = i + 1; k < 16; ++k) {
        if (k & 1)
          acc1 += sm[i * 16 + k] * x[k];
        else
          acc0 += sm[i * 16 + k] * x[k];
      }
      x[i] = i == c ? taul[i] : i < c ? -taul[i] * (acc0 + acc1) : 0.0;
    }
    double* T = jb.T[which] + (int64_t)t * 256;
#pragma unroll
    for (int i = 0; i < 16; ++i) T[i * 16 + c] = x[i];
  }
}

// Squared column norms of A0 (columns of M for dir > 0, rows for dir < 0): 64
// columns a group.
__global__ __launch_bounds__(256) void k_qj_norms0(const QjJob* __restrict__ jobs) {
  __shared__ double part[4][64];
  const QjJob& jb = jobs[blockIdx.y];
  const int j0 = blockIdx.x * 64;
  if (j0 >= jb.o) return;
  if (j0 == 0 && threadIdx.x == 0) *jb.last = -1;
  const int w = wave_id(), lane = threadIdx.x & 63;
  if (jb.dir < 0) {
    double acc = 0.0;
    if (j0 + lane < jb.o)
      for (int i = w; i < jb.n; i += 4) {
        const double v = jb.M[(int64_t)(j0 + lane) + (int64_t)i * jb.R];
        acc += v * v;
      }
    part[w][lane] = acc;
    __syncthreads();
    if (w == 0 && j0 + lane < jb.o) jb.nrm[j0 + lane] = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
  } else {
    for (int k = w; k < 64 && j0 + k < jb.o; k += 4) {
      double acc = 0.0;
      for (int i = lane; i < jb.n; i += 64) {
        const double v = jb.M[(int64_t)i + (int64_t)(j0 + k) * jb.R];
        acc += v * v;
      }
      for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
      if (lane == 0) jb.nrm[j0 + k] = acc;
    }
  }
}

// perm[rank of column j] = j, norms descending, ties by index.
__global__ __launch_bounds__(256) void k_qj_rank(const QjJob* __restrict__ jobs) {
  const QjJob& jb = jobs[blockIdx.y];
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (blockIdx.x * 256 >= jb.o) return;
  __shared__ double buf[256];
  const double x = j < jb.o ? jb.nrm[j] : 0.0;
  int rank = 0;
  for (int k0 = 0; k0 < jb.o; k0 += 256) {
    __syncthreads();
    if (k0 + threadIdx.x < jb.o) buf[threadIdx.x] = jb.nrm[k0 + threadIdx.x];
    __syncthreads();
    const int kn = min(256, jb.o - k0);
    for (int k = 0; k < kn; ++k) rank += buf[k] > x || (buf[k] == x && k0 + k < j);
  }
  if (j < jb.o) jb.perm[rank] = j;
}

// Panels of A0: sorted columns, scaled, zero-padded.
__global__ __launch_bounds__(256) void k_qj_gather(const QjJob* __restrict__ jobs, double scale) {
  const QjJob& jb = jobs[blockIdx.y];
  const int p = blockIdx.x;
  if (p >= blocks16(jb.o)) return;
  const int rb = blocks16(jb.n), c = threadIdx.x & 15, rr = threadIdx.x >> 4;
  const int col = p * 16 + c < jb.o ? jb.perm[p * 16 + c] : -1;
  double* dst = jb.A[0] + (int64_t)p * rb * 256 + threadIdx.x;
  const int64_t cs = jb.dir > 0 ? jb.R : 1, is = jb.dir > 0 ? 1 : jb.R;
  for (int b = blockIdx.z; b < rb; b += gridDim.z) {
    const int i = b * 16 + rr;
    dst[(int64_t)b * 256] = col >= 0 && i < jb.n ? scale * jb.M[col * cs + i * is] : 0.0;
  }
}

// One Jacobi round on A2: block pair k of the circle schedule per
// work-group.  Gram matrix of the 32 columns on the matrix cores, an
// approximate eigenbasis V of it in LDS, columns ordered by norm, and the
// product Y V on the matrix cores.  Pairs whose columns are orthogonal already
// (relative to tol; norms below `floor` count as `floor`) stop after the Gram
// matrix.  A sector stops when a whole cycle of its rounds rotated nothing.
__global__ __launch_bounds__(512) void k_qj_round(const QjJob* __restrict__ jobs, int step, double tol2,
                                                  double floor2) {
  constexpr int kW = 8, kU = 4, kLd = 33;  // waves, row blocks in flight per wave, leading dimension
  __shared__ double red[kW][3][256];
  __shared__ double G[2][32 * kLd], V[32 * kLd];
  __shared__ double cn[32];
  __shared__ int order[32];
  const QjJob& jb = jobs[blockIdx.y];
  const int rb = blocks16(jb.K), npan = max(2, rb), nb = (npan + 1) & ~1, nr = nb - 1;
  if ((int)blockIdx.x >= nb / 2 || step - *jb.last > nr) return;
  const int rnd = step % nr;
  auto player = [&](int i) { return i == 0 ? 0 : (i - 1 + rnd) % nr + 1; };
  int p = player(blockIdx.x), q = player(nb - 1 - blockIdx.x);
  if (p > q) {
    const int t = p;
    p = q;
    q = t;
  }
  if (q >= npan) return;
  double* Yp = jb.A[2] + (int64_t)p * rb * 256;
  double* Yq = jb.A[2] + (int64_t)q * rb * 256;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
  {
    double4_t pp = {0.0, 0.0, 0.0, 0.0}, pq = pp, qq = pp;
    for (int b0 = w; b0 < rb; b0 += kU * kW) {
      double x[kU][4], y[kU][4];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int64_t o = (int64_t)min(b0 + u * kW, rb - 1) * 256 + lane;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          x[u][r] = Yp[o + 64 * r];
          y[u][r] = Yq[o + 64 * r];
        }
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (b0 + u * kW < rb) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            pp = mfma(x[u][r], x[u][r], pp);
            pq = mfma(x[u][r], y[u][r], pq);
            qq = mfma(y[u][r], y[u][r], qq);
          }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      red[w][0][64 * r + lane] = pp[r];
      red[w][1][64 * r + lane] = pq[r];
      red[w][2][64 * r + lane] = qq[r];
    }
  }
  __syncthreads();
  for (int e = tid; e < 768; e += 512) {
    double t = 0.0;
    const int m = e >> 8, x = e & 255;
#pragma unroll
    for (int k = 0; k < kW; ++k) t += red[k][m][x];
    const int i = (x >> 4) + (m == 2 ? 16 : 0), j = (x & 15) + (m >= 1 ? 16 : 0);
    G[0][i * kLd + j] = t;
    if (m == 1) G[0][j * kLd + i] = t;
  }
  __syncthreads();
  constexpr double eps2 = 2.220446049250313e-16 * 2.220446049250313e-16;
  int act = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int i = (tid >> 5) + 16 * h, j = tid & 31;
    const double gi = G[0][i * kLd + i], gj = G[0][j * kLd + j], x = G[0][i * kLd + j];
    act |= i < j && x * x > tol2 * fmax(gi, gj) * fmax(fmin(gi, gj), floor2);
  }
  if (!__syncthreads_or(act)) return;
  if (tid == 0) *jb.last = step;
  // Inner solve, all pairs at once: X holds the Jacobi tangents of every pair
  // (scaled down where a column of X exceeds kCap in the 2-norm), V the
  // orthogonal polar factor of I + X by Newton-Schulz steps V += V (I - V^T V) / 2
  // on the matrix cores, repeated on V^T G V while the rotations were large.
  // Its off-diagonal rest is of second order, as after a cyclic sweep of
  // rotations, at a fraction of the latency: a sweep is 31 dependent rounds of
  // LDS traffic, 46000 cycles, this 8000 to 33000, and one outer sweep fewer
  // on the sectors of an m=1024 Heisenberg state.
  constexpr double kCap = 0.7, kSmall = 0.25;
  constexpr int kRepeats = 2, kNewton = 12;
  double* E = G[1];
  double* Vt = &red[0][0][0];      // the products so far
  double* Tm = Vt + 32 * kLd;      // scratch
  const int ti = (w >> 1) & 1, tj = w & 1;  // waves 0..3: a 16 x 16 tile each
  auto mul = [&](const double* A, bool tA, const double* B, double4_t acc) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int kk = 4 * k + g;
      acc = mfma(tA ? A[kk * kLd + 16 * ti + c] : A[(16 * ti + c) * kLd + kk], B[kk * kLd + 16 * tj + c], acc);
    }
    return acc;
  };
  auto get = [&](const double* D) {
    double4_t v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = D[(16 * ti + 4 * r + g) * kLd + 16 * tj + c];
    return v;
  };
  auto put = [&](double* D, double4_t v) {
#pragma unroll
    for (int r = 0; r < 4; ++r) D[(16 * ti + 4 * r + g) * kLd + 16 * tj + c] = v[r];
  };
  const double4_t zero4 = {0.0, 0.0, 0.0, 0.0};
  double cap = kCap;
  for (int it = 0; it < kRepeats;) {
    // tangents in single precision (any nearby V serves), and the order of the
    // columns by norm: the comparisons of a row are one ballot
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int i = (tid >> 5) + 16 * h, j = tid & 31;
      const double gi = G[0][i * kLd + i], gj = G[0][j * kLd + j], x = G[0][i * kLd + j], d = gj - gi;
      const bool go = i != j && x * x > fmax(eps2 * gi * gj, 1e-280);
      const float f = (float)(d * __builtin_amdgcn_rcp(go ? 2.0 * x : 1.0));
      const bool neg = f < 0.0f || (f == 0.0f && (i > j) != (x < 0.0));
      const float t = jacobi_tangent(fabsf(f));
      V[i * kLd + j] = i == j ? 1.0 : go ? (double)(neg ? -t : t) : 0.0;
      const unsigned long long m = __ballot(gj > gi || (gj == gi && j < i));
      if (j == 0) order[__popc((unsigned)(lane < 32 ? m : m >> 32))] = i;
    }
    __syncthreads();
    // X is skew: I - V^T V = X^2, and V + X^2 / 2 is orthogonal up to X^4 / 4
    double4_t v = zero4, e = zero4;
    if (w < 4) {
      v = get(V);
      e = mul(V, true, V, zero4);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool one = ti == tj && 4 * r + g == c;
        e[r] = (one ? 1.0 : 0.0) - e[r];
        if (one) cn[16 * ti + c] = -e[r];  // squared norms of the columns of X
      }
    }
    __syncthreads();
    double mx = 0.0;
#pragma unroll
    for (int k = 0; k < 32; ++k) mx = fmax(mx, cn[k]);
    const bool large = mx > kSmall * kSmall;
    if (w < 4) {
      const double a2 = mx > cap * cap ? cap * cap / mx : 1.0, a1 = sqrt(a2);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool one = ti == tj && 4 * r + g == c;
        v[r] = (one ? 1.0 : a1 * v[r]) + 0.5 * a2 * e[r];
      }
      put(V, v);
    }
    __syncthreads();
    // Newton-Schulz steps as many as |X|_2^2 = 2 mx asks for, the last one
    // checked: the deviation it found is squared by its update
    double dev = fmin(2.0 * mx, 1.0);
    dev *= 0.25 * dev;
    bool conv = dev < 1e-17;
    for (int nt = 0; nt < kNewton && !conv; ++nt) {
      int big = 0;
      if (w < 4) {
        e = mul(V, true, V, zero4);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          e[r] = (ti == tj && 4 * r + g == c ? 1.0 : 0.0) - e[r];
          big |= fabs(e[r]) > 1e-8;
        }
        put(E, 0.5 * e);
      }
      if (dev < 1e-8)
        conv = !__syncthreads_or(big);
      else
        __syncthreads();
      dev *= 0.75 * dev;
      if (w < 4) v = mul(V, false, E, get(V));
      __syncthreads();
      if (w < 4) put(V, v);
      __syncthreads();
    }
    if (!conv) {
      // |X|_2 above 1.8, where the steps do not converge (32 columns of equal
      // norms and products): at a quarter of the cap |X|_2 <= 0.7
      if (cap < kCap) return;
      cap *= 0.25;
      continue;
    }
    if (it > 0) {
      if (w < 4) v = mul(Vt, false, V, zero4);
      __syncthreads();
      if (w < 4) put(Vt, v);
    } else if (w < 4) {
      put(Vt, get(V));
    }
    if (!large || ++it == kRepeats) break;
    if (w < 4) put(Tm, mul(G[0], false, V, zero4));
    __syncthreads();
    if (w < 4) put(G[0], mul(V, true, Tm, zero4));
    __syncthreads();
  }
  __syncthreads();
  double vb[2][8];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int k = 0; k < 8; ++k)
      vb[h][k] = Vt[((k >> 2) * 16 + 4 * g + (k & 3)) * kLd + order[16 * h + c]];
  for (int b0 = w; b0 < rb; b0 += 2 * kW) {
    double2_t x[2][4];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t o = (int64_t)min(b0 + u * kW, rb - 1) * 256 + c * 16 + 4 * g;
      x[u][0] = *(const double2_t*)(Yp + o);
      x[u][1] = *(const double2_t*)(Yp + o + 2);
      x[u][2] = *(const double2_t*)(Yq + o);
      x[u][3] = *(const double2_t*)(Yq + o + 2);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (b0 + u * kW < rb) {
        double4_t yp = {0.0, 0.0, 0.0, 0.0}, yq = yp;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          yp = mfma(x[u][k >> 1][k & 1], vb[0][k], yp);
          yq = mfma(x[u][k >> 1][k & 1], vb[1][k], yq);
        }
        const int64_t o = (int64_t)(b0 + u * kW) * 256 + lane;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          Yp[o + 64 * r] = yp[r];
          Yq[o + 64 * r] = yq[r];
        }
      }
  }
}

// Column norms of A2: one panel a group, 16 per panel in nrm.
__global__ __launch_bounds__(256) void k_qj_norms3(const QjJob* __restrict__ jobs) {
  __shared__ double part[4][16];
  const QjJob& jb = jobs[blockIdx.y];
  const int rb = blocks16(jb.K), p = blockIdx.x;
  if (p >= rb) return;
  const int w = wave_id(), lane = threadIdx.x & 63;
  const double* P = jb.A[2] + (int64_t)p * rb * 256 + threadIdx.x;
  double acc = 0.0;
  for (int b = 0; b < rb; ++b) acc += P[(int64_t)b * 256] * P[(int64_t)b * 256];
  acc = sum_rows(acc);
  if (lane < 16) part[w][lane] = acc;
  __syncthreads();
  if (threadIdx.x < 16)
    jb.nrm[p * 16 + threadIdx.x] =
        sqrt(part[0][threadIdx.x] + part[1][threadIdx.x] + part[2][threadIdx.x] + part[3][threadIdx.x]);
}

// The kept vectors: 16 normalised columns of A2 a group, the block
// reflectors of the first factorisation applied to them from the last to the
// first in registers.
template <int NW, int TPW>
__global__ __launch_bounds__(NW * 64) void k_qj_back(const QjJob* __restrict__ jobs) {
  __shared__ double red[NW * 256], wl[256];
  const QrShared sh{red, wl, nullptr, nullptr, nullptr, nullptr};
  const QjJob& jb = jobs[blockIdx.y];
  const int k0 = blockIdx.x * 16;
  if (k0 >= jb.keep) return;
  const int rb = blocks16(jb.n), kb = blocks16(jb.K);
  const int w = wave_id(), lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int k = k0 + c;
  const int src = k < jb.keep ? jb.kcol[k] : -1;
  const double inv = k < jb.keep ? jb.kinv[k] : 0.0;
  const double* S = jb.A[2] + (int64_t)(max(src, 0) >> 4) * kb * 256 + (max(src, 0) & 15);
  double4_t a[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int b = w + NW * i;
#pragma unroll
    for (int r = 0; r < 4; ++r) a[i][r] = b < kb && src >= 0 ? inv * S[(int64_t)b * 256 + (4 * r + g) * 16] : 0.0;
  }
  const int m = 4 * (c & 3) + (c >> 2);
  for (int s = kb - 1; s >= 0; --s) {
    const double* V = jb.A[0] + (int64_t)s * rb * 256;
    const double* T = jb.T[0] + (int64_t)s * 256;
    // row blocks above s do not take part: their V is not stored
    double4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const int b = w + NW * i;
      const double z = b >= s && b < rb ? 1.0 : 0.0;
      const double* v = V + (int64_t)min(max(b, s), rb - 1) * 256 + lane;
#pragma unroll
      for (int r = 0; r < 4; ++r) acc = mfma(v[64 * r], z * a[i][r], acc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) red[w * 256 + 64 * r + lane] = acc[r];
    __syncthreads();
    if (threadIdx.x < 256) {
      double t = 0.0;
#pragma unroll
      for (int j = 0; j < NW; ++j) t += red[j * 256 + threadIdx.x];
      wl[threadIdx.x] = t;
    }
    __syncthreads();
    double4_t Y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int j = 0; j < 4; ++j) Y = mfma(T[m * 16 + 4 * j + g], wl[64 * j + lane], Y);
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const int b = w + NW * i;
      const double z = b >= s && b < rb ? -1.0 : 0.0;
      const double2_t* v = (const double2_t*)(V + (int64_t)min(max(b, s), rb - 1) * 256 + c * 16 + 4 * g);
      const double2_t v0 = v[0], v1 = v[1];
      a[i] = mfma(z * v0[0], Y[0], a[i]);
      a[i] = mfma(z * v0[1], Y[1], a[i]);
      a[i] = mfma(z * v1[0], Y[2], a[i]);
      a[i] = mfma(z * v1[1], Y[3], a[i]);
    }
  }
  if (k >= jb.keep) return;
#pragma unroll
  for (int i = 0; i < TPW; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * (w + NW * i) + 4 * r + g;
      if (row < jb.n) jb.out[row * jb.es + k * jb.vs] = a[i][r];
    }
}

// ------------------------------------------------------------------ host side
namespace {

// Rows of the tallest matrix a shape of the register-resident kernels takes.
template <int NW, int TPW>
constexpr int max_rows() {
  return 16 * NW * TPW;
}

void launch_qr_step(Context& c, const QjJob* dj, int rows, int which, int s, dim3 grid) {
  if (rows <= max_rows<8, 2>())
    hipLaunchKernelGGL((k_qj_qr<8, 2>), grid, dim3(512), 0, c.stream, dj, which, s);
  else if (rows <= max_rows<8, 4>())
    hipLaunchKernelGGL((k_qj_qr<8, 4>), grid, dim3(512), 0, c.stream, dj, which, s);
  else if (rows <= max_rows<16, 4>())
    hipLaunchKernelGGL((k_qj_qr<16, 4>), grid, dim3(1024), 0, c.stream, dj, which, s);
  else
    hipLaunchKernelGGL((k_qj_qr<16, 8>), grid, dim3(1024), 0, c.stream, dj, which, s);
}

void launch_back(Context& c, const QjJob* dj, int rows, dim3 grid) {
  if (rows <= max_rows<8, 2>())
    hipLaunchKernelGGL((k_qj_back<8, 2>), grid, dim3(512), 0, c.stream, dj);
  else if (rows <= max_rows<8, 4>())
    hipLaunchKernelGGL((k_qj_back<8, 4>), grid, dim3(512), 0, c.stream, dj);
  else if (rows <= max_rows<16, 4>())
    hipLaunchKernelGGL((k_qj_back<16, 4>), grid, dim3(1024), 0, c.stream, dj);
  else
    hipLaunchKernelGGL((k_qj_back<16, 8>), grid, dim3(1024), 0, c.stream, dj);
}

int up16(int n) { return (n + 15) / 16 * 16; }

}  // namespace

bool qj_fits(int64_t R, int64_t C) { return std::max(R, C) <= max_rows<16, 8>(); }

QjBatch::~QjBatch() {
  c.alloc.release(work);
  c.alloc.release(ints);
}

// Factorisations, Jacobi sweeps and column norms of all sectors; sigma and
// col of every sector receive the column norms (unscaled) in descending order
// and the column each belongs to.  Returns false when a sector did not
// converge within the sweep limit.
bool qj_solve(QjBatch& q, double norm2) {
  Context& c = q.c;
  std::vector<QjSector>& sec = q.sec;
  const int nj = (int)sec.size();
  // largest first: a launch's grid covers the jobs that still take part
  std::stable_sort(sec.begin(), sec.end(), [](const QjSector& a, const QjSector& b) { return a.o > b.o; });
  // powers of two, exact: norms of order one whatever the tensor's scale
  int ex = 0;
  (void)std::frexp(std::sqrt(norm2), &ex);
  const double scale = std::ldexp(1.0, -ex);
  // doubles: the norms of all sectors (one copy to the host), then the
  // matrices; ints: the round counters of all sectors, then the orders
  int64_t nd = 0, ni = nj, nn = 0;
  std::vector<int64_t> dof(nj), iof(nj), nof(nj);
  auto kcols = [](int K) { return (int64_t)std::max(up16(K), 32); };  // at least two panels
  for (int j = 0; j < nj; ++j) {
    const int64_t o = up16(sec[j].o), n = up16(sec[j].n), K = up16(sec[j].K), Kc = kcols(sec[j].K);
    nof[j] = nn;
    nn += o;
    dof[j] = nd;
    nd += n * o + o * Kc + K * Kc + 2 * 16 * K;
    iof[j] = ni;
    ni += o;
  }
  q.work = (double*)c.alloc.alloc((nn + nd) * sizeof(double));
  q.ints = (int*)c.alloc.alloc(ni * sizeof(int));
  launch_fill(c, q.work + nn, nd, 0.0);
  q.jobs.resize(nj);
  int maxo = 0, maxn = 0, maxK = 0;
  for (int j = 0; j < nj; ++j) {
    QjJob& b = q.jobs[j];
    const QjSector& s = sec[j];
    const int64_t o = up16(s.o), n = up16(s.n), K = up16(s.K), Kc = kcols(s.K);
    b = QjJob{};
    b.M = s.M;
    b.A[0] = q.work + nn + dof[j];
    b.A[1] = b.A[0] + n * o;
    b.A[2] = b.A[1] + o * Kc;
    b.T[0] = b.A[2] + K * Kc;
    b.T[1] = b.T[0] + 16 * K;
    b.nrm = q.work + nof[j];
    b.perm = q.ints + iof[j];
    b.last = q.ints + j;
    b.R = s.R;
    b.o = s.o;
    b.n = s.n;
    b.K = s.K;
    b.dir = s.dir;
    maxo = std::max(maxo, s.o);
    maxn = std::max(maxn, s.n);
    maxK = std::max(maxK, s.K);
  }
  auto* dj = (QjJob*)c.upload(q.jobs.data(), nj * sizeof(QjJob));
  const int pk = up16(maxK) / 16;
  hipLaunchKernelGGL(k_qj_norms0, dim3((maxo + 63) / 64, nj), dim3(256), 0, c.stream, dj);
  hipLaunchKernelGGL(k_qj_rank, dim3((maxo + 255) / 256, nj), dim3(256), 0, c.stream, dj);
  hipLaunchKernelGGL(k_qj_gather, dim3(up16(maxo) / 16, nj, std::min(16, up16(maxn) / 16)), dim3(256), 0, c.stream,
                     dj, scale);
  for (int which = 0; which < 2; ++which) {
    const int rows = which == 0 ? maxn : maxo;
    // slabs and panels of every job in this factorisation
    std::vector<int> slabs(nj), pans(nj);
    int np = 0;
    for (int j = 0; j < nj; ++j) {
      slabs[j] = up16(which == 0 ? sec[j].o : sec[j].K) / 16;
      pans[j] = std::min(up16(which == 0 ? sec[j].n : sec[j].o) / 16, slabs[j]);
      np = std::max(np, pans[j]);
    }
    for (int s = -1; s < np; ++s) {
      int gx = 0, gy = 0;
      for (int j = 0; j < nj; ++j)
        if (s < pans[j] && slabs[j] > s + 1) {
          gx = std::max(gx, s < 0 ? 1 : slabs[j] - s - 1);
          gy = j + 1;
        }
      if (gx > 0) launch_qr_step(c, dj, rows, which, s, dim3(gx, gy));
    }
  }
  HIP_OK(hipGetLastError());
  // Jacobi rounds, every sector on its own schedule; the state of all sectors
  // comes to the host after every half cycle of the largest while the next
  // half cycle is already queued
  const int nbmax = (std::max(2, pk) + 1) & ~1;
  const int chunk = nbmax / 2;
  const double tol = std::max(1e-14, 4.0 * 2.220446049250313e-16 * std::sqrt((double)maxK));
  const double fl = 1e-11;  // relative to |AA|, which the scaling puts in [1/2, 1)
  constexpr int kMaxSweeps = 40;
  int step = 0;
  bool done = false;
  int* hlast = (int*)c.host_sigma((nj + 1) / 2 + 1);
  auto rounds = [&]() {
    for (int k = 0; k < chunk; ++k, ++step)
      hipLaunchKernelGGL(k_qj_round, dim3(nbmax / 2, nj), dim3(512), 0, c.stream, dj, step, tol * tol, fl * fl);
  };
  for (int k = 0; k < 10 && step < 5 * (nbmax - 1); ++k) rounds();  // five sweeps are always needed
  while (!done && step < kMaxSweeps * (nbmax - 1)) {
    const int upto = step;
    HIP_OK(hipMemcpyAsync(hlast, q.ints, nj * sizeof(int), hipMemcpyDeviceToHost, c.stream));
    HIP_OK(hipEventRecord(c.poll, c.stream));
    rounds();
    HIP_OK(hipEventSynchronize(c.poll));
    done = true;
    for (int j = 0; j < nj; ++j) {
      const int nb = (std::max(2, up16(sec[j].K) / 16) + 1) & ~1;
      done = done && upto - 1 - hlast[j] >= nb - 1;
    }
  }
  HIP_OK(hipGetLastError());
  if (!done) return false;
  hipLaunchKernelGGL(k_qj_norms3, dim3(pk, nj), dim3(256), 0, c.stream, dj);
  double* h = c.host_sigma(nn);
  HIP_OK(hipMemcpyAsync(h, q.work, nn * sizeof(double), hipMemcpyDeviceToHost, c.stream));
  HIP_OK(hipStreamSynchronize(c.stream));
  for (int j = 0; j < nj; ++j) {
    QjSector& s = sec[j];
    const double* v = h + nof[j];
    s.col.resize(up16(s.K));
    for (int i = 0; i < (int)s.col.size(); ++i) s.col[i] = i;
    std::stable_sort(s.col.begin(), s.col.end(), [&](int a, int b) { return v[a] > v[b]; });
    s.col.resize(s.K);
    s.sigma.resize(s.K);
    s.inv.resize(s.K);
    for (int i = 0; i < s.K; ++i) {
      s.sigma[i] = v[s.col[i]] / scale;
      s.inv[i] = v[s.col[i]] > 0.0 ? 1.0 / v[s.col[i]] : 0.0;
    }
  }
  return true;
}

// The first `keep` vectors of every sector (keep, out, es, vs set by the
// caller) on the device.
void qj_vectors(QjBatch& q) {
  Context& c = q.c;
  UploadPack pk;
  const int nj = (int)q.sec.size();
  std::vector<size_t> oc(nj), oi(nj);
  int maxn = 0, maxkeep = 0;
  for (int j = 0; j < nj; ++j) {
    const QjSector& s = q.sec[j];
    oc[j] = pk.add(s.col.data(), s.keep * sizeof(int));
    oi[j] = pk.add(s.inv.data(), s.keep * sizeof(double));
    maxn = std::max(maxn, s.n);
    maxkeep = std::max(maxkeep, s.keep);
  }
  if (maxkeep == 0) return;
  char* base = pk.commit(c);
  for (int j = 0; j < nj; ++j) {
    const QjSector& s = q.sec[j];
    QjJob& b = q.jobs[j];
    b.kcol = (const int*)(base + oc[j]);
    b.kinv = (const double*)(base + oi[j]);
    b.out = s.out;
    b.es = s.es;
    b.vs = s.vs;
    b.keep = s.keep;
  }
  auto* dj = (QjJob*)c.upload(q.jobs.data(), nj * sizeof(QjJob));
  launch_back(c, dj, maxn, dim3((maxkeep + 15) / 16, nj));
  HIP_OK(hipGetLastError());
}

}  // namespace dmrj

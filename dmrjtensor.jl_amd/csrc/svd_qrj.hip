// Batched SVD of the larger charge sectors: QR-preconditioned block one-sided
// Jacobi on the FP64 matrix cores.
//
// The wanted orthonormal vectors of a sector M (R x C) are the left singular
// vectors of A0 = M (dir > 0: U) or A0 = M^T (dir < 0: V), an n x o matrix
// with K = min(n, o).  Two unpivoted Householder factorisations precede the
// Jacobi sweeps (the preconditioning of Drmac and Veselic, SIAM J. Matrix
// Anal. Appl. 29 (2008), with a column sort in place of the pivoting):
//   A0 P = Q0 R0, A1 = R0^H;  A1 = Q1 R1, A2 = R1^H
// (P orders the columns by decreasing norm).  Two-site tensors are graded on
// both sides, so every factorisation moves A_i closer to a diagonal matrix:
// on the 433 x 462 sector of an m=1024 Heisenberg state the sweeps fall from
// 20 (columns sorted, no factorisation) over 10 to 7, and the error of the
// singular values from 5e-14 to 1e-15 of the largest.  Jacobi sweeps then
// rotate the columns of A2 until they are orthogonal, A2 V = W D, so that
// R1 = V D W^H, A1 = Q1 V D W^H, R0 = W D (Q1 V)^H, and the vectors are
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
// 6.5 ms with this; m=2048 Hubbard (sectors to 1164): 134 and 28.6 ms.  A third
// factorisation (of A2) saves a sweep and costs its panels (7.3 against 7.1 ms,
// 30.7 against 31, 1.06 against 0.98 at a single 100 x 100 sector, when rounds
// were 5% slower).
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

// The value of lane J of every row of 16 lanes (DPP row_newbcast, one 64-bit
// move: a panel step 2% shorter than with two 32-bit ones).
template <int J>
__device__ __forceinline__ double row_bcast(double x) {
  const long long v = __builtin_bit_cast(long long, x);
  const long long r = __builtin_amdgcn_update_dpp(v, v, 0x150 + J, 0xf, 0xf, true);
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

// Generator of the Jacobi rotation from its cotangent of the double angle
// f >= 0 (1e-38 for the pairs of columns furthest apart: no overflow in f^2):
// the x for which the unitary polynomial of the round turns by the angle of the
// tangent t = 1 / (f + sqrt(f^2 + 1)), x = t - t^3 / 4 + ..., to 0.003 rad.
__device__ __forceinline__ float jacobi_generator(float f) {
  const float t = __builtin_amdgcn_rcpf(f + (f < 1e15f ? __builtin_amdgcn_sqrtf(fmaf(f, f, 1.0f)) : f));
  const float t2 = t * t;
  return t * (1.0f - t2 * (0.25f - 0.096f * t2));
}

// The wave's number in its work-group, in a scalar register.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

__device__ __forceinline__ int blocks16(int n) { return (n + 15) >> 4; }

constexpr int kGroup = 2;  // register tiles whose loads are in flight together

// Complex tensors (Z) hold every tile as a real and an imaginary 16 x 16
// plane, 512 doubles; their products are real products of the planes.
template <bool Z>
constexpr int kTile = Z ? 512 : 256;
template <bool Z>
struct Tile {  // a wave's registers of one tile (i: complex only)
  double4_t r, i;
};
constexpr double4_t kZero4 = {0.0, 0.0, 0.0, 0.0};

// acc += conj(a) b, acc += a b and acc -= a b, one MFMA step
template <bool Z>
__device__ __forceinline__ void mac_h(Tile<Z>& acc, double ar, double ai, double br, double bi) {
  acc.r = mfma(ar, br, acc.r);
  if constexpr (Z) {
    acc.r = mfma(ai, bi, acc.r);
    acc.i = mfma(ar, bi, acc.i);
    acc.i = mfma(-ai, br, acc.i);
  }
}
template <bool Z>
__device__ __forceinline__ void mac(Tile<Z>& acc, double ar, double ai, double br, double bi) {
  acc.r = mfma(ar, br, acc.r);
  if constexpr (Z) {
    acc.r = mfma(-ai, bi, acc.r);
    acc.i = mfma(ar, bi, acc.i);
    acc.i = mfma(ai, br, acc.i);
  }
}

struct QrShared {
  double* red;   // NW partial tiles
  double* w;     // a tile
  double* dots;  // 2 x NW x 16 (x 2 complex)
  double* piv;   // 2 x 16 (x 2)
  double* s;     // 256 (x 2): V^H V above the diagonal
  double* tau;   // 16 (x 2)
};

// W = V^H A over the register tiles of the work-group's slab (tiles of row
// blocks base + w + NW i, those from `first` on), summed over the waves; every
// lane returns its elements in the B operand layout.
template <bool Z, int NW, int TPW>
__device__ __forceinline__ Tile<Z> slab_vha(const double* V, int base, int first, int rb, const Tile<Z> (&a)[TPW],
                                            const QrShared& sh) {
  const int w = wave_id(), lane = threadIdx.x & 63;
  Tile<Z> acc = {kZero4, kZero4};
  // groups of tiles: the loads of a group are in flight together; tiles that
  // take no part are zeroed, so any tile of V will do for them
#pragma unroll
  for (int i0 = 0; i0 < TPW; i0 += kGroup)
    if (base + w + NW * i0 < rb && base + w + NW * (i0 + kGroup - 1) >= first) {
#pragma unroll
      for (int i = i0; i < i0 + kGroup; ++i) {
        const int b = base + w + NW * i;
        const double z = b >= first ? 1.0 : 0.0;  // (tiles past the end hold zeros)
        const double* v = V + (int64_t)min(max(b, first), rb - 1) * kTile<Z> + lane;
#pragma unroll
        for (int r = 0; r < 4; ++r) mac_h<Z>(acc, z * v[64 * r], Z ? z * v[256 + 64 * r] : 0.0, a[i].r[r], Z ? a[i].i[r] : 0.0);
      }
    }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    sh.red[w * kTile<Z> + 64 * r + lane] = acc.r[r];
    if constexpr (Z) sh.red[w * kTile<Z> + 256 + 64 * r + lane] = acc.i[r];
  }
  __syncthreads();
  if (threadIdx.x < kTile<Z>) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < NW; ++k) t += sh.red[k * kTile<Z> + threadIdx.x];
    sh.w[threadIdx.x] = t;
  }
  __syncthreads();
  Tile<Z> r = {kZero4, kZero4};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    r.r[k] = sh.w[64 * k + lane];
    if constexpr (Z) r.i[k] = sh.w[256 + 64 * k + lane];
  }
  return r;
}

// A -= V Y on the register tiles; Y's register s holds row 4 (l/16) + s of
// column l%16, the reduction index order of V's four consecutive elements.
template <bool Z, int NW, int TPW>
__device__ __forceinline__ void slab_sub(const double* V, int base, int first, int rb, Tile<Z> (&a)[TPW],
                                         const Tile<Z>& Y) {
  const int w = wave_id(), lane = threadIdx.x & 63;
#pragma unroll
  for (int i0 = 0; i0 < TPW; i0 += kGroup)
    if (base + w + NW * i0 < rb && base + w + NW * (i0 + kGroup - 1) >= first) {
#pragma unroll
      for (int i = i0; i < i0 + kGroup; ++i) {
        const int b = base + w + NW * i;
        const double z = b >= first && b < rb ? -1.0 : 0.0;  // other tiles stay as they are
        const double2_t* v = (const double2_t*)(V + (int64_t)min(max(b, first), rb - 1) * kTile<Z> +
                                                (lane & 15) * 16 + 4 * (lane >> 4));
        const double2_t v0 = v[0], v1 = v[1];
        double2_t u0 = {0.0, 0.0}, u1 = u0;
        if constexpr (Z) {
          u0 = v[128];
          u1 = v[129];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
          mac<Z>(a[i], z * (k < 2 ? v0[k & 1] : v1[k & 1]), z * (k < 2 ? u0[k & 1] : u1[k & 1]), Y.r[k],
                 Z ? Y.i[k] : 0.0);
      }
    }
}

// One column of a panel: Householder reflector of column J (pivot in row J of
// the pivot tile, tile 0 of the wave with `top`) and its application to the
// columns right of it.  One reduction gives the products of column J with all
// 16 columns: the norm, the update coefficients and the inner products of the
// reflectors that the triangular factor needs.
template <bool Z, int J, int NW, int TPW>
__device__ __forceinline__ void panel_column(Tile<Z> (&a)[TPW], int nt, bool top, const QrShared& sh) {
  constexpr int kP = Z ? 2 : 1;
  const int w = wave_id(), lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  double4_t dr = kZero4, di = kZero4;
#pragma unroll
  for (int i = 0; i < TPW; ++i)
    if (i < nt) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool out = i == 0 && top && 4 * r + g <= J;
        const double x = row_bcast<J>(a[i].r[r]);
        const double y = out ? 0.0 : a[i].r[r];
        dr[r] = fma(x, y, dr[r]);
        if constexpr (Z) {
          const double xi = row_bcast<J>(a[i].i[r]);
          const double yi = out ? 0.0 : a[i].i[r];
          dr[r] = fma(xi, yi, dr[r]);
          di[r] = fma(x, yi, di[r]);
          di[r] = fma(-xi, y, di[r]);
        }
      }
    }
  double* d = sh.dots + (J & 1) * NW * 16 * kP;
  double* pv = sh.piv + (J & 1) * 16 * kP;
  const double dot = sum_rows((dr[0] + dr[1]) + (dr[2] + dr[3]));
  if (g == 0) d[w * 16 + c] = dot;
  if (top && g == (J & 3)) pv[c] = a[0].r[J >> 2];
  if constexpr (Z) {
    const double dotz = sum_rows((di[0] + di[1]) + (di[2] + di[3]));
    if (g == 0) d[NW * 16 + w * 16 + c] = dotz;
    if (top && g == (J & 3)) pv[16 + c] = a[0].i[J >> 2];
  }
  __syncthreads();
  double part[4] = {0.0, 0.0, 0.0, 0.0}, partz[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    part[k & 3] += d[k * 16 + c];
    if constexpr (Z) partz[k & 3] += d[NW * 16 + k * 16 + c];
  }
  const double tot = (part[0] + part[1]) + (part[2] + part[3]);
  const double totz = (partz[0] + partz[1]) + (partz[2] + partz[3]);
  const double pr = pv[c], prz = Z ? pv[16 + c] : 0.0;
  const double xn = row_bcast<J>(tot), alpha = row_bcast<J>(pr);
  const double alphaz = Z ? row_bcast<J>(prz) : 0.0;
  double tau = 0.0, tauz = 0.0, beta = alpha, scale = 0.0, scalez = 0.0;
  const double xa = Z ? fma(alphaz, alphaz, xn) : xn;
  // a residual below 1e-145 of the sector's norm counts as zero (its elements are
  // dropped, coef = -1 below): squares near the subnormal range have too few
  // bits for a unitary reflector, and the reciprocals would overflow
  if (xa > 1e-290) {
    const double h = fma(alpha, alpha, xa);
    const double ri = copysign(fast_rsqrt(h), -alpha);  // 1 / beta
    beta = h * ri;
    tau = fma(-alpha, ri, 1.0);
    if constexpr (Z) {
      tauz = -alphaz * ri;
      const double u = alpha - beta, q = fast_rcp(fma(u, u, alphaz * alphaz));
      scale = u * q;
      scalez = -alphaz * q;
    } else {
      scale = fast_rcp(alpha - beta);
    }
  }
  // v_J^H column c (c < J: the column is v_c), and conj(tau) of it right of J
  double vc = fma(scale, tot, pr), vcz = 0.0;
  if constexpr (Z) {
    vc = fma(scalez, totz, vc);
    vcz = prz + scale * totz - scalez * tot;
  }
  double wc = tau * vc, wcz = 0.0;
  if constexpr (Z) {
    wc = fma(tauz, vcz, wc);
    wcz = tau * vcz - tauz * vc;
  }
  wc = c > J ? wc : 0.0;
  wcz = c > J ? wcz : 0.0;
  if (w == 0 && g == 0) {
    if (c < J) sh.s[c * 16 + J] = vc;
    if (c == J) sh.tau[J] = tau;
    if constexpr (Z) {
      if (c < J) sh.s[256 + c * 16 + J] = -vcz;
      if (c == J) sh.tau[16 + J] = tauz;
    }
  }
  // column J becomes the reflector, x + (scale - 1) x, the columns right of it
  // lose w_c scale x: one multiply-add with a coefficient per column.  The
  // broadcasts of the first pass are made again: held across the barrier they
  // would take as many registers as the tiles.
  const double coef = c == J ? scale - 1.0 : -(wc * scale - (Z ? wcz * scalez : 0.0));
  const double coefz = Z ? (c == J ? scalez : -(wc * scalez + wcz * scale)) : 0.0;
#pragma unroll
  for (int i = 0; i < TPW; ++i)
    if (i < nt) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * r + g;
        double x = a[i].r[r];
        asm volatile("" : "+v"(x));
        const double xj = row_bcast<J>(x);
        double y = fma(coef, xj, x);
        if constexpr (Z) {
          double z = a[i].i[r];
          asm volatile("" : "+v"(z));
          const double zj = row_bcast<J>(z);
          y = fma(-coefz, zj, y);
          const double yz = fma(coefz, xj, fma(coef, zj, z));
          if (i == 0 && top)
            a[i].i[r] = row > J ? yz : row == J ? (c == J ? 0.0 : z - wcz) : z;
          else
            a[i].i[r] = yz;
        }
        if (i == 0 && top)
          a[i].r[r] = row > J ? y : row == J ? (c == J ? beta : x - wc) : x;
        else
          a[i].r[r] = y;
      }
    }
}

template <bool Z, int J, int NW, int TPW>
__device__ __forceinline__ void panel_columns(Tile<Z> (&a)[TPW], int nt, bool top, const QrShared& sh) {
  if constexpr (J < 16) {
    panel_column<Z, J, NW, TPW>(a, nt, top, sh);
    panel_columns<Z, J + 1, NW, TPW>(a, nt, top, sh);
  }
}

}  // namespace

// One step of factorisation `which` (A[which] = Q R, A[which + 1] = R^H): the
// block reflector of panel s applied to the slabs right of it, and panel
// s + 1 factorised by its slab's group.  s = -1 factorises panel 0.
//
// A slab of 16 columns per work-group, its rows in registers (NW x TPW tiles
// of 16): read once, written once, V read from L2 twice (once per operand
// layout).  The step's length is that of the group that goes on to the
// panel: 16 columns of one reduction and one barrier each.
template <bool Z, int NW, int TPW>
__global__ __launch_bounds__(NW * 64) void k_qj_qr(const QjJob* __restrict__ jobs, int which, int s) {
  constexpr int kT = kTile<Z>, kP = Z ? 2 : 1;
  __shared__ double red[NW * kT], wl[kT], dots[2 * NW * 16 * kP], piv[32 * kP], sm[256 * kP], taul[16 * kP];
  const QrShared sh{red, wl, dots, piv, sm, taul};
  const QjJob& jb = jobs[blockIdx.y];
  const int rows = which == 0 ? jb.n : jb.o, cols = which == 0 ? jb.o : jb.K;
  const int rb = blocks16(rows), nb = blocks16(cols), np = min(rb, nb);
  const int t = s + 1 + blockIdx.x;
  if (s >= np || t >= nb) return;
  const int w = wave_id(), lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int base = max(s, 0);
  double* P = jb.A[which] + (int64_t)t * rb * kT;
  Tile<Z> a[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int b = base + w + NW * i;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      a[i].r[r] = b < rb ? P[(int64_t)b * kT + 64 * r + lane] : 0.0;
      if constexpr (Z) a[i].i[r] = b < rb ? P[(int64_t)b * kT + 256 + 64 * r + lane] : 0.0;
    }
  }
  double* An = jb.A[which + 1];
  const int rbn = nb;  // row blocks of the next matrix
  if (s >= 0) {
    const double* V = jb.A[which] + (int64_t)s * rb * kT;
    const double* T = jb.T[which] + (int64_t)s * kT;
    const Tile<Z> W = slab_vha<Z, NW, TPW>(V, base, base, rb, a, sh);
    // Y = T^H W, its rows ordered for slab_sub: row i = 4r + g of the product is row 4g + r of Y
    const int m = 4 * (c & 3) + (c >> 2);
    Tile<Z> Y = {kZero4, kZero4};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double* tk = T + (4 * k + g) * 16 + m;
      mac_h<Z>(Y, tk[0], Z ? tk[256] : 0.0, W.r[k], Z ? W.i[k] : 0.0);
    }
    slab_sub<Z, NW, TPW>(V, base, base, rb, a, Y);
    if (w == 0) {  // rows 16 s .. of R are final: conjugate-transposed into the next matrix
      double* q = An + ((int64_t)s * rbn + t) * kT + c * 16 + g;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        q[4 * r] = a[0].r[r];
        a[0].r[r] = 0.0;
        if constexpr (Z) {
          q[256 + 4 * r] = -a[0].i[r];
          a[0].i[r] = 0.0;
        }
      }
    }
  }
  const bool factor = t == s + 1 && t < np;
  const int pw = s >= 0 ? 1 : 0;  // wave of the pivot tile
  if (factor) {
    const bool top = w == pw;
    panel_columns<Z, 0, NW, TPW>(a, (rb - base - w + NW - 1) / NW, top, sh);
    if (top) {
      double* q = An + ((int64_t)t * rbn + t) * kT + c * 16 + g;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 4 * r + g;
        q[4 * r] = row <= c ? a[0].r[r] : 0.0;
        a[0].r[r] = row > c ? a[0].r[r] : row == c ? 1.0 : 0.0;
        if constexpr (Z) {
          q[256 + 4 * r] = row <= c ? -a[0].i[r] : 0.0;
          a[0].i[r] = row > c ? a[0].i[r] : 0.0;
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int b = base + w + NW * i;
    if (b < rb && !(s >= 0 && b == s)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        P[(int64_t)b * kT + 64 * r + lane] = a[i].r[r];
        if constexpr (Z) P[(int64_t)b * kT + 256 + 64 * r + lane] = a[i].i[r];
      }
    }
  }
  if (!factor) return;
  __syncthreads();
  // T = (diag(1/tau) + strictly upper V^H V)^-1, one column per lane
  if (w == 0 && g == 0) {
    double x[16], xz[16];
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      double acc[2] = {0.0, 0.0}, accz[2] = {0.0, 0.0};
#pragma unroll
      for (int k = i + 1; k < 16; ++k) {
        const double sr = sm[i * 16 + k];
        acc[k & 1] += sr * x[k];
        if constexpr (Z) {
          const double si = sm[256 + i * 16 + k];
          acc[k & 1] -= si * xz[k];
          accz[k & 1] += sr * xz[k] + si * x[k];
        }
      }
      const double sr = acc[0] + acc[1], si = accz[0] + accz[1];
      const double tr = taul[i], ti = Z ? taul[16 + i] : 0.0;
      x[i] = i == c ? tr : i < c ? -(tr * sr - ti * si) : 0.0;
      xz[i] = i == c ? ti : i < c ? -(tr * si + ti * sr) : 0.0;
    }
    double* T = jb.T[which] + (int64_t)t * kT;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      T[i * 16 + c] = x[i];
      if constexpr (Z) T[256 + i * 16 + c] = xz[i];
    }
  }
}

// Squared column norms of scale A0 (columns of M for dir > 0, rows for dir < 0): 16
// columns and 16 interleaved sequences of rows a group, which reads whole
// 128-byte lines in both directions (a wave a column or 64 columns a wave:
// 42 us at 400 x 400, 5 now).
template <bool Z>
__global__ __launch_bounds__(256) void k_qj_norms0(const QjJob* __restrict__ jobs, double scale) {
  __shared__ double part[256];
  const QjJob& jb = jobs[blockIdx.y];
  const int j0 = blockIdx.x * 16, lo = threadIdx.x & 15, hi = threadIdx.x >> 4;
  if (j0 >= jb.o) return;
  if (j0 == 0 && threadIdx.x == 0) *jb.last = -1;
  const int col = jb.dir > 0 ? hi : lo, i0 = jb.dir > 0 ? lo : hi, n = jb.n;
  const int64_t cs = jb.dir > 0 ? jb.R : 1, is = jb.dir > 0 ? 1 : jb.R;
  double acc = 0.0;
  if (j0 + col < jb.o) {
    const double* m = jb.M + (j0 + col) * cs;
    const int64_t plane = jb.plane;
#pragma unroll 8
    for (int i = i0; i < n; i += 16) {
      const double x = scale * m[i * is], y = Z ? scale * m[plane + i * is] : 0.0;
      acc += Z ? x * x + y * y : x * x;
    }
  }
  part[col * 16 + i0] = acc;
  __syncthreads();
  if (threadIdx.x < 16 && j0 + (int)threadIdx.x < jb.o) {
    double t = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += part[threadIdx.x * 16 + i];
    jb.nrm[j0 + threadIdx.x] = t;
  }
}

// perm[rank of column j] = j, norms descending, ties by index: 16 columns a
// group, a sixteenth of the comparisons a thread (a column a thread: 57 us at
// 1024 columns, 6 now).
__global__ __launch_bounds__(256) void k_qj_rank(const QjJob* __restrict__ jobs) {
  __shared__ int part[256];
  const QjJob& jb = jobs[blockIdx.y];
  const int lo = threadIdx.x & 15, hi = threadIdx.x >> 4, o = jb.o, j = blockIdx.x * 16 + lo;
  if ((int)blockIdx.x * 16 >= o) return;
  const double* nrm = jb.nrm;
  const double x = j < o ? nrm[j] : 0.0;
  int rank = 0;
#pragma unroll 8
  for (int k = hi; k < o; k += 16) {
    const double y = nrm[k];
    rank += (y > x) | ((y == x) & (k < j));
  }
  part[hi * 16 + lo] = rank;
  __syncthreads();
  if (hi == 0 && j < o) {
#pragma unroll
    for (int k = 1; k < 16; ++k) rank += part[k * 16 + lo];
    jb.perm[rank] = j;
  }
}

// Panels of A0: sorted columns, scaled, zero-padded.  `scale` brings the norm
// of the tensor to order one, the factor found here that of the sector: what
// the solver counts as zero is relative to the sector's own norm, so the values
// and vectors of a weak sector are as accurate as a strong one's (a factor for
// the whole tensor left sectors below 1e-11 of its norm unrotated).  The factor
// goes to the host behind the column norms.  Every group sums all norms itself;
// sectors below 1e-140 of the tensor's norm keep its factor.
template <bool Z>
__global__ __launch_bounds__(256) void k_qj_gather(const QjJob* __restrict__ jobs, double scale) {
  __shared__ double part[256], sums[16];
  const QjJob& jb = jobs[blockIdx.y];
  const int p = blockIdx.x;
  if (p >= blocks16(jb.o)) return;
  {
    double t = 0.0;
    for (int j = threadIdx.x; j < jb.o; j += 256) t += jb.nrm[j];
    part[threadIdx.x] = t;
    __syncthreads();
    if (threadIdx.x < 16) {
      t = 0.0;
#pragma unroll
      for (int i = 0; i < 16; ++i) t += part[threadIdx.x * 16 + i];
      sums[threadIdx.x] = t;
    }
    __syncthreads();
    t = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += sums[i];
    int ex = 0;
    if (t > 1e-280) (void)frexp(sqrt(t), &ex);
    const double factor = ldexp(1.0, -ex);
    if (p == 0 && blockIdx.z == 0 && threadIdx.x == 0) jb.nrm[16 * blocks16(jb.o)] = factor;
    scale *= factor;
  }
  const int rb = blocks16(jb.n), c = threadIdx.x & 15, rr = threadIdx.x >> 4;
  const int col = p * 16 + c < jb.o ? jb.perm[p * 16 + c] : -1;
  double* dst = jb.A[0] + (int64_t)p * rb * kTile<Z> + threadIdx.x;
  const int64_t cs = jb.dir > 0 ? jb.R : 1, is = jb.dir > 0 ? 1 : jb.R;
  for (int b = blockIdx.z; b < rb; b += gridDim.z) {
    const int i = b * 16 + rr;
    const bool in = col >= 0 && i < jb.n;
    const double* m = jb.M + col * cs + i * is;
    dst[(int64_t)b * kTile<Z>] = in ? scale * m[0] : 0.0;
    if constexpr (Z) dst[(int64_t)b * kTile<Z> + 256] = in ? scale * m[jb.plane] : 0.0;
  }
}

// One Jacobi round on A2: block pair k of the circle schedule per
// work-group.  Gram matrix of the 32 columns on the matrix cores, an
// approximate eigenbasis V of it in LDS, columns ordered by norm, and the
// product Y V on the matrix cores.  Pairs whose columns are orthogonal already
// (relative to tol; norms below `floor` count as `floor`) stop after the Gram
// matrix.  A sector stops when a whole cycle of its rounds rotated nothing.
template <bool Z>
__global__ __launch_bounds__(512) void k_qj_round(const QjJob* __restrict__ jobs, int step, double tol2,
                                                  double floor2) {
  // waves, row blocks in flight per wave, planes, leading dimension and size of a 32 x 32 matrix in LDS
  constexpr int kW = 8, kU = 2, kS = Z ? 1 : 2, kP = Z ? 2 : 1, kLd = 33, kM = 32 * kLd, kT = kTile<Z>;
  __shared__ double red[kW * 3 * kT];   // partial Gram tiles, then four matrices
  __shared__ double G[kP * kM];
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
  double* Yp = jb.A[2] + (int64_t)p * rb * kT;
  double* Yq = jb.A[2] + (int64_t)q * rb * kT;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
  {
    // real: the next row blocks are in flight while the current ones are multiplied
    Tile<Z> pp = {kZero4, kZero4}, pq = pp, qq = pp;
    double x[kS][kU][4 * kP], y[kS][kU][4 * kP];
    auto load = [&](int s, int b0) {
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int64_t o = (int64_t)min(b0 + u * kW, rb - 1) * kT + lane;
#pragma unroll
        for (int r = 0; r < 4 * kP; ++r) {
          x[s][u][r] = Yp[o + 64 * r];
          y[s][u][r] = Yq[o + 64 * r];
        }
      }
    };
    auto add = [&](int s, int b0) {
#pragma unroll
      for (int u = 0; u < kU; ++u)
        if (b0 + u * kW < rb) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const double xr = x[s][u][r], yr = y[s][u][r], xi = Z ? x[s][u][(4 + r) % (4 * kP)] : 0.0,
                         yi = Z ? y[s][u][(4 + r) % (4 * kP)] : 0.0;
            mac_h<Z>(pp, xr, xi, xr, xi);
            mac_h<Z>(pq, xr, xi, yr, yi);
            mac_h<Z>(qq, yr, yi, yr, yi);
          }
        }
    };
    load(0, w);
    for (int b0 = w; b0 < rb; b0 += kS * kU * kW) {
      if constexpr (kS == 2) {
        if (b0 + kU * kW < rb) load(1, b0 + kU * kW);
        add(0, b0);
        if (b0 + 2 * kU * kW < rb) load(0, b0 + 2 * kU * kW);
        add(kS - 1, b0 + kU * kW);
      } else {
        add(0, b0);
        if (b0 + kU * kW < rb) load(0, b0 + kU * kW);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double* d = red + w * 3 * kT + 64 * r + lane;
      d[0] = pp.r[r];
      d[kT] = pq.r[r];
      d[2 * kT] = qq.r[r];
      if constexpr (Z) {
        d[256] = pp.i[r];
        d[kT + 256] = pq.i[r];
        d[2 * kT + 256] = qq.i[r];
      }
    }
  }
  __syncthreads();
  for (int e = tid; e < 3 * kT; e += 512) {
    double t = 0.0;
    const int m = e / kT, im = Z ? (e >> 8) & 1 : 0, x = e & 255;
#pragma unroll
    for (int k = 0; k < kW; ++k) t += red[k * 3 * kT + e];
    const int i = (x >> 4) + (m == 2 ? 16 : 0), j = (x & 15) + (m >= 1 ? 16 : 0);
    G[im * kM + i * kLd + j] = t;
    if (m == 1) G[im * kM + j * kLd + i] = im ? -t : t;
  }
  __syncthreads();
  constexpr double eps2 = 2.220446049250313e-16 * 2.220446049250313e-16;
  int act = 0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int i = (tid >> 5) + 16 * h, j = tid & 31;
    const double gi = G[i * kLd + i], gj = G[j * kLd + j], x = G[i * kLd + j], y = Z ? G[(kP - 1) * kM + i * kLd + j] : 0.0;
    act |= i < j && x * x + y * y > tol2 * fmax(gi, gj) * fmax(fmin(gi, gj), floor2);
  }
  if (!__syncthreads_or(act)) return;
  if (tid == 0) *jb.last = step;
  // rows for the final product, the first block's fetched before the inner
  // solve and each next one's while the current is multiplied
  double2_t rows[2][4 * kP];
  auto fetch = [&](int s, int b) {
    const int64_t o = (int64_t)b * kT + c * 16 + 4 * g;
#pragma unroll
    for (int h = 0; h < kP; ++h) {
      rows[s][4 * h + 0] = *(const double2_t*)(Yp + o + 256 * h);
      rows[s][4 * h + 1] = *(const double2_t*)(Yp + o + 256 * h + 2);
      rows[s][4 * h + 2] = *(const double2_t*)(Yq + o + 256 * h);
      rows[s][4 * h + 3] = *(const double2_t*)(Yq + o + 256 * h + 2);
    }
  };
  fetch(0, min(w, rb - 1));
  // Inner solve, all pairs at once: X holds the Jacobi rotations of every pair
  // as a skew matrix (scaled down where a column of X exceeds kCap in the
  // 2-norm), V a unitary matrix near I + X, from a polynomial and
  // Newton-Schulz steps V += V (I - V^H V) / 2 on the matrix cores, repeated on
  // V^H G V while the rotations were large.  Its off-diagonal rest is of second
  // order, as after a cyclic sweep of rotations, at a fraction of the latency:
  // a sweep is 31 dependent rounds of LDS traffic, 46000 cycles, this 9000 on
  // average (20000 where the rotations are large), and one outer sweep fewer on
  // the sectors of an m=1024 Heisenberg state.  (A cosine applied to a
  // column would also scale it by its rounding error, and those factors add up
  // over the rounds: 3e-14 of the singular values of a 200 x 200 Gaussian
  // matrix, against 1.5e-15.)
  // The rest of an average round at 400 columns: 9200 cycles the Gram tiles,
  // 2000 their sum, 11100 the product, for 5400 and 7200 of FP64 MFMA time of
  // the CU's busiest SIMD; their loads are therefore in flight ahead.  Bond
  // steps with this and the polynomial against neither: 200 x 400 dense 4.23 to
  // 4.05 ms, m=510 Hubbard 2.90 to 2.70, m=2048 Hubbard 30.6 to 28.6.  Slicing
  // the rows of a pair over several work-groups (partial Gram tiles in a launch
  // of their own) was no faster at any size.
  constexpr double kCap = 0.85, kSmall = 0.25;
  constexpr int kRepeats = 2, kNewton = 12;
  double* V = red;             // this repeat's factor
  double* Vt = V + kP * kM;    // the products so far
  double* Tm = Vt + kP * kM;   // scratch
  double* E = Tm + kP * kM;    // (I - V^H V) / 2
  const int ti = (w >> 1) & 1, tj = w & 1;  // waves 0..3: a 16 x 16 tile each
  const bool mine = w < 4;
  auto mul = [&](const double* A, bool tA, const double* B, Tile<Z> acc) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int kk = 4 * k + g;
      const double* a = tA ? A + kk * kLd + 16 * ti + c : A + (16 * ti + c) * kLd + kk;
      const double* b = B + kk * kLd + 16 * tj + c;
      if (tA)
        mac_h<Z>(acc, a[0], Z ? a[(kP - 1) * kM] : 0.0, b[0], Z ? b[(kP - 1) * kM] : 0.0);
      else
        mac<Z>(acc, a[0], Z ? a[(kP - 1) * kM] : 0.0, b[0], Z ? b[(kP - 1) * kM] : 0.0);
    }
    return acc;
  };
  auto get = [&](const double* D) {
    Tile<Z> v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      v.r[r] = D[(16 * ti + 4 * r + g) * kLd + 16 * tj + c];
      v.i[r] = Z ? D[(kP - 1) * kM + (16 * ti + 4 * r + g) * kLd + 16 * tj + c] : 0.0;
    }
    return v;
  };
  auto put = [&](double* D, const Tile<Z>& v) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      D[(16 * ti + 4 * r + g) * kLd + 16 * tj + c] = v.r[r];
      if constexpr (Z) D[kM + (16 * ti + 4 * r + g) * kLd + 16 * tj + c] = v.i[r];
    }
  };
  const Tile<Z> zero = {kZero4, kZero4};
  double cap = kCap;
  for (int it = 0; it < kRepeats;) {
    // tangents in single precision (any nearby V serves), and the order of the
    // columns by norm: the comparisons of a row are one ballot
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int i = (tid >> 5) + 16 * h, j = tid & 31;
      const double gi = G[i * kLd + i], gj = G[j * kLd + j], x = G[i * kLd + j], d = gj - gi;
      if constexpr (Z) {
        const double y = G[kM + i * kLd + j], q2 = x * x + y * y;
        const bool go = i != j && q2 > fmax(eps2 * gi * gj, 1e-280);
        const double ri = fast_rsqrt(go ? q2 : 1.0);   // 1 / |g_ij|
        const float f = (float)(0.5 * d * ri);
        const bool neg = f < 0.0f || (f == 0.0f && i > j);
        const double t = go ? (double)jacobi_generator(fabsf(f)) * ri : 0.0;
        V[i * kLd + j] = i == j ? 1.0 : neg ? -t * x : t * x;
        V[kM + i * kLd + j] = i == j ? 0.0 : neg ? -t * y : t * y;
      } else {
        const bool go = i != j && x * x > fmax(eps2 * gi * gj, 1e-280);
        const float f = (float)(d * __builtin_amdgcn_rcp(go ? 2.0 * x : 1.0));
        const bool neg = f < 0.0f || (f == 0.0f && (i > j) != (x < 0.0));
        const float t = jacobi_generator(fabsf(f));
        V[i * kLd + j] = i == j ? 1.0 : go ? (double)(neg ? -t : t) : 0.0;
      }
      const unsigned long long m = __ballot(gj > gi || (gj == gi && j < i));
      if (j == 0) order[__popc((unsigned)(lane < 32 ? m : m >> 32))] = i;
    }
    __syncthreads();
    // X is skew, S = V^H V - I = X^H X = -X^2, and
    //   (I - S/2 + S^2/8) + X (I - S/4 + S^2/32)
    // is unitary up to S^5 / 1024 (the coefficients cancel S to S^4), so few
    // Newton-Schulz steps are left where |X|_2 is near one
    Tile<Z> v = zero, e = zero;
    if (mine) {
      e = mul(V, true, V, zero);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (ti == tj && 4 * r + g == c) {
          e.r[r] -= 1.0;
          cn[16 * ti + c] = e.r[r];  // squared norms of the columns of X
        }
      put(E, e);
    }
    __syncthreads();
    double mx = 0.0;
#pragma unroll
    for (int k = 0; k < 32; ++k) mx = fmax(mx, cn[k]);
    const bool large = mx > kSmall * kSmall;
    const double a2 = mx > cap * cap ? cap * cap / mx : 1.0, a1 = sqrt(a2);
    if (mine) {
      const Tile<Z> q = mul(E, true, E, zero);
      Tile<Z> d;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double one = ti == tj && 4 * r + g == c ? 1.0 : 0.0;
        d.r[r] = one - a2 * (0.25 * e.r[r] - 0.03125 * a2 * q.r[r]);
        v.r[r] = one - a2 * (0.5 * e.r[r] - 0.125 * a2 * q.r[r]) - a1 * d.r[r];
        if constexpr (Z) {
          d.i[r] = -a2 * (0.25 * e.i[r] - 0.03125 * a2 * q.i[r]);
          v.i[r] = -a2 * (0.5 * e.i[r] - 0.125 * a2 * q.i[r]) - a1 * d.i[r];
        }
        d.r[r] *= a1;
        d.i[r] *= a1;
      }
      put(Tm, d);
    }
    __syncthreads();
    if (mine) v = mul(V, false, Tm, v);  // V = I + X, the surplus D is in v already
    __syncthreads();
    if (mine) put(V, v);
    __syncthreads();
    // Newton-Schulz steps as many as |X|_2^2 = 2 mx asks for, the last one
    // checked: the deviation it found is squared by its update
    double dev = fmin(2.0 * a2 * mx, 1.0);
    dev = dev * dev * dev * dev * dev * (1.0 / 1024);
    bool conv = dev < 1e-17;
    for (int nt = 0; nt < kNewton && !conv; ++nt) {
      int big = 0;
      if (mine) {
        e = mul(V, true, V, zero);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          e.r[r] = (ti == tj && 4 * r + g == c ? 0.5 : 0.0) - 0.5 * e.r[r];
          big |= !(fabs(e.r[r]) <= 5e-9);  // (not a number after a divergence)
          if constexpr (Z) {
            e.i[r] *= -0.5;
            big |= !(fabs(e.i[r]) <= 5e-9);
          }
        }
        put(E, e);
      }
      if (dev < 1e-8)
        conv = !__syncthreads_or(big);
      else
        __syncthreads();
      dev *= 0.75 * dev;
      if (mine) v = mul(V, false, E, get(V));
      __syncthreads();
      if (mine) put(V, v);
      __syncthreads();
    }
    if (!conv) {
      // |X|_2 above 2.1, where the steps do not converge (32 columns of nearly
      // equal norms and products): at a quarter of the cap |X|_2 <= 1.2
      if (cap < kCap) return;
      cap *= 0.25;
      continue;
    }
    if (it > 0) {
      if (mine) v = mul(Vt, false, V, zero);
      __syncthreads();
      if (mine) put(Vt, v);
    } else if (mine) {
      put(Vt, get(V));
    }
    if (!large || ++it == kRepeats) break;
    if (mine) put(Tm, mul(G, false, V, zero));
    __syncthreads();
    if (mine) put(G, mul(V, true, Tm, zero));
    __syncthreads();
  }
  __syncthreads();
  double vb[2][8], vi[2][8];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int e = ((k >> 2) * 16 + 4 * g + (k & 3)) * kLd + order[16 * h + c];
      vb[h][k] = Vt[e];
      vi[h][k] = Z ? Vt[(kP - 1) * kM + e] : 0.0;
    }
  auto turn = [&](int s, int b) {
    Tile<Z> yp = zero, yq = zero;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const double xr = rows[s][k >> 1][k & 1], xi = Z ? rows[s][4 * (kP - 1) + (k >> 1)][k & 1] : 0.0;
      mac<Z>(yp, xr, xi, vb[0][k], vi[0][k]);
      mac<Z>(yq, xr, xi, vb[1][k], vi[1][k]);
    }
    const int64_t o = (int64_t)b * kT + lane;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      Yp[o + 64 * r] = yp.r[r];
      Yq[o + 64 * r] = yq.r[r];
      if constexpr (Z) {
        Yp[o + 256 + 64 * r] = yp.i[r];
        Yq[o + 256 + 64 * r] = yq.i[r];
      }
    }
  };
  for (int b = w; b < rb; b += 2 * kW) {
    if (b + kW < rb) fetch(1, b + kW);
    turn(0, b);
    if (b + 2 * kW < rb) fetch(0, b + 2 * kW);
    if (b + kW < rb) turn(1, b + kW);
  }
}

// Column norms of A2: one panel a group, 16 per panel in nrm.
template <bool Z>
__global__ __launch_bounds__(256) void k_qj_norms2(const QjJob* __restrict__ jobs) {
  __shared__ double part[4][16];
  const QjJob& jb = jobs[blockIdx.y];
  const int rb = blocks16(jb.K), p = blockIdx.x;
  if (p >= rb) return;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const double* P = jb.A[2] + (int64_t)p * rb * kTile<Z> + threadIdx.x;
  double acc = 0.0;
  for (int b = 0; b < rb * (Z ? 2 : 1); ++b) acc += P[(int64_t)b * 256] * P[(int64_t)b * 256];
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
template <bool Z, int NW, int TPW>
__global__ __launch_bounds__(NW * 64) void k_qj_back(const QjJob* __restrict__ jobs) {
  constexpr int kT = kTile<Z>;
  __shared__ double red[NW * kT], wl[kT];
  const QrShared sh{red, wl, nullptr, nullptr, nullptr, nullptr};
  const QjJob& jb = jobs[blockIdx.y];
  const int k0 = blockIdx.x * 16;
  if (k0 >= jb.keep) return;
  const int rb = blocks16(jb.n), kb = blocks16(jb.K);
  const int w = wave_id(), lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int k = k0 + c;
  const int src = k < jb.keep ? jb.kcol[k] : -1;
  const double inv = k < jb.keep ? jb.kinv[k] : 0.0;
  const double* S = jb.A[2] + (int64_t)(max(src, 0) >> 4) * kb * kT + (max(src, 0) & 15);
  Tile<Z> a[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int b = w + NW * i;
    const bool in = b < kb && src >= 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      a[i].r[r] = in ? inv * S[(int64_t)b * kT + (4 * r + g) * 16] : 0.0;
      if constexpr (Z) a[i].i[r] = in ? inv * S[(int64_t)b * kT + 256 + (4 * r + g) * 16] : 0.0;
    }
  }
  const int m = 4 * (c & 3) + (c >> 2);
  for (int s = kb - 1; s >= 0; --s) {
    const double* V = jb.A[0] + (int64_t)s * rb * kT;
    const double* T = jb.T[0] + (int64_t)s * kT + m * 16 + g;
    // row blocks above s do not take part: their V is not stored
    const Tile<Z> W = slab_vha<Z, NW, TPW>(V, 0, s, rb, a, sh);
    Tile<Z> Y = {kZero4, kZero4};
#pragma unroll
    for (int j = 0; j < 4; ++j) mac<Z>(Y, T[4 * j], Z ? T[256 + 4 * j] : 0.0, W.r[j], Z ? W.i[j] : 0.0);
    slab_sub<Z, NW, TPW>(V, 0, s, rb, a, Y);
  }
  if (k >= jb.keep) return;
#pragma unroll
  for (int i = 0; i < TPW; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * (w + NW * i) + 4 * r + g;
      if (row < jb.n) {
        jb.out[row * jb.es + k * jb.vs] = a[i].r[r];
        if constexpr (Z) jb.out[jb.oplane + row * jb.es + k * jb.vs] = a[i].i[r];
      }
    }
}

// ------------------------------------------------------------------ host side
namespace {

// Rows of the tallest matrix a shape of the register-resident kernels takes.
template <int NW, int TPW>
constexpr int max_rows() {
  return 16 * NW * TPW;
}

template <bool Z>
void launch_qr_step(Context& c, const QjJob* dj, int rows, int which, int s, dim3 grid) {
  if (rows <= max_rows<8, 2>())
    hipLaunchKernelGGL((k_qj_qr<Z, 8, 2>), grid, dim3(512), 0, c.stream, dj, which, s);
  else if (rows <= max_rows<8, 4>())
    hipLaunchKernelGGL((k_qj_qr<Z, 8, 4>), grid, dim3(512), 0, c.stream, dj, which, s);
  else if constexpr (Z)
    hipLaunchKernelGGL((k_qj_qr<true, 8, 8>), grid, dim3(512), 0, c.stream, dj, which, s);
  else if (rows <= max_rows<16, 4>())
    hipLaunchKernelGGL((k_qj_qr<false, 16, 4>), grid, dim3(1024), 0, c.stream, dj, which, s);
  else
    hipLaunchKernelGGL((k_qj_qr<false, 16, 8>), grid, dim3(1024), 0, c.stream, dj, which, s);
}

template <bool Z>
void launch_back(Context& c, const QjJob* dj, int rows, dim3 grid) {
  if (rows <= max_rows<8, 2>())
    hipLaunchKernelGGL((k_qj_back<Z, 8, 2>), grid, dim3(512), 0, c.stream, dj);
  else if (rows <= max_rows<8, 4>())
    hipLaunchKernelGGL((k_qj_back<Z, 8, 4>), grid, dim3(512), 0, c.stream, dj);
  else if constexpr (Z)
    hipLaunchKernelGGL((k_qj_back<true, 8, 8>), grid, dim3(512), 0, c.stream, dj);
  else if (rows <= max_rows<16, 4>())
    hipLaunchKernelGGL((k_qj_back<false, 16, 4>), grid, dim3(1024), 0, c.stream, dj);
  else
    hipLaunchKernelGGL((k_qj_back<false, 16, 8>), grid, dim3(1024), 0, c.stream, dj);
}

int up16(int n) { return (n + 15) / 16 * 16; }

}  // namespace

bool qj_fits(int64_t R, int64_t C, bool cplx) {
  return std::max(R, C) <= (cplx ? max_rows<8, 8>() : max_rows<16, 8>());
}

QjBatch::~QjBatch() {
  c.alloc.release(work);
  c.alloc.release(ints);
}

// Orders the sectors, allocates and stages the job table.
void qj_prepare(QjBatch& q) {
  if (q.sec.empty()) return;
  Context& c = q.c;
  std::vector<QjSector>& sec = q.sec;
  const int nj = (int)sec.size();
  // largest first: a launch's grid covers the jobs that still take part
  std::stable_sort(sec.begin(), sec.end(), [](const QjSector& a, const QjSector& b) { return a.o > b.o; });
  // doubles: the norms and the factor of all sectors (one copy to the host), then the
  // matrices; ints: the round counters of all sectors, then the orders
  const bool z = q.cplx;
  const int zf = z ? 2 : 1;
  int64_t nd = 0, ni = nj, nn = 0;
  std::vector<int64_t> dof(nj), iof(nj), nof(nj);
  auto kcols = [](int K) { return (int64_t)std::max(up16(K), 32); };  // at least two panels
  for (int j = 0; j < nj; ++j) {
    const int64_t o = up16(sec[j].o), n = up16(sec[j].n), K = up16(sec[j].K), Kc = kcols(sec[j].K);
    nof[j] = nn;
    nn += o + 16;
    dof[j] = nd;
    nd += zf * (n * o + o * Kc + K * Kc + 2 * 16 * K);
    iof[j] = ni;
    ni += o;
  }
  q.work = (double*)c.alloc.alloc((nn + nd) * sizeof(double));
  q.ints = (int*)c.alloc.alloc(ni * sizeof(int));
  q.nn = nn;
  q.nd = nd;
  q.jobs.resize(nj);
  for (int j = 0; j < nj; ++j) {
    QjJob& b = q.jobs[j];
    const QjSector& s = sec[j];
    const int64_t o = up16(s.o), n = up16(s.n), K = up16(s.K), Kc = kcols(s.K);
    b = QjJob{};
    b.M = s.M;
    b.A[0] = q.work + nn + dof[j];
    b.A[1] = b.A[0] + zf * n * o;
    b.A[2] = b.A[1] + zf * o * Kc;
    b.T[0] = b.A[2] + zf * K * Kc;
    b.T[1] = b.T[0] + zf * 16 * K;
    b.plane = z ? (int64_t)s.n * s.o : 0;
    b.nrm = q.work + nof[j];
    b.perm = q.ints + iof[j];
    b.last = q.ints + j;
    b.R = s.R;
    b.o = s.o;
    b.n = s.n;
    b.K = s.K;
    b.dir = s.dir;
  }
  q.dj = (QjJob*)c.stage_put(q.jobs.data(), nj * sizeof(QjJob));
}

// Factorisations, Jacobi sweeps and column norms of all sectors; sigma and
// col of every sector that converged within the sweep limit (ok) receive the
// column norms (unscaled) in descending order and the column each belongs to.
void qj_solve(QjBatch& q, double norm2) {
  Context& c = q.c;
  std::vector<QjSector>& sec = q.sec;
  const int nj = (int)sec.size();
  // powers of two, exact: norms of order one whatever the tensor's scale (k_qj_gather adds the sector's)
  int ex = 0;
  (void)std::frexp(std::sqrt(norm2), &ex);
  const double scale = std::ldexp(1.0, -ex);
  const bool z = q.cplx;
  const int64_t nn = q.nn;
  int maxo = 0, maxn = 0, maxK = 0;
  for (const QjSector& s : sec) {
    maxo = std::max(maxo, s.o);
    maxn = std::max(maxn, s.n);
    maxK = std::max(maxK, s.K);
  }
  QjJob* dj = q.dj;
  c.stage_flush();
  launch_fill(c, q.work + nn, q.nd, 0.0);
  const int pk = up16(maxK) / 16;
  const dim3 go((maxo + 15) / 16, nj);
  if (z)
    hipLaunchKernelGGL(k_qj_norms0<true>, go, dim3(256), 0, c.stream, dj, scale);
  else
    hipLaunchKernelGGL(k_qj_norms0<false>, go, dim3(256), 0, c.stream, dj, scale);
  hipLaunchKernelGGL(k_qj_rank, go, dim3(256), 0, c.stream, dj);
  const dim3 gg(up16(maxo) / 16, nj, std::min(16, up16(maxn) / 16));
  if (z)
    hipLaunchKernelGGL(k_qj_gather<true>, gg, dim3(256), 0, c.stream, dj, scale);
  else
    hipLaunchKernelGGL(k_qj_gather<false>, gg, dim3(256), 0, c.stream, dj, scale);
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
      if (gx > 0 && z)
        launch_qr_step<true>(c, dj, rows, which, s, dim3(gx, gy));
      else if (gx > 0)
        launch_qr_step<false>(c, dj, rows, which, s, dim3(gx, gy));
    }
  }
  HIP_OK(hipGetLastError());
  // Jacobi rounds, every sector on its own schedule; the state of all sectors
  // comes to the host after every half cycle of the largest while the next
  // half cycle is already queued
  const int nbmax = (std::max(2, pk) + 1) & ~1;
  const int chunk = nbmax / 2;
  const double tol = std::max(1e-14, 4.0 * 2.220446049250313e-16 * std::sqrt((double)maxK));
  const double fl = 1e-11;  // relative to the sector's norm, which the scaling puts in [1/2, 1)
  const int limit = c.jacobi_sweeps * (nbmax - 1);
  int step = 0;
  bool done = false;
  int* hlast = (int*)c.host_sigma((nj + 1) / 2 + 1);
  auto rounds = [&]() {
    for (int k = 0; k < chunk; ++k, ++step)
      if (z)
        hipLaunchKernelGGL(k_qj_round<true>, dim3(nbmax / 2, nj), dim3(512), 0, c.stream, dj, step, tol * tol, fl * fl);
      else
        hipLaunchKernelGGL(k_qj_round<false>, dim3(nbmax / 2, nj), dim3(512), 0, c.stream, dj, step, tol * tol, fl * fl);
  };
  while (step < std::min(limit, 5 * (nbmax - 1))) rounds();  // five sweeps are always needed
  for (bool more = true; more && !done;) {
    const int upto = step;
    HIP_OK(hipMemcpyAsync(hlast, q.ints, nj * sizeof(int), hipMemcpyDeviceToHost, c.stream));
    HIP_OK(hipEventRecord(c.poll, c.stream));
    more = step < limit;
    if (more) rounds();
    HIP_OK(hipEventSynchronize(c.poll));
    done = true;
    for (int j = 0; j < nj; ++j) {
      const int nb = (std::max(2, up16(sec[j].K) / 16) + 1) & ~1;
      sec[j].ok = upto - 1 - hlast[j] >= nb - 1;
      done = done && sec[j].ok;
    }
  }
  HIP_OK(hipGetLastError());
  if (z)
    hipLaunchKernelGGL(k_qj_norms2<true>, dim3(pk, nj), dim3(256), 0, c.stream, dj);
  else
    hipLaunchKernelGGL(k_qj_norms2<false>, dim3(pk, nj), dim3(256), 0, c.stream, dj);
  double* h = c.host_sigma(nn);
  HIP_OK(hipMemcpyAsync(h, q.work, nn * sizeof(double), hipMemcpyDeviceToHost, c.stream));
  HIP_OK(hipStreamSynchronize(c.stream));
  for (int j = 0; j < nj; ++j) {
    QjSector& s = sec[j];
    const double* v = h + (q.jobs[j].nrm - q.work);
    const double factor = v[up16(s.o)];
    for (int i = 0; i < up16(s.K); ++i) s.ok = s.ok && std::isfinite(v[i]);
    if (!s.ok) continue;
    s.col.resize(up16(s.K));
    for (int i = 0; i < (int)s.col.size(); ++i) s.col[i] = i;
    std::stable_sort(s.col.begin(), s.col.end(), [&](int a, int b) { return v[a] > v[b]; });
    s.col.resize(s.K);
    s.sigma.resize(s.K);
    s.inv.resize(s.K);
    for (int i = 0; i < s.K; ++i) {
      s.sigma[i] = v[s.col[i]] / factor / scale;
      s.inv[i] = v[s.col[i]] > 0.0 ? 1.0 / v[s.col[i]] : 0.0;
    }
  }
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
    b.oplane = s.oplane;
  }
  auto* dj = (QjJob*)c.stage_put(q.jobs.data(), nj * sizeof(QjJob));
  c.stage_flush();
  if (q.cplx)
    launch_back<true>(c, dj, maxn, dim3((maxkeep + 15) / 16, nj));
  else
    launch_back<false>(c, dj, maxn, dim3((maxkeep + 15) / 16, nj));
  HIP_OK(hipGetLastError());
}

}  // namespace dmrj

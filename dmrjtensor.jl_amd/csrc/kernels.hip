// Device kernels of libdmrjhip (gfx950 / CDNA4).
//
//  * k_gemm_f64<BM,BN>: persistent grouped GEMM over a flat tile list.  Every
//    task is C = beta*C + sum over K-segments of alpha*op(A)*op(B) with its own
//    pointers, leading dimensions and transpose flags, so one launch covers all
//    symmetry blocks of one contraction step.  FP64 MFMA
//    v_mfma_f64_16x16x4f64, 256 threads = 4 waves in a 2x2 arrangement, LDS
//    double buffer with register prefetch (one barrier per K step).
//  * k_mix: small dense "label" contraction with the MPO coefficients
//    (HBM-bound weighted sums of equally shaped blocks).
//  * k_copy: batched strided block copy with optional row/column scaling
//    (SVD sector gather and split).
//  * deterministic two-pass dot products and the scalar steps of the
//    two-vector Lanczos, all reading and writing device scalars so that a
//    Lanczos application needs no host round trip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "internal.h"

namespace dmrj {

typedef double double4_t __attribute__((ext_vector_type(4)));

#define HIP_OK(x)                                                                    \
  do {                                                                               \
    hipError_t e_ = (x);                                                             \
    if (e_ != hipSuccess) throw Error(-3, std::string("HIP: ") + hipGetErrorString(e_)); \
  } while (0)

constexpr int kThreads = 256;
constexpr int kBK = 16;
// LDS tiles are stored [row][k] with a pitch of kBK+1 doubles (34 banks): the
// 16 lanes of an MFMA operand read (consecutive rows, same k) and the 16-lane
// groups of the stores (consecutive k of one row, or consecutive rows of one k)
// each touch 16 distinct bank pairs.
constexpr int kPitch = kBK + 1;

// The 32x32 shape is held to 64 registers per lane (eight waves per SIMD,
// eight work-groups per CU as its LDS allows) without scratch; the larger
// shapes keep the compiler's allocation.
template <int BM, int BN>
__global__ __launch_bounds__(kThreads, (BM * BN <= 1024 ? 8 : 1)) void k_gemm_f64(const GemmTile* __restrict__ tiles,
                                                       int ntiles,
                                                       const GemmTask* __restrict__ tasks,
                                                       const GemmSeg* __restrict__ segs) {
  constexpr int WM = BM / 2, WN = BN / 2, FM = WM / 16, FN = WN / 16;
  constexpr int AE = BM * kBK / kThreads, BE = BN * kBK / kThreads;
  __shared__ double sA[2][BM * kPitch];
  __shared__ double sB[2][BN * kPitch];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int lr = lane & 15, lk = lane >> 4;
  int buf = 0;

  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const GemmTile tl = tiles[t];
    const GemmTask tk = tasks[tl.task];
    const int m0 = tl.m0, n0 = tl.n0;
    double4_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = double4_t{0.0, 0.0, 0.0, 0.0};

    for (int sidx = 0; sidx < tk.nseg; ++sidx) {
      const GemmSeg sg = segs[tk.seg0 + sidx];
      const bool tA = sg.flags & 1, tB = sg.flags & 2;
      const int K = sg.K;
      double ra[AE], rb[BE];
      // Per-thread element offsets of the first K step (k0 = 0); a K step adds
      // k0 * (stride along k).  A row (column) outside the task reads the
      // task's first row (column) instead and is written to LDS as zero, so
      // a K step that lies wholly inside K loads without per-element checks.
      const int64_t ska = tA ? 1 : sg.lda, skb = tB ? sg.ldb : 1;
      int64_t oa[AE], ob[BE];
      int ka[AE], kb[BE];
      bool va[AE], vb[BE];
#pragma unroll
      for (int r = 0; r < AE; ++r) {
        const int idx = tid + r * kThreads;
        int m, k;
        if (!tA) { m = idx % BM; k = idx / BM; } else { k = idx % kBK; m = idx / kBK; }
        va[r] = m0 + m < tk.M;
        const int gm = va[r] ? m0 + m : m0;
        ka[r] = k;
        oa[r] = tA ? (int64_t)k + (int64_t)gm * sg.lda : (int64_t)gm + (int64_t)k * sg.lda;
      }
#pragma unroll
      for (int r = 0; r < BE; ++r) {
        const int idx = tid + r * kThreads;
        int n, k;
        if (!tB) { k = idx % kBK; n = idx / kBK; } else { n = idx % BN; k = idx / BN; }
        vb[r] = n0 + n < tk.N;
        const int gn = vb[r] ? n0 + n : n0;
        kb[r] = k;
        ob[r] = tB ? (int64_t)gn + (int64_t)k * sg.ldb : (int64_t)k + (int64_t)gn * sg.ldb;
      }
      auto load = [&](int k0) {
        const double* pa = sg.A + (int64_t)k0 * ska;
        const double* pb = sg.B + (int64_t)k0 * skb;
        if (k0 + kBK <= K) {
#pragma unroll
          for (int r = 0; r < AE; ++r) ra[r] = ld_global(pa + oa[r]);
#pragma unroll
          for (int r = 0; r < BE; ++r) rb[r] = ld_global(pb + ob[r]);
        } else {
#pragma unroll
          for (int r = 0; r < AE; ++r) ra[r] = k0 + ka[r] < K ? ld_global(pa + oa[r]) : 0.0;
#pragma unroll
          for (int r = 0; r < BE; ++r) rb[r] = k0 + kb[r] < K ? ld_global(pb + ob[r]) : 0.0;
        }
      };
      // alpha is applied when the prefetched values are written to LDS, after
      // the products of the current step, so nothing waits on the loads early
      auto store = [&](int b) {
#pragma unroll
        for (int r = 0; r < AE; ++r) {
          const int idx = tid + r * kThreads;
          int m, k;
          if (!tA) { m = idx % BM; k = idx / BM; } else { k = idx % kBK; m = idx / kBK; }
          sA[b][m * kPitch + k] = va[r] ? ra[r] * sg.alpha : 0.0;
        }
#pragma unroll
        for (int r = 0; r < BE; ++r) {
          const int idx = tid + r * kThreads;
          int n, k;
          if (!tB) { k = idx % kBK; n = idx / kBK; } else { n = idx % BN; k = idx / BN; }
          sB[b][n * kPitch + k] = vb[r] ? rb[r] : 0.0;
        }
      };
      if (K <= 0) continue;
      load(0);
      for (int k0 = 0; k0 < K; k0 += kBK) {
        store(buf);
        __syncthreads();
        if (k0 + kBK < K) load(k0 + kBK);
#pragma unroll
        for (int kk = 0; kk < kBK / 4; ++kk) {
          double a[FM], b[FN];
#pragma unroll
          for (int i = 0; i < FM; ++i) a[i] = sA[buf][(wm * WM + i * 16 + lr) * kPitch + kk * 4 + lk];
#pragma unroll
          for (int j = 0; j < FN; ++j) b[j] = sB[buf][(wn * WN + j * 16 + lr) * kPitch + kk * 4 + lk];
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        buf ^= 1;
      }
    }
    // epilogue: accumulator item r of lane l holds row 4r + l/16, column l%16
    // of each 16x16 block (gfx950 v_mfma_f64_16x16x4f64 output layout)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = n0 + wn * WN + j * 16 + lr;
        if (col >= tk.N) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = m0 + wm * WM + i * 16 + r * 4 + lk;
          if (row < tk.M) {
            double* p = tk.C + (int64_t)row + (int64_t)col * tk.ldc;
            double v = acc[i][j][r];
            if (tk.beta != 0.0) v += tk.beta * *p;
            *p = v;
          }
        }
      }
  }
}

// ---------------------------------------------------------------------------
constexpr int kMixChunk = 2048;

__global__ __launch_bounds__(kThreads) void k_mix(const MixWork* __restrict__ work, int nwork,
                                                  const MixDst* __restrict__ dsts,
                                                  const MixTerm* __restrict__ terms) {
  for (int wi = blockIdx.x; wi < nwork; wi += gridDim.x) {
    const MixWork w = work[wi];
    const MixDst d = dsts[w.dst];
    const int64_t e1 = min(w.e0 + (int64_t)kMixChunk, d.n);
    for (int64_t e = w.e0 + threadIdx.x; e < e1; e += kThreads) {
      double acc = 0.0;
      for (int t = 0; t < d.nt; ++t) {
        const MixTerm tm = terms[d.t0 + t];
        acc += tm.coef * tm.src[e];
      }
      d.dst[e] = acc;
    }
  }
}

__global__ __launch_bounds__(kThreads) void k_copy(const CopyWork* __restrict__ work, int nwork,
                                                   const CopyOp* __restrict__ ops) {
  for (int wi = blockIdx.x; wi < nwork; wi += gridDim.x) {
    const CopyWork w = work[wi];
    const CopyOp op = ops[w.op];
    const int64_t n = (int64_t)op.rows * op.cols;
    const int64_t e1 = min(w.e0 + (int64_t)kMixChunk, n);
    for (int64_t e = w.e0 + threadIdx.x; e < e1; e += kThreads) {
      const int r = (int)(e % op.rows), c = (int)(e / op.rows);
      double v = 0.0;
      if (op.src) {
        v = op.alpha * op.src[(int64_t)r + (int64_t)c * op.lds];
        if (op.rscale) v *= op.rscale[r];
        if (op.cscale) v *= op.cscale[c];
      }
      op.dst[(int64_t)r + (int64_t)c * op.ldd] = v;
    }
  }
}

__global__ void k_fill(double* p, int64_t n, double v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// ---------------------------------------------------------------------------
constexpr int kDotBlocks = 256;

struct DotArgs {
  const double* x[4];
  const double* y[4];
};

__device__ inline double lane_get(double v, int i) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), i),
                          __builtin_amdgcn_readlane(__double2loint(v), i));
}

template <int CTRL, int ROWS>
__device__ inline double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, true);
  return v + __hiloint2double(hi, lo);
}

// sum over the wave, in every lane: inside the rows of 16 lanes by shifts,
// across them by broadcasts of their last lanes (six dependent additions of
// VALU latency instead of six of LDS-permute latency)
__device__ inline double wave_sum(double v) {
  v = dpp_add<0x111, 0xf>(v);
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);
  v = dpp_add<0x143, 0xc>(v);
  return lane_get(v, 63);
}

__global__ __launch_bounds__(kThreads) void k_dot_partial(DotArgs args, int64_t n, double* partial) {
  const int pair = blockIdx.y;
  const double* __restrict__ x = args.x[pair];
  const double* __restrict__ y = args.y[pair];
  double s = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)kThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kThreads)
    s += x[i] * y[i];
  __shared__ double red[kThreads / 64];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int i = 0; i < kThreads / 64; ++i) t += red[i];
    partial[pair * kDotBlocks + blockIdx.x] = t;
  }
}

__global__ __launch_bounds__(kThreads) void k_dot_final(const double* partial, double* out) {
  const int pair = blockIdx.x;
  double s = 0.0;
  for (int i = threadIdx.x; i < kDotBlocks; i += kThreads) s += partial[pair * kDotBlocks + i];
  __shared__ double red[kThreads / 64];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int i = 0; i < kThreads / 64; ++i) t += red[i];
    out[pair] = t;
  }
}

// ---------------------------------------------------------------- Krylov step
// Everything between two H_eff applications of a Krylov iteration: alpha_j =
// Re <v_j, w>, two classical Gram-Schmidt passes of w against v_0..v_j (the
// coefficients of a pass from the same w, then one subtraction; alpha_j is the
// real part of the first pass's last one), beta_j = |w|, v_{j+1} = w / beta_j
// (zero when beta_j <= 1e-10, the space is exhausted), written to V and to the
// fixed H_eff input xin.  Complex vectors: real plane then imaginary plane of
// n elements each, <v, w> = sum conj(v) w.
//
// A piece of w is held in LDS and every wave takes whole vectors of the basis
// (several waves one vector when there are few), so a pass has one barrier
// however many vectors there are.  One work-group up to 4096 stored elements
// (complex two-site step at m = 12: 11.9 us with one barrier pair per vector,
// 6.9 now), above that four launches (m = 96, 18432 complex elements: 57 us of
// 16 launches before, 35 now).

// acc[i P + part] (first piece: set, else add) = the dots of the m elements
// from e0 of v_0..v_{k-1} with the piece wl (imaginary plane at wl + ldw)
template <int NW>
__device__ inline void krylov_dots(const double* __restrict__ V, int64_t nv, int64_t n, int cplx, int k,
                                   const double* wl, int ldw, int64_t e0, int m, double2* acc, bool first) {
  const int P = k < NW ? NW / k : 1, wv = threadIdx.x >> 6, part = wv % P, lane = threadIdx.x & 63;
  for (int i = wv / P; i < k; i += NW / P) {
    const double* v = V + (int64_t)i * nv + e0;
    double re = 0.0, im = 0.0;
    if (cplx) {
#pragma unroll 4
      for (int e = 64 * part + lane; e < m; e += 64 * P) {
        const double vr = v[e], vi = v[n + e], wr = wl[e], wi = wl[ldw + e];
        re += vr * wr + vi * wi;
        im += vr * wi - vi * wr;
      }
      im = wave_sum(im);
    } else {
#pragma unroll 8
      for (int e = 64 * part + lane; e < m; e += 64 * P) re += v[e] * wl[e];
    }
    re = wave_sum(re);
    if (lane == 0) {
      double2* d = acc + i * P + part;
      *d = first ? make_double2(re, im) : make_double2(d->x + re, d->y + im);
    }
  }
}

// element e of sum_i coef_i v_i
__device__ inline double2 krylov_project(const double* __restrict__ V, int64_t nv, int64_t n, int cplx, int k,
                                         const double2* coef, int64_t e) {
  double ar = 0.0, ai = 0.0;
  const double* v = V + e;
  if (cplx) {
#pragma unroll 4
    for (int i = 0; i < k; ++i) {
      const double vr = v[(int64_t)i * nv], vi = v[(int64_t)i * nv + n];
      const double2 c = coef[i];
      ar += c.x * vr - c.y * vi;
      ai += c.x * vi + c.y * vr;
    }
  } else {
#pragma unroll 8
    for (int i = 0; i < k; ++i) ar += coef[i].x * v[(int64_t)i * nv];
  }
  return make_double2(ar, ai);
}

constexpr int kTailThreads = 1024;
constexpr size_t kKrylovTailLds = 60 << 10;  // dynamic LDS of the one-work-group kernel

// Short vectors: one launch of one work-group.  VL: the basis fits into LDS
// beside w, so that the one memory latency of the kernel is that of all loads
// at once.
template <bool VL>
__global__ __launch_bounds__(kTailThreads) void k_krylov_tail(double* __restrict__ Vg, int64_t nv, int j,
                                                              const double* __restrict__ w, int64_t n, int cplx,
                                                              double* __restrict__ sc, double* __restrict__ xin,
                                                              int last) {
  constexpr int NW = kTailThreads / 64;
  extern __shared__ double wl[];
  __shared__ double2 acc[64], coef[64];
  __shared__ double red[NW];
  const int tid = threadIdx.x, m = (int)n, ne = cplx ? 2 * m : m;
  const int k = last ? 1 : j + 1;  // the last iteration only asks for alpha_j
  const int P = k < NW ? NW / k : 1;
  const double* B = last ? Vg + (int64_t)j * nv : Vg;
  if constexpr (VL) {
    for (int e = tid; e < ne; e += kTailThreads) {
      wl[e] = w[e];
#pragma unroll 8
      for (int i = 0; i < k; ++i) wl[(i + 1) * ne + e] = B[(int64_t)i * nv + e];
    }
  } else {
    for (int e = tid; e < ne; e += kTailThreads) wl[e] = w[e];
  }
  const double* V = VL ? wl + ne : B;
  const int64_t ld = VL ? ne : nv;
  __syncthreads();
  double s2 = 0.0;
  for (int pass = 0; pass < 2; ++pass) {
    krylov_dots<NW>(V, ld, m, cplx, k, wl, m, 0, m, acc, true);
    __syncthreads();
    if (tid < k) {
      double2 t = acc[tid * P];
      for (int q = 1; q < P; ++q) {
        t.x += acc[tid * P + q].x;
        t.y += acc[tid * P + q].y;
      }
      coef[tid] = t;
      if (pass == 0 && tid == k - 1) sc[j] = t.x;
    }
    if (last) return;
    __syncthreads();
    for (int e = tid; e < m; e += kTailThreads) {
      const double2 a = krylov_project(V, ld, m, cplx, k, coef, e);
      const double x = wl[e] - a.x, y = cplx ? wl[m + e] - a.y : 0.0;
      wl[e] = x;
      if (cplx) wl[m + e] = y;
      if (pass == 1) s2 += x * x + y * y;
    }
    if (pass == 0) __syncthreads();
  }
  s2 = wave_sum(s2);
  if ((tid & 63) == 0) red[tid >> 6] = s2;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int i = 0; i < NW; ++i) t += red[i];
  const double b = sqrt(t);
  const double invb = b > 1e-10 ? 1.0 / b : 0.0;
  if (tid == 0) sc[64 + j] = b;
  double* vn = Vg + (int64_t)(j + 1) * nv;
  for (int e = tid; e < ne; e += kTailThreads) {
    const double x = wl[e] * invb;
    vn[e] = x;
    xin[e] = x;
  }
}

// Longer vectors: four launches over many work-groups, each of which owns the
// same range of elements in all of them.  A launch starts by summing the
// partial sums of the one before it (every work-group all of them, from L2):
//   0: dots of w                                      -> pa
//   1: coefficients from pa, subtract, dots of the new w -> pb
//   2: coefficients from pb, subtract, squared norm   -> pa
//   3: beta from pa, v_{j+1} and xin
constexpr int kKrylovPiece = 1024;

template <int STEP>
__global__ __launch_bounds__(kThreads) void k_krylov_step(double* __restrict__ V, int64_t nv, int j,
                                                          double* __restrict__ w, int64_t n, int cplx,
                                                          double* __restrict__ sc, double* __restrict__ xin,
                                                          const double2* __restrict__ pin,
                                                          double2* __restrict__ pout) {
  constexpr int NW = kThreads / 64;
  __shared__ double wl[2 * kKrylovPiece];
  __shared__ double2 acc[64], coef[64];
  __shared__ double red[NW];
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, k = j + 1;
  const int nblk = gridDim.x;
  const int64_t per = ((n + nblk - 1) / nblk + 63) / 64 * 64;
  const int64_t lo = min(n, blockIdx.x * per), hi = min(n, lo + per);
  if constexpr (STEP == 1 || STEP == 2) {
    for (int i = wv; i < k; i += NW) {
      double re = 0.0, im = 0.0;
      for (int b = lane; b < nblk; b += 64) {
        const double2 p = pin[(int64_t)i * nblk + b];
        re += p.x;
        im += p.y;
      }
      re = wave_sum(re);
      im = wave_sum(im);
      if (lane == 0) coef[i] = make_double2(re, im);
    }
    __syncthreads();
    if (STEP == 1 && blockIdx.x == 0 && tid == 0) sc[j] = coef[j].x;
  }
  if constexpr (STEP == 3) {
    double t = 0.0;
    for (int b = tid; b < nblk; b += kThreads) t += pin[b].x;
    t = wave_sum(t);
    if (lane == 0) red[wv] = t;
    __syncthreads();
    t = 0.0;
#pragma unroll
    for (int i = 0; i < NW; ++i) t += red[i];
    const double b = sqrt(t);
    const double invb = b > 1e-10 ? 1.0 / b : 0.0;
    if (blockIdx.x == 0 && tid == 0) sc[64 + j] = b;
    double* vn = V + (int64_t)(j + 1) * nv;
    for (int64_t e = lo + tid; e < hi; e += kThreads) {
      const double x = w[e] * invb;
      vn[e] = x;
      xin[e] = x;
      if (cplx) {
        const double y = w[n + e] * invb;
        vn[n + e] = y;
        xin[n + e] = y;
      }
    }
    return;
  }
  double s2 = 0.0;
  for (int64_t e0 = lo; e0 < hi; e0 += kKrylovPiece) {
    const int m = (int)min((int64_t)kKrylovPiece, hi - e0);
    if (e0 > lo) __syncthreads();
    for (int e = tid; e < m; e += kThreads) {
      double x = w[e0 + e], y = cplx ? w[n + e0 + e] : 0.0;
      if constexpr (STEP != 0) {
        const double2 a = krylov_project(V, nv, n, cplx, k, coef, e0 + e);
        x -= a.x;
        y -= a.y;
        w[e0 + e] = x;
        if (cplx) w[n + e0 + e] = y;
        if (STEP == 2) s2 += x * x + y * y;
      }
      if constexpr (STEP != 2) {
        wl[e] = x;
        wl[kKrylovPiece + e] = y;
      }
    }
    if constexpr (STEP != 2) {
      __syncthreads();
      krylov_dots<NW>(V, nv, n, cplx, k, wl, kKrylovPiece, e0, m, acc, e0 == lo);
    }
  }
  __syncthreads();
  if constexpr (STEP == 2) {
    s2 = wave_sum(s2);
    if (lane == 0) red[wv] = s2;
    __syncthreads();
    if (tid == 0) {
      double t = 0.0;
      for (int i = 0; i < NW; ++i) t += red[i];
      pout[blockIdx.x] = make_double2(t, 0.0);
    }
  } else if (tid < k) {
    const int P = k < NW ? NW / k : 1;
    double2 t = make_double2(0.0, 0.0);
    for (int q = 0; q < P && lo < hi; ++q) {
      t.x += acc[tid * P + q].x;
      t.y += acc[tid * P + q].y;
    }
    pout[(int64_t)tid * nblk + blockIdx.x] = t;
  }
}

void launch_krylov_step(Context& c, double* V, int64_t nv, int j, double* w, int64_t n, int cplx, double* sc,
                        double* xin, double* work) {
  if (j < 0 || j >= 64) throw Error(-1, "krylov step: vector index out of range");
  if (n <= 0) return;
  const int nblk = (int)std::min<int64_t>(kKrylovBlocks, (n + kKrylovPiece - 1) / kKrylovPiece);
  double2* pa = (double2*)work;
  double2* pb = pa + 64 * kKrylovBlocks;
  const dim3 g(nblk), t(kThreads);
  hipLaunchKernelGGL(k_krylov_step<0>, g, t, 0, c.stream, V, nv, j, w, n, cplx, sc, xin, pb, pa);
  hipLaunchKernelGGL(k_krylov_step<1>, g, t, 0, c.stream, V, nv, j, w, n, cplx, sc, xin, pa, pb);
  hipLaunchKernelGGL(k_krylov_step<2>, g, t, 0, c.stream, V, nv, j, w, n, cplx, sc, xin, pb, pa);
  hipLaunchKernelGGL(k_krylov_step<3>, g, t, 0, c.stream, V, nv, j, w, n, cplx, sc, xin, pa, pb);
  HIP_OK(hipGetLastError());
}

void launch_krylov_tail(Context& c, double* V, int64_t nv, int j, double* w, int64_t n, int cplx, double* sc,
                        double* xin, int last) {
  if (j < 0 || j >= 64 || (cplx ? 2 * n : n) > kKrylovTailMax)
    throw Error(-1, "krylov tail: vector index or length out of range");
  const size_t wb = (cplx ? 2 * n : n) * sizeof(double), vb = wb * (last ? 1 : j + 1);
  const dim3 t(kTailThreads);
  if (wb + vb <= kKrylovTailLds)
    hipLaunchKernelGGL(k_krylov_tail<true>, dim3(1), t, wb + vb, c.stream, V, nv, j, w, n, cplx, sc, xin, last);
  else
    hipLaunchKernelGGL(k_krylov_tail<false>, dim3(1), t, wb, c.stream, V, nv, j, w, n, cplx, sc, xin, last);
  HIP_OK(hipGetLastError());
}

// The first vector: V and xin = x / |x| (an imaginary plane of zeros when the
// basis is complex and x is not: ne > ns), the scalars of the iteration
// cleared.  NRM: |x|^2 of a short x by every work-group itself, else from *n2.
template <bool NRM>
__global__ __launch_bounds__(kTailThreads) void k_krylov_first(const double* __restrict__ x, int64_t ns, int64_t ne,
                                                               const double* __restrict__ n2, double* __restrict__ V,
                                                               double* __restrict__ xin, double* __restrict__ sc) {
  __shared__ double red[kTailThreads / 64];
  double t = 0.0;
  if constexpr (NRM) {
    for (int64_t e = threadIdx.x; e < ns; e += kTailThreads) t += x[e] * x[e];
    t = wave_sum(t);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
    __syncthreads();
    t = 0.0;
#pragma unroll
    for (int i = 0; i < kTailThreads / 64; ++i) t += red[i];
  } else {
    t = *n2;
  }
  const double inv = 1.0 / sqrt(t);
  for (int64_t e = blockIdx.x * (int64_t)kTailThreads + threadIdx.x; e < ne; e += (int64_t)gridDim.x * kTailThreads) {
    const double v = e < ns ? x[e] * inv : 0.0;
    V[e] = v;
    xin[e] = v;
  }
  if (blockIdx.x == 0 && threadIdx.x < 256) sc[threadIdx.x] = 0.0;
}

void launch_krylov_first(Context& c, const double* x, int64_t ns, int64_t ne, double* V, double* xin, double* sc) {
  const dim3 t(kTailThreads);
  if (ne <= kKrylovTailMax) {
    hipLaunchKernelGGL(k_krylov_first<true>, dim3(1), t, 0, c.stream, x, ns, ne, nullptr, V, xin, sc);
  } else {
    const double* xs[1] = {x};
    launch_dots(c, 1, xs, xs, ns, c.scal + S_OC);
    const int64_t g = std::min<int64_t>((ne + kTailThreads - 1) / kTailThreads, 4 * c.num_cu);
    hipLaunchKernelGGL(k_krylov_first<false>, dim3((unsigned)g), t, 0, c.stream, x, ns, ne, c.scal + S_OC, V, xin,
                       sc);
  }
  HIP_OK(hipGetLastError());
}

__global__ void k_axpy_dev(double* y, const double* x, int64_t n, const double* coef) {
  const double c = *coef;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] += c * x[i];
}

__global__ void k_scale_dev(double* x, int64_t n, const double* coef) {
  const double c = *coef;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    x[i] *= c;
}

// Scalar steps of algs/DMRG.jl:57-90 on device scalars.
__device__ inline void lz_scalar(double* s, int stage) {
  if (stage == 0) {            // normalise the orthogonality-centre tensor
    s[S_INVOC] = 1.0 / sqrt(s[S_OC]);
  } else if (stage == 1) {     // alpha1 = <AA|Hpsi>, AA = theta/|theta|
    const double nrm = sqrt(s[S_TT]);
    s[S_NRM] = nrm;
    s[S_A1] = s[S_TH] / nrm;
    s[S_CAXPY] = -s[S_A1] / nrm;   // psi2 = Hpsi - alpha1*theta/|theta|
  } else if (stage == 2) {     // beta1 = |psi2|
    const double b = sqrt(s[S_PP]);
    s[S_B1] = b;
    const bool go = b > 1e-10;
    s[S_FLAG] = go ? 1.0 : 0.0;
    s[S_INVB] = go ? 1.0 / b : 0.0;
  } else if (stage == 3) {     // 2x2 Rayleigh-Ritz, lowest eigenpair
    const double a1 = s[S_A1];
    if (s[S_FLAG] == 0.0) {
      s[S_E] = a1;
      s[S_CA] = 1.0 / s[S_NRM];
      s[S_CB] = 0.0;
      return;
    }
    const double b = s[S_B1], a2 = s[S_PHP];
    s[S_A2] = a2;
    const double dd = 0.5 * (a2 - a1);
    const double r = sqrt(dd * dd + b * b);
    const double lam = 0.5 * (a1 + a2) - r;
    double v1, v2;
    if (dd >= 0.0) { v1 = -(dd + r); v2 = b; } else { v1 = b; v2 = -(r - dd); }
    const double nv = sqrt(v1 * v1 + v2 * v2);
    v1 /= nv;
    v2 /= nv;
    s[S_E] = lam;
    s[S_CA] = v1 / s[S_NRM];
    s[S_CB] = v2;
  } else if (stage == 4) {     // FP64 Rayleigh quotient of the Ritz vector
    s[S_ELP] = s[S_E];
    const double e = s[S_RH] / s[S_RR];
    s[S_E] = e;
    s[S_NEGE] = -e;
  }
}

__global__ void k_lz_scalar(double* s, int stage) {
  if (threadIdx.x == 0 && blockIdx.x == 0) lz_scalar(s, stage);
}

// The vector work of the two-vector Lanczos step (algs/DMRG.jl:57-90) between
// its H_eff applications, th the state, y1 = H th, then y2 = H psi2:
//   0: tt = |th|^2 and <th, y1>
//   1: scalars of stage 1, y1 -= alpha1 th / |th|, |y1|^2
//   2: scalars of stage 2, y1 /= beta1 (psi2)
//   3: <y1, y2>
//   4: scalars of stage 3, y2 := the Ritz vector
// A launch begins with the sums of the one before it (every work-group sums all
// partials).  Short vectors: steps 0 to 2 and steps 3 and 4 in one work-group
// each, the vector in registers: eleven launches became two or five, 35 of 460
// us of a bond step at m = 16 and 0.7 of 25.7 ms of a sweep at m = 64.  Up to
// 16384 elements one work-group and five launches measure the same in a sweep,
// the single launch costs the host less.
constexpr int kLzThreads = 1024;

__device__ inline double2 lz_block_sum(double a, double b, double2* red) {
  a = wave_sum(a);
  b = wave_sum(b);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = make_double2(a, b);
  __syncthreads();
  double2 t = make_double2(0.0, 0.0);
#pragma unroll
  for (int i = 0; i < kLzThreads / 64; ++i) {
    t.x += red[i].x;
    t.y += red[i].y;
  }
  return t;
}

template <int STEP>
__global__ __launch_bounds__(kLzThreads) void k_lz_step(const double* __restrict__ th, double* __restrict__ y1,
                                                        double* __restrict__ y2, int64_t n, double* __restrict__ s,
                                                        double* __restrict__ partial) {
  __shared__ double2 red[kLzThreads / 64];
  __shared__ double loc[S_COUNT];
  const int tid = threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * kLzThreads, e0 = blockIdx.x * (int64_t)kLzThreads + tid;
  double* part = partial + (STEP & 1 ? 2 * kDotPartials : 0);        // read by the odd steps' successors
  const double* prev = partial + (STEP & 1 ? 0 : 2 * kDotPartials);  // written by the step before
  if constexpr (STEP == 1 || STEP == 2 || STEP == 4) {
    const double* p = STEP == 4 ? partial + 2 * kDotPartials : prev;
    const bool in = tid < (int)gridDim.x;
    const double2 t = lz_block_sum(in ? p[tid] : 0.0, STEP == 1 && in ? p[kDotPartials + tid] : 0.0, red);
    if (tid < S_COUNT) loc[tid] = s[tid];
    __syncthreads();
    if (tid == 0) {
      if constexpr (STEP == 1) {
        loc[S_TT] = t.x;
        loc[S_TH] = t.y;
      }
      if constexpr (STEP == 2) loc[S_PP] = t.x;
      if constexpr (STEP == 4) loc[S_PHP] = t.x;
      lz_scalar(loc, STEP == 4 ? 3 : STEP);
    }
    __syncthreads();
  }
  double a = 0.0, b = 0.0;
  if constexpr (STEP == 0) {
#pragma unroll 4
    for (int64_t e = e0; e < n; e += stride) {
      const double x = th[e];
      a += x * x;
      b += x * y1[e];
    }
  } else if constexpr (STEP == 1) {
    const double c = loc[S_CAXPY];
#pragma unroll 4
    for (int64_t e = e0; e < n; e += stride) {
      const double y = y1[e] + c * th[e];
      y1[e] = y;
      a += y * y;
    }
  } else if constexpr (STEP == 2) {
    const double c = loc[S_INVB];
#pragma unroll 4
    for (int64_t e = e0; e < n; e += stride) y1[e] *= c;
  } else if constexpr (STEP == 3) {
#pragma unroll 4
    for (int64_t e = e0; e < n; e += stride) a += y1[e] * y2[e];
  } else {
    const double u = loc[S_CA], v = loc[S_CB];
#pragma unroll 4
    for (int64_t e = e0; e < n; e += stride) y2[e] = u * th[e] + v * y1[e];
  }
  if constexpr (STEP == 0 || STEP == 1 || STEP == 3) {
    const double2 t = lz_block_sum(a, b, red);
    if (tid == 0) {
      part[blockIdx.x] = t.x;
      if constexpr (STEP == 0) part[kDotPartials + blockIdx.x] = t.y;
    }
  }
  // the scalars last: other work-groups may still read the old ones (they do
  // not use what this step sets)
  if constexpr (STEP == 1 || STEP == 2 || STEP == 4)
    if (blockIdx.x == 0 && tid < S_COUNT) s[tid] = loc[tid];
}

template <int E>
__global__ __launch_bounds__(kLzThreads) void k_lz_short(const double* __restrict__ th, double* __restrict__ y1,
                                                         double* __restrict__ y2, int n, double* __restrict__ s,
                                                         int second) {
  __shared__ double2 red[kLzThreads / 64];
  __shared__ double loc[S_COUNT];
  const int tid = threadIdx.x;
  if (tid < S_COUNT) loc[tid] = s[tid];
  double y[E], a = 0.0, b = 0.0;
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int e = tid + u * kLzThreads;
    y[u] = e < n ? y1[e] : 0.0;
    const double x = e < n ? (second ? y2 : th)[e] : 0.0;
    a += second ? 0.0 : x * x;
    b += x * y[u];
  }
  const double2 t = lz_block_sum(a, b, red);
  if (tid == 0) {
    loc[second ? S_PHP : S_TH] = t.y;
    if (!second) loc[S_TT] = t.x;
    lz_scalar(loc, second ? 3 : 1);
  }
  __syncthreads();
  if (!second) {
    const double c = loc[S_CAXPY];
    a = 0.0;
#pragma unroll
    for (int u = 0; u < E; ++u) {
      const int e = tid + u * kLzThreads;
      y[u] += c * (e < n ? th[e] : 0.0);
      a += y[u] * y[u];
    }
    const double2 p = lz_block_sum(a, 0.0, red);
    if (tid == 0) {
      loc[S_PP] = p.x;
      lz_scalar(loc, 2);
    }
    __syncthreads();
  }
  const double c0 = second ? loc[S_CA] : 0.0, c1 = loc[second ? S_CB : S_INVB];
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int e = tid + u * kLzThreads;
    if (e < n) {
      if (second)
        y2[e] = c0 * th[e] + c1 * y[u];
      else
        y1[e] = y[u] * c1;
    }
  }
  if (tid < S_COUNT) s[tid] = loc[tid];
}

// After the first (second = false) or the second H_eff application.
void launch_lanczos(Context& c, const double* th, double* y1, double* y2, int64_t n, bool second) {
  const dim3 t(kLzThreads);
  if (n <= 4 * kLzThreads) {
    hipLaunchKernelGGL(k_lz_short<4>, dim3(1), t, 0, c.stream, th, y1, y2, (int)n, c.scal, second ? 1 : 0);
  } else if (n <= kLzShort) {
    hipLaunchKernelGGL(k_lz_short<kLzShort / kLzThreads>, dim3(1), t, 0, c.stream, th, y1, y2, (int)n, c.scal,
                       second ? 1 : 0);
  } else {
    const dim3 g((unsigned)std::min<int64_t>(kDotPartials, (n + 4 * kLzThreads - 1) / (4 * kLzThreads)));
    if (!second) {
      hipLaunchKernelGGL(k_lz_step<0>, g, t, 0, c.stream, th, y1, y2, n, c.scal, c.partial);
      hipLaunchKernelGGL(k_lz_step<1>, g, t, 0, c.stream, th, y1, y2, n, c.scal, c.partial);
      hipLaunchKernelGGL(k_lz_step<2>, g, t, 0, c.stream, th, y1, y2, n, c.scal, c.partial);
    } else {
      hipLaunchKernelGGL(k_lz_step<3>, g, t, 0, c.stream, th, y1, y2, n, c.scal, c.partial);
      hipLaunchKernelGGL(k_lz_step<4>, g, t, 0, c.stream, th, y1, y2, n, c.scal, c.partial);
    }
  }
  HIP_OK(hipGetLastError());
}

// Lane-layout probes of v_mfma_f64_16x16x4f64 (one wave, in-bounds):
//  mode 0: a = lane+1, b = 1      -> each output is a row sum of A
//  mode 1: a = 1, b = lane+1      -> each output is a column sum of B
//  mode 2: A[:,0] = i+1, A[:,1] = 1, B[0,:] = 1, B[1,:] = 1000(j+1) under the
//          layout A[i][k] <- lane i+16k, B[k][j] <- lane j+16k, giving
//          D[i][j] = (i+1) + 1000(j+1), found in item r of lane l for
//          i = 4r + l/16, j = l%16
__global__ void k_mfma_probe(double* out) {
  const int l = threadIdx.x;
  const int r16 = l & 15, k = l >> 4;
  for (int mode = 0; mode < 3; ++mode) {
    double a, b;
    if (mode == 0) {
      a = (double)(l + 1);
      b = 1.0;
    } else if (mode == 1) {
      a = 1.0;
      b = (double)(l + 1);
    } else {
      a = k == 0 ? (double)(r16 + 1) : (k == 1 ? 1.0 : 0.0);
      b = k == 0 ? 1.0 : (k == 1 ? 1000.0 * (r16 + 1) : 0.0);
    }
    double4_t acc = double4_t{0.0, 0.0, 0.0, 0.0};
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
    for (int r = 0; r < 4; ++r) out[mode * 256 + l * 4 + r] = acc[r];
  }
}

void launch_mfma_probe(Context& c, double* out) {
  hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, c.stream, out);
  HIP_OK(hipGetLastError());
}

// out[i] = sum_j c[j] V[j ld + i]; with out2: out2[i] = sum_j c[k + j] V[j ld + i] beside it
__global__ void k_combine(double* __restrict__ out, double* __restrict__ out2, const double* __restrict__ V,
                          int64_t ld, int64_t n, const double* __restrict__ c, int k) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    double a = 0.0, b = 0.0;
#pragma unroll 4
    for (int j = 0; j < k; ++j) {
      const double v = V[(int64_t)j * ld + i];
      a += c[j] * v;
      if (out2) b += c[k + j] * v;
    }
    out[i] = a;
    if (out2) out2[i] = b;
  }
}

// Coefficients of the Krylov exponential / Ritz vector on the device (one
// wave; the Krylov dimension is at most 64, typically 2..12):
//   k = the Krylov dimension used (first beta_j <= 1e-10 ends the space),
//   T = Q diag(lam) Q^T by the QL algorithm with implicit shifts (Dubrulle,
//   Martin and Wilkinson, Numer. Math. 12 (1968); FP64, the tridiagonal of alpha in sc[0..], beta in sc[64..]),
//   c = Q exp(pf lam) Q^T e1 with the complex prefactor pf = (pf_re, pf_im),
//   or (ritz) the eigenvector of the lowest lam signed to c_1 >= 0.
// coef: real Krylov vectors: c_re[0..r), c_im[r..2r); complex Krylov vectors
// (split planes, basis planes 2j = Re v_j, 2j+1 = Im v_j): the plane weights
// of Re out in [0..2r) and of Im out in [2r..4r).  Entries j >= k are zero.
// outs: {lowest Ritz value, k, 1 if an alpha/beta was non-finite}.
//
// Bound by the latency of the chain of plane rotations, about 0.85 k^2 of
// them: diagonal and off-diagonal live in the lanes (entry i in lane i, read as
// scalars), every lane runs the same chain and turns its own row of Q.  39 us
// at k = 12 against 86 of a parallel-order Jacobi in LDS.
__device__ inline double rsqrt_newton(double h) {
  double y = __builtin_amdgcn_rsq(h);
  y = fma(0.5 * y, fma(-h * y, y, 1.0), y);
  return fma(0.5 * y, fma(-h * y, y, 1.0), y);
}

__global__ __launch_bounds__(64) void k_krylov_coef(const double* __restrict__ sc, int r, double pf_re,
                                                     double pf_im, int ritz, int zv, double* __restrict__ coef,
                                                     double* __restrict__ outs) {
  __shared__ double Q[64 * 64];  // Q[i][t]: component t of eigenvector i
  const int t = threadIdx.x;
  double d = t < r ? sc[t] : 0.0, e = t + 1 < r ? sc[64 + t] : 0.0;
  const unsigned long long ends = __ballot(t + 1 < r && e <= 1e-10);
  const int k = ends ? __builtin_ctzll(ends) + 1 : r;
  const bool bad = __ballot(t < k && t + 1 < r && (!isfinite(d) || !isfinite(e))) != 0;
  if (t >= k) d = 0.0;
  if (t + 1 >= k) e = 0.0;
  for (int i = 0; i < k; ++i) Q[i * 64 + t] = i == t ? 1.0 : 0.0;
  // a power of two that brings the largest entry to order one
  double mx = fmax(fabs(d), fabs(e));
  for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
  int ex = 0;
  if (mx > 0.0 && mx < 1e308) (void)frexp(mx, &ex);
  ex = max(-1000, min(1000, ex));
  d = ldexp(d, -ex);
  e = ldexp(e, -ex);
  for (int l = 0; l < k && !bad; ++l) {
    for (int iter = 0; iter < 80; ++iter) {
      // the block [l, m] ends at the first negligible coupling (a NaN ends it too)
      const double dn = __shfl_down(d, 1, 64);
      const unsigned long long neg =
          __ballot(!(fabs(e) > 2.220446049250313e-16 * (fabs(d) + fabs(dn))) || t >= k - 1) >> l;
      const int m = l + __builtin_ctzll(neg);
      if (m == l) break;
      const double dl = lane_get(d, l), el = lane_get(e, l);
      double g = (lane_get(d, l + 1) - dl) / (2.0 * el);
      g = lane_get(d, m) - dl + el / (g + copysign(sqrt(g * g + 1.0), g));
      double s = 1.0, c = 1.0, p = 0.0, z = Q[m * 64 + t];
      int i = m - 1;
      for (; i >= l; --i) {
        const double ei = lane_get(e, i), di = lane_get(d, i), dj = lane_get(d, i + 1), zi = Q[i * 64 + t];
        const double f = s * ei, b = c * ei, h = f * f + g * g;
        if (!(h > 1e-280)) {  // the rotation is undefined: the block splits here
          if (t == i + 1) {
            d = dj - p;
            e = 0.0;
          }
          Q[(i + 1) * 64 + t] = z;
          break;
        }
        const double y = rsqrt_newton(h);
        s = f * y;
        c = g * y;
        g = dj - p;
        const double q = (di - g) * s + 2.0 * c * b;
        p = s * q;
        if (t == i + 1) {
          d = g + p;
          e = h * y;
        }
        g = c * q - b;
        Q[(i + 1) * 64 + t] = s * zi + c * z;
        z = c * zi - s * z;
      }
      if (t == m) e = 0.0;
      if (i < l) {
        Q[l * 64 + t] = z;
        if (t == l) {
          d = dl - p;
          e = g;
        }
      }
    }
  }
  __syncthreads();
  d = ldexp(d, ex);
  // lowest value, the first of equal ones; not a number if any is not finite
  double emin = t < k ? d : __builtin_inf();
  int imin = t;
  for (int o = 32; o > 0; o >>= 1) {
    const double v = __shfl_xor(emin, o, 64);
    const int i = __shfl_xor(imin, o, 64);
    if (v < emin || (v == emin && i < imin)) {
      emin = v;
      imin = i;
    }
  }
  emin = lane_get(emin, 0);
  imin = __builtin_amdgcn_readfirstlane(imin);
  if (__ballot(t < k && !isfinite(d)) != 0) emin = __builtin_nan("");
  if (t == 0) {
    outs[0] = emin;
    outs[1] = (double)k;
    outs[2] = bad ? 1.0 : 0.0;
  }
  double cre = 0.0, cim = 0.0;
  if (ritz) {
    if (t < k) cre = Q[imin * 64] >= 0.0 ? Q[imin * 64 + t] : -Q[imin * 64 + t];
    if (emin != emin) cre = emin;
  } else {
    const double mag = t < k ? exp(pf_re * d) * Q[t * 64] : 0.0;
    const double wr = mag * cos(pf_im * d), wi = mag * sin(pf_im * d);
    for (int i = 0; i < k; ++i) {
      const double q = Q[i * 64 + t];
      cre += q * lane_get(wr, i);
      cim += q * lane_get(wi, i);
    }
  }
  if (t >= k) cre = cim = 0.0;
  if (t >= r) return;
  if (!zv) {
    coef[t] = cre;
    coef[r + t] = cim;
  } else {
    coef[2 * t] = cre;           // Re out += Re c Re v - Im c Im v
    coef[2 * t + 1] = -cim;
    coef[2 * r + 2 * t] = cim;   // Im out += Im c Re v + Re c Im v
    coef[2 * r + 2 * t + 1] = cre;
  }
}

// ---------------------------------------------------------------------------
static int grid_for(int64_t n, int per = kThreads * 4) {
  int64_t g = (n + per - 1) / per;
  if (g < 1) g = 1;
  if (g > 4096) g = 4096;
  return (int)g;
}

int choose_gemm_cfg(const std::vector<GemmTask>& tasks, int num_cu) {
  // Heuristic used when the autotuner is off: the largest square tile whose
  // tile count still fills the chip ~2x; small blocks fall back to smaller
  // tiles.
  for (int cfg = 2; cfg >= 1; --cfg) {
    int64_t tiles = 0, waste = 0, useful = 0;
    for (const auto& t : tasks) {
      const int bm = kGemmShapes[cfg].bm, bn = kGemmShapes[cfg].bn;
      const int64_t tm = (t.M + bm - 1) / bm, tn = (t.N + bn - 1) / bn;
      tiles += tm * tn;
      useful += (int64_t)t.M * t.N;
      waste += tm * bm * tn * bn;
    }
    if (tiles >= 2 * num_cu && useful * 10 >= waste * 7) return cfg;
  }
  return 1;
}

double gemm_flops(const std::vector<GemmTask>& tasks, const std::vector<GemmSeg>& segs) {
  double f = 0.0;
  for (const auto& t : tasks)
    for (int s = 0; s < t.nseg; ++s) f += 2.0 * t.M * (double)t.N * segs[t.seg0 + s].K;
  return f;
}

double gemm_bytes(const std::vector<GemmTask>& tasks, const std::vector<GemmSeg>& segs) {
  double bytes = 0.0;  // compulsory: every operand block read once, C written once
  for (const auto& t : tasks) {
    bytes += 8.0 * t.M * (double)t.N;
    for (int q = 0; q < t.nseg; ++q) bytes += 8.0 * segs[t.seg0 + q].K * ((double)t.M + t.N);
  }
  return bytes;
}

template <int BM, int BN>
static void gemm_f64_kernel_launch(Context& c, const GemmLaunch& g) {
  if (c.ext_a)
    hipExtLaunchKernelGGL((k_gemm_f64<BM, BN>), dim3(g.grid), dim3(kThreads), 0, c.stream, c.ext_a, c.ext_b, 0,
                          g.tiles, g.ntiles, g.tasks, g.segs);
  else
    hipLaunchKernelGGL((k_gemm_f64<BM, BN>), dim3(g.grid), dim3(kThreads), 0, c.stream, g.tiles, g.ntiles,
                       g.tasks, g.segs);
}

static const void* gemm_f64_kernel_ptr(int cfg) {
  switch (cfg) {
    case 0: return (const void*)k_gemm_f64<32, 32>;
    case 1: return (const void*)k_gemm_f64<64, 64>;
    case 2: return (const void*)k_gemm_f64<128, 128>;
    case 3: return (const void*)k_gemm_f64<64, 128>;
    default: return (const void*)k_gemm_f64<128, 64>;
  }
}

int gemm_occupancy_f64(int cfg) {
  int nb = 0;
  HIP_OK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, gemm_f64_kernel_ptr(cfg), kThreads, 0));
  return std::max(nb, 1);
}

void issue_gemm_f64(Context& c, const GemmLaunch& g) {
  if (g.ntiles <= 0) return;
  c.stage_flush();
  switch (g.cfg) {
    case 0: gemm_f64_kernel_launch<32, 32>(c, g); break;
    case 1: gemm_f64_kernel_launch<64, 64>(c, g); break;
    case 2: gemm_f64_kernel_launch<128, 128>(c, g); break;
    case 3: gemm_f64_kernel_launch<64, 128>(c, g); break;
    default: gemm_f64_kernel_launch<128, 64>(c, g); break;
  }
  HIP_OK(hipGetLastError());
}

void launch_gemm(Context& c, const std::vector<GemmTask>& tasks, const std::vector<GemmSeg>& segs,
                 int cfg) {
  launch_gemm_arith(c, tasks, segs, cfg, 0);
}

MixLaunch prepare_mix(Context& c, const std::vector<MixDst>& dsts, const std::vector<MixTerm>& terms) {
  MixLaunch m;
  if (dsts.empty()) return m;
  std::vector<MixWork> work;
  for (size_t i = 0; i < dsts.size(); ++i)
    for (int64_t e = 0; e < dsts[i].n; e += kMixChunk) work.push_back({(int)i, 0, e});
  if (work.empty()) return m;
  UploadPack up;
  const size_t ow = up.add(work.data(), work.size() * sizeof(MixWork));
  const size_t od = up.add(dsts.data(), dsts.size() * sizeof(MixDst));
  const size_t ot = up.add(terms.data(), terms.size() * sizeof(MixTerm));
  char* base = up.commit(c);
  m.work = (const MixWork*)(base + ow);
  m.dsts = (const MixDst*)(base + od);
  m.terms = (const MixTerm*)(base + ot);
  m.nwork = (int)work.size();
  m.grid = (int)std::min<size_t>(work.size(), (size_t)c.num_cu * 8);
  for (const auto& d : dsts) {
    m.bytes += 8.0 * d.n * (1.0 + d.nt);
    m.flops += 2.0 * d.n * d.nt;
  }
  return m;
}

void issue_mix(Context& c, const MixLaunch& m) {
  if (m.nwork <= 0) return;
  c.stage_flush();
  hipLaunchKernelGGL(k_mix, dim3(m.grid), dim3(kThreads), 0, c.stream, m.work, m.nwork, m.dsts, m.terms);
  HIP_OK(hipGetLastError());
}

// Region marker for kernel traces: a one-wave kernel that does nothing; its
// dispatches bracket a region of interest in a profiler's dispatch list.
__global__ void k_region_marker(int id, double* sink) {
  if (id < 0 && threadIdx.x == 0) sink[0] = (double)id;
}

// The marker's id is also its work-group count, so kernel traces (which
// record grid sizes, not arguments) tell the markers apart.
void launch_marker(Context& c, int id) {
  hipLaunchKernelGGL(k_region_marker, dim3(std::max(1, id)), dim3(64), 0, c.stream, id, c.partial);
  HIP_OK(hipGetLastError());
}

void issue_mix_timed(Context& c, const MixLaunch& m) {
  if (m.nwork <= 0) return;
  const int ps = c.prof_begin();
  issue_mix(c, m);
  if (ps >= 0) c.prof_end(ps, KIND_MIX, m.flops, m.bytes);
}

void launch_mix(Context& c, const std::vector<MixDst>& dsts, const std::vector<MixTerm>& terms) {
  issue_mix_timed(c, prepare_mix(c, dsts, terms));
}

CopyLaunch prepare_copy(Context& c, const std::vector<CopyOp>& ops) {
  CopyLaunch l;
  std::vector<CopyWork> work;
  for (size_t i = 0; i < ops.size(); ++i) {
    const int64_t n = (int64_t)ops[i].rows * ops[i].cols;
    for (int64_t e = 0; e < n; e += kMixChunk) work.push_back({(int)i, 0, e});
  }
  if (work.empty()) return l;
  UploadPack up;
  const size_t ow = up.add(work.data(), work.size() * sizeof(CopyWork));
  const size_t oo = up.add(ops.data(), ops.size() * sizeof(CopyOp));
  char* base = up.commit(c);
  l.work = (const CopyWork*)(base + ow);
  l.ops = (const CopyOp*)(base + oo);
  l.nwork = (int)work.size();
  l.grid = (int)std::min<size_t>(work.size(), (size_t)c.num_cu * 8);
  for (const auto& o : ops) l.bytes += 8.0 * o.rows * (double)o.cols * (o.src ? 2.0 : 1.0);
  return l;
}

void issue_copy(Context& c, const CopyLaunch& l) {
  if (l.nwork <= 0) return;
  c.stage_flush();
  const int ps = c.prof_begin();
  hipLaunchKernelGGL(k_copy, dim3(l.grid), dim3(kThreads), 0, c.stream, l.work, l.nwork, l.ops);
  HIP_OK(hipGetLastError());
  if (ps >= 0) c.prof_end(ps, KIND_COPY, 0.0, l.bytes);
}

void launch_copy(Context& c, const std::vector<CopyOp>& ops) { issue_copy(c, prepare_copy(c, ops)); }

void launch_fill(Context& c, double* p, int64_t n, double v) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(kThreads), 0, c.stream, p, n, v);
  HIP_OK(hipGetLastError());
}

static_assert(kDotBlocks == kDotPartials, "partials per pair");

void launch_dots_buf(Context& c, int npairs, const double* const* xs, const double* const* ys, int64_t n,
                     double* out, double* partial) {
  if (npairs < 1 || npairs > 4) throw Error(-2, "launch_dots: 1..4 pairs");
  DotArgs a{};
  for (int i = 0; i < npairs; ++i) {
    a.x[i] = xs[i];
    a.y[i] = ys[i];
  }
  hipLaunchKernelGGL(k_dot_partial, dim3(kDotBlocks, npairs), dim3(kThreads), 0, c.stream, a, n, partial);
  HIP_OK(hipGetLastError());
  hipLaunchKernelGGL(k_dot_final, dim3(npairs), dim3(kThreads), 0, c.stream, partial, out);
  HIP_OK(hipGetLastError());
}

void launch_dots(Context& c, int npairs, const double* const* xs, const double* const* ys,
                 int64_t n, double* out) {
  launch_dots_buf(c, npairs, xs, ys, n, out, c.partial);
}

void launch_axpy_dev(Context& c, double* y, const double* x, int64_t n, const double* coef) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_axpy_dev, dim3(grid_for(n)), dim3(kThreads), 0, c.stream, y, x, n, coef);
  HIP_OK(hipGetLastError());
}

void launch_scale_dev(Context& c, double* x, int64_t n, const double* coef) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_scale_dev, dim3(grid_for(n)), dim3(kThreads), 0, c.stream, x, n, coef);
  HIP_OK(hipGetLastError());
}

void launch_krylov_coef(Context& c, const double* sc, int r, double pf_re, double pf_im, int ritz, int zv,
                        double* coef, double* outs) {
  if (r < 1 || r > 64) throw Error(-1, "launch_krylov_coef: Krylov dimension must be 1..64");
  hipLaunchKernelGGL(k_krylov_coef, dim3(1), dim3(64), 0, c.stream, sc, r, pf_re, pf_im, ritz, zv, coef, outs);
  HIP_OK(hipGetLastError());
}

void launch_combine(Context& c, double* out, double* out2, const double* V, int64_t ld, int64_t n,
                    const double* coef, int k) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_combine, dim3(grid_for(n)), dim3(kThreads), 0, c.stream, out, out2, V, ld, n, coef, k);
  HIP_OK(hipGetLastError());
}

void launch_lz_scalar(Context& c, int stage) {
  hipLaunchKernelGGL(k_lz_scalar, dim3(1), dim3(64), 0, c.stream, c.scal, stage);
  HIP_OK(hipGetLastError());
}

}  // namespace dmrj

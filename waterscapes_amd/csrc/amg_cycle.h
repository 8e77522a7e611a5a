// AMG V-cycle machinery shared by the single-instance solver (krylov.hip)
// and the batched solver (batch.hip): level SpMM kernels on node-interleaved
// NC-column vectors, Chebyshev smoothing, dense coarsest solves, and the
// block-diagonal MPET preconditioner built on them.
//
// Replaces the hypre BoomerAMG V-cycle behind PETSc's "hypre_amg"
// preconditioner of the MINRES solve (mpet/mpettotalpressuresolver.py:448).
#pragma once
#include "mpet_ops.h"
#include <hip/hip_fp16.h>
#include <vector>
#include <stdio.h>

namespace mpet {

constexpr int NT = 256;            // threads per block everywhere
constexpr int MAX_PARTIALS = 8192; // per-block partial sums of one reduction
constexpr int MAXLEV = 16;
constexpr int MAXDEG = 16;

// Work skipped by the level kernels: everything when *all is set; the rows
// of instance k when inst[k] is set (grp: row -> instance of the level).
struct Skip {
  const int* all = nullptr;
  const int* inst = nullptr;
};
__device__ __forceinline__ bool row_skipped(const Skip& sk, const int* __restrict__ grp, int r) {
  return sk.inst && grp && sk.inst[grp[r]];
}

// ---------------------------------------------------------------------------
// reductions
// ---------------------------------------------------------------------------
// All lanes of an aligned group of G lanes get the group sum.
template <int G, typename T>
__device__ __forceinline__ T group_allsum(T v) {
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Block sum of v, valid in thread 0.
__device__ __forceinline__ double block_sum(double v) {
  __shared__ double sh[NT / 64];
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0) sh[w] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0)
    for (int i = 0; i < NT / 64; ++i) r += sh[i];
  return r;
}

// Fixed-order sum of p[lo, hi) by the threads of a block into four
// accumulators per thread (four loads in flight); per-thread value.
__device__ __forceinline__ double thread_sum(const double* __restrict__ p, int lo, int hi) {
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
  int i = lo + threadIdx.x;
  for (; i + 3 * NT < hi; i += 4 * NT) {
    a0 += p[i];
    a1 += p[i + NT];
    a2 += p[i + 2 * NT];
    a3 += p[i + 3 * NT];
  }
  for (; i < hi; i += NT) a0 += p[i];
  return (a0 + a1) + (a2 + a3);
}

// Fixed-order sum of n partials by one block; valid in thread 0.
__device__ __forceinline__ double sum_partials(const double* __restrict__ p, int n) {
  return block_sum(thread_sum(p, 0, n));
}

static int grid_for(long long items, int per_block, int cap) {
  long long b = (items + per_block - 1) / per_block;
  if (b < 1) b = 1;
  return (int)(b < cap ? b : cap);
}

// Where the finest pressure level's result goes: position r (field-major,
// r = f nP1 + c) to the vectors' node-interleaved DOF F c + f, or through a
// map; identity when both are off.
struct OutMap {
  int nP1 = 0, F = 0;
  const int* map = nullptr;        // explicit places (batches)
  __device__ __forceinline__ long long operator()(int r) const {
    return map ? map[r] : (F ? (long long)(r % nP1) * F + r / nP1 : r);
  }
};

// ---------------------------------------------------------------------------
// AMG level kernels on NC-column node-interleaved vectors (NC = 3 for the
// displacement block: one scalar matrix, three components; NC = 1 for the
// pressure blocks).  LPR lanes per row; after an xor all-reduce, lane c of
// the row group finishes component c.
// MODE 0: y = A x        MODE 1: y = b - A x       MODE 2: y += A x
// MODE 3: Chebyshev step d' = cd d + cr Dinv (b - A x); y = x + d'; d is
//         read only when cd != 0 (not by the first step from x), d' is
//         written to y2 when y2 is given (not by the last step of a
//         smoothing sequence; y2 may be d: each entry is read, then written,
//         by one thread)
// MODE 4: restriction entering the coarse level's smoother: y = A x, then
//         its first Chebyshev step from zero d = y2 = cr Dinv y (dinv and
//         cr of the coarse level)
// ---------------------------------------------------------------------------
template <typename T, int NC, int LPR, int MODE, bool COMPACT = false>
__global__ void __launch_bounds__(NT)
spmm_kernel(int nrows, const int* __restrict__ rp, const int* __restrict__ ci,
            const T* __restrict__ val, const T* __restrict__ x, const T* __restrict__ b,
            T* __restrict__ y, const T* __restrict__ dinv, T* d, T cd, T cr,
            const uint8_t* __restrict__ mask, Skip sk, const int* __restrict__ grp,
            T* y2, OutMap om, const __half* __restrict__ val16 = nullptr,
            const int16_t* __restrict__ dci = nullptr, T vscale = (T)1) {
  // COMPACT: values stored as half precision times 1/vscale, columns as
  // signed 16-bit offsets from the row (half the bytes per nonzero)
  static_assert(NC <= LPR, "one lane per component in the epilogue");
  if (sk.all && *sk.all) return;
  long long gid = (long long)blockIdx.x * NT + threadIdx.x;
  int r = (int)(gid / LPR);
  int lane = (int)(gid % LPR);
  if (r >= nrows || row_skipped(sk, grp, r)) return;   // whole row groups leave
  T acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0;
  const int kb = rp[r], ke = rp[r + 1];
  auto value = [&](int k) -> T {
    if constexpr (COMPACT) return (T)__half2float(val16[k]);
    else return val[k];
  };
  auto column = [&](int k) -> long long {
    if constexpr (COMPACT) return (long long)NC * (r + (int)dci[k]);
    else return (long long)NC * ci[k];
  };
  // the epilogue operands are loaded first (by every lane, at clamped
  // indices, so that no branch splits the loads) and their latency overlaps
  // the row loop
  const long long o = (long long)NC * r + (lane < NC ? lane : NC - 1);
  T pb = 0, px = 0, pd = 0, pdinv = 0;
  if constexpr (MODE == 1 || MODE == 3) pb = b[o];
  if constexpr (MODE == 2) px = y[o];
  if constexpr (MODE == 3) {
    px = x[o];
    if (cd != (T)0) pd = d[o];
    pdinv = dinv[r];
  }
  if constexpr (MODE == 4) pdinv = dinv[r];
  const int mrow = mask ? (int)mask[r] : 0;
  // U nonzeros per lane per trip: every index, value and gather load of a
  // trip is issued before the first use (a missing nonzero reloads the
  // row's last one and contributes 0).  A lane's nonzeros are summed in the
  // order k, k + LPR, k + 2 LPR, ... (the same order for any unrolling).
  constexpr int U = (NC == 3 && LPR <= 4) ? 8 : 4;
  for (int k = kb + lane; k < ke; k += U * LPR) {
    T a[U];
    long long cc[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int kk = k + j * LPR;
      const int kc = kk < ke ? kk : ke - 1;
      const T v = value(kc);
      cc[j] = column(kc);
      a[j] = kk < ke ? v : (T)0;
    }
    T xv[U][NC];
#pragma unroll
    for (int j = 0; j < U; ++j) load_nc<T, NC>(x + cc[j], xv[j]);
#pragma unroll
    for (int j = 0; j < U; ++j)
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[c] += a[j] * xv[j][c];
  }
  if constexpr (COMPACT) {
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] *= vscale;
  }
  T mine = 0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    T v = group_allsum<LPR>(acc[c]);
    if (lane == c) mine = v;
  }
  if (lane >= NC) return;
  const bool m = mrow != 0;
  if (MODE == 0) {
    y[o] = m ? (T)0 : mine;
  } else if (MODE == 1) {
    y[o] = m ? (T)0 : pb - mine;
  } else if (MODE == 2) {
    if (!m) y[o] = px + mine;
  } else if (MODE == 4) {
    y[o] = mine;
    const T v = cr * pdinv * mine;
    d[o] = v;
    y2[o] = v;
  } else {
    T dd = m ? (T)0 : cd * pd + cr * pdinv * (pb - mine);
    if (y2) y2[o] = dd;
    y[NC == 1 ? om(r) : o] = m ? (T)0 : px + dd;
  }
}

// The same SpMM modes with one thread per row doing all NC columns (rows of
// a few nonzeros, such as the prolongator from the P1 level: no lanes idle
// on short rows).  Nonzeros are summed in row order.
template <typename T, int NC, int MODE>
__global__ void __launch_bounds__(NT)
spmm_row_kernel(int nrows, const int* __restrict__ rp, const int* __restrict__ ci,
                const T* __restrict__ val, const T* __restrict__ x, const T* __restrict__ b,
                T* __restrict__ y, const T* __restrict__ dinv, T* d, T cd, T cr,
                const uint8_t* __restrict__ mask, Skip sk, const int* __restrict__ grp,
                T* y2) {
  if (sk.all && *sk.all) return;
  const int r = blockIdx.x * NT + threadIdx.x;
  if (r >= nrows || row_skipped(sk, grp, r)) return;
  T acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0;
  const int kb = rp[r], ke = rp[r + 1];
  int k = kb;
  for (; k + 1 < ke; k += 2) {
    const T va = val[k], vb = val[k + 1];
    const long long ca = (long long)NC * ci[k], cb = (long long)NC * ci[k + 1];
    T xa[NC], xb[NC];
    load_nc<T, NC>(x + ca, xa);
    load_nc<T, NC>(x + cb, xb);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      acc[c] += va * xa[c];
      acc[c] += vb * xb[c];
    }
  }
  if (k < ke) {
    const T va = val[k];
    T xa[NC];
    load_nc<T, NC>(x + (long long)NC * ci[k], xa);
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] += va * xa[c];
  }
  const bool m = mask ? mask[r] != 0 : false;
  const T di = (MODE == 3 || MODE == 4) ? dinv[r] : (T)0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const long long o = (long long)NC * r + c;
    const T mine = acc[c];
    if (MODE == 0) {
      y[o] = m ? (T)0 : mine;
    } else if (MODE == 1) {
      y[o] = m ? (T)0 : b[o] - mine;
    } else if (MODE == 2) {
      if (!m) y[o] = y[o] + mine;
    } else if (MODE == 4) {
      y[o] = mine;
      const T v = cr * di * mine;
      d[o] = v;
      y2[o] = v;
    } else {
      const T dp = cd != (T)0 ? cd * d[o] : (T)0;
      const T dd = m ? (T)0 : dp + cr * di * (b[o] - mine);
      if (y2) y2[o] = dd;
      y[o] = m ? (T)0 : x[o] + dd;
    }
  }
}


// ---------------------------------------------------------------------------
// Fused transfers.  With k pre-smoothing steps from zero ending in x and the
// residual r = b - A x, restriction and residual are one product
//     R r = R b - (R A) x,
// and prolongation of the coarse correction e and the first post-smoothing
// step from x' = x + P e are one product as well,
//     b - A x' = r - (A P) e:  d = cr D^-1 (r - (A P) e),  x'' = x + P e + d,
// with R A and A P formed at set-up.  Each saves a dependent launch; which
// level takes which follows from their bytes (levels.py): on the P2 level A P
// has 0.28 of A's nonzeros (7.2 against 25.4 M at 48^3) and replaces a product
// with A, while R A would only add to the residual, which the post-smoothing
// needs anyway.
//   one smoothing step (x = c D^-1 b):  W = R - c (R A) D^-1 acts on b alone
//     and Q = P - c D^-1 (A P) on e alone;
//   more steps: W = [-R A, R] acts on [x; b] (one buffer), Q holds the pairs
//     ((A P)_ij, P_ij) on the pattern of A P.
// Lanes per row are run-time powers of two (2^lg).
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T lanes_allsum(T v, int lanes) {
  for (int off = lanes >> 1; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// This lane's part of row r of a CSR (or compact) matrix times x, in the
// order k, k + lanes, ..; four nonzeros in flight as in spmm_kernel.
template <typename T, int NC, bool COMPACT>
__device__ __forceinline__ void row_part(const int* __restrict__ rp, const int* __restrict__ ci,
                                         const T* __restrict__ val,
                                         const __half* __restrict__ val16,
                                         const int16_t* __restrict__ dci,
                                         const T* __restrict__ x, int r, int lane, int lanes,
                                         T (&acc)[NC]) {
  constexpr int U = 4;
  const int kb = rp[r], ke = rp[r + 1];
  for (int k = kb + lane; k < ke; k += U * lanes) {
    T a[U];
    long long cc[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int kk = k + j * lanes;
      const int kc = kk < ke ? kk : ke - 1;
      T v;
      if constexpr (COMPACT) {
        v = (T)__half2float(val16[kc]);
        cc[j] = (long long)NC * (r + (int)dci[kc]);
      } else {
        v = val[kc];
        cc[j] = (long long)NC * ci[kc];
      }
      a[j] = kk < ke ? v : (T)0;
    }
    T xv[U][NC];
#pragma unroll
    for (int j = 0; j < U; ++j) load_nc<T, NC>(x + cc[j], xv[j]);
#pragma unroll
    for (int j = 0; j < U; ++j)
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[c] += a[j] * xv[j][c];
  }
}

// ---------------------------------------------------------------------------
// Sliced rows (SELL-64): one thread per row and all NC columns, slices of 64
// rows padded to their longest.  Rows are ordered by length within windows
// of 512 (the P2 rows alternate between 65 and 17-29 nonzeros: padding 5%
// instead of 49%), so a slice's rows stay neighbours: at the k-th nonzero
// the 64 lanes read 64 nearby columns, where lanes sharing a row read 8
// scattered ones.  Columns are 16-bit offsets from the slice's smallest, which
// padding entries read times zero: a batch's slices hold one instance's rows,
// so that a NaN stays in its instance.
// Used where one thread per row fills the chip (65,536 rows, levels.py).
// ---------------------------------------------------------------------------
// Runs of 16 consecutive blocks (4,096 rows) go to one XCD, so that its L2
// serves a run's gathered planes (48^3 iteration 490 against 495 us without).
constexpr int SELL_CHUNK = 16;

template <typename T>
struct Sell {
  const int* off = nullptr;        // first entry of each slice / 64 (nslice + 1)
  const int* base = nullptr;       // smallest column of each slice
  const int* row = nullptr;        // row of each (slice, lane), -1: none
  const uint16_t* dc = nullptr;    // column - base; null for packed values
  const void* v = nullptr;         // T, pairs of T, or packed: half | offset << 16
};
enum SellValues { SELL_PLAIN = 0, SELL_PACKED = 1, SELL_PAIR = 2 };

// Sums of one row: s1 (and s2 of the second values of pairs).
template <typename T, int NC, int VK>
__device__ __forceinline__ void sell_part(const Sell<T>& M, int slice, int lane,
                                          const T* __restrict__ x, T (&s1)[NC], T (&s2)[NC]) {
  const int o = M.off[slice], w = M.off[slice + 1] - o;
  const T* __restrict__ xb = x + (long long)NC * M.base[slice];
  constexpr int U = 8;             // entries in flight (4: 495 against 490 us)
  auto entry = [&](int j, T& a, T& p, int& c) {
    const long long k = ((long long)(o + j) << 6) + lane;
    if constexpr (VK == SELL_PACKED) {
      const uint32_t q = ((const uint32_t*)M.v)[k];
      const uint16_t h = (uint16_t)(q & 0xffffu);
      __half hv;
      __builtin_memcpy(&hv, &h, 2);
      a = (T)__half2float(hv);
      p = (T)0;
      c = (int)(q >> 16);
    } else if constexpr (VK == SELL_PAIR) {
      T v[2];
      load_nc<T, 2>((const T*)M.v + 2 * k, v);
      a = v[0];
      p = v[1];
      c = M.dc[k];
    } else {
      a = ((const T*)M.v)[k];
      p = (T)0;
      c = M.dc[k];
    }
  };
  for (int j = 0; j < w; j += U) {          // w is the wave's own: no divergence
    T a[U], p[U], xv[U][NC];
    int c[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int jj = j + i < w ? j + i : w - 1;
      entry(jj, a[i], p[i], c[i]);
    }
#pragma unroll
    for (int i = 0; i < U; ++i) load_nc<T, NC>(xb + NC * c[i], xv[i]);
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const T ai = j + i < w ? a[i] : (T)0;
      const T pi = j + i < w ? p[i] : (T)0;
#pragma unroll
      for (int q = 0; q < NC; ++q) {
        s1[q] += ai * xv[i][q];
        if constexpr (VK == SELL_PAIR) s2[q] += pi * xv[i][q];
      }
    }
  }
}

// Vectors of a sliced kernel's epilogue, by mode:
//   1: y = b - A x      3: d' = cd d + cr Dinv (b - A x), y = x + d', y2 = d'
//   6: y = xs + cr Dinv b + A x (post_kernel, one step)
//   7: d' = cr Dinv (b - A x), y = xs + P x + d', y2 = d' (pairs)
template <typename T>
struct SellEpi {
  const T *b, *xs, *dinv, *d;
  T cd, cr, vscale;
  T *y, *y2;
  const uint8_t* mask;
  OutMap om;
  const int* grp;
};

template <typename T, int NC, int VK, int MODE>
__device__ __forceinline__ void sell_rows(const Sell<T>& M, int nslice, int slice, int lane,
                                          const T* __restrict__ x, const SellEpi<T>& E,
                                          const Skip& sk) {
  if (slice >= nslice) return;
  const int r = M.row[slice * 64 + lane];
  T pb[NC], px[NC], pd[NC];
  const long long o = (long long)NC * (r < 0 ? 0 : r);
  load_nc<T, NC>(E.b + o, pb);
  if constexpr (MODE == 3) load_nc<T, NC>(x + o, px);
  if constexpr (MODE >= 6) load_nc<T, NC>(E.xs + o, px);
#pragma unroll
  for (int q = 0; q < NC; ++q) pd[q] = 0;
  if constexpr (MODE == 3)
    if (E.cd != (T)0) load_nc<T, NC>(E.d + o, pd);
  T di = 0;
  if constexpr (MODE != 1) di = E.cr * E.dinv[r < 0 ? 0 : r];
  const bool m = r >= 0 && E.mask && E.mask[r] != 0;
  T s1[NC], s2[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) { s1[q] = 0; s2[q] = 0; }
  sell_part<T, NC, VK>(M, slice, lane, x, s1, s2);
  if (r < 0 || row_skipped(sk, E.grp, r)) return;
  T out[NC], dd[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    T t = s1[q];
    if constexpr (VK == SELL_PACKED) t *= E.vscale;
    dd[q] = 0;
    if constexpr (MODE == 1) {
      out[q] = m ? (T)0 : pb[q] - t;
    } else if constexpr (MODE == 3) {
      dd[q] = m ? (T)0 : E.cd * pd[q] + di * (pb[q] - t);
      out[q] = m ? (T)0 : px[q] + dd[q];
    } else if constexpr (MODE == 6) {
      out[q] = m ? (T)0 : px[q] + di * pb[q] + t;
    } else {
      dd[q] = m ? (T)0 : di * (pb[q] - t);
      out[q] = m ? (T)0 : px[q] + s2[q] + dd[q];
    }
  }
  if constexpr (MODE == 3 || MODE == 7)
    if (E.y2) __builtin_memcpy(E.y2 + o, dd, sizeof(T) * NC);
  __builtin_memcpy(E.y + (NC == 1 ? E.om(r) : o), out, sizeof(T) * NC);
}

template <typename T, int NC, int VK, int MODE>
__global__ void __launch_bounds__(NT)
sell_kernel(Sell<T> M, int nslice, const T* __restrict__ x, SellEpi<T> E, Skip sk) {
  if (sk.all && *sk.all) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = xcd_tile(blockIdx.x, gridDim.x, SELL_CHUNK);
  sell_rows<T, NC, VK, MODE>(M, nslice, tile * (NT / 64) + wave, threadIdx.x & 63, x, E, sk);
}

// Arguments of the two halves of transfer_kernel.
template <typename T>
struct DownArgs {           // bc = W v; with dinv: d = y2 = cr Dinv bc (the coarse
  int n, lg;                // level's first Chebyshev step)
  const int *rp, *ci;
  const T *val, *v;
  T* bc;
  const T* dinv;
  T cr;
  T *d, *y2;
  const int* grp;
};
template <typename T>
struct ResArgs {            // r = b - A x, rows with mask 0
  int n, lg;
  const int *rp, *ci;
  const T* val;
  const __half* val16;
  const int16_t* dci;
  T vscale;
  const T *x, *b;
  T* r;
  const uint8_t* mask;
  const int* grp;
};

// One row group of the restriction half.
template <typename T, int NC>
__device__ __forceinline__ void down_rows(const DownArgs<T>& w, int block, const Skip& sk) {
  T acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0;
  const long long gid = (long long)block * NT + threadIdx.x;
  const int r = (int)(gid >> w.lg), lanes = 1 << w.lg;
  const int lane = (int)(gid & (lanes - 1));
  if (r >= w.n || row_skipped(sk, w.grp, r)) return;     // whole row groups leave
  const T di = w.dinv ? w.cr * w.dinv[r] : (T)0;
  row_part<T, NC, false>(w.rp, w.ci, w.val, nullptr, nullptr, w.v, r, lane, lanes, acc);
  T mine = 0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const T v = lanes_allsum(acc[c], lanes);
    if (lane == c) mine = v;
  }
  if (lane >= NC) return;
  const long long o = (long long)NC * r + lane;
  w.bc[o] = mine;
  if (w.dinv) {
    w.d[o] = di * mine;
    w.y2[o] = di * mine;
  }
}

// One row group of the residual half.
template <typename T, int NC, bool COMPACT>
__device__ __forceinline__ void res_rows(const ResArgs<T>& a, int block, const Skip& sk) {
  T acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0;
  const long long gid = (long long)block * NT + threadIdx.x;
  const int r = (int)(gid >> a.lg), lanes = 1 << a.lg;
  const int lane = (int)(gid & (lanes - 1));
  if (r >= a.n || row_skipped(sk, a.grp, r)) return;
  const long long o = (long long)NC * r + (lane < NC ? lane : NC - 1);
  const T pb = a.b[o];
  const int m = a.mask ? (int)a.mask[r] : 0;
  row_part<T, NC, COMPACT>(a.rp, a.ci, a.val, a.val16, a.dci, a.x, r, lane, lanes, acc);
  T mine = 0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const T v = lanes_allsum(acc[c], lanes);
    if (lane == c) mine = v;
  }
  if (lane >= NC) return;
  if constexpr (COMPACT) mine *= a.vscale;
  a.r[o] = m ? (T)0 : pb - mine;
}

// Blocks [0, nbw) form the coarse right-hand side, the rest the residual:
// both read only x and b, so one launch holds both (a launch of its own
// costs 3-5 us, more than the rows of every level but the finest).
template <typename T, int NC, bool COMPACT>
__global__ void __launch_bounds__(NT)
transfer_kernel(DownArgs<T> w, ResArgs<T> a, int nbw, Skip sk) {
  if (sk.all && *sk.all) return;
  if ((int)blockIdx.x < nbw) down_rows<T, NC>(w, blockIdx.x, sk);
  else res_rows<T, NC, COMPACT>(a, (int)blockIdx.x - nbw, sk);
}

// The same with the residual's rows sliced.
template <typename T, int NC, int VK>
__global__ void __launch_bounds__(NT)
transfer_sell_kernel(DownArgs<T> w, Sell<T> M, int nslice, const T* __restrict__ x,
                     SellEpi<T> E, int nbw, Skip sk) {
  if (sk.all && *sk.all) return;
  if ((int)blockIdx.x < nbw) {
    down_rows<T, NC>(w, blockIdx.x, sk);
    return;
  }
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = xcd_tile((int)blockIdx.x - nbw, (int)gridDim.x - nbw, SELL_CHUNK);
  sell_rows<T, NC, VK, 1>(M, nslice, tile * (NT / 64) + wave, threadIdx.x & 63, x, E, sk);
}

// Prolongation with the first post-smoothing step.  One step in all
// (PAIR false): y = x + cr Dinv r + Q e.  More (PAIR): d = cr Dinv (r -
// (A P) e), y = x + P e + d; d is stored for the next step.
template <typename T>
struct PostArgs {
  int n, lg;
  const int *rp, *ci;
  const T *val, *e, *x, *r, *dinv;
  T cr;
  T *y, *d;
  const uint8_t* mask;
  OutMap om;
  const int* grp;
};
template <typename T, int NC, bool PAIR>
__device__ __forceinline__ void post_rows(const PostArgs<T>& A, int block, const Skip& sk) {
  const int n = A.n, lg = A.lg;
  const int *__restrict__ rp = A.rp, *__restrict__ ci = A.ci;
  const T *__restrict__ val = A.val, *__restrict__ e = A.e;
  const T *x = A.x, *r_ = A.r, *__restrict__ dinv = A.dinv;
  const T cr = A.cr;
  T *y = A.y, *d = A.d;
  const uint8_t* __restrict__ mask = A.mask;
  const int* __restrict__ grp = A.grp;
  const OutMap om = A.om;
  const long long gid = (long long)block * NT + threadIdx.x;
  const int r = (int)(gid >> lg), lanes = 1 << lg;
  const int lane = (int)(gid & (lanes - 1));
  if (r >= n || row_skipped(sk, grp, r)) return;
  const long long o = (long long)NC * r + (lane < NC ? lane : NC - 1);
  const T px = x[o], pr = r_[o], di = cr * dinv[r];
  const int m = mask ? (int)mask[r] : 0;
  constexpr int U = 4;
  const int kb = rp[r], ke = rp[r + 1];
  T s1[NC], s2[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) { s1[c] = 0; s2[c] = 0; }
  for (int k = kb + lane; k < ke; k += U * lanes) {
    T a[U], p[U];
    long long cc[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int kk = k + j * lanes;
      const int kc = kk < ke ? kk : ke - 1;
      T v[2];
      if constexpr (PAIR) load_nc<T, 2>(val + 2ll * kc, v);
      else { v[0] = val[kc]; v[1] = 0; }
      cc[j] = (long long)NC * ci[kc];
      a[j] = kk < ke ? v[0] : (T)0;
      p[j] = kk < ke ? v[1] : (T)0;
    }
    T xv[U][NC];
#pragma unroll
    for (int j = 0; j < U; ++j) load_nc<T, NC>(e + cc[j], xv[j]);
#pragma unroll
    for (int j = 0; j < U; ++j)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        s1[c] += a[j] * xv[j][c];
        if constexpr (PAIR) s2[c] += p[j] * xv[j][c];
      }
  }
  T m1 = 0, m2 = 0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const T v = lanes_allsum(s1[c], lanes);
    if (lane == c) m1 = v;
    if constexpr (PAIR) {
      const T u = lanes_allsum(s2[c], lanes);
      if (lane == c) m2 = u;
    }
  }
  if (lane >= NC) return;
  const long long oo = NC == 1 ? om(r) : o;
  if constexpr (PAIR) {
    const T dd = m ? (T)0 : di * (pr - m1);
    if (d) d[o] = dd;
    y[oo] = m ? (T)0 : px + m2 + dd;
  } else {
    y[oo] = m ? (T)0 : px + di * pr + m1;
  }
}
template <typename T, int NC, bool PAIR>
__global__ void __launch_bounds__(NT)
post_kernel(PostArgs<T> A, Skip sk) {
  if (sk.all && *sk.all) return;
  post_rows<T, NC, PAIR>(A, blockIdx.x, sk);
}

// A MINRES vector update fused into the first kernels of a preconditioner
// apply that read its input (off when y is null): the input entry i is
// r[i] = y[i] - (alfa / beta) r2o[i], computed where it is first read and
// stored to r[i] for the later readers.
template <typename T>
struct K2In {
  const T* y = nullptr;
  const T* r2o = nullptr;
  T* r = nullptr;
  const double* alfa = nullptr;
  const double* beta = nullptr;
  __device__ __forceinline__ T make(long long i) const {
    const T c = (T)(*alfa / *beta);
    const T v = y[i] - c * r2o[i];
    r[i] = v;
    return v;
  }
};

// First Chebyshev step from x0 = 0: d = y = cr * Dinv * (scale * b) (d
// only when given); the scaled right-hand side is kept in bcopy when given;
// with k2 on, b is made by k2 (and b itself is not read).
template <typename T, int NC>
__device__ __forceinline__ void cheb0_rows(int block, int nrows, const T* b, T scale,
                                           const T* __restrict__ dinv, T cr, T* __restrict__ d,
                                           T* __restrict__ y, T* __restrict__ bcopy,
                                           const uint8_t* __restrict__ mask, const Skip& sk,
                                           const int* __restrict__ grp, const K2In<T>& k2) {
  long long i = (long long)block * NT + threadIdx.x;
  if (i >= (long long)NC * nrows) return;
  int r = (int)(i / NC);
  if (row_skipped(sk, grp, r)) return;
  T bv = scale * (k2.y ? k2.make(i) : b[i]);
  if (bcopy) bcopy[i] = bv;
  T v = (mask && mask[r]) ? (T)0 : cr * dinv[r] * bv;
  if (d) d[i] = v;
  y[i] = v;
}
template <typename T, int NC>
__global__ void __launch_bounds__(NT)
cheb0_kernel(int nrows, const T* b, T scale, const T* __restrict__ dinv, T cr,
             T* __restrict__ d, T* __restrict__ y, T* __restrict__ bcopy,
             const uint8_t* __restrict__ mask, Skip sk, const int* __restrict__ grp,
             K2In<T> k2 = K2In<T>()) {
  if (sk.all && *sk.all) return;
  cheb0_rows<T, NC>(blockIdx.x, nrows, b, scale, dinv, cr, d, y, bcopy, mask, sk, grp, k2);
}

// This lane's part of a dense row times b (NC columns): 16 bytes of the row
// per load, U loads (and their b values) in flight; the last n mod V columns
// one per lane.  With K2, b = y - kc r2o.  (Single-word loads: 3,859 rows in
// FP32 23 us, now 15; 1,972 rows of three columns 12 us, now 9.)
template <typename T, int NC, bool K2 = false>
__device__ __forceinline__ void dense_part(const T* __restrict__ row, const T* __restrict__ b,
                                           int n, int lane, T (&acc)[NC],
                                           const T* __restrict__ r2o = nullptr, T kc = 0) {
  constexpr int V = 16 / (int)sizeof(T), U = NC == 1 ? 4 : 2;
  const int full = n / V;
  for (int g0 = lane; g0 < full; g0 += 64 * U) {
    T a[U][V], bv[U][V * NC];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int g = g0 + 64 * j;
      const int gc = g < full ? g : full - 1;
      load_nc<T, V>(row + (long long)V * gc, a[j]);
      load_nc<T, V * NC>(b + (long long)V * NC * gc, bv[j]);
      if constexpr (K2) {
        T rv[V * NC];
        load_nc<T, V * NC>(r2o + (long long)V * NC * gc, rv);
#pragma unroll
        for (int i = 0; i < V * NC; ++i) bv[j][i] -= kc * rv[i];
      }
    }
#pragma unroll
    for (int j = 0; j < U; ++j)
      if (g0 + 64 * j < full)
#pragma unroll
        for (int v = 0; v < V; ++v)
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[c] += a[j][v] * bv[j][NC * v + c];
  }
  const int k = V * full + lane;
  if (k < n) {
    const T a = row[k];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      T v = b[(long long)NC * k + c];
      if constexpr (K2) v -= kc * r2o[(long long)NC * k + c];
      acc[c] += a * v;
    }
  }
}

// Dense coarsest solve x = Cinv (scale b) (NC columns), one wave per row over
// the row's nonzero columns rng (two runs; null: all): the pressure fields do
// not couple in the preconditioner, so a row of F fields has 1 / F of them,
// its field's columns and, further on, those of aggregates formed last.  The 64 MiB
// this can be are read once an apply.  Whole rows / runs, us per iteration:
// mixed 8^3 (A = 4, 3,645 rows) 76.3 / 47.8, 6^3 48.6 / 39.3, direct 8^3 (A =
// 2) 60.7 / 48.8; the FP64 preconditioner at 16^3 75.7 / 68.7 us an apply.
template <typename T, int NC>
__device__ __forceinline__ void coarse_rows(int block, int n, const T* __restrict__ cinv,
                                            const int* __restrict__ rng, const T* b,
                                            T* __restrict__ x, T scale, const OutMap& om,
                                            const K2In<T>& k2) {
  const int r = block * (NT / 64) + threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  if (r >= n) return;
  T acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0;
  const T* __restrict__ row = cinv + (long long)r * n;
  const bool own = om.F || om.map;
  const T kc2 = k2.y ? (T)(*k2.alfa / *k2.beta) : (T)0;
  const int runs = rng ? 2 : 1;
#pragma unroll 1
  for (int run = 0; run < runs; ++run) {
    const int c0 = rng ? rng[4 * r + 2 * run] : 0, c1 = rng ? rng[4 * r + 2 * run + 1] : n;
    if (c0 >= c1) continue;
    if (!own && k2.y) {
      dense_part<T, NC, true>(row + c0, k2.y + (long long)NC * c0, c1 - c0, lane, acc,
                              k2.r2o + (long long)NC * c0, kc2);
    } else if (!own) {
      dense_part<T, NC>(row + c0, b + (long long)NC * c0, c1 - c0, lane, acc);
    } else {
      for (int k0 = c0 + lane; k0 < c1; k0 += 256) {
        T a[4], bv[4][NC];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int k = k0 + 64 * j;
          const int kc = k < c1 ? k : c1 - 1;
          a[j] = k < c1 ? row[kc] : (T)0;
          const long long o = NC == 1 ? om(kc) : (long long)NC * kc;
          if (k2.y) {
            T yv[NC], rv[NC];
            load_nc<T, NC>(k2.y + o, yv);
            load_nc<T, NC>(k2.r2o + o, rv);
#pragma unroll
            for (int c = 0; c < NC; ++c) bv[j][c] = yv[c] - kc2 * rv[c];
          } else {
            load_nc<T, NC>(b + o, bv[j]);
          }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[c] += a[j] * bv[j][c];
      }
    }
  }
  const long long o = NC == 1 ? om(r) : (long long)NC * r;
  if (k2.y && lane < NC) k2.make(o + lane);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    T v = group_allsum<64>(acc[c]);
    if (lane == c) x[o + c] = scale * v;
  }
}
template <typename T, int NC>
__global__ void __launch_bounds__(NT)
coarse_kernel(int n, const T* __restrict__ cinv, const int* __restrict__ rng, const T* b,
              T* __restrict__ x, const int* __restrict__ skip, T scale, OutMap om, K2In<T> k2) {
  if (skip && *skip) return;
  coarse_rows<T, NC>(blockIdx.x, n, cinv, rng, b, x, scale, om, k2);
}

// The gather with the first Chebyshev step of the finest pressure level from
// zero: b = the gathered entry, x = cr Dinv b (and the direction d when
// given), each at the entry's place in the hierarchy (field-major, or map).
template <typename T>
struct EnterArgs {
  long long np;
  int nP1, F;
  const int* map;
  const T* src;
  T* b;
  const T* dinv;
  T cr;
  T *d, *x;
  const uint8_t* mask;
  const int* grp;
  K2In<T> k2;
};
template <typename T>
__device__ __forceinline__ void enter_rows(const EnterArgs<T>& E, int block, const Skip& sk) {
  const long long i = (long long)block * NT + threadIdx.x;
  if (i >= E.np) return;
  const int q = E.map ? E.map[i] : (int)((i % E.F) * E.nP1 + i / E.F);
  if (row_skipped(sk, E.grp, q)) return;
  const T bv = E.k2.y ? E.k2.make(i) : E.src[i];
  E.b[q] = bv;
  const T v = (E.mask && E.mask[q]) ? (T)0 : E.cr * E.dinv[q] * bv;
  if (E.d) E.d[q] = v;
  E.x[q] = v;
}
template <typename T>
__global__ void __launch_bounds__(NT)
p_enter_kernel(EnterArgs<T> E, Skip sk) {
  if (sk.all && *sk.all) return;
  enter_rows(E, blockIdx.x, sk);
}
// Block-diagonal dense coarsest solve (many independent instances): row r
// lies in block blk[r] spanning rows off[b] .. off[b+1]-1, whose dense
// inverse is stored row-major at inv + ioff[b].
template <typename T, int NC>
__device__ __forceinline__ void blockdiag_rows(int block, int n, const int* __restrict__ blk,
                                               const int* __restrict__ off,
                                               const int64_t* __restrict__ ioff,
                                               const T* __restrict__ inv,
                                               const T* __restrict__ b, T* __restrict__ x,
                                               const Skip& sk, const int* __restrict__ grp) {
  const int r = block * (NT / 64) + threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  if (r >= n || row_skipped(sk, grp, r)) return;
  const int bk = blk[r];
  const int o = off[bk], sz = off[bk + 1] - o;
  const T* row = inv + ioff[bk] + (long long)(r - o) * sz;
  T acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0;
  dense_part<T, NC>(row, b + (long long)NC * o, sz, lane, acc);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    T v = group_allsum<64>(acc[c]);
    if (lane == c) x[NC * r + c] = v;
  }
}
template <typename T, int NC>
__global__ void __launch_bounds__(NT)
coarse_blockdiag_kernel(int n, const int* __restrict__ blk, const int* __restrict__ off,
                        const int64_t* __restrict__ ioff, const T* __restrict__ inv,
                        const T* __restrict__ b, T* __restrict__ x, Skip sk,
                        const int* __restrict__ grp) {
  if (sk.all && *sk.all) return;
  blockdiag_rows<T, NC>(blockIdx.x, n, blk, off, ioff, inv, b, x, sk, grp);
}

// ---------------------------------------------------------------------------
// Joint launches.  On small systems a V-cycle kernel takes 3-5 us whatever
// its rows, and forking the pressure blocks onto a second stream costs more
// than it hides (12^3, four networks: 94.7 us per iteration forked, 87.7 in
// one chain); there the i-th step of the displacement cycle and the i-th of
// the pressure cycle, which are independent, share a launch.  A step is one
// of the kernels above, named by its kind; lanes per row at run time.
// ---------------------------------------------------------------------------
enum StepKind { STEP_NONE, STEP_FIRST, STEP_ENTER, STEP_CHEB, STEP_DOWN, STEP_POST, STEP_DENSE,
                STEP_BLOCKS };

template <typename T>
struct Step {
  int kind = STEP_NONE, blocks = 0, nbw = 0, n = 0;
  bool compact = false, pair = false;
  ResArgs<T> a{};                  // matrix and rows (CHEB, DOWN)
  DownArgs<T> w{};
  PostArgs<T> p{};
  EnterArgs<T> e{};
  const T *b = nullptr, *dinv = nullptr;
  T cd = 0, cr = 0, scale = 1;
  T *d = nullptr, *y = nullptr, *y2 = nullptr, *bcopy = nullptr;
  OutMap om;
  K2In<T> k2;
  const T* cinv = nullptr;
  const int *blk = nullptr, *off = nullptr;
  const int64_t* ioff = nullptr;
};

// Chebyshev step d' = cd d + cr Dinv (b - A x), y = x + d' (spmm_kernel mode
// 3) of one row group; S.a.x and S.a.b hold x and b.
template <typename T, int NC, bool COMPACT>
__device__ __forceinline__ void cheb_rows(const Step<T>& S, int block, const Skip& sk) {
  const ResArgs<T>& a = S.a;
  const long long gid = (long long)block * NT + threadIdx.x;
  const int r = (int)(gid >> a.lg), lanes = 1 << a.lg;
  const int lane = (int)(gid & (lanes - 1));
  if (r >= a.n || row_skipped(sk, a.grp, r)) return;
  const long long o = (long long)NC * r + (lane < NC ? lane : NC - 1);
  const T pb = a.b[o], px = a.x[o], pd = S.cd != (T)0 ? S.d[o] : (T)0, di = S.dinv[r];
  const int m = a.mask ? (int)a.mask[r] : 0;
  T acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = 0;
  row_part<T, NC, COMPACT>(a.rp, a.ci, a.val, a.val16, a.dci, a.x, r, lane, lanes, acc);
  T mine = 0;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const T v = lanes_allsum(acc[c], lanes);
    if (lane == c) mine = v;
  }
  if (lane >= NC) return;
  if constexpr (COMPACT) mine *= a.vscale;
  const T dd = m ? (T)0 : S.cd * pd + S.cr * di * (pb - mine);
  if (S.y2) S.y2[o] = dd;
  S.y[NC == 1 ? S.om(r) : o] = m ? (T)0 : px + dd;
}

template <typename T, int NC>
__device__ __forceinline__ void run_step(const Step<T>& S, int block, const Skip& sk) {
  switch (S.kind) {
    case STEP_FIRST:
      cheb0_rows<T, NC>(block, S.n, S.b, S.scale, S.dinv, S.cr, S.d, S.y, S.bcopy, S.a.mask, sk,
                        S.a.grp, S.k2);
      break;
    case STEP_ENTER:
      if constexpr (NC == 1) enter_rows(S.e, block, sk);
      break;
    case STEP_CHEB:
      if constexpr (sizeof(T) == 4) {
        if (S.compact) { cheb_rows<T, NC, true>(S, block, sk); break; }
      }
      cheb_rows<T, NC, false>(S, block, sk);
      break;
    case STEP_DOWN:
      if (block < S.nbw) { down_rows<T, NC>(S.w, block, sk); break; }
      if constexpr (sizeof(T) == 4) {
        if (S.compact) { res_rows<T, NC, true>(S.a, block - S.nbw, sk); break; }
      }
      res_rows<T, NC, false>(S.a, block - S.nbw, sk);
      break;
    case STEP_POST:
      if (S.pair) post_rows<T, NC, true>(S.p, block, sk);
      else post_rows<T, NC, false>(S.p, block, sk);
      break;
    case STEP_DENSE:
      coarse_rows<T, NC>(block, S.n, S.cinv, S.off, S.b, S.y, S.scale, S.om, S.k2);
      break;
    case STEP_BLOCKS:
      blockdiag_rows<T, NC>(block, S.n, S.blk, S.off, S.ioff, S.cinv, S.b, S.y, sk, S.a.grp);
      break;
    default: break;
  }
}

template <typename T>
__global__ void __launch_bounds__(NT)
joint_kernel(Step<T> u, Step<T> p, Skip sk) {
  if (sk.all && *sk.all) return;
  if ((int)blockIdx.x < u.blocks) run_step<T, 3>(u, blockIdx.x, sk);
  else run_step<T, 1>(p, (int)blockIdx.x - u.blocks, sk);
}

// inv[map[i]] = i (map a permutation of 0 .. n - 1).  A template, so that the
// translation units including this header share one instance.
template <typename I>
__global__ void __launch_bounds__(NT)
invert_map_kernel_t(int n, const I* __restrict__ map, I* __restrict__ inv) {
  const int i = blockIdx.x * NT + threadIdx.x;
  if (i < n) inv[map[i]] = i;
}

// Pressure vectors through an explicit map: dst[map[i]] = src[i] (gather
// into hierarchy order) and dst[i] = src[map[i]] (scatter back).
template <typename T>
__global__ void __launch_bounds__(NT)
p_gather_map_kernel(long long np, const int* __restrict__ map, const T* __restrict__ src,
                    T* __restrict__ dst, const int* __restrict__ skip) {
  if (skip && *skip) return;
  long long i = (long long)blockIdx.x * NT + threadIdx.x;
  if (i < np) dst[map[i]] = src[i];
}
template <typename T>
__global__ void __launch_bounds__(NT)
p_scatter_map_kernel(long long np, const int* __restrict__ map, const T* __restrict__ src,
                     T* __restrict__ dst, const int* __restrict__ skip) {
  if (skip && *skip) return;
  long long i = (long long)blockIdx.x * NT + threadIdx.x;
  if (i < np) dst[i] = src[map[i]];
}

}  // namespace mpet

// --- host side ---
using namespace mpet;

#define HIPCHK(expr)                                                        \
  do {                                                                      \
    hipError_t _e = (expr);                                                 \
    if (_e != hipSuccess) {                                                 \
      char _m[400];                                                         \
      snprintf(_m, sizeof(_m), "%s: %s", #expr, hipGetErrorString(_e));     \
      mpet_set_error(_m);                                                   \
      return ERR_HIP;                                                       \
    }                                                                       \
  } while (0)

static void chebyshev(double lmin, double lmax, int deg, double* cd, double* cr) {
  double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin);
  double sigma = theta / delta, rho = 1.0 / sigma;
  cd[0] = 0.0;
  cr[0] = 1.0 / theta;
  for (int i = 1; i < deg; ++i) {
    double rn = 1.0 / (2.0 * sigma - rho);
    cd[i] = rn * rho;
    cr[i] = 2.0 * rn / delta;
    rho = rn;
  }
}

template <typename T>
struct LevelDev {
  int n = 0, nc = 0;
  const int *rp = nullptr, *ci = nullptr;
  const T *v = nullptr, *dinv = nullptr;
  const int *Prp = nullptr, *Pci = nullptr, *Rrp = nullptr, *Rci = nullptr;
  const T *Pv = nullptr, *Rv = nullptr;
  const uint8_t* mask = nullptr;
  // row -> instance of this level and of the next coarser one (batches)
  const int *grp = nullptr, *grpc = nullptr;
  // optional compact copy of the level operator (half values times 1/vscale,
  // 16-bit column offsets from the row), used by the level SpMMs when set
  const __half* v16 = nullptr;
  const int16_t* dci = nullptr;
  double vscale = 1.0;
  int deg = 2;                     // Chebyshev degree of this level's smoother
  double cd[MAXDEG], cr[MAXDEG];
  int lpr = 8, lprP = 4, lprR = 8;
  // fused transfers (transfer_kernel, post_kernel; null: the separate ones),
  // log2 lanes per row
  const int *Wrp = nullptr, *Wci = nullptr, *Qrp = nullptr, *Qci = nullptr;
  const T *Wv = nullptr, *Qv = nullptr;
  int lgW = 3, lgQ = 2;
  // sliced copies of the level operator and of Q (off null: none), their slices
  Sell<T> As, Qs;
  int nAs = 0, nQs = 0;
  T *B = nullptr, *X = nullptr, *R = nullptr, *E = nullptr, *S1 = nullptr, *S2 = nullptr,
    *D = nullptr;
};

// One AMG hierarchy applied to NC-column vectors.
template <typename T>
struct Hier {
  int nlev = 0, deg = 2, NC = 1;
  LevelDev<T> lev[MAXLEV];
  const T* cinv = nullptr;
  // block-diagonal coarsest level (batched instances); cblk null: one dense
  // block, coff its rows' column ranges (null: whole rows)
  const int *cblk = nullptr, *coff = nullptr;
  const int64_t* cioff = nullptr;
  double scale = 1.0;      // the V-cycle approximates (scale * A0)^-1
};

template <typename T>
struct Precond {
  Hier<T> u, p;
  int nP1 = 0, F = 0;
  long long nu = 0;
  const int* pmap = nullptr;           // explicit pressure order (batches)
  int* pinv = nullptr;                 // its inverse
  bool joint = false;                  // both cycles in joint launches, no fork
  // optional second stream: the pressure V-cycle runs beside the
  // displacement one (fork / join through the two events; inside a captured
  // graph these become parallel branches)
  hipStream_t ps = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
};

// Create the fork stream and events of P (default priority, no timing).
template <typename T>
static int make_fork(Precond<T>& P) {
  if (P.joint) return OK;
  if (hipStreamCreateWithFlags(&P.ps, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&P.ev_fork, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&P.ev_join, hipEventDisableTiming) != hipSuccess) {
    mpet_set_error("preconditioner stream / event creation failed");
    return ERR_HIP;
  }
  return OK;
}
template <typename T>
static void free_fork(Precond<T>& P) {
  if (P.ev_fork) (void)hipEventDestroy(P.ev_fork);
  if (P.ev_join) (void)hipEventDestroy(P.ev_join);
  if (P.ps) (void)hipStreamDestroy(P.ps);
  P.ev_fork = P.ev_join = nullptr;
  P.ps = nullptr;
}

template <typename T, int NC, int MODE>
static void spmm(const LevelDev<T>& L, int which, const T* x, const T* b, T* y, T* d, T cd,
                 T cr, Skip sk, hipStream_t s, const T* dinv = nullptr, T* y2 = nullptr,
                 OutMap om = OutMap()) {
  // which: 0 level operator, 1 prolongator (rows n), 2 restriction (rows nc);
  // dinv: the diagonal inverse used by the epilogue (default the level's)
  int nrows = which == 2 ? L.nc : L.n;
  const int* rp = which == 0 ? L.rp : (which == 1 ? L.Prp : L.Rrp);
  const int* ci = which == 0 ? L.ci : (which == 1 ? L.Pci : L.Rci);
  const T* v = which == 0 ? L.v : (which == 1 ? L.Pv : L.Rv);
  int lpr = which == 0 ? L.lpr : (which == 1 ? L.lprP : L.lprR);
  if constexpr (MODE == 1 || MODE == 3) {
    if (which == 0 && L.As.off) {
      const int ns = L.nAs, nb = (ns + NT / 64 - 1) / (NT / 64);
      const SellEpi<T> E{b, nullptr, dinv ? dinv : L.dinv, d, cd, cr, (T)L.vscale, y, y2, L.mask,
                         om, L.grp};
      if (L.As.dc)
        hipLaunchKernelGGL((sell_kernel<T, NC, SELL_PLAIN, MODE>), dim3(nb), dim3(NT), 0, s,
                           L.As, ns, x, E, sk);
      else if constexpr (sizeof(T) == 4)
        hipLaunchKernelGGL((sell_kernel<T, NC, SELL_PACKED, MODE>), dim3(nb), dim3(NT), 0, s,
                           L.As, ns, x, E, sk);
      return;
    }
  }
  const bool compact = which == 0 && L.v16;
  if (NC > 1 && lpr == 1 && !compact) {     // one thread per row, all columns
    const int blocks1 = (nrows + NT - 1) / NT;
    if (blocks1 == 0) return;
    hipLaunchKernelGGL((spmm_row_kernel<T, NC, MODE>), dim3(blocks1), dim3(NT), 0, s, nrows,
                       rp, ci, v, x, b, y, dinv ? dinv : L.dinv, d, cd, cr,
                       which == 2 ? nullptr : L.mask, sk, which == 2 ? L.grpc : L.grp, y2);
    return;
  }
  if (lpr < NC) lpr = NC == 3 ? 4 : NC;
  const uint8_t* mask = which == 2 ? nullptr : L.mask;
  const int* grp = which == 2 ? L.grpc : L.grp;
  if (!dinv) dinv = L.dinv;
  long long threads = (long long)nrows * lpr;
  int blocks = (int)((threads + NT - 1) / NT);
  if (blocks == 0) return;
  if (which == 0 && L.v16) {
    if constexpr (sizeof(T) == 4 && MODE != 4) {
#define SPMM_CASE(LP)                                                                          \
  case LP:                                                                                     \
    hipLaunchKernelGGL((spmm_kernel<T, NC, (LP < NC ? 4 : LP), MODE, true>), dim3(blocks),     \
                       dim3(NT), 0, s, nrows, rp, ci, v, x, b, y, dinv, d, cd, cr, mask, sk, grp, \
                       y2, om, L.v16, L.dci, (T)L.vscale);                                     \
    break;
      switch (lpr) {
        SPMM_CASE(4) SPMM_CASE(8) SPMM_CASE(16) SPMM_CASE(32) SPMM_CASE(64)
        default: hipLaunchKernelGGL((spmm_kernel<T, NC, (NC > 4 ? 8 : 4), MODE, true>),
                                    dim3((unsigned)(((long long)nrows * (NC > 4 ? 8 : 4) + NT - 1) / NT)),
                                    dim3(NT), 0, s, nrows, rp, ci, v, x, b, y, dinv, d, cd, cr,
                                    mask, sk, grp, y2, om, L.v16, L.dci, (T)L.vscale);
      }
#undef SPMM_CASE
      return;
    }
  }
#define SPMM_CASE(LP)                                                                          \
  case LP:                                                                                     \
    hipLaunchKernelGGL((spmm_kernel<T, NC, (LP < NC ? 4 : LP), MODE>), dim3(blocks), dim3(NT), \
                       0, s, nrows, rp, ci, v, x, b, y, dinv, d, cd, cr, mask, sk, grp, y2, om);  \
    break;
  switch (lpr) {
    SPMM_CASE(1) SPMM_CASE(2) SPMM_CASE(4) SPMM_CASE(8) SPMM_CASE(16) SPMM_CASE(32)
    SPMM_CASE(64)
    default: break;
  }
#undef SPMM_CASE
}

// Buffer of the first Chebyshev step from zero on a level whose smoothing
// result goes to out.
template <typename T>
static T* first_dst(const LevelDev<T>& L, T* out) {
  return L.deg == 1 ? out : L.S1;
}

// Chebyshev steps i0 .. of level L from cur, the last one into out (through
// om); the direction of step i0 - 1 is in L.D when i0 > 0.
template <typename T, int NC>
static void smooth_steps(const LevelDev<T>& L, const T* b, const T* cur, int i0, T* out,
                         Skip sk, hipStream_t s, OutMap om = OutMap()) {
  T* bufs[2] = {L.S1, L.S2};
  int flip = i0 & 1;
  for (int i = i0; i < L.deg; ++i) {
    const bool last = i == L.deg - 1;
    T* dst = last ? out : bufs[flip];
    if (dst == cur) dst = bufs[flip ^ 1];
    // the last step's direction is not needed again
    spmm<T, NC, 3>(L, 0, cur, b, dst, L.D, (T)L.cd[i], (T)L.cr[i], sk, s, nullptr,
                   last ? nullptr : L.D, last ? om : OutMap());
    cur = dst;
    flip ^= 1;
  }
}

// Pre-smoothing from zero of level l into L.X; b scaled by bscale and
// copied to bcopy when given; entered: the first step is already in
// first_dst (made by the restriction or the pressure gather).
template <typename T, int NC>
static void smooth_from_zero(const LevelDev<T>& L, const T* b, T bscale, T* bcopy, Skip sk,
                             hipStream_t s, bool entered, K2In<T> k2) {
  T* dst = first_dst(L, L.X);
  const int blocks = (int)(((long long)NC * L.n + NT - 1) / NT);
  if (!entered)
    hipLaunchKernelGGL((cheb0_kernel<T, NC>), dim3(blocks), dim3(NT), 0, s, L.n, b, bscale,
                       L.dinv, (T)L.cr[0], L.deg == 1 ? nullptr : L.D, dst, bcopy, L.mask, sk,
                       L.grp, k2);
  smooth_steps<T, NC>(L, bcopy ? bcopy : b, dst, 1, L.X, sk, s);
}

// Blocks of n rows at 2^lg lanes each.
static int row_blocks(int n, int lg) {
  return (int)((((long long)n << lg) + NT - 1) / NT);
}
template <typename T>
static DownArgs<T> down_args(const Hier<T>& H, int l, const T* b) {
  const LevelDev<T>& L = H.lev[l];
  const LevelDev<T>& C = H.lev[l + 1];
  const bool enter = l + 1 < H.nlev - 1;
  return DownArgs<T>{L.nc, L.lgW, L.Wrp, L.Wci, L.Wv, L.deg == 1 ? b : L.X, C.B,
                     enter ? C.dinv : nullptr, (T)C.cr[0], C.D,
                     enter ? first_dst(C, C.X) : nullptr, L.grpc};
}
// log2 of a level's lanes per row (three columns: at least 4 lanes).
template <typename T>
static int level_lg(const LevelDev<T>& L, int NC) {
  int lg = NC == 3 ? 2 : 0;
  while ((1 << lg) < L.lpr) ++lg;
  return lg;
}
template <typename T>
static ResArgs<T> res_args(const LevelDev<T>& L, const T* b, int NC) {
  return ResArgs<T>{L.n, level_lg(L, NC), L.rp, L.ci, L.v, L.v16, L.dci, (T)L.vscale, L.X, b,
                    L.R, L.mask, L.grp};
}

// Fused restriction (into level l + 1's right-hand side and first step) and
// residual of level l after its pre-smoothing, one launch.
template <typename T, int NC>
static void fused_down(const Hier<T>& H, int l, const T* b, Skip sk, hipStream_t s) {
  const LevelDev<T>& L = H.lev[l];
  const DownArgs<T> w = down_args(H, l, b);
  const ResArgs<T> a = res_args(L, b, NC);
  const int nbw = row_blocks(w.n, w.lg), nba = row_blocks(a.n, a.lg);
  if (L.As.off) {
    const int ns = L.nAs, nbs = (ns + NT / 64 - 1) / (NT / 64);
    const SellEpi<T> E{b, nullptr, nullptr, nullptr, 0, 0, (T)L.vscale, L.R, nullptr, L.mask,
                       OutMap(), L.grp};
    if (L.As.dc)
      hipLaunchKernelGGL((transfer_sell_kernel<T, NC, SELL_PLAIN>), dim3(nbw + nbs), dim3(NT),
                         0, s, w, L.As, ns, (const T*)L.X, E, nbw, sk);
    else if constexpr (sizeof(T) == 4)
      hipLaunchKernelGGL((transfer_sell_kernel<T, NC, SELL_PACKED>), dim3(nbw + nbs), dim3(NT),
                         0, s, w, L.As, ns, (const T*)L.X, E, nbw, sk);
    return;
  }
  const dim3 grid(nbw + nba);
  if constexpr (sizeof(T) == 4) {
    if (L.v16) {
      hipLaunchKernelGGL((transfer_kernel<T, NC, true>), grid, dim3(NT), 0, s, w, a, nbw, sk);
      return;
    }
  }
  hipLaunchKernelGGL((transfer_kernel<T, NC, false>), grid, dim3(NT), 0, s, w, a, nbw, sk);
}

template <typename T>
static PostArgs<T> post_args(const LevelDev<T>& L, const T* e, T* y, T* d, OutMap om) {
  return PostArgs<T>{L.n, L.lgQ, L.Qrp, L.Qci, L.Qv, e, L.X, L.R, L.dinv, (T)L.cr[0], y, d,
                     L.mask, om, L.grp};
}

// Prolongation of C.E with level l's post-smoothing into out.
template <typename T, int NC>
static void fused_up(const Hier<T>& H, int l, const T* b, T* out, Skip sk,
                     hipStream_t s, OutMap om) {
  const LevelDev<T>& L = H.lev[l];
  const T* e = H.lev[l + 1].E;
  const bool one = L.deg == 1;
  T* dst = one ? out : L.S1;
  const OutMap dm = one ? om : OutMap();
  if (L.Qs.off) {
    const int ns = L.nQs, nb = (ns + NT / 64 - 1) / (NT / 64);
    const SellEpi<T> E{L.R, L.X, L.dinv, nullptr, 0, (T)L.cr[0], (T)1, dst, one ? nullptr : L.D,
                       L.mask, dm, L.grp};
    if (one)
      hipLaunchKernelGGL((sell_kernel<T, NC, SELL_PLAIN, 6>), dim3(nb), dim3(NT), 0, s, L.Qs, ns,
                         e, E, sk);
    else
      hipLaunchKernelGGL((sell_kernel<T, NC, SELL_PAIR, 7>), dim3(nb), dim3(NT), 0, s, L.Qs, ns,
                         e, E, sk);
  } else {
    const int blocks = (int)((((long long)L.n << L.lgQ) + NT - 1) / NT);
    const PostArgs<T> A = post_args(L, e, dst, one ? nullptr : L.D, dm);
    if (one)
      hipLaunchKernelGGL((post_kernel<T, NC, false>), dim3(blocks), dim3(NT), 0, s, A, sk);
    else
      hipLaunchKernelGGL((post_kernel<T, NC, true>), dim3(blocks), dim3(NT), 0, s, A, sk);
  }
  if (!one) smooth_steps<T, NC>(L, b, L.S1, 1, out, sk, s, om);
}

// Copy of a level's right-hand side: where it is scaled, and where the fused
// restriction reads [x; b] as one buffer.
template <typename T>
static T* vcycle_bcopy(const LevelDev<T>& L, const T* b, T bscale) {
  const bool stacked = L.Wv && L.deg > 1;
  return (bscale != (T)1 || (stacked && b != L.B)) ? L.B : nullptr;
}

template <typename T, int NC>
static void vcycle(const Hier<T>& H, int l, const T* b, T bscale, T* out, Skip sk,
                   hipStream_t s, bool entered = false, K2In<T> k2 = K2In<T>(),
                   OutMap om = OutMap()) {
  const LevelDev<T>& L = H.lev[l];
  if (l == H.nlev - 1) {
    const int blocks = (L.n + NT / 64 - 1) / (NT / 64);
    if (H.cblk && bscale != (T)1) {  // scale into L.B first
      hipLaunchKernelGGL((cheb0_kernel<T, NC>), dim3((int)(((long long)NC * L.n + NT - 1) / NT)),
                         dim3(NT), 0, s, L.n, b, bscale, L.dinv, (T)0, L.D, L.X, L.B, L.mask, sk,
                         L.grp);
      b = L.B;
    }
    if (H.cblk)
      hipLaunchKernelGGL((coarse_blockdiag_kernel<T, NC>), dim3(blocks), dim3(NT), 0, s, L.n,
                         H.cblk, H.coff, H.cioff, H.cinv, b, out, sk, L.grp);
    else
      hipLaunchKernelGGL((coarse_kernel<T, NC>), dim3(blocks), dim3(NT), 0, s, L.n, H.cinv,
                         H.coff, b, out, sk.all, bscale, om, k2);
    return;
  }
  T* bcopy = vcycle_bcopy(L, b, bscale);
  smooth_from_zero<T, NC>(L, b, bscale, bcopy, sk, s, entered, k2);
  const T* bb = bcopy ? bcopy : b;
  const LevelDev<T>& C = H.lev[l + 1];
  const bool enter = l + 1 < H.nlev - 1;
  if (L.Wv) {
    fused_down<T, NC>(H, l, bb, sk, s);
  } else {
    spmm<T, NC, 1>(L, 0, L.X, bb, L.R, nullptr, 0, 0, sk, s);
    // restriction with the coarse level's first smoothing step (its
    // pre-smoothing writes to C.X)
    if (enter)
      spmm<T, NC, 4>(L, 2, L.R, nullptr, C.B, C.D, 0, (T)C.cr[0], sk, s, C.dinv,
                     first_dst(C, C.X));
    else
      spmm<T, NC, 0>(L, 2, L.R, nullptr, C.B, nullptr, 0, 0, sk, s);
  }
  vcycle<T, NC>(H, l + 1, C.B, (T)1, C.E, sk, s, enter);
  if (L.Qv) {
    fused_up<T, NC>(H, l, bb, out, sk, s, om);
  } else {
    spmm<T, NC, 2>(L, 1, C.E, nullptr, L.X, nullptr, 0, 0, sk, s);
    smooth_steps<T, NC>(L, bb, L.X, 0, out, sk, s, om);
  }
}

// Whether precond_apply can take a fused input update (k2): single
// instances, whose first kernels read the input directly.
template <typename T>
static bool k2_fusable(const Precond<T>& P) {
  return !P.pmap;
}

template <typename T>
static EnterArgs<T> enter_args(const Precond<T>& P, const T* r, K2In<T> k2) {
  const LevelDev<T>& L0 = P.p.lev[0];
  return EnterArgs<T>{(long long)P.F * P.nP1, P.nP1, P.F, P.pmap, r + P.nu, L0.B, L0.dinv,
                      (T)L0.cr[0], L0.deg == 1 ? nullptr : L0.D, first_dst(L0, L0.X), L0.mask,
                      L0.grp, k2};
}
template <typename T>
static OutMap pressure_map(const Precond<T>& P) {
  OutMap om;
  if (P.pmap) om.map = P.pinv;
  else { om.nP1 = P.nP1; om.F = P.F; }
  return om;
}

// Pressure block of precond_apply on stream s.
template <typename T>
static void precond_pressure(const Precond<T>& P, const T* r, T* z, Skip sk, hipStream_t s,
                             K2In<T> k2) {
  const long long np = (long long)P.F * P.nP1;
  const int eb = (int)((np + NT - 1) / NT);
  const LevelDev<T>& L0 = P.p.lev[0];
  const OutMap om = pressure_map(P);
  if (P.p.nlev > 1) {
    hipLaunchKernelGGL((p_enter_kernel<T>), dim3(eb), dim3(NT), 0, s, enter_args(P, r, k2), sk);
    vcycle<T, 1>(P.p, 0, L0.B, (T)1, z + P.nu, sk, s, true, K2In<T>(), om);
  } else if (!P.p.cblk) {
    vcycle<T, 1>(P.p, 0, r + P.nu, (T)1, z + P.nu, sk, s, false, k2, om);
  } else {
    hipLaunchKernelGGL((p_gather_map_kernel<T>), dim3(eb), dim3(NT), 0, s, np, P.pmap, r + P.nu,
                       L0.B, sk.all);
    vcycle<T, 1>(P.p, 0, L0.B, (T)1, L0.X, sk, s);
    hipLaunchKernelGGL((p_scatter_map_kernel<T>), dim3(eb), dim3(NT), 0, s, np, P.pmap, L0.X,
                       z + P.nu, sk.all);
  }
}

// The steps of a V-cycle from level l (as vcycle; fused transfers on every
// level but the coarsest).
template <typename T, int NC>
static void cycle_smooth(std::vector<Step<T>>& out, const LevelDev<T>& L, const T* b,
                         const T* cur, T* dst_last, OutMap om) {
  T* bufs[2] = {L.S1, L.S2};
  int flip = 1;
  for (int i = 1; i < L.deg; ++i) {
    const bool last = i == L.deg - 1;
    T* dst = last ? dst_last : bufs[flip];
    if (dst == cur) dst = bufs[flip ^ 1];
    Step<T> S;
    S.kind = STEP_CHEB;
    S.a = res_args(L, b, NC);
    S.a.x = cur;
    S.compact = L.v16 != nullptr;
    S.blocks = row_blocks(L.n, S.a.lg);
    S.dinv = L.dinv;
    S.cd = (T)L.cd[i];
    S.cr = (T)L.cr[i];
    S.d = L.D;
    S.y = dst;
    S.y2 = last ? nullptr : L.D;
    if (last) S.om = om;
    out.push_back(S);
    cur = dst;
    flip ^= 1;
  }
}
template <typename T, int NC>
static void cycle_steps(std::vector<Step<T>>& out, const Hier<T>& H, int l, const T* b, T bscale,
                        T* z, bool entered, K2In<T> k2, OutMap om) {
  const LevelDev<T>& L = H.lev[l];
  Step<T> S;
  if (l == H.nlev - 1) {
    S.kind = H.cblk ? STEP_BLOCKS : STEP_DENSE;
    S.blocks = (L.n + NT / 64 - 1) / (NT / 64);
    S.n = L.n;
    S.cinv = H.cinv;
    S.blk = H.cblk;
    S.off = H.coff;
    S.ioff = H.cioff;
    S.b = b;
    S.y = z;
    S.scale = bscale;
    S.om = om;
    S.k2 = k2;
    S.a.grp = L.grp;
    out.push_back(S);
    return;
  }
  T* bcopy = vcycle_bcopy(L, b, bscale);
  T* first = first_dst(L, L.X);
  if (!entered) {
    S.kind = STEP_FIRST;
    S.blocks = (int)(((long long)NC * L.n + NT - 1) / NT);
    S.n = L.n;
    S.b = b;
    S.scale = bscale;
    S.dinv = L.dinv;
    S.cr = (T)L.cr[0];
    S.d = L.deg == 1 ? nullptr : L.D;
    S.y = first;
    S.bcopy = bcopy;
    S.a.mask = L.mask;
    S.a.grp = L.grp;
    S.k2 = k2;
    out.push_back(S);
  }
  const T* bb = bcopy ? bcopy : b;
  cycle_smooth<T, NC>(out, L, bb, first, L.X, OutMap());
  S = Step<T>();
  S.kind = STEP_DOWN;
  S.w = down_args(H, l, bb);
  S.a = res_args(L, bb, NC);
  S.compact = L.v16 != nullptr;
  S.nbw = row_blocks(S.w.n, S.w.lg);
  S.blocks = S.nbw + row_blocks(L.n, S.a.lg);
  out.push_back(S);
  const LevelDev<T>& C = H.lev[l + 1];
  cycle_steps<T, NC>(out, H, l + 1, C.B, (T)1, C.E, l + 1 < H.nlev - 1, K2In<T>(), OutMap());
  const bool one = L.deg == 1;
  S = Step<T>();
  S.kind = STEP_POST;
  S.pair = !one;
  S.p = post_args(L, C.E, one ? z : L.S1, one ? nullptr : L.D, one ? om : OutMap());
  S.blocks = row_blocks(L.n, L.lgQ);
  out.push_back(S);
  if (!one) cycle_smooth<T, NC>(out, L, bb, L.S1, z, om);
}

// Whether both cycles can run as steps, and should: every level below the
// coarsest has fused transfers and none is sliced (the sliced levels are
// the large ones, where the second stream pays; between 50,000 and 120,000 P2
// rows either is within 10%, the figures are at levels.py SLICE_ROWS).
template <typename T>
static bool joint_ok(const Precond<T>& P) {
  for (const Hier<T>* H : {&P.u, &P.p}) {
    for (int l = 0; l + 1 < H->nlev; ++l)
      if (!H->lev[l].Wv || !H->lev[l].Qv || H->lev[l].As.off || H->lev[l].Qs.off) return false;
    if (H->nlev == 1 && H->cblk) return false;
  }
  return true;
}

template <typename T>
static void precond_joint(const Precond<T>& P, const T* r, T* z, Skip sk, hipStream_t s,
                          K2In<T> ku, K2In<T> kp) {
  std::vector<Step<T>> u, p;
  u.reserve(32);
  p.reserve(32);
  cycle_steps<T, 3>(u, P.u, 0, r, (T)(1.0 / P.u.scale), z, false, ku, OutMap());
  const OutMap om = pressure_map(P);
  if (P.p.nlev > 1) {
    Step<T> S;
    S.kind = STEP_ENTER;
    S.e = enter_args(P, r, kp);
    S.blocks = (int)((S.e.np + NT - 1) / NT);
    p.push_back(S);
    cycle_steps<T, 1>(p, P.p, 0, P.p.lev[0].B, (T)1, z + P.nu, true, K2In<T>(), om);
  } else {
    cycle_steps<T, 1>(p, P.p, 0, r + P.nu, (T)1, z + P.nu, false, kp, om);
  }
  const Step<T> none;
  for (size_t i = 0; i < u.size() || i < p.size(); ++i) {
    const Step<T>& a = i < u.size() ? u[i] : none;
    const Step<T>& b = i < p.size() ? p[i] : none;
    hipLaunchKernelGGL((joint_kernel<T>), dim3(a.blocks + b.blocks), dim3(NT), 0, s, a, b, sk);
  }
}

// z = M^-1 r; with k2 (k2_fusable only) r is first made as k2 describes.
template <typename T>
static void precond_apply(const Precond<T>& P, const T* r, T* z, Skip sk, hipStream_t s,
                          const K2In<T>* k2 = nullptr) {
  K2In<T> ku, kp;
  if (k2 && k2->y) {
    ku = *k2;
    kp = K2In<T>{k2->y + P.nu, k2->r2o + P.nu, k2->r + P.nu, k2->alfa, k2->beta};
  }
  if (P.joint) {
    precond_joint(P, r, z, sk, s, ku, kp);
    return;
  }
  hipStream_t sp = s;
  if (P.ps) {                      // pressure blocks on the second stream
    (void)hipEventRecord(P.ev_fork, s);
    (void)hipStreamWaitEvent(P.ps, P.ev_fork, 0);
    sp = P.ps;
  }
  vcycle<T, 3>(P.u, 0, r, (T)(1.0 / P.u.scale), z, sk, s, false, ku);
  precond_pressure(P, r, z, sk, sp, kp);
  if (P.ps) {
    (void)hipEventRecord(P.ev_join, P.ps);
    (void)hipStreamWaitEvent(s, P.ev_join, 0);
  }
}
template <typename T>
static void precond_apply(const Precond<T>& P, const T* r, T* z, const int* skip,
                          hipStream_t s) {
  Skip sk;
  sk.all = skip;
  precond_apply(P, r, z, sk, s);
}

// Lanes per row of the levels' SpMMs from an MpetTuning table (0 keeps).
static bool lpr_ok(int v) {
  return v == 0 || v == 1 || v == 2 || v == 4 || v == 8 || v == 16 || v == 32 || v == 64;
}
static bool tuning_ok(const MpetTuning* t) {
  if (!t) return false;
  for (int l = 0; l < MPET_MAXLEV; ++l)
    for (int k = 0; k < 3; ++k)
      if (!lpr_ok(t->u_lpr[l][k]) || !lpr_ok(t->p_lpr[l][k])) return false;
  return true;
}
template <typename T>
static void set_hier_lpr(Hier<T>& H, const int32_t (*lpr)[3]) {
  for (int l = 0; l < H.nlev && l < MPET_MAXLEV; ++l) {
    if (lpr[l][0] > 0) H.lev[l].lpr = lpr[l][0];
    if (lpr[l][1] > 0) H.lev[l].lprP = lpr[l][1];
    if (lpr[l][2] > 0) {
      H.lev[l].lprR = lpr[l][2];
      // of the fused restriction where there is one (three columns: one lane
      // per component)
      int lg = H.NC == 3 ? 2 : 0;
      while ((1 << lg) < lpr[l][2]) ++lg;
      H.lev[l].lgW = lg;
    }
  }
}
template <typename T>
static void set_precond_tuning(Precond<T>& P, const MpetTuning* t) {
  set_hier_lpr(P.u, t->u_lpr);
  set_hier_lpr(P.p, t->p_lpr);
}

template <typename T>
static int alloc_dev(std::vector<void*>& allocs, T** p, size_t count) {
  void* q = nullptr;
  if (hipMalloc(&q, sizeof(T) * (count ? count : 1)) != hipSuccess) {
    mpet_set_error("hipMalloc failed (out of device memory)");
    return ERR_OOM;
  }
  allocs.push_back(q);
  *p = (T*)q;
  return OK;
}

static inline int slice_count(const MpetSlices& s, int n) {
  return s.count > 0 ? s.count : (n + 63) / 64;
}
template <typename T>
static int build_hier(std::vector<void*>& allocs, const MpetHierDesc* d, int NC,
                      Hier<T>& H) {
  H.nlev = d->nlev;
  H.deg = d->degree;
  H.NC = NC;
  H.scale = d->scale != 0.0 ? d->scale : 1.0;
  if (H.nlev < 1 || H.nlev > MAXLEV || H.deg < 1 || H.deg > MAXDEG) {
    mpet_set_error("invalid hierarchy description");
    return ERR_INVALID;
  }
  for (int l = 0; l < H.nlev; ++l) {
    const MpetAmgLevelDesc& ld = d->lev[l];
    LevelDev<T>& L = H.lev[l];
    L.n = ld.n;
    L.nc = ld.nc;
    L.rp = ld.A_rp; L.ci = ld.A_ci; L.v = (const T*)ld.A_v; L.dinv = (const T*)ld.dinv;
    L.Prp = ld.P_rp; L.Pci = ld.P_ci; L.Pv = (const T*)ld.P_v;
    L.Rrp = ld.R_rp; L.Rci = ld.R_ci; L.Rv = (const T*)ld.R_v;
    L.mask = l == 0 ? d->mask0 : nullptr;
    L.grp = ld.grp;
    L.v16 = (const __half*)ld.A_v16;
    L.dci = ld.A_dci;
    L.vscale = ld.A_vscale != 0.0 ? ld.A_vscale : 1.0;
    L.lpr = ld.lpr ? ld.lpr : 8;
    L.lprP = ld.lprP ? ld.lprP : 4;
    L.lprR = ld.lprR ? ld.lprR : 8;
    L.deg = d->level_degree[l] > 0 ? d->level_degree[l] : H.deg;
    if (L.deg > MAXDEG) {
      mpet_set_error("invalid hierarchy description");
      return ERR_INVALID;
    }
    double lmax = ld.rho * d->eig_safety;
    chebyshev(lmax / d->eig_ratio, lmax, L.deg, L.cd, L.cr);
    size_t m = (size_t)NC * L.n;
    int rc;
    // X and B adjacent: the fused restriction of several smoothing steps
    // reads them as one vector
    if ((rc = alloc_dev(allocs, &L.X, 2 * m)) ||
        (rc = alloc_dev(allocs, &L.R, m)) || (rc = alloc_dev(allocs, &L.E, m)) ||
        (rc = alloc_dev(allocs, &L.S1, m)) || (rc = alloc_dev(allocs, &L.S2, m)) ||
        (rc = alloc_dev(allocs, &L.D, m)))
      return rc;
    L.B = L.X + m;
    if (ld.A_s.off) {
      if (!ld.A_s.base || !ld.A_s.row || !ld.A_sv || (!ld.A_s.dc && sizeof(T) != 4)) {
        mpet_set_error("invalid hierarchy description (sliced level)");
        return ERR_INVALID;
      }
      L.As = Sell<T>{ld.A_s.off, ld.A_s.base, ld.A_s.row, ld.A_s.dc, ld.A_sv};
      L.nAs = slice_count(ld.A_s, L.n);
    }
    if (l + 1 < H.nlev && (ld.W_v || ld.Q_v)) {
      const int lo = NC == 3 ? 2 : 0;
      if ((ld.W_v && (!ld.W_rp || !ld.W_ci || ld.lgW < lo || ld.lgW > 6)) ||
          (ld.Q_v && !ld.Q_s.off && (!ld.Q_rp || !ld.Q_ci || ld.lgQ < lo || ld.lgQ > 6)) ||
          (ld.Q_v && ld.Q_s.off && (!ld.Q_s.base || !ld.Q_s.row || !ld.Q_s.dc))) {
        mpet_set_error("invalid hierarchy description (fused transfers)");
        return ERR_INVALID;
      }
      L.Wrp = ld.W_rp; L.Wci = ld.W_ci; L.Wv = (const T*)ld.W_v;
      L.Qrp = ld.Q_rp; L.Qci = ld.Q_ci; L.Qv = (const T*)ld.Q_v;
      L.lgW = ld.lgW;
      L.lgQ = ld.lgQ;
      if (ld.Q_s.off) {
        L.Qs = Sell<T>{ld.Q_s.off, ld.Q_s.base, ld.Q_s.row, ld.Q_s.dc, ld.Q_v};
        L.nQs = slice_count(ld.Q_s, L.n);
      }
    }
  }
  for (int l = 0; l + 1 < H.nlev; ++l) H.lev[l].grpc = H.lev[l + 1].grp;
  H.cinv = (const T*)d->coarse_inv;
  H.cblk = d->coarse_blk;
  H.coff = d->coarse_blk ? d->coarse_off : d->coarse_rng;
  H.cioff = d->coarse_ioff;
  return OK;
}

template <typename T>
static int build_precond(std::vector<void*>& allocs, long long nu, const MpetPrecDesc* d,
                         Precond<T>& P) {
  int rc;
  if ((rc = build_hier(allocs, &d->u, 3, P.u)) || (rc = build_hier(allocs, &d->p, 1, P.p)))
    return rc;
  P.nP1 = d->nP1;
  P.F = d->F;
  P.nu = nu;
  P.pmap = d->pmap;
  if (P.u.lev[0].n * 3ll != nu || (long long)P.p.lev[0].n != (long long)P.F * P.nP1) {
    mpet_set_error("preconditioner sizes do not match the operator");
    return ERR_INVALID;
  }
  P.joint = joint_ok(P);
  if (P.pmap) {                    // the batch's pressure order, inverted
    const int np = P.F * P.nP1;
    if ((rc = alloc_dev(allocs, &P.pinv, (size_t)np))) return rc;
    hipLaunchKernelGGL((invert_map_kernel_t<int>), dim3((np + NT - 1) / NT), dim3(NT), 0, 0, np, P.pmap,
                       P.pinv);
    HIPCHK(hipDeviceSynchronize());
  }
  return OK;
}

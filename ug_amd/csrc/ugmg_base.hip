// Base-level set-up on the device: the band LU of EXPreProcess
// (EXDecomposeMatrixDOUBLE, gm/evm.cc:1400-1418, or EXDecomposeMatrixFLOAT,
// 1355-1373, for ex $f: no pivoting, a zero pivot fails) and the explicit
// inverse, one column per unit vector pushed through EXApplyLUDOUBLE
// (gm/evm.cc:1493-1510; EXApplyLUFLOAT, 1448-1466, is the same double
// arithmetic on the FLOAT factors).
//
// Every value is formed by the same operations in the same order as the host
// loops of build_base, with products and differences rounded separately (no
// contraction into fused multiply-adds), so the factors and the inverse are
// bit-identical to the host's.
//
// Band storage is UG's EX_MAT (gm/evm.h:392): entry (i, j) at
// band[2 bw i + j], |i - j| <= bw, rows and columns in band positions (BFS
// order, b consecutive scalar unknowns per vector).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ugmg_kernels.h"

namespace ugmg {

namespace {

__device__ __forceinline__ double &bandref(double *m, int bw, int i, int j) {
  return m[2 * (size_t)bw * i + j];
}

// Pivot step i (i < n - 1): a_jk <- a_jk - (a_ji / a_ii) a_ik for j, k in
// (i, min(i + bw, n - 1)].  The same launch stores the multipliers of step
// i - 1 into column i - 1, which no thread of step i reads.  Step n - 1 only
// stores the last multipliers.  A zero pivot sets *failed and leaves the
// band as it is (the host loop stops there).
// R = float: EXDecomposeMatrixFLOAT (gm/evm.cc:1355-1373) on a band of
// FLOAT values held as doubles: every operation in float arithmetic, the
// results stored back exactly.
template <typename R>
__global__ __launch_bounds__(256) void k_band_lu_step(double *__restrict__ band, int bw, int n,
                                                      int i, int *__restrict__ failed) {
#pragma clang fp contract(off)
  if (*failed) return;
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i < n - 1) {
    const R d = (R)bandref(band, bw, i, i);
    if (d == (R)0) {
      if (idx == 0) *failed = 1;
      return;
    }
    const int jmax = min(i + bw, n - 1);
    const int m = jmax - i;
    if (idx < (long long)m * m) {
      const int j = i + 1 + (int)(idx / m);
      const int k = i + 1 + (int)(idx % m);
      const R f = (R)bandref(band, bw, j, i) / d;
      const R p = f * (R)bandref(band, bw, i, k);
      bandref(band, bw, j, k) = (double)((R)bandref(band, bw, j, k) - p);
    }
  }
  if (i > 0) {
    const int q = i - 1;
    const int mp = min(q + bw, n - 1) - q;
    if (idx < mp) {
      const int j = q + 1 + (int)idx;
      bandref(band, bw, j, q) = (double)((R)bandref(band, bw, j, q) / (R)bandref(band, bw, q, q));
    }
  }
}

// Blocked LU.  The step kernel above costs one launch per pivot (4913 of
// them, 6.3 us each, for a 17^3 base level, each touching bw^2 entries).  A panel of kNb pivots is two launches instead: k_band_panel
// eliminates inside the panel's columns and rows, k_band_trail subtracts the
// panel's kNb terms from the entries behind it.  An entry still receives its
// terms one by one in ascending pivot order, each product and difference
// rounded by itself, so the factors are the step kernel's bit for bit.
// 17^3 base level (n 4913, bw 907): 31 -> 5.1 ms (24 us a panel, 9 us behind it).
constexpr int kNb = 32;
constexpr size_t kLdsBytes = 160 * 1024;

// the value of v in lane s (a constant of the unrolled loops)
__device__ __forceinline__ float lane_value(float v, int s) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), s));
}
__device__ __forceinline__ double lane_value(double v, int s) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)b, s);
  const long long hi = __builtin_amdgcn_readlane((int)(b >> 32), s);
  return __longlong_as_double((hi << 32) | lo);
}

// Panel of pivots p .. p + kNb - 1 (kNb <= bw).  Every workgroup, one wave,
// eliminates the panel's kNb x kNb diagonal block for itself: lane r holds
// row r, pivot rows are passed on by readlane.  Its 64 threads then take one
// row each below the block (mr rows) or one column each right of it (mc
// columns, the workgroups behind) through the block's factors in LDS.  Workgroup 0
// leaves the factored block in `block`; the next launch stores it, when
// nobody reads the band's copy any more.  Bound by the chain of kNb pivots.
template <typename R>
__global__ __launch_bounds__(64) void k_band_panel(double *__restrict__ band, int bw, int n, int p,
                                                   int mr, int mc, R *__restrict__ block,
                                                   int *__restrict__ failed) {
#pragma clang fp contract(off)
  __shared__ R f[kNb][kNb];
  if (*failed) return;
  const int t = threadIdx.x;
  const int np = min(kNb, n - p);        // columns and rows of the panel
  {
    R a[kNb];
    const int r = min(t, kNb - 1);
#pragma unroll
    for (int s = 0; s < kNb; ++s) a[s] = r < np && s < np ? (R)bandref(band, bw, p + r, p + s) : (R)1;
#pragma unroll
    for (int s = 0; s < kNb - 1; ++s) {
      const R d = lane_value(a[s], s);
      if (s < np - 1 || p + kNb < n) {   // a pivot below n - 1
        if (d == (R)0) {
          if (blockIdx.x == 0 && t == 0) *failed = 1;
          return;
        }
        const bool below = r > s && r < np;
        const R m = a[s] / d;
        a[s] = below ? m : a[s];
#pragma unroll
        for (int k = s + 1; k < kNb; ++k) {
          const R q = m * lane_value(a[k], s);
          const R v = a[k] - q;
          a[k] = below ? v : a[k];
        }
      }
    }
    // the last pivot has no row below it in the block, but behind it
    if (p + kNb < n && lane_value(a[kNb - 1], kNb - 1) == (R)0) {
      if (blockIdx.x == 0 && t == 0) *failed = 1;
      return;
    }
    if (t < kNb)
#pragma unroll
      for (int s = 0; s < kNb; ++s) {
        f[t][s] = a[s];
        if (blockIdx.x == 0) block[t * kNb + s] = a[s];
      }
  }
  __syncthreads();
  const int nrow = (mr + 63) / 64;
  if ((int)blockIdx.x < nrow) {
    const int j = p + kNb + 64 * blockIdx.x + t;   // row j: pivots i >= j - bw
    if (j >= p + kNb + mr) return;
    const int first = j - bw - p;
    R a[kNb];
#pragma unroll
    for (int s = 0; s < kNb; ++s) a[s] = s >= first ? (R)bandref(band, bw, j, p + s) : (R)0;
#pragma unroll
    for (int s = 0; s < kNb; ++s)
      if (s >= first) {
        const R m = a[s] / f[s][s];
        a[s] = m;
#pragma unroll
        for (int k = s + 1; k < kNb; ++k) {
          const R q = m * f[s][k];
          a[k] = a[k] - q;
        }
      }
#pragma unroll
    for (int s = 0; s < kNb; ++s)
      if (s >= first) bandref(band, bw, j, p + s) = (double)a[s];
    return;
  }
  const int k = p + kNb + 64 * ((int)blockIdx.x - nrow) + t;
  if (k >= p + kNb + mc) return;
  const int first = k - bw - p;          // the column's first row in the band
  R u[kNb];
#pragma unroll
  for (int s = 0; s < kNb; ++s) u[s] = s >= first ? (R)bandref(band, bw, p + s, k) : (R)0;
#pragma unroll
  for (int s = 0; s < kNb; ++s)
    if (s >= first)
#pragma unroll
      for (int r = s + 1; r < kNb; ++r) {
        const R q = f[r][s] * u[s];
        u[r] = u[r] - q;
      }
#pragma unroll
  for (int s = 1; s < kNb; ++s)
    if (s >= first) bandref(band, bw, p + s, k) = (double)u[s];
}

// Stores the panel's diagonal block, and
// a_jk -= sum of the panel's terms l_ji u_ik with both factors in the band
// (i >= max(j, k) - bw), i ascending, for the mr rows j and the mc columns k
// behind the panel that its pivots reach: one workgroup per 32 x 32 entries, four rows per thread.
template <typename R>
__global__ __launch_bounds__(256) void k_band_trail(double *__restrict__ band, int bw, int n, int p, int mr, int mc,
                                                    const R *__restrict__ block,
                                                    const int *__restrict__ failed) {
#pragma clang fp contract(off)
  __shared__ R l[32][kNb + 1], u[kNb][32];
  if (*failed) return;
  if (blockIdx.x == 0 && blockIdx.y == 0) {
    const int np = min(kNb, n - p);
    for (int q = threadIdx.x; q < kNb * kNb; q += 256)
      if (q / kNb < np && q % kNb < np) bandref(band, bw, p + q / kNb, p + q % kNb) = (double)block[q];
    if (mr <= 0 || mc <= 0) return;
  }
  const int j0 = p + kNb + 32 * blockIdx.y, k0 = p + kNb + 32 * blockIdx.x;
  const int jlast = p + kNb + mr - 1, klast = p + kNb + mc - 1;
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int q = y + 8 * r;
    const int j = j0 + q, i = p + x;     // row j, pivot column i
    l[q][x] = j <= jlast && j - i <= bw ? (R)bandref(band, bw, j, i) : (R)0;
    const int k = k0 + x, iu = p + q;    // pivot row iu, column k
    u[q][x] = k <= klast && k - iu <= bw ? (R)bandref(band, bw, iu, k) : (R)0;
  }
  __syncthreads();
  const int k = k0 + x;
  R a[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int j = j0 + y + 8 * r;
    a[r] = j <= jlast && k <= klast ? (R)bandref(band, bw, j, k) : (R)0;
  }
  if (max(j0, k0) + 31 - bw <= p) {      // every pivot of the panel reaches the tile
#pragma unroll
    for (int i = 0; i < kNb; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const R q = l[y + 8 * r][i] * u[i][x];
        a[r] = a[r] - q;
      }
  } else {
#pragma unroll
    for (int i = 0; i < kNb; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const R q = l[y + 8 * r][i] * u[i][x];
        const R d = a[r] - q;
        a[r] = i >= max(j0 + y + 8 * r, k) - bw - p ? d : a[r];
      }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int j = j0 + y + 8 * r;
    if (j <= jlast && k <= klast) bandref(band, bw, j, k) = (double)a[r];
  }
}

// acc - sum_{k0 <= k < k1} row[k] x[k ldx], subtracting term by term in
// ascending k (each product rounded, then the difference), in chunks of
// 64 terms.  The band row is wave-uniform: lane j loads row[k + j] in one
// coalesced load and each term takes its factor with readlane, while the
// 64 column entries of a chunk are loaded before any of them is used, so a
// chunk costs one memory round trip; only the subtractions form the
// dependent chain.
template <bool TAIL>
__device__ __forceinline__ double band_chunk_sub(int llo, int lhi, const double *__restrict__ x,
                                                 size_t ldx, int k, int k1, double acc) {
#pragma clang fp contract(off)
  constexpr int kCh = 64;
  double xv[kCh];
#pragma unroll
  for (int j = 0; j < kCh; ++j) xv[j] = x[(size_t)(TAIL ? min(k + j, k1 - 1) : k + j) * ldx];
  // keep the scheduler from sinking each load next to its use
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < kCh; ++j) {
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane(llo, j);
    const long long hi = __builtin_amdgcn_readlane(lhi, j);
    const double lj = __longlong_as_double((hi << 32) | lo);
    const double p = lj * xv[j];
    const double t = acc - p;
    // terms past k1 (last chunk only) are discarded by a select, not a
    // branch, which would let the compiler sink each load into its block
    acc = (!TAIL || k + j < k1) ? t : acc;
  }
  return acc;
}

__device__ __forceinline__ double band_row_sub(const double *__restrict__ row,
                                               const double *__restrict__ x, size_t ldx, int k0,
                                               int k1, double acc) {
  constexpr int kCh = 64;
  const int lane = threadIdx.x & 63;
  int k = k0;
  for (; k + kCh <= k1; k += kCh) {
    const long long lb = __double_as_longlong(row[k + lane]);
    acc = band_chunk_sub<false>((int)lb, (int)(lb >> 32), x, ldx, k, k1, acc);
  }
  if (k < k1) {
    const long long lb = __double_as_longlong(row[min(k + lane, k1 - 1)]);
    acc = band_chunk_sub<true>((int)lb, (int)(lb >> 32), x, ldx, k, k1, acc);
  }
  return acc;
}

// Columns c0 .. c0 + 63 of the inverse in band positions, one lane per
// column c (the unit vector e_c).  The 64 columns of one wave are stored
// row by row in one contiguous panel (entry (k, c) at
// X[(c / 64) n 64 + 64 k + c % 64]), so the rows a substitution step reads
// are a few consecutive pages rather than one page per row.  Forward
// substitution from row c0 + 1 (rows below a lane's own c hold zeros, so
// the extra terms of lanes with c > c0 subtract zeros and change nothing),
// then backward substitution over every row, as EXApplyLUDOUBLE.
__global__ __launch_bounds__(64) void k_band_inverse(const double *__restrict__ band, int bw, int n,
                                                     double *__restrict__ X,
                                                     const int *__restrict__ failed) {
#pragma clang fp contract(off)
  if (*failed) return;
  const int c0 = blockIdx.x * 64;
  const int c = c0 + (int)threadIdx.x;
  const size_t ldx = 64;
  double *x = X + (size_t)blockIdx.x * n * 64 + threadIdx.x;
  for (int k = 0; k < n; ++k) x[(size_t)k * ldx] = k == c ? 1.0 : 0.0;
  for (int i = c0 + 1; i < n; ++i)
    x[(size_t)i * ldx] = band_row_sub(band + 2 * (size_t)bw * i, x, ldx, max(i - bw, c0), i,
                                      x[(size_t)i * ldx]);
  for (int i = n - 1; i >= 0; --i) {
    const double *__restrict__ Ui = band + 2 * (size_t)bw * i;
    const double acc = band_row_sub(Ui, x, ldx, i + 1, min(i + bw, n - 1) + 1, x[(size_t)i * ldx]);
    x[(size_t)i * ldx] = acc / Ui[i];
  }
}

// The same substitutions with the window of solution rows in LDS.  NC
// columns per workgroup of four waves, W = bw rounded up to 16 rows in a ring
// (row k in slot k mod W, so runs of 16 rows starting at a multiple of 16 are
// contiguous).
//
// Forward, 16 rows at a time: every wave takes four rows through the terms
// of the rows before the block (two rows per half wave, sharing the reads of
// the ring), then one wave finishes the block's triangle in registers.
// Backward the order of the terms (ascending from the row's own successor)
// makes each column one chain: one wave walks it, 16 terms a time with the
// operands of the next 16 on their way from LDS and the next row of U on its
// way from memory.  That wave bounds the kernel: 29 cycles a term, of which
// the dependent subtraction takes 8; the reads and products that it issues
// besides take the rest, while the other three waves are done.
// Terms a chunk covers beyond the row's range are discarded by a select.
//
// Elimination fills a row only from its first to its last column of the
// matrix' own envelope: lfirst[q] is the first column of rows 16 q .. 16 q +
// 15 of L, ulast[i] the last of row i of U (about half of bw on the average
// in BFS order, whose level sets grow and shrink); the terms outside are
// zeros.  (Zero times a solution entry: where one overflowed, the host's
// substitutions give NaN in more places than these.)
// 17^3 base level (n 4913, bw 907), 246 workgroups of 20 columns: 175 -> 43 ms
// (forward 7, backward 36).
constexpr int kCh = 16;

// One chunk of the backward chain: acc minus the products p, whose places
// take the next chunk's products u x, whose places take the operands of the
// chunk after that.  So a product is ready a chunk before its subtraction
// and its operands were asked for a chunk before that.  The empty asm and
// the barriers keep the compiler from pairing each product with its own subtraction, from
// gathering the reads and from joining two reads of the ring to one
// ds_read2_b64 (which takes about 20 cycles, a ds_read_b64 4).
// PART: only the terms lo <= j < hi are taken.
template <int NC, bool PART>
__device__ __forceinline__ double band_step(double acc, double (&p)[kCh], double (&x)[kCh],
                                            double2 (&u)[kCh / 2], const double *ring,
                                            const double2 *f, int lo = 0, int hi = kCh) {
#pragma clang fp contract(off)
#pragma unroll
  for (int j = 0; j < kCh; ++j) {
    const double d = acc - p[j];
    acc = !PART || (j >= lo && j < hi) ? d : acc;
    p[j] = (j & 1 ? u[j / 2].y : u[j / 2].x) * x[j];
    asm volatile("" : "+v"(acc), "+v"(p[j]));   // both are formed here
    __builtin_amdgcn_sched_barrier(0);
    x[j] = ring[j * NC];
    if (j & 1) u[j / 2] = f[j / 2];
    __builtin_amdgcn_sched_barrier(0);
  }
  return acc;
}

// rows of the ring
__host__ __device__ inline int band_ring(int bw) { return bw < kCh ? kCh : (bw + kCh - 1) / kCh * kCh; }
constexpr int kKc = 64;                  // columns of L staged at a time
constexpr int kKs = kKc + 2;             // (the rows of a wave's halves on other banks)
constexpr int kStage = 16;               // a row of U in 64 kStage doubles

template <int NC>
__global__ __launch_bounds__(256) void k_band_inverse_lds(const double *__restrict__ band, int bw, int n,
                                                          const int *__restrict__ lfirst,
                                                          const int *__restrict__ ulast,
                                                          double *__restrict__ X,
                                                          const int *__restrict__ failed) {
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  static_assert(NC <= 32, "a half wave holds the columns");
  if (*failed) return;
  const int W = band_ring(bw);
  double *ring = lds;                    // W x NC
  double *fac = lds + (size_t)W * NC;    // 2 x kCh x kKs of L, then 2 rows of U
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int col = min(lane & 31, NC - 1);
  const int c0 = blockIdx.x * NC, c = c0 + col;
  // column c at X[(c / 64) n 64 + 64 k + c % 64]
  double *x = X + (size_t)(c >> 6) * n * 64 + (c & 63);

  // rows i0 .. i0 + 15 of L from column k0 (the first one of the block's
  // first row, or c0) to the block's own triangle, kKc columns a time, the
  // next ones on their way while these are used
  const int ibeg = c0 & ~(kCh - 1);
  auto first = [&](int i0) { return max(lfirst[i0 / kCh], ibeg) & ~(kCh - 1); };
  double st4[4];
  auto fetch_l = [&](int i0, int k) {
    const int i = min(i0 + (tid >> 4), n - 1);
    const double *row = band + 2 * (size_t)bw * i;
#pragma unroll
    for (int q = 0; q < 4; ++q) st4[q] = row[min(max(k + (tid & 15) * 4 + q, i - bw), i)];
  };
  fetch_l(ibeg, ibeg);
  int buf = 0;
  for (int i0 = ibeg; i0 < n; i0 += kCh) {
    const int k0 = first(i0);
    constexpr int NR = 2;                // rows of a half wave
    const int r0 = 4 * wave + 2 * (lane >> 5);
    double acc[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] = i0 + r0 + r == c ? 1.0 : 0.0;
    int slot = k0 % W;
    const double *tri = fac;
    for (int kc = k0; kc < i0 + kCh; kc += kKc) {
      double *fb = fac + buf * (kCh * kKs);
      buf ^= 1;
#pragma unroll
      for (int q = 0; q < 4; ++q) fb[(tid >> 4) * kKs + (tid & 15) * 4 + q] = st4[q];
      __syncthreads();
      if (kc + kKc < i0 + kCh) fetch_l(i0, kc + kKc);
      else if (i0 + kCh < n) fetch_l(i0 + kCh, first(i0 + kCh));
      tri = fb + (i0 - kc);              // (of the last columns: the triangle)
      for (int k = kc; k < min(kc + kKc, i0); k += kCh) {
        const double *xr = ring + (size_t)slot * NC + col;
        slot += kCh;
        if (slot == W) slot = 0;
        double xv[kCh];
#pragma unroll
        for (int j = 0; j < kCh; ++j) xv[j] = xr[j * NC];
        double fv[NR][kCh];
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int j = 0; j < kCh; ++j) fv[r][j] = fb[(r0 + r) * kKs + (k - kc) + j];
#pragma unroll
        for (int r = 0; r < NR; ++r)
#pragma unroll
          for (int j = 0; j < kCh; ++j) fv[r][j] = fv[r][j] * xv[j];
        __builtin_amdgcn_sched_barrier(0);
        // the last row of the block sets in at i0 + 15 - bw
        if (k < i0 + kCh - 1 - bw) {
#pragma unroll
          for (int j = 0; j < kCh; ++j)
#pragma unroll
            for (int r = 0; r < NR; ++r) {
              const double d = acc[r] - fv[r][j];
              acc[r] = j >= i0 + r0 + r - bw - k ? d : acc[r];
            }
        } else {
#pragma unroll
          for (int j = 0; j < kCh; ++j)
#pragma unroll
            for (int r = 0; r < NR; ++r) acc[r] = acc[r] - fv[r][j];
        }
      }
    }
    __syncthreads();                     // the ring was read
    double *blk = ring + (size_t)(i0 % W) * NC + col;
#pragma unroll
    for (int r = 0; r < NR; ++r) blk[(r0 + r) * NC] = acc[r];
    __syncthreads();
    if (wave == 0) {
      double v[kCh];
#pragma unroll
      for (int r = 0; r < kCh; ++r) v[r] = blk[r * NC];
#pragma unroll
      for (int s = 0; s < kCh; ++s)
#pragma unroll
        for (int r = s + 1; r < kCh; ++r) {
          const double q = tri[r * kKs + s] * v[s];
          const double d = v[r] - q;
          v[r] = r - s <= bw ? d : v[r];
        }
#pragma unroll
      for (int r = 0; r < kCh; ++r) {
        blk[r * NC] = v[r];
        if (i0 + r < n && c < n) x[(size_t)(i0 + r) * 64] = v[r];
      }
    }
    // (the next block reads these rows after its first barrier)
  }
  __syncthreads();
  if (wave != 0) return;

  // rows before c0 are zeros of the forward substitution, the others come
  // from memory, where this wave wrote them
  double st[kStage];
  const bool live = c < n;
  const int nst = (bw + 2 * kCh + 63) / 64;
  // vector loads of what every lane shares: a scalar load in flight would
  // make each wait for LDS a wait for it
  int zero;
  asm("v_mov_b32 %0, 0" : "=v"(zero));
  auto staged = [&](int i, int last) { return (last - ((i + 1) & ~(kCh - 1)) + 64) / 64; };
  auto fetch = [&](int i, int last, double &y, double &d) {
    if (i < 0) return;
    const double *row = band + 2 * (size_t)bw * i;
    const int k = ((i + 1) & ~(kCh - 1)) + lane, m = staged(i, last);
#pragma unroll
    for (int j = 0; j < kStage; ++j)
      if (j < m) st[j] = row[max(min(k + 64 * j, last), i)];
    d = row[i + zero];
    y = i >= c0 && live ? x[(size_t)i * 64] : 0.0;
  };
  double y = 0.0, d = 1.0;
  int last = ulast[n - 1], vnext = ulast[max(n - 2, 0) + zero];
  fetch(n - 1, last, y, d);
  for (int i = n - 1; i >= 0; --i) {
    double *u = fac + (i & 1) * (size_t)(64 * nst);
    const int m = staged(i, last);
#pragma unroll
    for (int j = 0; j < kStage; ++j)
      if (j < m) u[lane + 64 * j] = st[j];
    double acc = y;
    const double di = d;
    const int ka = (i + 1) & ~(kCh - 1), ke = last + 1;
    last = __builtin_amdgcn_readfirstlane(vnext);
    vnext = ulast[max(i - 2, 0) + zero];
    fetch(i - 1, last, y, d);
    int slot = ka % W;
    const double2 *f = (const double2 *)u;
    // the first chunk sets in at i + 1, the last ends at ke; operands of up
    // to two more chunks are read (within LDS) and not used
    const double *rp = ring + (size_t)slot * NC + col;
    auto next = [&] {
      slot += kCh;
      if (slot == W) slot = 0;
      rp = ring + (size_t)slot * NC + col;
      f += kCh / 2;
    };
    int left = ke - ka;                  // terms from ka on
    if (left > i + 1 - ka) {
      double xv[kCh], p[kCh];
      double2 uv[kCh / 2];
#pragma unroll
      for (int j = 0; j < kCh; ++j) {
        xv[j] = rp[j * NC];
        if (j & 1) uv[j / 2] = f[j / 2];
      }
      next();
#pragma unroll
      for (int j = 0; j < kCh; ++j) p[j] = (j & 1 ? uv[j / 2].y : uv[j / 2].x) * xv[j];
#pragma unroll
      for (int j = 0; j < kCh; ++j) {
        xv[j] = rp[j * NC];
        if (j & 1) uv[j / 2] = f[j / 2];
      }
      next();
      acc = band_step<NC, true>(acc, p, xv, uv, rp, f, i + 1 - ka, left);
      next();
      for (left -= kCh; left >= kCh; left -= kCh) {
        acc = band_step<NC, false>(acc, p, xv, uv, rp, f);
        next();
      }
#pragma unroll
      for (int j = 0; j < kCh; ++j) {
        const double d = acc - p[j];
        acc = j < left ? d : acc;
      }
    }
    acc = acc / di;
    ring[(size_t)(i % W) * NC + col] = acc;
    if (live) x[(size_t)i * 64] = acc;
  }
}

// bytes of LDS for NC columns: the ring, and the staged rows of L or U
inline size_t band_inverse_lds(int bw, int nc) {
  const size_t l = 2 * (size_t)kCh * kKs, u = 2 * (size_t)((bw + 2 * kCh + 63) / 64 * 64);
  return ((size_t)band_ring(bw) * nc + std::max(l, u + 2 * kCh)) * sizeof(double);
}

template <int NC>
void launch_band_inverse_lds(hipStream_t st, const double *band, int bw, int n, const int *lfirst,
                             const int *ulast, double *X, const int *failed) {
  const size_t bytes = band_inverse_lds(bw, NC);
  (void)hipFuncSetAttribute((const void *)k_band_inverse_lds<NC>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)kLdsBytes);
  k_band_inverse_lds<NC><<<(n + NC - 1) / NC, 256, bytes, st>>>(band, bw, n, lfirst, ulast, X, failed);
}

// inv[r][u] = entry (pos[r], pos[u]) of the panels (list order rows and
// columns)
__global__ __launch_bounds__(256) void k_band_inverse_out(const double *__restrict__ X,
                                                          const int *__restrict__ pos, int n,
                                                          double *__restrict__ inv,
                                                          const int *__restrict__ failed) {
  if (*failed) return;
  const int u = blockIdx.x * 256 + threadIdx.x;
  const int r = blockIdx.y;
  if (u >= n) return;
  const int q = pos[u];
  inv[(size_t)r * n + u] = X[(size_t)(q >> 6) * n * 64 + (size_t)pos[r] * 64 + (q & 63)];
}

}  // namespace

void launch_base_factor(hipStream_t st, double *band, const HostBase &B, const int *pos, const int *lfirst,
                        const int *ulast, double *X, double *inv, int *failed) {
  const int n = B.n, bw = B.bw;
  if (n <= 0) return;
  // panels need bw >= kNb: a pivot row reaches past its panel's columns (then
  // n > kNb, and X, free until the substitutions, holds the diagonal block)
  const bool panels = bw >= kNb;
  for (int p = 0; panels && p < n; p += kNb) {
    const int e = std::min(p + kNb, n) - 1;            // the panel's last pivot
    const int mr = std::max(B.llast[e] - e, 0), mc = std::max(B.ulast[e] - e, 0);
    const int nw = (mr + 63) / 64 + (mc + 63) / 64;
    const dim3 g(std::max((mc + 31) / 32, 1), std::max((mr + 31) / 32, 1));
    if (B.fmode) {
      k_band_panel<float><<<std::max(nw, 1), 64, 0, st>>>(band, bw, n, p, mr, mc, (float *)X, failed);
      k_band_trail<float><<<g, 256, 0, st>>>(band, bw, n, p, mr, mc, (const float *)X, failed);
    } else {
      k_band_panel<double><<<std::max(nw, 1), 64, 0, st>>>(band, bw, n, p, mr, mc, X, failed);
      k_band_trail<double><<<g, 256, 0, st>>>(band, bw, n, p, mr, mc, X, failed);
    }
  }
  for (int i = 0; !panels && i < n; ++i) {
    const int m = i < n - 1 ? std::min(i + bw, n - 1) - i : 0;
    const long long work = std::max<long long>({(long long)m * m, (long long)bw, 1LL});
    const unsigned nb = (unsigned)((work + 255) / 256);
    if (B.fmode) k_band_lu_step<float><<<nb, 256, 0, st>>>(band, bw, n, i, failed);
    else k_band_lu_step<double><<<nb, 256, 0, st>>>(band, bw, n, i, failed);
  }
  // as many columns as leave the ring in LDS (32 up to a bandwidth of 560, 20
  // up to 912, 16 up to 992): the time is one column's chain, so fewer columns
  // gain nothing until the workgroups outnumber the CUs (17^3: 246 of 20
  // columns, 308 of 16 would take two rounds).  A row of U has to fit the
  // staging registers; wider bands keep the window in memory.
  const bool row = bw + 2 * kCh <= 64 * kStage;
  auto fits = [&](int nc) { return row && band_inverse_lds(bw, nc) <= kLdsBytes; };
  if (fits(32)) launch_band_inverse_lds<32>(st, band, bw, n, lfirst, ulast, X, failed);
  else if (fits(20)) launch_band_inverse_lds<20>(st, band, bw, n, lfirst, ulast, X, failed);
  else if (fits(16)) launch_band_inverse_lds<16>(st, band, bw, n, lfirst, ulast, X, failed);
  else k_band_inverse<<<(n + 63) / 64, 64, 0, st>>>(band, bw, n, X, failed);
  k_band_inverse_out<<<dim3((n + 255) / 256, n), 256, 0, st>>>(X, pos, n, inv, failed);
}

}  // namespace ugmg

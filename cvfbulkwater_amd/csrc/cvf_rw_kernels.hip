// Histogram reweighting kernels: the per-cell log-sum over simulations of
// Calcula_Histograma (HistogramReweighting/histogram_reweighting_mixed_
// paramSI_norm_x.f90:1003-1124) for many targets in one launch, and the
// per-target max / log-sum-exp / normalization reductions.
//
// The reference's argument for cell c, target t and simulation j is
//   arg_j = beta_t (E + p_t V) - beta_j (E + p_j V) - c_j + lm_j = t1 + u_j,
// so the target only shifts a cell's sum: log sum_j exp(arg_j) =
// t1 + log sum_j exp(u_j).  k_rw_cells evaluates the n_sim terms u_j once
// per cell and then serves every target of its row with a few flops.
// The reference's two cut-offs are kept exactly:
//  - a cell's sum switches to the max-shifted form that drops terms more
//    than 10 below the largest once any |arg_j| > 10 (f90:1048-1078); the
//    switch depends on the target through t1 (t1 + max u > 10 or
//    t1 + min u < -10), the dropped set does not, so both sums (all terms,
//    and the terms within 10 of the largest) are formed once per cell;
//  - log_Z drops cells more than 10 below the largest log_P (1106-1118).
// Factoring t1 out rounds differently from the reference's left-to-right
// sum: log_P moves by about |t1| x 1e-16 (1e-10 for L = 8).
//
// No kernel stores log_P: it is a few flops from the cell's sum, so every
// pass forms it again from 33 bytes per cell (which stay in the caches)
// instead of writing and reading 8 bytes per cell and target.  At the
// production shape (710,000 cells, 11 simulations) a constants' sweep went
// from three launches of 31.8 + 17.8 + 6.0 us to two of 26.0 + 17.7 (the sweeps
// of few, near simulations now multiply tables, see k_rw_sweep_cells), and a
// scan of 64 targets x 3 angles from 1.17 ms of kernels over 363 MB of
// densities to 0.57 ms.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "cvf_rw_kernels.h"

namespace cvf {
namespace {

constexpr double kUnderflow = -700.0;  // log densities above it are positive doubles, see k_rw_sum

// max and min of doubles, one instruction each (fmax and fmin put a
// canonicalizing one before it where an operand's origin is unknown); a NaN
// operand gives the other one
__device__ inline double max1(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ inline double min1(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// x of lane ^ m (m a power of two, known when compiled): moves within and
// between rows of lanes, without the trip through LDS that a shuffle makes (a
// reduction of a sweep's partial results is a chain of six of them)
__device__ inline uint32_t lane_xor(uint32_t x, int m) {
  const auto half = [&](auto r, uint32_t bit) { return (threadIdx.x & bit) ? (uint32_t)r[0] : (uint32_t)r[1]; };
  switch (m) {
    case 1: return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, true);  // quad_perm 1 0 3 2
    case 2: return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xF, 0xF, true);  // quad_perm 2 3 0 1
    case 4:  // row_half_mirror, then quad_perm 3 2 1 0: lane ^ 7 ^ 3
      return (uint32_t)__builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xF, 0xF, true), 0x1B, 0xF, 0xF,
                                                true);
    case 8: return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x128, 0xF, 0xF, true);  // row_ror 8
    case 16: return half(__builtin_amdgcn_permlane16_swap(x, x, false, false), 16u);
    default: return half(__builtin_amdgcn_permlane32_swap(x, x, false, false), 32u);
  }
}
__device__ inline double lane_xor(double v, int m) {
  const uint64_t x = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = lane_xor((uint32_t)x, m), hi = lane_xor((uint32_t)(x >> 32), m);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

__device__ inline double wave_max(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, lane_xor(v, o));
  return v;
}

__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += lane_xor(v, o);
  return v;
}

// block-wide reduction, result in every thread (red: one entry per wave)
template <bool kMax>
__device__ inline double block_reduce(double v, double* red) {
  v = kMax ? wave_max(v) : wave_sum(v);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double r = red[0];
  for (int i = 1; i < nw; ++i) r = kMax ? fmax(r, red[i]) : r + red[i];
  __syncthreads();
  return r;
}

// exp(d) for d <= 0 (or NaN): d = k ln2 + r, |r| <= ln2 / 2, and the degree-11
// Chebyshev interpolant of e^r there (1.6e-17 relative; coefficients computed
// for this file to 60 digits).  Seven instructions fewer than the library's
// exp, which also serves large arguments: a third of a pass is exponentials.
__device__ inline double exp_le0(double d) {
  const double k = __builtin_rint(d * 0x1.71547652b82fep+0);
  double r = __builtin_fma(k, -0x1.62e42fefa39efp-1, d);
  r = __builtin_fma(k, -0x1.abc9e3b39803fp-56, r);
  double p = 0x1.af632a0f7e2cep-26;
  p = __builtin_fma(p, r, 0x1.28b4101c77212p-22);
  p = __builtin_fma(p, r, 0x1.71ddf56d8deb5p-19);
  p = __builtin_fma(p, r, 0x1.a01991a10d9aep-16);
  p = __builtin_fma(p, r, 0x1.a01a01b1461c5p-13);
  p = __builtin_fma(p, r, 0x1.6c16c1880029fp-10);
  p = __builtin_fma(p, r, 0x1.111111110f21ep-7);
  p = __builtin_fma(p, r, 0x1.555555554f0bap-5);
  p = __builtin_fma(p, r, 0x1.555555555555ap-3);
  p = __builtin_fma(p, r, 0x1.0000000000011p-1);
  p = __builtin_fma(p, r, 1.0);
  p = __builtin_fma(p, r, 1.0);
  // below -745.14 the result is zero (and k may be no int)
  return d < -746.0 ? 0.0 : __builtin_ldexp(p, (int)k);
}

// (a & m) | (b & ~m) of the bits of two doubles, m all ones or all zeros (a
// conditional between two elements of an array would become an indexed read
// of it, a chain of selects over all its elements)
__device__ inline double pick_bits(uint32_t m, double a, double b) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
  const uint32_t lo = ((uint32_t)x & m) | ((uint32_t)y & ~m);
  const uint32_t hi = ((uint32_t)(x >> 32) & m) | ((uint32_t)(y >> 32) & ~m);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// Sums (or maxima) of N values over the wavefront, N a power of two: value i
// ends in the lanes whose bits 5, 4, ... spell i from its highest bit on.
// Each step halves the values that a lane still carries, so N values cost
// N - 1 + log2(64 / N) exchanges and not 6 N.
template <int N, bool kMax>
__device__ inline void wave_reduce(double (&v)[N]) {
  int m = 32;
#pragma unroll
  for (int n = N; n > 1; n /= 2, m /= 2) {
    const uint32_t up = (threadIdx.x & m) ? ~0u : 0u;
#pragma unroll
    for (int i = 0; i < n / 2; ++i) {
      const double keep = pick_bits(up, v[i + n / 2], v[i]), give = pick_bits(up, v[i], v[i + n / 2]);
      const double got = lane_xor(give, m);
      v[i] = kMax ? max1(keep, got) : keep + got;
    }
  }
#pragma unroll
  for (; m > 0; m /= 2) {
    const double got = lane_xor(v[0], m);
    v[0] = kMax ? max1(v[0], got) : v[0] + got;
  }
}
// the value that a lane holds after wave_reduce<N>, and whether it is the
// first lane of those that hold it
template <int N>
__device__ inline int reduced_index() {
  int i = 0;
  for (int n = N, m = 32; n > 1; n /= 2, m /= 2) i += (threadIdx.x & m) ? n / 2 : 0;
  return i;
}
template <int N>
__device__ inline bool reduced_first() {
  return (threadIdx.x & (64 / N - 1)) == 0;
}

// The wavefronts' results red[slot][wave] of a workgroup combined, four lanes
// per slot: valid in the threads 4 slot .. 4 slot + 3 that the call covers.
template <bool kMax>
__device__ inline double combine_waves(const double (*red)[16]) {
  const int nw = blockDim.x >> 6, slot = threadIdx.x >> 2, q = threadIdx.x & 3;
  double v = kMax ? -INFINITY : 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int wv = 4 * i + q;
    const double x = red[slot][wv < nw ? wv : q];  // (q < nw: at least four wavefronts)
    if (wv < nw) v = kMax ? fmax(v, x) : v + x;
  }
#pragma unroll
  for (int m = 1; m < 4; m *= 2) {
    const double x = lane_xor(v, m);
    v = kMax ? fmax(v, x) : v + x;
  }
  return v;
}

// T partial results of nblk workgroups each, kRwRow apart (p[i * kRwRow + k]):
// their sums or maxima into out[0..T), all threads loading at once (one
// latency, not one per result).  red: 16 x 16 of LDS; out(k, result) runs in
// one thread per result.
template <int T, bool kMax, class Out>
__device__ inline void reduce_partials(const double* p, int nblk, double (*red)[16], Out&& out) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double v = kMax ? -INFINITY : 0.0;
  // eight loads on their way at once (past the end the last one again)
  const int stride = blockDim.x / T;
  for (int i0 = threadIdx.x / T; i0 < nblk; i0 += 8 * stride) {
    double x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = p[min(i0 + u * stride, nblk - 1) * kRwRow + (threadIdx.x & (T - 1))];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (i0 + u * stride < nblk) v = kMax ? fmax(v, x[u]) : v + x[u];
  }
#pragma unroll
  for (int m = T; m < 64; m *= 2) {
    const double x = lane_xor(v, m);
    v = kMax ? fmax(v, x) : v + x;
  }
  if (lane < T) red[lane][wave] = v;
  __syncthreads();
  if ((int)threadIdx.x < 4 * T) {
    v = combine_waves<kMax>(red);
    if ((threadIdx.x & 3) == 0) out((int)(threadIdx.x >> 2), v);
  }
}

// u_j = -beta_j (E + p_j V) - c_j + lm_j; s = {beta, p, c, lm}
__device__ inline double rw_u(double E, double V, const double* s) { return -(s[0] * (E + s[1] * V)) - s[2] + s[3]; }

// log_P of a cell for one target: t1 shifts the cell's sum, and picks it
// where the targets of a row disagree (a mixed cell).
__device__ inline double rw_t1(double E, double V, double2 bp) { return bp.x * (E + bp.y * V); }
__device__ inline bool rw_cut(double t1, double umax, double umin) { return t1 + umax > 10.0 || t1 + umin < -10.0; }

// 0, unknown to the compiler: an LDS index that includes it is read where it
// stands, in each round of the loop, instead of all targets' values being
// held in registers across it (which spills)
__device__ inline int opaque_zero() {
  int z = 0;
  asm volatile("" : "+v"(z));
  return z;
}

// A thread's first cell of the grid-stride walk: a wavefront's 64 cells
// together, the workgroups' first wavefronts before their second ones, so
// that the last, partial round is spread over all CUs.
__device__ inline int64_t first_cell() {
  return ((int64_t)(threadIdx.x >> 6) * gridDim.x + blockIdx.x) * 64 + (threadIdx.x & 63);
}

struct CellIn {
  double E, V, lh, S;
  bool mixed;
};
__device__ inline CellIn cell_in(const RwCells& c, const RwWork& w, int row, int64_t b) {
  return CellIn{c.en[b], c.vn[b], c.lh[b], w.sum[(int64_t)row * c.n + b], w.mixed[(int64_t)row * c.n + b] != 0};
}
__device__ inline double cell_sum(const CellIn& c, const RwWork& w, int64_t b, double t1) {
  if (!c.mixed) return c.S;
  const RwMixed m = w.mix[b];
  return rw_cut(t1, m.umax, m.umin) ? m.near : m.all;
}
__device__ inline double cell_logp(const CellIn& c, const RwWork& w, int64_t b, double2 bp) {
  const double t1 = rw_t1(c.E, c.V, bp);
  return c.lh - (t1 + cell_sum(c, w, b, t1));
}

// The cells' sums over the simulations for a row of kRwRow targets
// (blockIdx.y), and the row's partial maxima of log_P.  A sweep of the
// constants takes them from the previous sweep's partial sums (`ps`, not
// null), each workgroup reducing them for itself, so that no launch lies
// between two sweeps but k_rw_sum; workgroup 0 writes them to `used`.
// Bound by FP64 issue (n_sim exponentials per cell); a thread takes several
// cells, so that the maxima are reduced across lanes once per workgroup and
// not once per cell (those shuffles cost as much as the exponentials).
template <int R>
__global__ __launch_bounds__(1024) void k_rw_cells(RwCells cells, const RwSim* __restrict__ sims,
                                                   const double* __restrict__ ctes, int32_t n_sim, RwTargets tg,
                                                   RwWork w, const double* __restrict__ ps,
                                                   const double* __restrict__ mx, double* __restrict__ used) {
  constexpr int kGroup = R < 4 ? R : 4;
  extern __shared__ double sl[];  // 4 per simulation: beta, p, c, lm; then log_Z of each
  __shared__ double red[16][16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int j = threadIdx.x; j < n_sim; j += blockDim.x) {
    sl[4 * j] = sims[j].beta;
    sl[4 * j + 1] = sims[j].pres;
    if (!ps) sl[4 * j + 2] = ctes[j];
    sl[4 * j + 3] = sims[j].lm;
  }
  const int64_t lanes = (int64_t)gridDim.x * blockDim.x, b0 = first_cell();
  // the next cell, loaded a round ahead, the first one before the reduction (a
  // full row has no registers for that)
  double En = 0, Vn = 0, lhn = 0;
  if (R < kRwRow && b0 < cells.n) En = cells.en[b0], Vn = cells.vn[b0], lhn = cells.lh[b0];
  // the row's targets, the last one repeated to fill it: the loop over them
  // below then has no branch, and no global load stalls it
  const int row = blockIdx.y, t0 = row * kRwRow, nt = min(tg.n - t0, kRwRow);
  __shared__ double2 bps[R];
  if ((int)threadIdx.x < R) bps[threadIdx.x] = tg.bp[t0 + min((int)threadIdx.x, nt - 1)];
  // log_Z of the sweep before, and from it this sweep's constants (a sweep's
  // targets are its simulations: n_sim <= R where R < kRwRow)
  const auto log_z = [](double st, double m) { return (st != 0 ? log(st) : 0.0) + m; };
  if (R < kRwRow && ps) {
    // its results are in the lanes of the first wavefront (a full row has no
    // registers for that)
    const int jm = min((int)(threadIdx.x >> 2), n_sim - 1);
    const double m = mx[jm];
    reduce_partials<R, false>(ps, w.nblk, red, [&](int k, double st) {
      const double lz = log_z(st, m);
      const uint64_t x = __builtin_bit_cast(uint64_t, lz);
      const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x);
      const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
      const double c = lz - __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
      if (k < n_sim) {
        sl[4 * k + 2] = c;
        if (blockIdx.x == 0 && blockIdx.y == 0) used[k] = c;
      }
    });
  } else if (ps) {
    double* lz = sl + 4 * n_sim;
    for (int j0 = 0; j0 < n_sim; j0 += R) {
      reduce_partials<R, false>(ps + (int64_t)j0 * w.nblk, w.nblk, red, [&](int k, double st) {
        if (j0 + k < n_sim) lz[j0 + k] = log_z(st, mx[j0 + k]);
      });
      __syncthreads();
    }
    for (int j = threadIdx.x; j < n_sim; j += blockDim.x) {
      const double c = lz[j] - lz[0];
      sl[4 * j + 2] = c;
      if (blockIdx.x == 0 && blockIdx.y == 0) used[j] = c;
    }
  }
  __syncthreads();
  double top[R];
#pragma unroll
  for (int k = 0; k < R; ++k) top[k] = -INFINITY;
  if (R == kRwRow && b0 < cells.n) En = cells.en[b0], Vn = cells.vn[b0], lhn = cells.lh[b0];
  for (int64_t b = b0; b < cells.n; b += lanes) {
    const double E = En, V = Vn, lh = lhn;
    if (b + lanes < cells.n) En = cells.en[b + lanes], Vn = cells.vn[b + lanes], lhn = cells.lh[b + lanes];
    double umax = -INFINITY, umin = INFINITY, sa = 0, st = 0;
    const double* sp = sl + opaque_zero();
    for (int j = 0; j < n_sim; ++j) {
      const double u = rw_u(E, V, sp + 4 * j);
      umax = fmax(umax, u);
      umin = fmin(umin, u);
    }
    // four at a time, so that four chains interleave, then the rest
    int j = 0;
    for (; j + 4 <= n_sim; j += 4) {
      double d[4], e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        d[i] = rw_u(E, V, sp + 4 * (j + i)) - umax;
        e[i] = exp_le0(d[i]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        sa = sa + e[i];
        if (-d[i] < 10.0) st = st + e[i];
      }
    }
    for (; j < n_sim; ++j) {
      const double d = rw_u(E, V, sp + 4 * j) - umax;
      const double e = exp_le0(d);
      sa = sa + e;
      if (-d < 10.0) st = st + e;
    }
    const double near = log(st) + umax;  // log sum_j exp(u_j) over the terms within 10 of the largest
    // (each target's t1, and its log_P with the sum that the cell's targets
    // mostly use; a cell whose targets may not all be cut, as a bound of t1
    // says, is looked at again target by target)
    double all = near;  // log sum_j exp(u_j); not needed by a cell whose targets are all cut
    bool any_cut = true, any_all = false;
    const double2* bp = bps + opaque_zero();
    double t_lo = INFINITY;
#pragma unroll
    for (int k0 = 0; k0 < R; k0 += kGroup)
      if (k0 < nt) {
#pragma unroll
        for (int k = k0; k < k0 + kGroup; ++k) t_lo = fmin(t_lo, rw_t1(E, V, bp[k]));
      }
    if (__ballot(!(t_lo + umax > 10.0))) {
      all = log(sa) + umax;
      any_cut = false;
      for (int k = 0; k < nt; ++k) {
        const bool cut = rw_cut(rw_t1(E, V, bp[k]), umax, umin);
        any_cut = any_cut || cut;
        any_all = any_all || !cut;
      }
    }
    const double S = any_cut ? near : all;
    if (__ballot(any_cut && any_all)) {
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const double t1 = rw_t1(E, V, bp[k]);
        top[k] = fmax(top[k], lh - (t1 + (rw_cut(t1, umax, umin) ? near : all)));
      }
    } else {
#pragma unroll
      for (int k0 = 0; k0 < R; k0 += kGroup)
        if (k0 < nt) {
#pragma unroll
          for (int k = k0; k < k0 + kGroup; ++k) top[k] = fmax(top[k], lh - (rw_t1(E, V, bp[k]) + S));
        }
    }
    w.sum[(int64_t)row * cells.n + b] = S;
    w.mixed[(int64_t)row * cells.n + b] = any_cut && any_all;
    if (any_cut && any_all) w.mix[b] = RwMixed{near, all, umax, umin};  // the same in every row
  }
  wave_reduce<R, true>(top);
  if (reduced_first<R>()) red[reduced_index<R>()][wave] = top[0];
  __syncthreads();
  if ((int)threadIdx.x < 4 * R) {
    const double m = combine_waves<true>(red);
    const int k = threadIdx.x >> 2;
    if ((threadIdx.x & 3) == 0 && k < nt) w.pmax[((int64_t)row * w.nblk + blockIdx.x) * kRwRow + k] = m;
  }
}

__device__ inline void cell_er(const RwGeom& g, uint32_t c, double& e, double& r) {
  const uint32_t i = c >> 16, w = c & 0xFFFFu;
  e = g.e_min + ((int)(i + 1) - 0.5) * g.de;
  r = g.rho_min + ((int)(w + 1) - 0.5) * g.drho;
}

// For a tile of T targets (blockIdx.y): their max log_P m from the partial
// maxima, then over the workgroup's cells the partial sums of
// x = exp(log_P - m): over the cells within 10 of the max (for log_Z); with
// kMode >= kRwDensity over all cells (for the normalization); with kRwScan
// also of x e^2, x e^4, x rho^2, x rho^4 (the Binder cumulants are ratios, so
// any scale serves).  A scan's workgroup also says which targets have a
// cell with log_P - m <= -700 (or not a number): for the others every
// density exp(log_P - log_Z) / norm is surely positive (0 <= log_Z - m <=
// log of the cell count, and the norm is that sum times the cell's area), so
// the order parameter's range is that of the grid's cells, whatever the
// target.  T: what the accumulators leave of the registers at four waves
// per SIMD.
template <int T, int kMode>
__global__ __launch_bounds__(1024) void k_rw_sum(RwCells cells, RwTargets tg, RwWork w, RwGeom g) {
  constexpr int V = kMode == kRwSweep ? 1 : kMode == kRwDensity ? 2 : kRwScanSums;
  constexpr int kRed = V * T > 16 ? V * T : 16, kGroup = T < 4 ? T : 4;
  __shared__ double red[kRed][16];
  __shared__ double ms[T];
  __shared__ double2 bps[T];
  __shared__ uint32_t low_s;
  const int wave = threadIdx.x >> 6;
  const int t0 = blockIdx.y * T, nt = min(tg.n - t0, T), row = t0 / kRwRow;
  if (threadIdx.x == 0) low_s = 0;
  if ((int)threadIdx.x < T) bps[threadIdx.x] = tg.bp[t0 + min((int)threadIdx.x, nt - 1)];
  const int64_t lanes = (int64_t)gridDim.x * blockDim.x, b0 = first_cell();
  // the first cell on its way while the maxima are reduced, later ones a round
  // ahead, where the registers allow it
  constexpr bool kAhead = kMode == kRwSweep && T <= 8;
  CellIn next{0, 0, 0, 0, false};
  if (kAhead && b0 < cells.n) next = cell_in(cells, w, row, b0);
  reduce_partials<T, true>(w.pmax + (int64_t)row * w.nblk * kRwRow + (t0 - row * kRwRow), w.nblk, red,
                           [&](int k, double m) {
                             ms[k] = k < nt ? m : 0.0;
                             if (blockIdx.x == 0 && k < nt) w.mx[t0 + k] = m;
                           });
  __syncthreads();
  double s[V][T];
#pragma unroll
  for (int k = 0; k < T; ++k)
#pragma unroll
    for (int v = 0; v < V; ++v) s[v][k] = 0;
  uint32_t low = 0;
  // the cells whose targets all use one sum, then (if there are any) the
  // mixed ones, so that the usual loop has no branch between its exponentials
  int saw_mixed = 0;
  for (int pass = 0; pass < 2; ++pass) {
    for (int64_t b = b0; b < cells.n; b += lanes) {
      const CellIn c = kAhead ? next : cell_in(cells, w, row, b);
      if (kAhead && b + lanes < cells.n) next = cell_in(cells, w, row, b + lanes);
      if (pass == 0) saw_mixed |= c.mixed;
      if (c.mixed != (pass != 0)) continue;
      RwMixed m{c.S, c.S, 0, 0};
      if (pass) m = w.mix[b];
      double e2 = 0, r2 = 0, e4 = 0, r4 = 0;
      if (kMode == kRwScan) {
        double e, r;
        cell_er(g, g.cell[b], e, r);
        e2 = e * e;
        r2 = r * r;
        e4 = e2 * e2;
        r4 = r2 * r2;
      }
      const auto add = [&](int k, int z) {
        const double t1 = rw_t1(c.E, c.V, bps[k + z]);
        double S = c.S;
        if (pass) S = rw_cut(t1, m.umax, m.umin) ? m.near : m.all;
        const double d = (c.lh - (t1 + S)) - ms[k + z];
        const double x = exp_le0(d);
        if (-d < 10.0) s[0][k] = s[0][k] + x;
        if (kMode >= kRwDensity) s[1 % V][k] = s[1 % V][k] + x;
        if (kMode == kRwScan) {
          if (!(d > kUnderflow)) low |= 1u << k;
          s[2 % V][k] = s[2 % V][k] + e2 * x;
          s[3 % V][k] = s[3 % V][k] + e4 * x;
          s[4 % V][k] = s[4 % V][k] + r2 * x;
          s[5 % V][k] = s[5 % V][k] + r4 * x;
        }
      };
      // four targets at a time: their chains interleave, and a last tile of
      // few targets skips the groups that hold none (the spare members of a
      // group repeat its last target and are not stored; a group of one is
      // taken alone)
#pragma unroll
      for (int k0 = 0; k0 < T; k0 += kGroup)
        if (k0 < nt) {
          const int z = opaque_zero();
          if (kMode == kRwSweep && k0 + 1 == nt) {
            add(k0, z);
          } else {
#pragma unroll
            for (int k = k0; k < k0 + kGroup; ++k) add(k, z);
          }
        }
    }
    if (pass == 0 && !__syncthreads_or(saw_mixed)) break;
    if (kAhead && b0 < cells.n) next = cell_in(cells, w, row, b0);
  }
  if (kMode == kRwScan && low) atomicOr(&low_s, low);
#pragma unroll
  for (int v = 0; v < V; ++v) {
    wave_reduce<T, false>(s[v]);
    if (reduced_first<T>()) red[reduced_index<T>() * V + v][wave] = s[v][0];
  }
  __syncthreads();
  if ((int)threadIdx.x < 4 * nt * V) {
    const double x = combine_waves<false>(red);
    const int k = (threadIdx.x >> 2) / V, v = (threadIdx.x >> 2) - k * V;
    if ((threadIdx.x & 3) == 0) w.ps[(((int64_t)v * w.rows + row) * w.nblk + blockIdx.x) * kRwRow + (t0 + k - row * kRwRow)] = x;
  }
  if (kMode == kRwScan && (int)threadIdx.x < nt)
    w.plow[(int64_t)(t0 + threadIdx.x) * w.nblk + blockIdx.x] = (low_s >> threadIdx.x) & 1u;
}

// One wavefront per target: log_Z = log(truncated sum) + max; with kMode >=
// kRwDensity the normalization sum exp(log_P - log_Z) de drho; of a scan the
// Binder cumulants 1 - <x^4> / (3 <x^2>^2) of the marginals and whether
// some cell's density may have underflowed.
template <int kMode>
__global__ __launch_bounds__(64) void k_rw_finish(RwWork w, double de, double drho,
                                                  double* __restrict__ binder_ed) {
  constexpr int V = kMode == kRwSweep ? 1 : kMode == kRwDensity ? 2 : kRwScanSums;
  const int t = blockIdx.x, lane = threadIdx.x;
  double s[V];
#pragma unroll
  for (int v = 0; v < V; ++v) s[v] = 0;
  uint32_t low = 0;
  // (all sums' loads of a round together)
  for (int i = lane; i < w.nblk; i += 64) {
#pragma unroll
    for (int v = 0; v < V; ++v)
      s[v] += w.ps[(((int64_t)v * w.rows + t / kRwRow) * w.nblk + i) * kRwRow + t % kRwRow];
    if (kMode == kRwScan) low |= w.plow[(int64_t)t * w.nblk + i];
  }
#pragma unroll
  for (int v = 0; v < V; ++v) s[v] = wave_sum(s[v]);
  low = __ballot(low != 0) != 0;
  if (lane) return;
  const double z = (s[0] != 0 ? log(s[0]) : 0.0) + w.mx[t];
  w.lz[t] = z;
  if (kMode >= kRwDensity) w.norm[t] = s[1 % V] * exp(w.mx[t] - z) * de * drho;
  if (kMode == kRwScan) {
    const double m0 = s[1 % V], e2 = s[2 % V] / m0, r2 = s[4 % V] / m0;
    binder_ed[2 * t] = 1.0 - (s[3 % V] / m0) / (3.0 * e2 * e2);
    binder_ed[2 * t + 1] = 1.0 - (s[5 % V] / m0) / (3.0 * r2 * r2);
    w.low[t] = low;
  }
}

// ------------------------------------------------- sweeps of the constants
// The tables of a solve (RwTables), the cells' histograms among them.
__global__ __launch_bounds__(256) void k_rw_tables(RwCells cells, const RwSim* __restrict__ sims, int32_t n_sim,
                                                   RwGeom g, int32_t N, RwTables tb) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < cells.n) {
    tb.h[i] = exp(cells.lh[i]);
    return;
  }
  i -= cells.n;
  const auto energy = [&](int k) { return (g.e_min + ((k + 1) - 0.5) * g.de) * N; };
  const auto volume = [&](int k) { return (double)0.018f / (g.rho_min + ((k + 1) - 0.5) * g.drho) * N; };
  const double e0 = energy(g.nb / 2), v0 = volume(g.nb / 2);
  const int64_t per = 2 * (int64_t)g.nb;
  if (i >= n_sim * (per + 1)) return;
  const int j = (int)(i / (per + 1)), k = (int)(i - j * (per + 1));
  // beta p to twice the digits: the product's rounding would be the same in
  // every cell
  const double b0 = sims[0].beta, p0 = sims[0].pres, b = sims[j].beta, p = sims[j].pres;
  const double q0 = b0 * p0, q = b * p;
  const double db = b - b0, dq = (q - q0) + (__builtin_fma(b, p, -q) - __builtin_fma(b0, p0, -q0));
  const auto put = [&](double2* t, int at, double x) {
    (&t[(size_t)(j / 2) * g.nb + at].x)[j & 1] = exp(x);
  };
  if (k < g.nb)
    put(tb.row, k, -(db * (energy(k) - e0)));
  else if (k < per)
    put(tb.col, k - g.nb, -(dq * (volume(k - g.nb) - v0)));
  else
    tb.sc[j] = double2{db * e0 + dq * v0, sims[j].lm};
}

constexpr double kExpM10 = 0x1.7cd79b5647c9bp-15;  // e^-10: the cut-offs of both sums

template <int N>
constexpr int kPad = N <= 2 ? 2 : N <= 4 ? 4 : N <= 8 ? 8 : 16;

// exp(x_j) of a cell for each of N simulations, two to a load: a gather costs
// by its lanes, not its bytes.
template <int N>
__device__ inline void cell_shifts(const RwTables& tb, uint32_t c, double (&D)[N]) {
  const double2 *row = tb.row + (c >> 16), *col = tb.col + (c & 0xFFFFu);
#pragma unroll
  for (int j = 0; j < N; j += 2) {
    const double2 r = row[(size_t)(j / 2 * tb.nb)], q = col[(size_t)(j / 2 * tb.nb)];
    D[j] = r.x * q.x;
    if (j + 1 < N) D[j + 1] = r.y * q.y;
  }
}

// A sweep's first launch, as k_rw_cells, on the tables: with D_j = exp(x_j)
// and W_j = exp(w_j - max w) a cell's terms are W_j D_j, its sum S over them
// (all, or those above e^-10 of the largest) gives R = h / S, and exp(log_P)
// of target t is R D_t exp(-(g_t + max w)), whose last factor no cell needs.
// The targets are the simulations, so every D_j serves twice and a cell costs
// N gathers of 16 bytes from tables in the L2s, a quotient and about 6 N FP64
// instructions, instead of N exponentials here and N more in k_rw_sum.  The
// exponents are differences between simulations, of order 1 to 100 where
// beta E is 10^5: against 80-bit arithmetic (6 simulations, 24,000 cells, 15
// sweeps) the constants are 3.5e-14 off, 1.1e-11 with exponentials.
// Bound by the gathers (one value at a time, twice as many: 27.0 us a sweep)
// and, for few cells, by the launches and their reductions.  A sweep of 11
// simulations and 710,000 cells 41.8 -> 22.6 us; 5 and 31,000 14.1 -> 9.3;
// 12 and 122,000 22.5 -> 11.8; 2 and 2,700 10.6 -> 8.2.  (In squares of 32 x 32
// cells a wavefront's gathers share lines: 21.4 us, for a sort on the host
// that costs more than a solve gains.)
// Stores R, negative where the cell's targets use different sums (mix[cell]:
// h / near, h / all, largest and smallest term).
template <int N>
__global__ __launch_bounds__(1024) void k_rw_sweep_cells(RwTables tb, int64_t n, RwWork w,
                                                         const double* __restrict__ ps, double* __restrict__ used) {
  constexpr int P = kPad<N>;
  __shared__ double red[16][16];
  __shared__ double lz[16], W[N], cut_hi[N], cut_lo[N];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t lanes = (int64_t)gridDim.x * blockDim.x, b0 = first_cell();
  uint32_t cn = 0;
  double hn = 0;
  if (b0 < n) cn = tb.cell[b0], hn = tb.h[b0];
  if (ps) {
    const double m = w.mx[min((int)(threadIdx.x >> 2), N - 1)];
    reduce_partials<P, false>(ps, w.nblk, red, [&](int k, double st) {
      if (k < N) lz[k] = (st != 0 ? log(st) : 0.0) + m;
    });
    __syncthreads();
  }
  if (wave == 0) {
    const int k = min(lane, N - 1);
    const double c = ps ? lz[k] - lz[0] : 0.0;
    const double2 s = tb.sc[k];
    const double wk = (s.y - s.x) - c, top = wave_max(wk), K = s.x + top;
    if (lane < N) {
      // arg_j of target t is log(W_j D_j) + K_t - x_t: above 10 where
      // W_j D_j > D_t exp(10 - K_t), below -10 where less than
      // D_t exp(-10 - K_t).  (Beyond 700 the comparison with any term has the
      // result that it has at 700: |x| <= kRwMaxShift, and the largest W is 1.)
      const double hi = exp(fmin(fmax(10.0 - K, -700.0), 700.0)), lo = exp(fmin(fmax(-10.0 - K, -700.0), 700.0));
      W[k] = exp(wk - top);
      cut_hi[k] = hi;
      cut_lo[k] = lo;
      if (blockIdx.x == 0) {
        used[k] = c;
        tb.kt[k] = K;
        tb.kt[kRwRow + k] = hi;
        tb.kt[2 * kRwRow + k] = lo;
      }
    }
  }
  __syncthreads();
  double top[P];
#pragma unroll
  for (int k = 0; k < P; ++k) top[k] = 0;
  for (int64_t b = b0; b < n; b += lanes) {
    const uint32_t c = cn;
    const double h = hn;
    if (b + lanes < n) cn = tb.cell[b + lanes], hn = tb.h[b + lanes];
    double D[N];
    cell_shifts<N>(tb, c, D);
    const double* Wp = W + opaque_zero();
    double M = 0, m = INFINITY, all = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const double t = D[j] * Wp[j];
      M = max1(M, t);
      m = min1(m, t);
      all = all + t;
    }
    double S = all, near = all;
    bool mixed = false;
    const bool split = !(m > M * kExpM10);  // the sums differ
    if (__ballot(split)) {
      near = 0;
      bool any_cut = false, any_all = false;
      const double *hi = cut_hi + opaque_zero(), *lo = cut_lo + opaque_zero();
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const double t = D[j] * Wp[j];
        if (t > M * kExpM10) near = near + t;
        const bool cut = M > D[j] * hi[j] || m < D[j] * lo[j];
        any_cut = any_cut || cut;
        any_all = any_all || !cut;
      }
      S = any_cut ? near : all;
      mixed = split && any_cut && any_all;
    }
    const double R = h / S;
    if (__ballot(mixed)) {
      const double Ra = h / all;
      const double *hi = cut_hi + opaque_zero(), *lo = cut_lo + opaque_zero();
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const bool cut = M > D[k] * hi[k] || m < D[k] * lo[k];
        top[k] = max1(top[k], D[k] * (!mixed || cut ? R : Ra));
      }
      if (mixed) w.mix[b] = RwMixed{R, Ra, M, m};
    } else {
#pragma unroll
      for (int k = 0; k < N; ++k) top[k] = max1(top[k], D[k] * R);
    }
    w.sum[b] = mixed ? -R : R;
  }
  wave_reduce<P, true>(top);
  if (reduced_first<P>()) red[reduced_index<P>()][wave] = top[0];
  __syncthreads();
  if ((int)threadIdx.x < 4 * P) {
    const double m = combine_waves<true>(red);
    const int k = threadIdx.x >> 2;
    if ((threadIdx.x & 3) == 0 && k < N) w.pmax[(int64_t)blockIdx.x * kRwRow + k] = m;
  }
}

// Its second launch: per target the sum of R D_t over the cells within e^-10
// of the largest; w.mx takes log of the factor left out.
template <int N>
__global__ __launch_bounds__(1024) void k_rw_sweep_sum(RwTables tb, int64_t n, RwWork w) {
  constexpr int P = kPad<N>;
  __shared__ double red[16][16];
  __shared__ double low[N], cut_hi[N], cut_lo[N];
  const int wave = threadIdx.x >> 6;
  const int64_t lanes = (int64_t)gridDim.x * blockDim.x, b0 = first_cell();
  uint32_t cn = 0;
  double rn = 0;
  if (b0 < n) cn = tb.cell[b0], rn = w.sum[b0];
  if ((int)threadIdx.x < N) {
    cut_hi[threadIdx.x] = tb.kt[kRwRow + threadIdx.x];
    cut_lo[threadIdx.x] = tb.kt[2 * kRwRow + threadIdx.x];
    if (blockIdx.x == 0) w.mx[threadIdx.x] = -tb.kt[threadIdx.x];
  }
  reduce_partials<P, true>(w.pmax, w.nblk, red, [&](int k, double m) {
    if (k < N) low[k] = m * kExpM10;
  });
  __syncthreads();
  double s[P];
#pragma unroll
  for (int k = 0; k < P; ++k) s[k] = 0;
  for (int64_t b = b0; b < n; b += lanes) {
    const uint32_t c = cn;
    const double R = rn;
    if (b + lanes < n) cn = tb.cell[b + lanes], rn = w.sum[b + lanes];
    double D[N];
    cell_shifts<N>(tb, c, D);
    const double* lp = low + opaque_zero();
    if (__ballot(R < 0)) {
      const bool mixed = R < 0;
      RwMixed m{R, R, 0, 0};
      if (mixed) m = w.mix[b];
      const double *hi = cut_hi + opaque_zero(), *lo = cut_lo + opaque_zero();
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const bool cut = m.umax > D[k] * hi[k] || m.umin < D[k] * lo[k];
        const double x = D[k] * (cut ? m.near : m.all);
        if (x > lp[k]) s[k] = s[k] + x;
      }
    } else {
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const double x = D[k] * R;
        if (x > lp[k]) s[k] = s[k] + x;
      }
    }
  }
  wave_reduce<P, false>(s);
  if (reduced_first<P>()) red[reduced_index<P>()][wave] = s[0];
  __syncthreads();
  if ((int)threadIdx.x < 4 * P) {
    const double x = combine_waves<false>(red);
    const int k = threadIdx.x >> 2;
    if ((threadIdx.x & 3) == 0 && k < N) w.ps[(int64_t)blockIdx.x * kRwRow + k] = x;
  }
}

// densities exp(log_P - log_Z) / norm, one target per blockIdx.y
__global__ __launch_bounds__(kRwBlock) void k_rw_dist(RwCells cells, RwTargets tg, RwWork w,
                                                      double* __restrict__ dens) {
  const int t = blockIdx.y;
  const int64_t b = (int64_t)blockIdx.x * kRwBlock + threadIdx.x;
  if (b >= cells.n) return;
  const double lp = cell_logp(cell_in(cells, w, t / kRwRow, b), w, b, tg.bp[t]);
  dens[(int64_t)t * cells.n + b] = exp(lp - w.lz[t]) / w.norm[t];
}

// ------------------------------------------------------------ projections
// Each workgroup of a projection takes one contiguous range of cells, so
// every sum below runs in an order fixed by the launch shape alone.
__device__ inline void block_range(int64_t n, int64_t& lo, int64_t& hi) {
  const int64_t per = (n + gridDim.x - 1) / gridDim.x;
  lo = (int64_t)blockIdx.x * per;
  hi = lo + per < n ? lo + per : n;
}

// Min and max of x = e sin(a) + rho cos(a) over a workgroup's cells: with
// blockIdx.y < n_a over all cells at angle blockIdx.y, the range of every
// target whose densities are all positive; beyond that, for target and
// angle blockIdx.y - n_a, over its cells of positive density, left out for
// the targets that the first kind serves.
__global__ __launch_bounds__(kRwBlock) void k_rw_xrange(RwGeom g, RwCells cells, RwTargets tg, RwWork w,
                                                        RwScan sc) {
  __shared__ double red[kRwBlock / 64];
  const int y = blockIdx.y;
  const bool own = y >= sc.n_a;
  const int t = own ? (y - sc.n_a) / sc.n_a : 0, a = own ? (y - sc.n_a) - t * sc.n_a : y;
  if (own && !w.low[t]) return;
  const double2 q = sc.angle[a], bp = own ? tg.bp[t] : double2{0, 0};
  int64_t lo, hi;
  block_range(g.n, lo, hi);
  double mn = INFINITY, mx = -INFINITY;
  for (int64_t b = lo + threadIdx.x; b < hi; b += kRwBlock) {
    if (own) {
      const double lp = cell_logp(cell_in(cells, w, t / kRwRow, b), w, b, bp);
      if (!(exp(lp - w.lz[t]) / w.norm[t] > 0)) continue;
    }
    double e, r;
    cell_er(g, g.cell[b], e, r);
    const double x = e * q.x + r * q.y;
    mn = fmin(mn, x);
    mx = fmax(mx, x);
  }
  mn = -block_reduce<true>(-mn, red);
  mx = block_reduce<true>(mx, red);
  if (threadIdx.x == 0) sc.range[(int64_t)y * gridDim.x + blockIdx.x] = double2{mn, mx};
}

// Bins from the range of x over the occupied cells, two empty ones on each
// side (f90:1420-1429): of the grid's cells at angle blockIdx.x < n_a (gbin),
// then of pair blockIdx.x - n_a, which are the grid's where all its
// densities are positive; one wavefront each.
__global__ __launch_bounds__(64) void k_rw_bins(RwWork w, RwScan sc, int32_t nm) {
  const bool pair = (int)blockIdx.x >= sc.n_a;
  const int ta = (int)blockIdx.x - sc.n_a, t = pair ? ta / sc.n_a : 0;
  const int at = pair && !w.low[t] ? ta - t * sc.n_a : (int)blockIdx.x;  // whose range
  const double2* r = sc.range + (int64_t)at * sc.n_proj;
  double xmin = (double)1E12f, xmax = (double)-1E12f;
  for (int i = threadIdx.x; i < sc.n_proj; i += 64) {
    xmin = fmin(xmin, r[i].x);
    xmax = fmax(xmax, r[i].y);
  }
  xmin = -wave_max(-xmin);
  xmax = wave_max(xmax);
  if (threadIdx.x) return;
  if (pair) sc.code[ta] = xmax >= xmin ? 0u : kRwNoCell;
  double range = xmax - xmin, width = range / nm;
  range = range + 4 * width;
  xmin = xmin - 2 * width;
  width = range / nm;
  (pair ? sc.bin[ta] : sc.gbin[blockIdx.x]) = double2{xmin, width};
}

// Bin of X: (int)((X - x0) / w) (f90:1440-1452), kRwNoBin outside the bins.
constexpr uint32_t kRwNoBin = 255;  // n_bin_mixed <= 215
__device__ inline uint32_t order_bin(double X, double2 bi, int nm) {
  const double y = X - bi.x, d = y / bi.y;
  if (fabs(d) < 1073741824.0 && (int)d >= 0 && (int)d < nm) return (uint32_t)(int)d;
  return fabs(y) < (double)1E-10f ? 0u : kRwNoBin;
}

// The cells' bins at NA angles, a byte each, for every target whose bins
// are the grid's (blockIdx.y: group of angles).
template <int NA>
__device__ inline uint32_t cell_bins(const RwGeom& g, uint32_t id, const RwScan& sc, const double2* bin, int a0, int na) {
  double e, r;
  cell_er(g, id, e, r);
  uint32_t v = 0;
#pragma unroll
  for (int a = 0; a < NA; ++a)
    if (a < na) {
      const double2 q = sc.angle[a0 + a];
      v |= order_bin(e * q.x + r * q.y, bin[a0 + a], g.nm) << (8 * a);
    }
  return v;
}
template <int NA>
__global__ __launch_bounds__(kRwBlock) void k_rw_cell_bins(RwGeom g, RwScan sc) {
  const int64_t b = (int64_t)blockIdx.x * kRwBlock + threadIdx.x;
  if (b >= g.n) return;
  const int a0 = blockIdx.y * NA;
  sc.cbin[(int64_t)blockIdx.y * g.n + b] = cell_bins<NA>(g, g.cell[b], sc, sc.gbin, a0, min(NA, sc.n_a - a0));
}

// Histograms of x over the bins of NA angles (blockIdx.y = target and group
// of NA angles), weighted by the density, one wavefront per workgroup.  A
// cell's exponential serves all NA angles.  kRwRows lanes apart share a row
// of the wavefront's histogram and add to it one group of kRwRows lanes
// after the other, so every sum runs in an order fixed by the launch shape:
// LDS additions of one wavefront are done in order, and no two lanes of a
// group share a row.  The densities are left unnormalized unless some
// underflow: the histogram is normalized after.
// Bound by FP64 issue and those additions.  A row per lane and angle (30 KB
// at 59 bins) with each lane reading, adding and writing back: 489 us for 64
// targets x 3 angles at 710,000 cells; 275 us in this form, with its exponentials.
constexpr int kRwXhistBatch = 4;  // cells per lane whose loads are issued together
constexpr int kRwRows = 16;

template <int NA>
__global__ __launch_bounds__(64) void k_rw_xhist(RwGeom g, RwCells cells, RwTargets tg, RwWork w, RwScan sc) {
  extern __shared__ double hl[];  // [NA][kRwRows][stride]
  const int ng = (sc.n_a + NA - 1) / NA, t = blockIdx.y / ng, a0 = (blockIdx.y - t * ng) * NA;
  const int na = min(NA, sc.n_a - a0), lane = threadIdx.x, nm = g.nm, stride = nm | 1;
  for (int i = lane; i < NA * kRwRows * stride; i += 64) hl[i] = 0;
  __syncthreads();
  const double2 bp = tg.bp[t];
  const double lz = w.lz[t], norm = w.norm[t];
  const bool own = w.low[t] != 0;  // the target has its own bins
  double* row = hl + (lane & (kRwRows - 1)) * stride;
  const uint32_t* cb = sc.cbin + (int64_t)(a0 / NA) * g.n;
  int64_t lo, hi;
  block_range(g.n, lo, hi);
  uint32_t bad = 0;
  for (int64_t b0 = lo; b0 < hi; b0 += 64 * kRwXhistBatch) {
    // the batch's loads first (an index past the end re-reads the last cell)
    CellIn c[kRwXhistBatch];
    uint32_t kb[kRwXhistBatch];
    double x[kRwXhistBatch];
#pragma unroll
    for (int u = 0; u < kRwXhistBatch; ++u) {
      const int64_t b = b0 + 64 * u + lane, bc = b < hi ? b : hi - 1;
      c[u] = cell_in(cells, w, t / kRwRow, bc);
      kb[u] = own ? cell_bins<NA>(g, g.cell[bc], sc, sc.bin + t * sc.n_a, a0, na) : cb[bc];
    }
#pragma unroll
    for (int u = 0; u < kRwXhistBatch; ++u) {
      const int64_t b = b0 + 64 * u + lane, bc = b < hi ? b : hi - 1;
      x[u] = exp_le0(cell_logp(c[u], w, bc, bp) - lz);  // log_Z is at least the largest log_P
      if (own) x[u] = x[u] / norm;
      if (b >= hi) x[u] = 0;
    }
#pragma unroll
    for (int u = 0; u < kRwXhistBatch; ++u) {
      const bool on = x[u] > 0;
      double* h[NA];
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        const uint32_t k = (kb[u] >> (8 * a)) & 255u;
        if (on && k == kRwNoBin) bad |= 1u << a;
        h[a] = row + a * kRwRows * stride + (k == kRwNoBin ? 0u : k);
      }
#pragma unroll
      for (int s = 0; s < 64 / kRwRows; ++s) {
        if (on && lane / kRwRows == s) {
#pragma unroll
          for (int a = 0; a < NA; ++a)
            __hip_atomic_fetch_add(h[a], x[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        asm volatile("" ::: "memory");  // the groups' turns stay apart
      }
    }
  }
#pragma unroll
  for (int a = 0; a < NA; ++a)
    if (a < na && ((bad >> a) & 1u)) atomicOr(&sc.code[t * sc.n_a + a0 + a], kRwOutside);
  __syncthreads();
  for (int i = lane; i < na * nm; i += 64) {
    const int a = i / nm, k = i - a * nm;
    double s = 0;
    for (int l = 0; l < kRwRows; ++l) s += hl[(a * kRwRows + l) * stride + k];
    sc.hist[((int64_t)(t * sc.n_a + a0 + a) * gridDim.x + blockIdx.x) * nm + k] = s;
  }
}

// ---------------------------------------------------- order parameter
// The rest of a pair's order parameter on its own wavefront, lane l taking
// bins l, l + 64, ... (kRwBinsPerLane of them: n_bin_mixed <= 215): the
// workgroups' histograms added in order, then Calcula_Histograma_Rotado_normX
// after binning (f90:1466-1617), binder (2580-2608) and the Ising scores
// (2042-2182), the steps of finish_order_parameter and cvf_rw_ising_scores on
// the host with sums taken across the lanes.  On the host the 192 pairs of a
// 64 x 3 scan took about 0.4 ms.
constexpr int kRwBinsPerLane = 4;
struct Bins {
  double x[kRwBinsPerLane], p[kRwBinsPerLane], w[kRwBinsPerLane];
};
template <class F>
__device__ inline double bins_sum(int nm, F f) {
  double s = 0;
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i)
    if ((int)threadIdx.x + 64 * i < nm) s += f(i);
  return wave_sum(s);
}
// norm 1, mean 0, variance 1; the mean removed and the scale applied
__device__ inline void bins_standardize(Bins& h, int nm, double& mean, double& a1) {
  const double norma = bins_sum(nm, [&](int i) { return h.p[i] * h.w[i]; });
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i) h.p[i] = h.p[i] / norma;
  mean = bins_sum(nm, [&](int i) { return h.x[i] * h.p[i] * h.w[i]; });
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i) h.x[i] = h.x[i] - mean;
  const double n2 = bins_sum(nm, [&](int i) { return h.p[i] > 0 ? h.p[i] * h.w[i] : 0.0; });
  const double var = bins_sum(nm, [&](int i) { return h.p[i] > 0 ? h.x[i] * h.x[i] * h.p[i] * h.w[i] : 0.0; });
  a1 = sqrt(n2 / var);
  const double a2 = 1 / (n2 * a1);
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i) {
    h.x[i] = h.x[i] * a1;
    h.w[i] = h.w[i] * a1;
    h.p[i] = h.p[i] * a2;
  }
}
// the reference's own check (f90:1510-1533)
__device__ inline bool bins_standard(const Bins& h, int nm) {
  const auto pos = [&](int i, double v) { return h.p[i] > 0 ? v : 0.0; };
  const double norma = bins_sum(nm, [&](int i) { return pos(i, h.p[i] * h.w[i]); });
  const double mean = bins_sum(nm, [&](int i) { return pos(i, h.x[i] * h.p[i] * h.w[i]); });
  const double var = bins_sum(nm, [&](int i) { return pos(i, h.x[i] * h.x[i] * h.p[i] * h.w[i]); }) - mean * mean;
  const double tol = (double)1E-10f;
  return !(fabs(mean) > tol || fabs(norma - 1) > tol || fabs(var - 1) > tol);
}
__device__ inline double ising2d(double z) {
  const double a = (double)0.058137f, b = (double)-2.68949f, c = (double)-0.11235f, d = (double)2.884162f;
  const double z2 = z * z, z4 = z2 * z2, z8 = z4 * z4, z16 = z8 * z8;
  return exp(-(a * z16 + b * z * z + c * fabs(z) + d));
}
__device__ inline double ising3d(double z) {
  const double a = (double)0.196f, c = (double)0.807f, M0 = (double)1.141059404f, A0 = (double)0.436591191f;
  const double q = z * z / (M0 * M0) - 1;
  return A0 * exp(-q * q * (a * z * z / (M0 * M0) + c));
}
// the first bin in order with the largest key (v, then lowest index): its
// index, or -1 where no lane has one (i < 0)
__device__ inline int wave_first_max(double v, int i) {
  for (int o = 32; o > 0; o >>= 1) {
    const double v2 = __shfl_xor(v, o);
    const int i2 = __shfl_xor(i, o);
    if (i2 >= 0 && (i < 0 || v2 > v || (v2 == v && i2 < i))) v = v2, i = i2;
  }
  return i;
}
// the bin's value from the lane that holds it
__device__ inline double bin_value(const double (&v)[kRwBinsPerLane], int k) {
  double r = 0;
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i) r = k >> 6 == i ? v[i] : r;
  return __shfl(r, k & 63);
}

__global__ __launch_bounds__(64) void k_rw_order(RwScan sc, int32_t nm, double peak2d, double peak3d, RwScanOut out) {
  __shared__ double xs[64 * kRwBinsPerLane];
  const int ta = blockIdx.x, lane = threadIdx.x;
  const double2 bin = sc.bin[ta];
  Bins h;
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i) {
    const int k = lane + 64 * i;
    double s = 0;
    if (k < nm)
#pragma unroll 32
      for (int b = 0; b < sc.n_proj; ++b) s += sc.hist[((int64_t)ta * sc.n_proj + b) * nm + k];
    h.p[i] = s;
    h.x[i] = bin.x + ((k + 1) - 0.5) * bin.y;
    h.w[i] = k < nm ? bin.y : 0.0;
  }
  double media, a1, unused;
  bins_standardize(h, nm, media, a1);
  uint32_t code = sc.code[ta];
  if (!bins_standard(h, nm)) code |= kRwMoments;
  // sine stretch of the axis (f90:1530-1534), then norm / mean / variance
  // again with the stretched bin widths (1538-1617)
  const double b = (double)1.53f, pi = (double)3.14159f;
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i) {
    h.x[i] = b * b * sin(pi * h.x[i] / b) / (pi * pi) + h.x[i];
    xs[lane + 64 * i] = h.x[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i) {
    const int k = lane + 64 * i;
    h.w[i] = k >= nm ? 0.0 : k == 0 ? xs[1] - xs[0] : k == nm - 1 ? xs[k] - xs[k - 1] : (xs[k + 1] - xs[k - 1]) / 2.0;
  }
  bins_standardize(h, nm, unused, a1);
  if (!bins_standard(h, nm)) code |= kRwStretched;
  // cumulant of M = x / a1 + media
  const double s = bins_sum(nm, [&](int i) { return h.p[i]; });
  const auto m2 = [&](int i) {
    const double m = (h.x[i] / a1) + media;
    return m * m;
  };
  const double u2 = bins_sum(nm, [&](int i) { return m2(i) * h.p[i] / s; });
  const double u4 = bins_sum(nm, [&](int i) { return m2(i) * m2(i) * h.p[i] / s; });
  // Ising scores
  double f2[kRwBinsPerLane], f3[kRwBinsPerLane];
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i) {
    f2[i] = ising2d(h.x[i]);
    f3[i] = ising3d(h.x[i]);
  }
  const auto on = [&](int i, double v) { return h.p[i] == 0 ? 0.0 : v; };
  const double n_liu = bins_sum(nm, [&](int i) { return on(i, 1.0); });
  const double kl2 = bins_sum(nm, [&](int i) { return on(i, f2[i] > 0 ? (log(f2[i]) - log(h.p[i])) * f2[i] : 0.0); });
  const double kl3 = bins_sum(nm, [&](int i) { return on(i, f3[i] > 0 ? (log(f3[i]) - log(h.p[i])) * f3[i] : 0.0); });
  const double liu2 = bins_sum(nm, [&](int i) { return on(i, sqrt(h.p[i]) * fabs(h.p[i] - f2[i])); });
  const double liu3 = bins_sum(nm, [&](int i) { return on(i, sqrt(h.p[i]) * fabs(h.p[i] - f3[i])); });
  // ZeroTest: the lowest bin with |x| < 1; HeightTest: the highest bin of
  // each side (the first of equals)
  double zv = 0, v1 = 0, v2 = 0;
  int zi = -1, i1 = -1, i2 = -1;
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i) {
    const int k = lane + 64 * i;
    if (k >= nm) continue;
    const double x = h.x[i], p = h.p[i];
    if (x > -1 && x < 1 && p < (double)1E12f && (zi < 0 || -p > zv)) zv = -p, zi = k;
    if (x < 0 && p > -10 && (i1 < 0 || p > v1)) v1 = p, i1 = k;
    if (!(x < 0) && p > -10 && (i2 < 0 || p > v2)) v2 = p, i2 = k;
  }
  zi = wave_first_max(zv, zi);
  i1 = wave_first_max(v1, i1);
  i2 = wave_first_max(v2, i2);
  const double k = (double)(6.0f / 0.8f);
  double zero = (double)1E3f, height = (double)1E3f;
  if (zi >= 0) {
    const double d = bin_value(h.p, zi) - ising3d(0.0), x = bin_value(h.x, zi);
    zero = d * d;
    zero = zero * k * k;
    zero = zero + x * x;
  }
  if (i1 >= 0 && i2 >= 0) {
    const double x1 = (double)-1.14f, x2 = (double)1.14f;
    const double d1 = bin_value(h.p, i1) - ising3d(x1), d2 = bin_value(h.p, i2) - ising3d(x2);
    const double y1 = bin_value(h.x, i1) - x1, y2 = bin_value(h.x, i2) - x2;
    height = d1 * d1 * k * k;
    height = height + d2 * d2 * k * k;
    height = height + y1 * y1;
    height = height + y2 * y2;
  }
#pragma unroll
  for (int i = 0; i < kRwBinsPerLane; ++i) {
    const int kk = lane + 64 * i;
    if (kk < nm) {
      out.x[(int64_t)ta * nm + kk] = h.x[i];
      out.p[(int64_t)ta * nm + kk] = h.p[i];
    }
  }
  if (lane) return;
  out.code[ta] = code;
  double *stats3 = out.stats3, *scores6 = out.scores6;
  stats3[3 * ta] = media;
  stats3[3 * ta + 1] = a1;
  stats3[3 * ta + 2] = 1.0 - u4 / (3.0 * u2 * u2);
  scores6[6 * ta] = kl2;
  scores6[6 * ta + 1] = kl3;
  scores6[6 * ta + 2] = liu2 / ((peak2d - ising2d(0.0)) * n_liu);
  scores6[6 * ta + 3] = liu3 / ((peak3d - ising3d(0.0)) * n_liu);
  scores6[6 * ta + 4] = zero;
  scores6[6 * ta + 5] = height;
}

template <int T, int kMode>
void sum_launch(const RwCells& cells, const RwTargets& tg, const RwWork& w, const RwGeom& g, hipStream_t st) {
  hipLaunchKernelGGL((k_rw_sum<T, kMode>), dim3((unsigned)w.nblk, (unsigned)((tg.n + T - 1) / T)), dim3(w.threads), 0,
                     st, cells, tg, w, g);
}

template <int N>
void sweep_launch(const RwTables& tb, int64_t n, int32_t n_sim, const RwWork& w, bool chain, double* used,
                  hipStream_t st) {
  if constexpr (N < kRwRow)
    if (n_sim > N) return sweep_launch<N + 1>(tb, n, n_sim, w, chain, used, st);
  hipLaunchKernelGGL(k_rw_sweep_cells<N>, dim3((unsigned)w.nblk), dim3(w.threads), 0, st, tb, n, w,
                     chain ? w.ps : nullptr, used);
  hipLaunchKernelGGL(k_rw_sweep_sum<N>, dim3((unsigned)w.nblk), dim3(w.threads), 0, st, tb, n, w);
}

template <int NA>
hipError_t xhist_launch(const RwGeom& g, const RwCells& cells, const RwTargets& tg, const RwWork& w, const RwScan& sc,
                        hipStream_t st) {
  const unsigned groups = (unsigned)((sc.n_a + NA - 1) / NA);
  hipLaunchKernelGGL(k_rw_cell_bins<NA>, dim3((unsigned)((g.n + kRwBlock - 1) / kRwBlock), groups), dim3(kRwBlock), 0,
                     st, g, sc);
  const size_t lds = sizeof(double) * NA * kRwRows * (size_t)(g.nm | 1);
  hipLaunchKernelGGL(k_rw_xhist<NA>, dim3((unsigned)sc.n_proj, (unsigned)tg.n * groups), dim3(64), lds, st, g,
                     cells, tg, w, sc);
  return hipGetLastError();
}

// Angles per wavefront: as many (up to 4) as keep five wavefronts on a CU, one
// at least (27 KB of LDS for 215 bins).
int angles_per_wave(int nm, int n_a) {
  const int fit = (int)(32 * 1024 / (sizeof(double) * kRwRows * (size_t)(nm | 1)));
  return std::max(1, std::min({fit, n_a, 4}));
}

}  // namespace

int32_t rw_angle_groups(int32_t nm, int32_t n_a) {
  const int per = angles_per_wave(nm, n_a);
  return (n_a + per - 1) / per;
}

// At most 256 workgroups per row of targets, since every workgroup of the
// next launch reduces their partial results for itself, and at most one of
// 1024 threads per CU; small grids take smaller workgroups, so that they
// spread over the CUs.  With several rows each takes its share of the CUs
// and a thread more cells: the reductions at the end of a workgroup cost as
// much as about four cells.
void rw_shape(int64_t n_cells, int32_t n_targets, RwWork* w) {
  w->rows = (n_targets + kRwRow - 1) / kRwRow;
  w->threads = n_cells > 163840 ? 1024 : n_cells > 65536 ? 512 : 256;
  const int64_t need = (n_cells + w->threads - 1) / w->threads;
  w->nblk = (int32_t)std::min<int64_t>(need, std::max<int64_t>(kRwMaxBlocks / w->rows, 32));
}

hipError_t launch_rw_pass(const RwCells& cells, const RwSim* sims, const double* ctes, int32_t n_sim,
                          const RwTargets& tg, const RwWork& w, const RwGeom& g, int mode, bool chain, double* used,
                          hipStream_t stream) {
  const unsigned rows = (unsigned)((tg.n + kRwRow - 1) / kRwRow);
  const size_t lds = sizeof(double) * 5 * (size_t)n_sim;
  // (the last row of many may hold fewer targets: it repeats one)
  auto* k = tg.n <= 2 ? k_rw_cells<2> : tg.n <= 4 ? k_rw_cells<4> : tg.n <= 8 ? k_rw_cells<8> : k_rw_cells<kRwRow>;
  hipLaunchKernelGGL(k, dim3((unsigned)w.nblk, rows), dim3(w.threads), lds, stream, cells, sims, ctes, n_sim, tg, w,
                     chain ? w.ps : nullptr, w.mx, used);
  // a sweep over few cells leaves the card idle: its targets go to more
  // workgroups (12 simulations, 30,578 / 61,945 / 158,675 cells: 19.1 / 21.8 / 28.4 us a
  // sweep in tiles of 4, 20.1 / 21.7 / 26.5 of 8, 21.5 / 22.6 / 27.6 of 16; 323,311 cells
  // 34.3 / 32.1 / 29.7)
  const int tile = tg.n <= 2 ? 2 : tg.n <= 4 || cells.n <= 81920 ? 4 : tg.n <= 8 || cells.n <= 163840 ? 8 : kRwRow;
  if (mode == kRwSweep)
    tile == 2   ? sum_launch<2, kRwSweep>(cells, tg, w, g, stream)
    : tile == 4 ? sum_launch<4, kRwSweep>(cells, tg, w, g, stream)
    : tile == 8 ? sum_launch<8, kRwSweep>(cells, tg, w, g, stream)
                : sum_launch<kRwRow, kRwSweep>(cells, tg, w, g, stream);
  else if (mode == kRwDensity)
    sum_launch<8, kRwDensity>(cells, tg, w, g, stream);
  else
    sum_launch<4, kRwScan>(cells, tg, w, g, stream);
  return hipGetLastError();
}

hipError_t launch_rw_tables(const RwCells& cells, const RwSim* sims, int32_t n_sim, const RwGeom& g, int32_t N,
                            const RwTables& tb, hipStream_t st) {
  const int64_t items = cells.n + n_sim * (2 * (int64_t)g.nb + 1);
  hipLaunchKernelGGL(k_rw_tables, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, st, cells, sims, n_sim, g, N,
                     tb);
  return hipGetLastError();
}

hipError_t launch_rw_sweep(const RwTables& tb, int64_t n_cells, int32_t n_sim, const RwWork& w, bool chain,
                           double* used, hipStream_t st) {
  sweep_launch<2>(tb, n_cells, n_sim, w, chain, used, st);
  return hipGetLastError();
}

hipError_t launch_rw_finish(const RwTargets& tg, const RwWork& w, const RwGeom& g, int mode, double* binder_ed,
                            hipStream_t st) {
  auto* k = mode == kRwSweep ? k_rw_finish<kRwSweep> : mode == kRwDensity ? k_rw_finish<kRwDensity>
                                                                          : k_rw_finish<kRwScan>;
  hipLaunchKernelGGL(k, dim3((unsigned)tg.n), dim3(64), 0, st, w, g.de, g.drho, binder_ed);
  return hipGetLastError();
}

hipError_t launch_rw_dist(const RwCells& cells, const RwTargets& tg, const RwWork& w, double* dens, hipStream_t st) {
  const unsigned nb = (unsigned)((cells.n + kRwBlock - 1) / kRwBlock);
  hipLaunchKernelGGL(k_rw_dist, dim3(nb, (unsigned)tg.n), dim3(kRwBlock), 0, st, cells, tg, w, dens);
  return hipGetLastError();
}

int32_t rw_proj_blocks(int64_t n_cells, int32_t n_targets) {
  const int64_t fill = std::min<int64_t>(1792 / n_targets, n_cells / 1024) / 32 * 32;
  return (int32_t)std::max<int64_t>(kRwProjBlocks, std::min<int64_t>(kRwMaxBlocks, fill));
}

hipError_t launch_rw_project(const RwCells& cells, const RwTargets& tg, const RwWork& w, const RwGeom& g,
                             const RwScan& sc, double peak2d, double peak3d, const RwScanOut& out, hipStream_t st) {
  const unsigned nta = (unsigned)(tg.n * sc.n_a);
  hipLaunchKernelGGL(k_rw_xrange, dim3((unsigned)sc.n_proj, (unsigned)sc.n_a + nta), dim3(kRwBlock), 0, st, g, cells, tg, w,
                     sc);
  hipLaunchKernelGGL(k_rw_bins, dim3((unsigned)sc.n_a + nta), dim3(64), 0, st, w, sc, g.nm);
  const int na = angles_per_wave(g.nm, sc.n_a);
  const hipError_t e = na >= 4   ? xhist_launch<4>(g, cells, tg, w, sc, st)
                       : na == 3 ? xhist_launch<3>(g, cells, tg, w, sc, st)
                       : na == 2 ? xhist_launch<2>(g, cells, tg, w, sc, st)
                                 : xhist_launch<1>(g, cells, tg, w, sc, st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_rw_order, dim3(nta), dim3(64), 0, st, sc, g.nm, peak2d, peak3d, out);
  return hipGetLastError();
}

}  // namespace cvf

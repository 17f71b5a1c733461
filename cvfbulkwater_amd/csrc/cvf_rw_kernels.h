// Device side of the histogram reweighting (include/cvf_reweight.h): the
// per-cell log-sum over simulations, the per-target reductions and the
// projections of a scan.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace cvf {

constexpr int kRwBlock = 256;
constexpr int kRwRow = 16;          // targets that share one pass over the cells' simulation sums
constexpr int kRwProjBlocks = 64;   // the fewest workgroups per target (or pair) of a projection
// what a pass is for: a sweep of the constants (log_Z alone), densities
// (and the normalization), a scan (and the moments of the marginals)
enum { kRwSweep = 0, kRwDensity = 1, kRwScan = 2 };
constexpr int kRwScanSums = 6;

// One simulation of the reweighting sums: beta_j = 1000/(0.2293 T_j) in
// mol/kJ, p_j = 100 P_j in kPa, lm_j = log(real(medidas_j)).
struct RwSim {
  double beta, pres, lm, pad;
};

// Occupied cells of the (e, rho) grid, structure of arrays in HBM.
struct RwCells {
  const double* en;  // e * N at the cell centre (kJ/mol)
  const double* vn;  // V * N = 0.018 N / rho (m^3/mol)
  const double* lh;  // log of the summed normalized histograms
  int64_t n;
};

struct RwTargets {
  const double2* bp;  // (beta, p) of each target
  int32_t n;
};

// Both sums of a cell and the bounds that pick one.
struct RwMixed {
  double near, all, umax, umin;
};

// Buffers of one reweighting pass over n targets.
struct RwWork {
  double* sum;     // [row][cell]: the simulation sum that the row's targets use
  uint8_t* mixed;  // [row][cell]: the row's targets use different ones (mix[cell])
  RwMixed* mix;    // [cell], written where mixed
  double* pmax;    // [row][block][target of the row] partial maxima of log_P
  double* mx;      // [target] max log_P
  double* ps;      // [sum][row][block][target of the row] partial sums
  uint32_t* plow;  // [target][block] of a scan: a density may have underflowed
  uint32_t* low;   // [target] the same
  double* lz;      // [target] log_Z
  double* norm;    // [target] sum of exp(log_P - log_Z) * de * drho
  int32_t rows, nblk, threads;  // rows of targets; launch shape (rw_shape)
};

// What the sweeps of the constants take from tables instead of exponentials.
// With x_j(c) = -(beta_j - beta_0)(E - E0) - (beta_j p_j - beta_0 p_0)(V - V0),
// E0 and V0 of the grid's middle, exp(x_j) is a factor of the cell's energy row
// times one of its density column, and exp(u_j) = exp(x_j + w_j - t1_0) with
// w_j = lm_j - g_j - c_j the same for all cells.
struct RwTables {
  double2 *row, *col;    // [pair of simulations][nb]
  double2* sc;           // [simulation]: g_j = (beta_j - beta_0) E0 + (beta_j p_j - beta_0 p_0) V0, and lm_j
  double* kt;            // [3][kRwRow] of a sweep: g_t + max w, and the bounds of the cut (k_rw_sweep_cells)
  double* h;             // [cell]: summed normalized histograms
  const uint32_t* cell;  // i << 16 | w
  int32_t nb;
};
// The largest |x_j| that the tables serve, and the largest |log| of a cell's
// histogram: no product or quotient of a sweep leaves the range of a double.
constexpr double kRwMaxShift = 150, kRwMaxLogHist = 100;

// Grid geometry for the projections: cell = i << 16 | w (nb < 2^16), energy
// e_min + (i + 1/2) de (kJ/mol), density rho_min + (w + 1/2) drho (kg/m^3).
struct RwGeom {
  const uint32_t* cell;
  int64_t n;
  int32_t nb, nm;
  double e_min, de, rho_min, drho;
};

// Buffers of a scan's projections; pair ta = target * n_a + angle.
struct RwScan {
  const double2* angle;  // (sin, cos) per angle
  int32_t n_a;
  double2* range;  // [n_a + pairs][n_proj]: min and max of x
  double2* bin;    // [pair]: first bin's lower edge, bin width
  double2* gbin;   // [n_a]: the same over all the grid's cells
  uint32_t* cbin;  // [group of up to 4 angles][cell]: the cell's bins, a byte per angle
  double* hist;    // [pair][n_proj][nm]
  uint32_t* code;  // [pair]: kRwNoCell, kRwOutside
  int32_t n_proj;  // workgroups per target (or pair) of a projection
};
// As many workgroups per target as fill the card with histograms (one
// wavefront each, seven on a CU), a thousand cells each at least; 64 of them
// left most CUs idle for a few targets.  One angle, 710,000 cells, 1 / 5 / 10 / 16
// targets: 64 workgroups 217 / 235 / 248 / 262 us, so many 131 / 150 / 178 / 210.
int32_t rw_proj_blocks(int64_t n_cells, int32_t n_targets);
// Groups of angles that a pass over the cells takes together (RwScan::cbin).
int32_t rw_angle_groups(int32_t nm, int32_t n_a);
// What went wrong with a pair: no cell of positive density, an x outside its
// bins, moments off before or after the axis stretch.
enum : uint32_t { kRwNoCell = 1, kRwOutside = 2, kRwMoments = 4, kRwStretched = 8 };
// A scan's results, written straight to pinned host memory.
struct RwScanOut {
  double *binder_ed, *x, *p, *stats3, *scores6;
  uint32_t* code;
};

// Fills in the launch shape of a pass over n_cells cells.
constexpr int kRwMaxBlocks = 256;  // workgroups per row of targets
void rw_shape(int64_t n_cells, int32_t n_targets, RwWork* w);

// One pass over the cells for every target (Calcula_Histograma over all
// targets): the cells' sums, then the partial sums of `mode`.  chain: the
// constants are log_Z(t) - log_Z(0) of the pass before (a kRwSweep pass over
// the same targets, the simulations themselves), written to `used`.
hipError_t launch_rw_pass(const RwCells& cells, const RwSim* sims, const double* ctes, int32_t n_sim,
                          const RwTargets& tg, const RwWork& w, const RwGeom& g, int mode, bool chain, double* used,
                          hipStream_t stream);
// The tables of n_sim simulations (2 .. kRwRow) for molecules N, and a sweep
// with them: chain as above, else from constants of zero.
hipError_t launch_rw_tables(const RwCells& cells, const RwSim* sims, int32_t n_sim, const RwGeom& g, int32_t N,
                            const RwTables& tb, hipStream_t st);
hipError_t launch_rw_sweep(const RwTables& tb, int64_t n_cells, int32_t n_sim, const RwWork& w, bool chain,
                           double* used, hipStream_t st);
// log_Z, norm and (kRwScan) the Binder cumulants {energy, density} per target
hipError_t launch_rw_finish(const RwTargets& tg, const RwWork& w, const RwGeom& g, int mode, double* binder_ed,
                            hipStream_t st);
// dens[target][cell] = exp(log_P - log_Z) / norm
hipError_t launch_rw_dist(const RwCells& cells, const RwTargets& tg, const RwWork& w, double* dens, hipStream_t st);
// The order parameter of every pair (Calcula_Histograma_Rotado_normX, binder,
// ConfrontIsing, ZeroTest, HeightTest) after a finished kRwScan pass.
hipError_t launch_rw_project(const RwCells& cells, const RwTargets& tg, const RwWork& w, const RwGeom& g,
                             const RwScan& sc, double peak2d, double peak3d, const RwScanOut& out, hipStream_t st);

}  // namespace cvf

// Device-side data structures and the host launchers of the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "cvf_core.h"

namespace cvf {

constexpr int kNumXcd = 8;  // MI355X: 8 XCDs, workgroups dispatched round-robin

// Immutable per-state-point description (device copy).
struct PointDev {
  uint64_t seed;
  uint32_t L, N, hL;
  uint32_t woff;       // offset of the point's words in the state array
  uint32_t loff;       // offset of the point's 6N labels
  uint32_t shell_off;  // offset of its shell table
  int32_t jeff_sign;   // sign of Jeff (SW covalent rule, gpu_water3D.cu:2399-2424)
  uint32_t pad;
  VolParams vp;
  uint64_t thr_sigma[33];  // index (eta*dhb + 1)*11 + dsig + 5
  uint64_t thr_eta[9];     // index DeltaN_HB + 4
  uint64_t thr_sw[2];      // covalent, intra-molecule link activation
};

// Mutable per-state-point device state.
struct PointState {
  uint64_t step;  // next MC step index of this point
  VolState vol;
};

// One workgroup's work: the state point, the first work item, and every
// per-point scalar the kernels need, so that one scalar load of the entry
// starts a workgroup (96 bytes).
struct BlockEnt {
  int32_t point;  // -1: padding entry
  uint32_t start;  // first work item (or first plane of a slab)
  uint32_t L, N, woff, loff;
  uint32_t seed_lo, seed_hi;
  uint32_t mL, mH, mQ;  // fast-division multipliers for L, L/2, L/4
  int32_t jeff_sign;
  uint32_t thb_lo, thb_hi, ts_lo, ts_hi;  // SW link thresholds
  uint32_t mLL, mP8, mP4, mC;  // multipliers for L^2, L^2/8, L^2/4, L^2/16
  uint32_t T;                  // slab thickness (planes) of the fused kernel
  uint32_t flags;              // kEntNoChess: the point runs without the chessboard
  uint32_t pad[2];
};

constexpr uint32_t kEntNoChess = 1;

constexpr int kChunk = 6;      // half-sweeps per fused kernel (default)
constexpr int kMaxChunk = 12;  // half-sweeps per fused kernel at most: a whole Metropolis pass
constexpr int kMaxSlab = 16;  // planes per slab of the fused kernel

struct Launch {
  const BlockEnt* tab;
  uint32_t nblocks;      // padded to a multiple of kNumXcd
  uint32_t block;        // threads per workgroup
  const uint64_t* step;  // the group's step counter (first step of the captured sequence)
  uint32_t step_off;     // this launch's step within the sequence
};

// Per-kernel timing for profiling: while set, launches go through
// hipExtLaunchKernelGGL with these start/stop events (nullptr to clear).
void set_launch_timing(hipEvent_t start, hipEvent_t stop);

// Launchers (all asynchronous on `st`).
// after nsteps lattice steps of a group: *gstep += nsteps and, with `moves`,
// the device volume moves of those steps for the listed points
void launch_vol_chain(hipStream_t st, const PointDev* pts, const int32_t* plist, int npts, PointState* ps,
                      uint64_t* gstep, uint32_t nsteps, const float* dist, const int32_t* freq,
                      int precision, int moves);
void launch_eta(hipStream_t st, Launch ln, const PointDev* pts, uint32_t* words, int family);
void launch_sigma(hipStream_t st, Launch ln, const PointDev* pts, uint32_t* words, uint32_t sub);
// one colour pass of the fast schedule (pass = 2 x Metropolis iteration +
// colour), over the half-sweep table (N/8 quads per point)
void launch_sigma_f(hipStream_t st, Launch ln, const PointDev* pts, uint32_t* words, uint32_t pass);
// Fused z-slab kernel: optional eta sweep + half-sweeps k0 .. k0+nk-1 of the
// step on LDS-staged slabs, reading `src` and writing `dst`; any_nc: the
// table holds non-chessboard slabs.
void launch_chunk(hipStream_t st, Launch ln, const PointDev* pts, const uint32_t* src, uint32_t* dst,
                  uint32_t k0, uint32_t nk, int with_eta, uint32_t lds_bytes, bool any_nc);
// largest dynamic LDS a fused launch may use
uint32_t chunk_lds_limit();
// One workgroup of the tile kernel (cvf_tile.hip): the core box of tx x ty x
// tz quads at quad (x0, y0, z0) of a point folded over its quadrants, x0 + tx
// and y0 + ty <= L/2, z0 + tz <= L.  point < 0: padding.
struct TileEnt {
  int32_t point;
  uint32_t L, woff, seed_lo, seed_hi;
  uint32_t x0, y0, z0, tx, ty, tz, nc;  // nc: runs without the chessboard
};
constexpr int kMaxTileWin = 64;  // quads along one axis of a window
constexpr uint32_t kMaxTile = kMaxTileWin - 2 * kMaxChunk - 2;
constexpr uint32_t kTileMinBlock = 64 + 3 * kMaxTileWin;  // threads: a wavefront, and one per entry of the axes' tables
// quads of the largest window of a tile for nk half-sweeps (and the cube
// sweep; nc: of a non-chessboard point)
uint32_t tile_window_quads(uint32_t tx, uint32_t ty, uint32_t tz, uint32_t nk, bool nc);
// largest dynamic LDS of a tile workgroup
constexpr uint32_t tile_lds_limit() { return 160 * 1024 - 4096; }
// As launch_chunk, on the ntiles (a multiple of kNumXcd) boxes of `tab`;
// workgroups of at least kTileMinBlock threads.
void launch_tile(hipStream_t st, const TileEnt* tab, uint32_t ntiles, uint32_t block, const uint64_t* stepp,
                 uint32_t step_off, const PointDev* pts, const uint32_t* src, uint32_t* dst, uint32_t k0, uint32_t nk,
                 int with_eta, uint32_t lds_bytes, bool any_nc);
void launch_zero_u32(hipStream_t st, uint32_t* p, size_t n);
void launch_zero3_u32(hipStream_t st, uint32_t* a, size_t na, uint32_t* b, size_t nb, uint32_t* c, size_t nc);
// Cells per k_observe workgroup (a multiple of 1024): small handles spread
// over more workgroups (L = 32: 32 of them), large ones keep the host's sum of
// the partial results short.
constexpr uint32_t observe_span(size_t total_cells) { return total_cells < (1u << 20) ? 1024 : 4096; }
// A sample's results in host memory (pinned, device-visible): per workgroup
// of the table the pair (2 N_HB, N_sigma) of its cells, every point's
// mutable state and the resident kernel's abort flag.
struct ObsOut {
  uint2* part;
  PointState* ps;
  uint32_t* status;
};
void launch_observe(hipStream_t st, const BlockEnt* tab, uint32_t nblocks, const uint32_t* words, uint32_t span,
                    const PointState* ps, const uint32_t* rstatus, const ObsOut& out, uint8_t* bonds);
// Capped counts of n non-chessboard points (no larger than maxL) from the bond
// bytes that launch_observe left at `bonds` + woff (null there if the handle
// has no such point); they are used up.  2 N_HB of a point goes to out[point].
struct CappedEnt {
  int32_t point;
  uint32_t L, woff, mH;  // mH: fast-division multiplier for L / 2
};
constexpr uint32_t kCappedLds = 160 * 1024 - 256;
void launch_capped_hb(hipStream_t st, const CappedEnt* ent, uint32_t n, uint32_t maxL, uint8_t* bonds, uint32_t* out);
// The words W of a point (N cells) as sigma and eta arrays (6N bytes each).
void launch_config_out(hipStream_t st, const uint32_t* W, uint32_t N, uint8_t* sigma, uint8_t* eta);
// sigma and eta arrays to the words W through `scratch` (L^3 words): *first
// (all ones before) tells the first value out of range, then W is not
// written; *inconsistent counts up the cubes whose eta was not a solution.
// *flag is the resident launches' abort flag: if it is set, neither scratch nor
// W is written.
void launch_config_in(hipStream_t st, const uint8_t* sigma, const uint8_t* eta, uint32_t L, int chessboard,
                      uint32_t* scratch, uint32_t* W, uint32_t* first, uint32_t* inconsistent,
                      const uint32_t* rstatus, uint32_t* flag);
void launch_sw_local(hipStream_t st, Launch ln, const uint32_t* words, uint32_t* parent, uint8_t* cov,
                     uint32_t jc);
void launch_sw_union(hipStream_t st, Launch ln, uint32_t* parent, const uint8_t* cov);
void launch_sw_flip(hipStream_t st, Launch ln, uint32_t* words, uint32_t* parent, uint32_t jc);
// sigma histogram as kHistReplicas partial histograms of 6 counters
// (kHistWords counters, zeroed by the caller) that the caller sums; *flag: the
// resident launches' abort flag (with rstatus)
constexpr int kHistReplicas = 8;
constexpr int kHistWords = 6 * kHistReplicas;
void launch_sigma_hist(hipStream_t st, const uint32_t* W, uint32_t N, unsigned long long* counts,
                       const uint32_t* rstatus, unsigned long long* flag);
// the same into slot (*gstep + step_off - *base) of a per-step series of
// `span` histograms (graph-replayable: the slot is read on the device)
void launch_sigma_hist_slot(hipStream_t st, const uint32_t* W, uint32_t N, unsigned long long* series,
                            const uint32_t* rstatus, unsigned long long* flag, const uint64_t* gstep,
                            uint32_t step_off, const uint64_t* base, uint32_t span);
// cluster statistics of one point (labels at `label`, 6N nodes)
// Per cluster root the cluster's other nodes (others[0..nn) zero before).
void launch_cluster_sizes(hipStream_t st, const uint32_t* label, uint32_t nn, int32_t* others);
// A labelling's clusters in host memory (pinned): their count, the sum and sum
// of squares of their sizes, the largest two, the percolation slots taken and
// the percolating ones; the resident launches' abort flag.
struct ClusterSums {
  uint64_t sum, squares;
  uint32_t largest, second, clusters, slots, percolating, aborted;
};
// Counts and moments per workgroup of kCompactSpan nodes (bcount and 4 words
// each of bmom, compact_blocks(nn) of them) and a slot for each cluster of at
// least minsize nodes; then, after the percolation test, the counts' offsets
// and the sums, and, with the offsets, the sizes in label order.
constexpr uint32_t kCompactSpan = 4096;
uint32_t compact_blocks(uint32_t nn);
void launch_compact_count(hipStream_t st, const uint32_t* label, const int32_t* others, uint32_t nn, uint32_t* bcount,
                          uint64_t* bmom, uint32_t minsize, int32_t* slot, uint32_t* nslot, uint32_t max_slots);
void launch_compact_scan(hipStream_t st, uint32_t* bcount, uint32_t nn, const uint64_t* bmom,
                         const uint32_t* nslot_nperc, const uint32_t* rstatus, ClusterSums* out);
void launch_compact_write(hipStream_t st, const uint32_t* label, const int32_t* others, uint32_t nn,
                          const uint32_t* bcount, int32_t* out);
void launch_perc_cover(hipStream_t st, const uint32_t* label, uint32_t nn, uint32_t L, const int32_t* others,
                       uint32_t minsize, const int32_t* slot, const uint32_t* nslot, uint32_t* cover,
                       uint32_t max_slots);
void launch_perc_count(hipStream_t st, const uint32_t* cover, const uint32_t* nslot, uint32_t L,
                       uint32_t max_slots, uint32_t* nperc);
void launch_vdw_eval(hipStream_t st, const float* dist, const int32_t* freq, int nshell,
                     float r_cutoff, int N, const double* r, int n_r, int precision, double* out);
// vdW pair form (validation of the shell table): per-workgroup partial sums
// over ordered pairs, vdw_pair_blocks(L) per radius, radius-major in `part`
uint32_t vdw_pair_blocks(int L);
void launch_vdw_pairs(hipStream_t st, int L, float r_cutoff, const double* r, int n_r, int precision, double* part);
// the events set by set_launch_timing (nullptr when launches are not timed)
void get_launch_timing(hipEvent_t* start, hipEvent_t* stop);

// ------------------------------------------------- resident Metropolis kernel
// One z-slab of one state point held in a resident workgroup's LDS
// (cvf_resident.hip), worked on by its own waves of the workgroup.  Its
// window: the ghost of the plane below, its T planes, the ghost of the
// plane above (no ghosts when ns = 1: the whole lattice, periodic in LDS).  Its rings in `rings` (words): [ring, ring +
// 2 kRingHalf L^2) its bottom plane as published for the slab below, then
// its top plane for the slab above, each a step-parity half of kRingHalf
// L^2-word slots holding 64-bit tagged words (two slots per plane);
// versions ver[2 i] (bottom), ver[2 i + 1] (top) for slab i.
struct RSlab {
  int32_t point;
  uint32_t L, z0, T, ns;      // ns: slabs of the point
  uint32_t woff, lds;         // the point's words; the window's first LDS word
  uint32_t seed_lo, seed_hi;
  uint32_t mH, mQ, mP8, mP4, mQQ;  // fast-division multipliers of L/2, L/4, L^2/8, L^2/4, (L/4)^2
  int32_t above, below;       // neighbouring slabs (ns > 1), indices into the slab array
  uint32_t ring;              // this slab's rings
  uint32_t ring_hi, ring_lo;  // the rings of `above` and `below`
  uint32_t w0, nw;            // its waves [w0, w0 + nw) of the workgroup
  // a lane's walk over a phase's items advances by 64 nw items: dp planes
  // and du items of L^2/8 (in-plane quads), L^2/4 (z quads) or (L/4)^2
  // (four-cube items) per plane
  uint32_t dp8, du8, dp4, du4, dpc, duc;
  uint32_t mS;  // fast-division multiplier of that stride, 64 nw
};
static_assert(sizeof(RSlab) % 16 == 0, "RSlab is copied in words");
// Workgroup g of a resident launch takes slabs [first, first + count).
struct RGroupEnt {
  uint32_t first, count;
};
constexpr uint32_t kMaxRSlabs = 8;   // slabs per resident workgroup
constexpr uint32_t kRingHalf = 32;   // ring slots per step parity: 2k, 2k + 1 after half-sweep k; 30, 31 at step end
constexpr uint32_t kResidentStatic = 6144;  // static LDS reserved for a resident workgroup
// largest dynamic LDS of a resident workgroup (its static arrays take the
// rest of the CU's 160 KB; each further workgroup on a CU takes another
// kResidentStatic)
uint32_t resident_lds_limit();
// resident workgroups of `block` threads and `lds_bytes` of dynamic LDS that
// fit on one CU at once
hipError_t resident_occupancy(int* per_cu, uint32_t block, uint32_t lds_bytes, bool fine, bool fast);
// fine: the instantiation for plans of thin slabs (at most two planes):
// in-plane half-sweeps whose quads fit half of a slab's lanes run two cells
// per lane (one, below 64 quads), cube families whose cubes fit the lanes one cube per lane, and
// z half-sweeps one cell per lane where that fits, else two where that
// does, instead of one quad (one four-cube item) per lane
// The launch's first step is *stepp + step_off, or step_off itself without
// stepp; with step_out (then no stepp) the step after its last goes there.
// The lattice that it starts from stays in `kept` (null: that of an earlier
// launch serves), for the steps to be done again if a wait times out: then
// status[0] is not zero, and status[1] the launch_mark of the first step of the
// launch whose start `kept` holds.  Launches after it with `kept` do nothing.
constexpr uint32_t launch_mark(uint64_t step) { return (uint32_t)(step + 1) | 0x80000000u; }
void launch_resident(hipStream_t st, const RGroupEnt* grp, uint32_t ngroups, uint32_t block, uint32_t lds_bytes,
                     const RSlab* slabs, const PointDev* pts, uint32_t* words, uint32_t* kept, uint32_t* rings,
                     uint64_t* ver, const uint64_t* stepp, uint64_t step_off, uint32_t nsteps, uint64_t* step_out, uint32_t* status,
                     bool fine, bool fast);
// The same for plans of the reference schedule whose workgroups hold one
// one-plane slab each (cvf_plane.hip), the moves of `per` half-sweeps (a
// divisor of 12) laid out at a time in plane_lds_bytes of dynamic LDS.
uint32_t plane_lds_bytes(uint32_t L, uint32_t per);
hipError_t plane_occupancy(int* per_cu, uint32_t block, uint32_t lds_bytes);
void launch_plane(hipStream_t st, const RGroupEnt* grp, uint32_t ngroups, uint32_t block, uint32_t lds_bytes,
                  const RSlab* slabs, const PointDev* pts, uint32_t* words, uint32_t* kept, uint32_t* rings,
                  uint64_t* ver, const uint64_t* stepp, uint64_t step_off, uint32_t nsteps, uint64_t* step_out, uint32_t* status,
                  uint32_t per);

}  // namespace cvf

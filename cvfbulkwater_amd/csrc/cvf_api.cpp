// C ABI of the engine (include/cvf_api.h): handle management, state
// packing, block tables, hipGraph capture of one MC step, observables and
// cluster statistics.
#include "cvf_api.h"

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "cvf_core.h"
#include "cvf_gate.h"
#include "cvf_host.h"
#include "cvf_kernels.h"

using namespace cvf;

namespace {

thread_local std::string g_err;

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}

#define HIPC(expr)                                                                  \
  do {                                                                              \
    hipError_t e_ = (expr);                                                         \
    if (e_ != hipSuccess)                                                           \
      return fail(CVF_EDEVICE, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), \
                  __FILE__, __LINE__);                                              \
  } while (0)

template <class T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { reset(); }
  void reset() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
  hipError_t alloc(size_t count) {
    reset();
    n = count;
    return hipMalloc((void**)&p, std::max<size_t>(count, 1) * sizeof(T));
  }
};

// Pinned host memory that kernels write directly.
template <class T>
struct PinBuf {
  T* p = nullptr;
  size_t n = 0;
  PinBuf() = default;
  PinBuf(const PinBuf&) = delete;
  PinBuf& operator=(const PinBuf&) = delete;
  ~PinBuf() { reset(); }
  void reset() {
    if (p) (void)hipHostFree(p);
    p = nullptr;
    n = 0;
  }
  hipError_t alloc(size_t count) {
    reset();
    n = count;
    return hipHostMalloc((void**)&p, std::max<size_t>(count, 1) * sizeof(T), hipHostMallocDefault);
  }
};

struct PointHost {
  cvf_params prm;
  uint32_t L, N, woff, loff, shell_off;
  Thresholds thr;
  std::vector<float> dist;
  std::vector<int32_t> freq;
  VolState vol;  // host copy (authoritative in host-volume mode)
  VolParams vp;
  int32_t group = 0;    // stream group under the current tuning
  uint32_t slab_T = 0;  // planes per slab of its fused launches (0: unfused kernels)
};

// A group of state points advanced by its own stream: its own block tables,
// step slot and captured graphs.  Groups share nothing mutable, so their
// launch sequences overlap on separate hardware queues.  A handle's only group
// uses the handle's main stream: the card has few hardware queues, and a stream
// that is never used still takes one, so that the launches of two handles
// end up in the same one, behind each other.
struct Group {
  std::vector<int> points;
  hipStream_t stream = nullptr;
  bool own_stream = false;
  hipEvent_t done = nullptr;
  DevBuf<BlockEnt> tab_half, tab_cube, tab_cell, tab_slab;
  DevBuf<int32_t> plist;
  uint32_t nb_half = 0, nb_cube = 0, nb_cell = 0, nb_slab = 0;
  bool fused = false;        // eta + sigma through the fused slab kernel
  uint32_t chunk_lds = 0;    // dynamic LDS bytes of a fused launch
  uint32_t chunk_lds_long = 0;  // the same for kMaxChunk half-sweeps; 0 if that does not fit
  uint32_t chunk_lds_eta = 0;   // the same for the eta sweep alone (fast schedule)
  bool any_nc = false;          // some point runs the non-chessboard rule
  // fused launches on tiles instead of slabs (chunk_lds, chunk_lds_long hold
  // their LDS then)
  bool tiled = false;
  DevBuf<TileEnt> tab_tile;
  uint32_t nb_tile = 0;
  size_t sigma_cells = 0;    // cells swept per fused launch
  // resident Metropolis kernel (tuning fused = 2): slabs dealt to at most one
  // workgroup per CU, their neighbour rings and versions
  bool resident = false;
  DevBuf<RSlab> rslabs;
  DevBuf<RGroupEnt> rgroups;
  DevBuf<uint32_t> rings;
  DevBuf<uint64_t> rver;
  uint32_t r_ngroups = 0, r_lds = 0;
  bool r_fine = false;  // every slab at most two planes: the fine instantiation
  uint32_t r_per = 0;   // one plane per workgroup: the plane kernel, this many half-sweeps at a time (0: not)
  // a second stream beside `stream` for the device volume chain of a
  // resident sequence, which never reads the lattice (fork / join events), and
  // for the capture of a resident group's graphs
  hipStream_t side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  // captured step sequences, longest first: graph_steps, then the powers of
  // two below it, so any step count is a few graph launches
  std::vector<int> gsteps;
  std::vector<hipGraph_t> graphs;
  std::vector<hipGraphExec_t> gexecs;
  // the same sequences with a sigma histogram of one point after every
  // step (cvf_step_histograms), captured on demand
  std::vector<hipGraph_t> rgraphs;
  std::vector<hipGraphExec_t> rgexecs;
  size_t cells = 0;
  void drop_rec_graphs() {
    for (auto e : rgexecs)
      if (e) (void)hipGraphExecDestroy(e);
    for (auto g : rgraphs)
      if (g) (void)hipGraphDestroy(g);
    rgraphs.clear();
    rgexecs.clear();
  }
  void drop_graphs() {
    drop_rec_graphs();
    for (auto e : gexecs)
      if (e) (void)hipGraphExecDestroy(e);
    for (auto g : graphs)
      if (g) (void)hipGraphDestroy(g);
    gsteps.clear();
    graphs.clear();
    gexecs.clear();
  }
  ~Group() {
    drop_graphs();
    if (done) (void)hipEventDestroy(done);
    if (fork) (void)hipEventDestroy(fork);
    if (join) (void)hipEventDestroy(join);
    if (side) (void)hipStreamDestroy(side);
    if (own_stream) (void)hipStreamDestroy(stream);
  }
};

}  // namespace

namespace cvf {
int set_error(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}
}  // namespace cvf

// Resident launches of several handles (cvf_gate.h).
struct HipStreams {
  using Event = hipEvent_t;
  using Stream = hipStream_t;
  static bool idle(Stream st) { return hipStreamQuery(st) == hipSuccess; }
  static int after(Stream st, Stream other, Event e) {
    if (hipError_t err = hipEventRecord(e, other)) return err;
    return hipStreamWaitEvent(st, e, 0);
  }
};
ResidentGate<HipStreams> g_resident_gate;
using GateUser = ResidentGate<HipStreams>::User;

struct ResidentTurn {
  GateUser* u = nullptr;
  hipError_t take(GateUser* user) {
    const hipError_t e = (hipError_t)g_resident_gate.enter(user);
    if (e == hipSuccess) u = user;
    return e;
  }
  ~ResidentTurn() {
    if (u) g_resident_gate.leave(u);
  }
};

struct cvf_sim {
  int device = 0;
  hipStream_t stream = nullptr;  // main stream: uploads, observables, statistics
  hipEvent_t start_ev = nullptr;
  int npts = 0;
  int nm = 1, nc = 0, precision = CVF_FP64, vol_device = 0, sched = CVF_SCHED_REFERENCE;
  std::vector<PointHost> ph;
  size_t total_cells = 0, total_nodes = 0;
  cvf_tuning tune{};

  DevBuf<uint32_t> words, words2, parent, cover, nslot_nperc;  // words2: ping-pong partner
  DevBuf<uint8_t> cov, cfg_bytes;
  DevBuf<int32_t> csize, slot, cclusters;  // clusters' nodes but their roots, percolation slots, compacted sizes
  DevBuf<uint32_t> cblock;                  // per-workgroup cluster counts of the compaction
  DevBuf<uint64_t> cmom;                    // per-workgroup size moments (4 words each)
  DevBuf<PointDev> pts;
  DevBuf<PointState> pst;
  DevBuf<float> dist;
  DevBuf<int32_t> freq;
  DevBuf<uint64_t> cur_steps;          // one slot per group
  DevBuf<BlockEnt> tab_cell_all;       // every point's cells, for observables
  // sigma histogram of one point, per-step histograms (kHistWords counters
  // each, the abort flag before them)
  DevBuf<unsigned long long> hist, hist_series;
  DevBuf<uint64_t> hist_base;              // step count at the first recorded step
  DevBuf<uint32_t> rstatus;                // abort flag of the resident kernel, launch_mark of the launch
  bool resident_used = false;              // some launch ran the resident kernel
  GateUser turn;                           // of its resident plan, if it has one
  uint64_t hist_base_host = 0;
  int rec_pt = -1;                         // point recorded by the groups' rec graphs
  uint32_t nb_cell_all = 0;
  std::vector<std::unique_ptr<Group>> groups;
  uint32_t max_slots = 0;

  int64_t steps = 0;
  int64_t obs_at = -1;
  bool sw_labels = false;  // the labels hold a Swendsen-Wang step's (all zero before the first)
  // the sample of step obs_at: written by k_observe, the partial sums added
  // up per point
  // (one allocation, which is most of what they cost: 70 us each)
  PinBuf<uint64_t> pinned;
  ClusterSums* csums = nullptr;
  uint2* obs_part = nullptr;
  PointState* obs_ps = nullptr;
  uint32_t *obs_status = nullptr, *obs_capped = nullptr;
  // non-chessboard points: their table, bond bytes (one per cell of the
  // handle) and capped counts (by point)
  DevBuf<CappedEnt> tab_capped;
  uint32_t n_capped = 0, capped_L = 0;
  DevBuf<uint8_t> bonds;
  std::vector<int32_t> obs_point;  // point of each k_observe workgroup (-1: padding)
  std::vector<int64_t> obs_nhb2, obs_nsig;

  void drop_graphs() {
    for (auto& g : groups) g->drop_graphs();
  }
  ~cvf_sim() {
    g_resident_gate.remove(&turn);
    if (turn.event) (void)hipEventDestroy(turn.event);
    groups.clear();
    if (start_ev) (void)hipEventDestroy(start_ev);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

int validate(const cvf_params& p) {
  if (p.L < 4 || p.L % 4 != 0 || p.L > kMaxL)
    return fail(CVF_EINVAL, "L=%d: the chessboard needs a cubic lattice with L %% 4 == 0 (4..%d)",
                p.L, kMaxL);
  if (!(p.T > 0.f)) return fail(CVF_EINVAL, "T must be > 0");
  if (p.n_metropolis < 0 || p.n_cluster < 0) return fail(CVF_EINVAL, "negative step counts");
  if (p.n_metropolis > 4096 || p.n_cluster > 4096) return fail(CVF_EINVAL, "step counts too large");
  if (p.flag_chessboard != 0 && p.flag_chessboard != 1)
    return fail(CVF_EINVAL, "Error: Wrong value for flag_chessboard = %d (0 or 1)", p.flag_chessboard);
  if (p.flag_config < 0 || p.flag_config > 2)
    return fail(CVF_EINVAL, "Error: Wrong value for flag_config = %d", p.flag_config);
  if (p.precision != CVF_FP64 && p.precision != CVF_FP32_COMPENSATED)
    return fail(CVF_EINVAL, "unknown precision %d", p.precision);
  if (p.precision == CVF_FP32_COMPENSATED && p.volume_mode != CVF_VOLUME_DEVICE)
    return fail(CVF_EINVAL, "the FP32-compensated vdW form runs the volume move on the device");
  if (p.volume_mode != CVF_VOLUME_HOST && p.volume_mode != CVF_VOLUME_DEVICE)
    return fail(CVF_EINVAL, "unknown volume mode %d", p.volume_mode);
  if (!(p.r_cutoff > 0.f)) return fail(CVF_EINVAL, "R_cutoff must be > 0");
  if (p.schedule != CVF_SCHED_REFERENCE && p.schedule != CVF_SCHED_FAST)
    return fail(CVF_EINVAL, "unknown schedule %d", p.schedule);
  // a colour pass would let two cells move one neighbour's counter at once
  if (p.schedule == CVF_SCHED_FAST && !p.flag_chessboard)
    return fail(CVF_EINVAL, "the fast schedule needs flag_chessboard = 1");
  return CVF_OK;
}

// corner cell of the cube with origin (ox,oy,oz) at local corner b
inline uint32_t corner_cell(uint32_t L, uint32_t ox, uint32_t oy, uint32_t oz, int b) {
  const uint32_t x = (ox + (b & 1)) % L, y = (oy + ((b >> 1) & 1)) % L, z = (oz + ((b >> 2) & 1)) % L;
  return x + L * (y + L * z);
}

// rewrite the eta bits of one cube from a solution mask
void set_cube_eta(std::vector<uint32_t>& w, uint32_t L, uint32_t ox, uint32_t oy, uint32_t oz,
                  uint32_t M) {
  for (int b = 0; b < 8; ++b) {
    const int bx = b & 1, by = (b >> 1) & 1, bz = (b >> 2) & 1;
    const uint32_t c = corner_cell(L, ox, oy, oz, b);
    const uint32_t own = (1u << bx) | (1u << (2 + by)) | (1u << (4 + bz));
    const uint32_t bits = (((M >> corner_edge(b, 0)) & 1u) << bx) |
                          (((M >> corner_edge(b, 1)) & 1u) << (2 + by)) |
                          (((M >> corner_edge(b, 2)) & 1u) << (4 + bz));
    w[c] = (w[c] & ~(own << kEtaShift)) | (bits << kEtaShift);
  }
}

template <class F>
void for_each_cube(uint32_t L, F f) {
  const uint32_t hL = L / 2;
  for (uint32_t fam = 0; fam < 2; ++fam)
    for (uint32_t k = 0; k < hL; ++k)
      for (uint32_t j = 0; j < hL; ++j)
        for (uint32_t i = 0; i < hL; ++i) {
          const uint32_t oz = 2 * k + fam;
          f(2 * i + fam, 2 * j + fam, oz, i + hL * j + hL * hL * oz);
        }
}

// Per-cell HB counters of the non-chessboard mode (gpu_water3D.cu:845-862):
// the number of arms whose sigma equals the facing arm of the neighbour,
// weighted by eta, into bits 24-31.
void set_nhb(uint32_t L, std::vector<uint32_t>& w) {
  const uint32_t N = L * L * L;
  std::vector<uint32_t> n(N);
  for (uint32_t c = 0; c < N; ++c) {
    const uint32_t x = c % L, y = (c / L) % L, z = c / (L * L);
    const uint32_t nb[6] = {(x + 1) % L + L * (y + L * z), (x + L - 1) % L + L * (y + L * z),
                            x + L * ((y + 1) % L + L * z), x + L * ((y + L - 1) % L + L * z),
                            x + L * (y + L * ((z + 1) % L)), x + L * (y + L * ((z + L - 1) % L))};
    uint32_t acc = 0;
    for (int a = 0; a < 6; ++a)
      acc += eta_of(w[c], a) * (sigma_of(w[c], a) == sigma_of(w[nb[a]], a ^ 1));
    n[c] = acc & 0xFF;
  }
  for (uint32_t c = 0; c < N; ++c) w[c] = (w[c] & kLowBits) | (n[c] << kNhbShift);
}

// Initial state of one point (gpu_water3D.cu:639-826 with Philox streams).
void init_words(const PointHost& P, std::vector<uint32_t>& w) {
  const uint32_t L = P.L, N = P.N;
  const uint64_t seed = P.prm.seed;
  w.assign(N, 0);
  if (P.prm.flag_config == 2) {
    const U4 r = draw(seed, kStInitSigma, 0, 0, 2);
    const uint32_t v = uniform_int(r.x, 6);
    for (uint32_t c = 0; c < N; ++c) w[c] = v * kFieldLsb;
  } else {
    for (uint32_t c = 0; c < N; ++c) {
      const U4 r0 = draw(seed, kStInitSigma, c, 0, 0), r1 = draw(seed, kStInitSigma, c, 0, 1);
      const uint32_t rw[6] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y};
      uint32_t s = 0;
      for (int a = 0; a < 6; ++a) s |= uniform_int(rw[a], 6) << (3 * a);
      w[c] = s;
    }
  }
  if (!P.prm.flag_chessboard) {
    // every bond active (gpu_water3D.cu:721-724)
    for (uint32_t c = 0; c < N; ++c) w[c] |= 0x3Fu << kEtaShift;
    set_nhb(L, w);
    return;
  }
  for_each_cube(L, [&](uint32_t ox, uint32_t oy, uint32_t oz, uint32_t cube) {
    const U4 r = draw(seed, kStInitCube, cube, 0, 0);
    set_cube_eta(w, L, ox, oy, oz, sol_mask(uniform_int(r.x, 9)));
  });
}

int upload_point_words(cvf_sim* s, int pt, const std::vector<uint32_t>& w) {
  HIPC(hipStreamSynchronize(s->stream));
  HIPC(hipMemcpyAsync(s->words.p + s->ph[pt].woff, w.data(), w.size() * 4, hipMemcpyHostToDevice,
                      s->stream));
  HIPC(hipStreamSynchronize(s->stream));
  s->obs_at = -1;
  return CVF_OK;
}

// Configurations of fewer cells than this are brought to the host as words and
// unpacked there, and their arrays go down in one copy: the runtime takes about
// 1 us per KB for copies of less than 64 KB, so the 12 bytes per cell of the
// arrays cost more than the host's work.  get_config of L = 8 / 16 / 24 / 28: 30 / 40 / 68
// / 90 us (first call of a handle 43 / 50 / 79 / 103), unpacked on the device 55 / 74 / 130 /
// 65 - 170 (63 / 90 / 137 / 180); L = 32 / 40: 122 / 106 (137 / 214) and 71 / 87 (80 / 124).
constexpr uint32_t kSmallConfig = 1u << 15;

// Device copy of a point's sigma and eta bytes, kept for the next call
// (sized for the largest point that asked), and after them what becomes of an
// input: first value out of range, inconsistent cubes, abort flag.
constexpr size_t kConfigResults = 3 * sizeof(uint32_t);
int reserve_config(cvf_sim* s, size_t n6) {
  if (2 * n6 + kConfigResults > s->cfg_bytes.n) HIPC(s->cfg_bytes.alloc(2 * n6 + kConfigResults));
  return CVF_OK;
}

// ------------------------------------------------- resident kernel plan
// LDS words of a slab's window: T planes plus a ghost plane on each side when
// the point is split, the whole periodic lattice otherwise.
uint32_t window_words(uint32_t L, uint32_t T, bool whole) { return (whole ? T : T + 2) * L * L; }

struct RDeal {
  std::vector<RSlab> slabs;   // in workgroup order
  std::vector<RGroupEnt> groups;
  uint32_t lds_bytes = 0;
  size_t ring_words = 0;
};

// Waves of a workgroup for slabs of the given cells: one each, the rest by
// largest remainder in proportion to the cells.  False if there are more
// slabs than waves.
bool split_waves(const std::vector<double>& cells, uint32_t wpg, std::vector<uint32_t>& nw) {
  const size_t n = cells.size();
  if (n == 0 || n > wpg) return false;
  double sum = 0;
  for (double c : cells) sum += c;
  nw.assign(n, 1);
  for (uint32_t left = wpg - (uint32_t)n; left > 0; --left) {
    size_t best = 0;
    double bd = -1e300;
    for (size_t j = 0; j < n; ++j) {
      const double d = (double)wpg * cells[j] / sum - (double)nw[j];
      if (d > bd) {
        bd = d;
        best = j;
      }
    }
    ++nw[best];
  }
  return true;
}

struct Piece {
  int point;
  uint32_t z0, T, wg;
};

// Modeled length of one MC step of a workgroup whose slabs (lattice L,
// first plane z0, T planes, split or whole) have nw waves each, in
// consecutive wave ranges: per phase, the busiest SIMD's wave iterations
// (waves w run on SIMD w % 4; a wave of a slab with n items and v waves
// makes ceil((n - 64 j) / (64 v)) iterations, j its rank in the slab)
// times the phase's VALU instructions per iteration, summed over the two
// cube families, eight in-plane and four z half-sweeps (two of each
// parity), the expected phases of a step, or the fast schedule's two passes.
struct SlabShape {
  uint32_t L, z0, T;
  bool split;
};
double workgroup_step_model(const std::vector<SlabShape>& sl, const std::vector<uint32_t>& nw, bool fast) {
  constexpr double kInPlane = 190, kZ = 176, kCube = 614;  // VALU per iteration
  double total = 0;
  for (int ph = 0; ph < (fast ? 3 : 5); ++ph) {
    // 0, 1: cube families; 2: in-plane (x8); 3, 4: z of parity 0, 1 (x2)
    double simd[4] = {0, 0, 0, 0};
    uint32_t w0 = 0;
    for (size_t j = 0; j < sl.size(); ++j) {
      const SlabShape& x = sl[j];
      const uint32_t LL = x.L * x.L;
      uint64_t n = 0;
      double cost = 0;
      if (ph < 2) {
        const int zlo = x.split ? -1 : 0;
        const int first = zlo + ((((int)x.z0 + zlo + (int)x.L) & 1) == ph ? 0 : 1);
        const uint32_t npl = first <= (int)x.T - 1 ? (uint32_t)((int)x.T - 1 - first) / 2 + 1 : 0u;
        n = (uint64_t)npl * (x.L / 4) * (x.L / 4);
        cost = kCube;
      } else if (ph == 2) {
        n = (uint64_t)x.T * LL / 8;
        cost = (fast ? 12 : 8) * kInPlane;  // (fast: two passes of six arms)
      } else {
        const uint32_t first = (x.z0 & 1u) == (uint32_t)(ph - 3) ? 0u : 1u;
        const uint32_t npl = first < x.T ? (x.T - first + 1) / 2 : 0u;
        n = (uint64_t)npl * LL / 4;
        cost = 2 * kZ;
      }
      const uint64_t span = 64ull * nw[j];
      for (uint32_t i = 0; i < nw[j]; ++i) {
        const uint64_t start = 64ull * i;
        const uint64_t it = n > start ? (n - start + span - 1) / span : 0;
        simd[(w0 + i) & 3] += (double)it * cost;
      }
      w0 += nw[j];
    }
    total += std::max(std::max(simd[0], simd[1]), std::max(simd[2], simd[3]));
  }
  return total;
}

// The model's lengths of the workgroups that one plan has asked for, by their
// slabs' (L, first plane's parity, T, split) in order: the points of a scan
// share few sizes, and the bisection asks for most of them again (creating
// 96 points of L = 16 .. 48: 76.4 -> 70.2 ms).
struct StepLengths {
  uint32_t wpg;
  bool fast;
  std::map<std::vector<uint32_t>, double> known;
  std::vector<uint32_t> key, nw;
  // of slabs `sl` with `cells` each; infinite if there are more slabs than waves
  double of(const std::vector<SlabShape>& sl, const std::vector<double>& cells) {
    key.clear();
    for (const SlabShape& x : sl) key.push_back(x.L << 10 | (x.z0 & 1u) << 9 | x.T << 1 | (x.split ? 1u : 0u));
    const auto it = known.find(key);
    if (it != known.end()) return it->second;
    const double len = split_waves(cells, wpg, nw) ? workgroup_step_model(sl, nw, fast) : INFINITY;
    known.emplace(key, len);
    return len;
  }
};

// Fill workgroups in order with z-pieces of the points (in `order`): a
// workgroup takes the thickest piece that keeps its modeled step length
// (workgroup_step_model) within W, its windows within cap words and its
// slabs within max_slabs; pieces are at least min_T planes, and so is what
// a cut leaves of the point.  False if the points do not fit in nwg
// workgroups.
bool fill_workgroups(const cvf_sim* s, const std::vector<int>& order, double W, int nwg, uint32_t wpg, uint32_t cap,
                     uint32_t min_T, uint32_t max_T, StepLengths& lengths, std::vector<Piece>& pc) {
  pc.clear();
  const uint32_t max_slabs = std::min<uint32_t>(kMaxRSlabs, wpg);
  uint32_t wg = 0, used = 0;
  std::vector<double> cells;
  std::vector<SlabShape> shapes;
  for (int p : order) {
    const uint32_t L = s->ph[p].L, LL = L * L, tcap = max_T ? std::min(max_T, L) : L;
    uint32_t z = 0;
    while (z < L) {
      const uint32_t rest = L - z;
      uint32_t take = 0;
      if (shapes.size() < max_slabs)
        for (uint32_t t = std::min(rest, tcap); t >= 1; --t) {
          if (t < rest && (t < min_T || rest - t < min_T)) continue;
          const uint32_t need = window_words(L, t, t == L);
          if (used + need > cap) continue;
          cells.push_back((double)t * LL);
          shapes.push_back(SlabShape{L, z, t, t < L});
          const bool ok = lengths.of(shapes, cells) <= W;
          cells.pop_back();
          shapes.pop_back();
          if (ok) {
            take = t;
            break;
          }
        }
      if (take == 0) {
        // the next workgroup; an empty one that takes nothing cannot help
        if (shapes.empty() || wg + 1 == (uint32_t)nwg) return false;
        ++wg;
        used = 0;
        cells.clear();
        shapes.clear();
        continue;
      }
      pc.push_back(Piece{p, z, take, wg});
      cells.push_back((double)take * LL);
      shapes.push_back(SlabShape{L, z, take, take < L});
      used += window_words(L, take, take == L);
      z += take;
    }
  }
  return true;
}

// The resident plan of a group on at most nwg workgroups of wpg waves and
// cap LDS words each: the points, largest lattice first, cut into z-pieces
// that fill the workgroups in order (fill_workgroups), with the smallest
// bound on any workgroup's modeled step length for which they fit, found
// by bisection (the neighbour exchange paces every slab of a point to the
// slowest workgroup).  A
// point in one piece is a whole-lattice window; the pieces of a split point
// are slabs of at least two planes (one with max_T = 1) and at most max_T
// planes when max_T > 0.  Each workgroup's waves go to its slabs in
// proportion to their cells, at least one each.  False when the group's
// points cannot run resident (several Metropolis sweeps per step, the
// non-chessboard rule) or do not fit.
bool plan_resident(const cvf_sim* s, const Group& g, int nwg, uint32_t wpg, uint32_t cap, uint32_t max_T,
                   RDeal& out) {
  if (s->nm != 1 || nwg <= 0 || wpg == 0) return false;
  std::vector<int> order = g.points;
  for (int p : order)
    if (!s->ph[p].prm.flag_chessboard) return false;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return s->ph[a].L > s->ph[b].L; });
  const uint32_t min_T = max_T == 1 ? 1u : 2u;
  StepLengths lengths{wpg, s->sched == CVF_SCHED_FAST, {}, {}, {}};
  std::vector<Piece> pc, trial;
  double lo = 0, hi = 1e300;
  if (!fill_workgroups(s, order, hi, nwg, wpg, cap, min_T, max_T, lengths, pc)) return false;
  hi = 1;  // the smallest power of two bound that fits
  while (!fill_workgroups(s, order, hi, nwg, wpg, cap, min_T, max_T, lengths, trial)) {
    lo = hi;
    hi *= 2;
  }
  pc.swap(trial);
  for (int it = 0; it < 30 && hi - lo > 0.002 * hi; ++it) {
    const double mid = 0.5 * (lo + hi);
    if (fill_workgroups(s, order, mid, nwg, wpg, cap, min_T, max_T, lengths, trial)) {
      hi = mid;
      pc.swap(trial);
    } else {
      lo = mid;
    }
  }
  const uint32_t wg = pc.empty() ? 0 : pc.back().wg;
  out = RDeal();
  std::vector<std::vector<size_t>> members(wg + 1);
  for (size_t i = 0; i < pc.size(); ++i) members[pc[i].wg].push_back(i);
  std::vector<uint32_t> pieces_of(s->ph.size(), 0);
  for (const Piece& x : pc) ++pieces_of[x.point];
  size_t ring = 0;
  for (uint32_t w = 0; w <= wg; ++w) {
    const auto& m = members[w];
    if (m.empty()) continue;
    // waves in proportion to cells (largest remainders), at least one each
    std::vector<double> cw;
    for (size_t i : m) cw.push_back((double)pc[i].T * s->ph[pc[i].point].L * s->ph[pc[i].point].L);
    std::vector<uint32_t> nw;
    if (!split_waves(cw, wpg, nw)) return false;
    RGroupEnt ge{(uint32_t)out.slabs.size(), (uint32_t)m.size()};
    uint32_t lds = 0, w0 = 0;
    for (size_t j = 0; j < m.size(); ++j) {
      const Piece& x = pc[m[j]];
      const PointHost& P = s->ph[x.point];
      const uint32_t L = P.L;
      const bool whole = pieces_of[x.point] == 1;
      RSlab r;
      memset(&r, 0, sizeof r);
      r.point = x.point;
      r.L = L;
      r.z0 = x.z0;
      r.T = x.T;
      r.ns = pieces_of[x.point];
      r.woff = P.woff;
      r.lds = lds;
      lds += window_words(L, x.T, whole);
      r.seed_lo = (uint32_t)P.prm.seed;
      r.seed_hi = (uint32_t)(P.prm.seed >> 32);
      r.mH = make_fastdiv(L / 2).m;
      r.mQ = make_fastdiv(L / 4).m;
      r.mP8 = make_fastdiv(L * L / 8).m;
      r.mP4 = make_fastdiv(L * L / 4).m;
      r.mQQ = make_fastdiv((L / 4) * (L / 4)).m;
      r.above = r.below = -1;
      r.w0 = w0;
      r.nw = nw[j];
      w0 += nw[j];
      const uint32_t stride = 64 * r.nw, Q8 = L * L / 8, Q4 = L * L / 4, Qc = (L / 4) * (L / 4);
      r.dp8 = stride / Q8;
      r.du8 = stride % Q8;
      r.dp4 = stride / Q4;
      r.du4 = stride % Q4;
      r.dpc = stride / Qc;
      r.duc = stride % Qc;
      r.mS = make_fastdiv(stride).m;
      if (!whole) {
        r.ring = (uint32_t)ring;
        ring += 4 * (size_t)kRingHalf * L * L;
      }
      out.slabs.push_back(r);
    }
    if (lds > cap) return false;
    out.lds_bytes = std::max(out.lds_bytes, lds * 4);
    out.groups.push_back(ge);
  }
  if (ring >= 0xFFFFFFFFull || out.groups.size() > (size_t)nwg) return false;
  out.ring_words = ring;
  // neighbours: the slabs of the same point above and below
  std::vector<std::vector<int32_t>> by_point(s->ph.size());
  for (size_t j = 0; j < out.slabs.size(); ++j) by_point[out.slabs[j].point].push_back((int32_t)j);
  for (auto& r : out.slabs) {
    if (r.ns == 1) continue;
    const uint32_t up = (r.z0 + r.T) % r.L;
    for (int32_t j : by_point[r.point]) {
      const RSlab& o = out.slabs[j];
      if (o.z0 == up) r.above = j;
      if ((o.z0 + o.T) % o.L == r.z0) r.below = j;
    }
    if (r.above < 0 || r.below < 0) return false;
  }
  for (auto& r : out.slabs)
    if (r.ns > 1) {
      r.ring_hi = out.slabs[r.above].ring;
      r.ring_lo = out.slabs[r.below].ring;
    }
  return true;
}

// Consistency of a resident plan, checked before it is used: every point of
// the group covered by its slabs exactly once, each slab's waves a
// non-empty range of its workgroup's wpg waves, disjoint from the others',
// windows packed in order within cap words, neighbours above and below of
// the same point adjacent in z, rings inside the ring buffer.
bool resident_plan_valid(const cvf_sim* s, const Group& g, const RDeal& d, uint32_t wpg, uint32_t cap) {
  std::vector<std::vector<uint8_t>> cov(s->ph.size());
  std::vector<uint32_t> nslab(s->ph.size(), 0);
  for (int p : g.points) cov[p].assign(s->ph[p].L, 0);
  for (const RSlab& r : d.slabs) {
    if (r.point < 0 || (size_t)r.point >= s->ph.size() || cov[r.point].empty()) return false;
    ++nslab[r.point];
  }
  for (const RGroupEnt& ge : d.groups) {
    if (ge.count == 0 || ge.count > kMaxRSlabs || (size_t)ge.first + ge.count > d.slabs.size()) return false;
    uint64_t waves = 0;
    uint32_t lds = 0;
    for (uint32_t j = ge.first; j < ge.first + ge.count; ++j) {
      const RSlab& r = d.slabs[j];
      const uint32_t L = s->ph[r.point].L, LL = L * L;
      if (r.L != L || r.T == 0 || r.z0 + r.T > L || r.ns != nslab[r.point]) return false;
      for (uint32_t z = r.z0; z < r.z0 + r.T; ++z)
        if (cov[r.point][z]++) return false;
      if (r.nw == 0 || r.w0 + r.nw > wpg || r.nw > 16) return false;
      const uint64_t mine = ((1ull << r.nw) - 1) << r.w0;
      if (waves & mine) return false;
      waves |= mine;
      if (r.lds != lds) return false;
      lds += window_words(L, r.T, r.ns == 1);
      const uint32_t stride = 64 * r.nw;
      if (r.dp8 * (LL / 8) + r.du8 != stride || r.du8 >= LL / 8 || r.dp4 * (LL / 4) + r.du4 != stride ||
          r.du4 >= LL / 4 || r.dpc * (L / 4) * (L / 4) + r.duc != stride || r.duc >= (L / 4) * (L / 4))
        return false;
      if (r.ns > 1) {
        if (r.above < 0 || r.below < 0 || (size_t)r.above >= d.slabs.size() || (size_t)r.below >= d.slabs.size())
          return false;
        const RSlab& a = d.slabs[r.above];
        const RSlab& b = d.slabs[r.below];
        if (a.point != r.point || b.point != r.point || a.z0 != (r.z0 + r.T) % L || (b.z0 + b.T) % L != r.z0)
          return false;
        if ((size_t)r.ring + 4 * (size_t)kRingHalf * LL > d.ring_words || r.ring_hi != a.ring || r.ring_lo != b.ring)
          return false;
      }
    }
    if (lds > cap || lds * 4 > d.lds_bytes) return false;
  }
  for (int p : g.points)
    for (uint8_t c : cov[p])
      if (c != 1) return false;
  return true;
}

template <class T>
int upload_vec(DevBuf<T>& buf, const std::vector<T>& v);

int side_stream(Group& g) {
  if (!g.side) HIPC(hipStreamCreateWithFlags(&g.side, hipStreamNonBlocking));
  return CVF_OK;
}

// With fused = 2, `streams` is the number of resident workgroups per CU (1
// or 2) and slab_planes caps the slab thickness (0: automatic): every
// workgroup of the launch must be resident at once, so the plan is checked
// against the occupancy the runtime reports for its workgroup size and LDS,
// and falls back to fused slab launches otherwise.
int build_resident(cvf_sim* s, Group& g) {
  g.resident = false;
  int ncu = 0;
  HIPC(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, s->device));
  if (ncu <= 0) return CVF_OK;
  const int per_cu = std::min(s->tune.slab_planes == 1 ? 4 : 2, std::max(1, s->tune.streams));
  const uint32_t cap = (resident_lds_limit() - (uint32_t)(per_cu - 1) * kResidentStatic) / (uint32_t)per_cu / 4u;
  const uint32_t wpg = (uint32_t)s->tune.block_chunk / 64u;
  RDeal d;
  if (!plan_resident(s, g, ncu * per_cu, wpg, cap, (uint32_t)std::max(0, s->tune.slab_planes), d)) return CVF_OK;
  if (!resident_plan_valid(s, g, d, wpg, cap)) return fail(CVF_EINVAL, "internal: the resident plan is inconsistent");
  int occ = 0;
  // the fine instantiation for plans of slabs of at most two planes of
  // which one has a phase that takes a fine path (two lanes for each of its
  // in-plane quads, or the cubes of its smaller family's items, fit its
  // lanes and at most 512 of them); otherwise the instantiation without
  // those paths
  bool thin = true, fine_phase = false;
  for (const auto& r : d.slabs) {
    thin = thin && r.T <= 2;
    const uint64_t lanes = std::min<uint64_t>(64ull * r.nw, 512), LL = (uint64_t)r.L * r.L;
    fine_phase = fine_phase || 2 * (uint64_t)r.T * (LL / 8) <= lanes || 4 * ((r.T + 1) / 2) * (LL / 16) <= lanes ||
                 (s->sched == CVF_SCHED_FAST && r.T * LL / 2 <= 128ull * r.nw);
  }
  const bool fine = thin && fine_phase;
  // one plane per workgroup: the kernel for that, while its phases are short
  // (one point of L = 12 / 32 / 48 / 56: 7.2 / 10.3 / 16.5 / 21.0 us per step of a long run,
  // the general kernel 13.7 / 15.8 / 22.3 / 23.6; L = 64, 64 steps a call: 25.9 and 24.4)
  bool planes = s->sched == CVF_SCHED_REFERENCE;
  uint32_t maxL = 0;
  for (const auto& r : d.slabs) {
    planes = planes && r.T == 1 && r.nw == wpg && r.L <= 56;
    maxL = std::max(maxL, r.L);
  }
  // as many half-sweeps laid out at a time as a workgroup's share of LDS holds
  // (its threads of the 1024 that the kernels' registers allow a CU: the
  // records take no CU from other launches)
  uint32_t per = 12;
  const uint32_t share = std::min<uint32_t>(4 * cap, 160 * (uint32_t)s->tune.block_chunk - 512);
  for (uint32_t next : {6u, 4u, 3u, 2u, 1u})
    if (plane_lds_bytes(maxL, per) > share) per = next;
  planes = planes && plane_lds_bytes(maxL, per) <= 4 * cap;
  if (planes) {
    d.lds_bytes = plane_lds_bytes(maxL, per);
    HIPC(plane_occupancy(&occ, (uint32_t)s->tune.block_chunk, d.lds_bytes));
  } else {
    HIPC(resident_occupancy(&occ, (uint32_t)s->tune.block_chunk, d.lds_bytes, fine, s->sched == CVF_SCHED_FAST));
  }
  if (occ < per_cu) return CVF_OK;
  int rc;
  if ((rc = upload_vec(g.rslabs, d.slabs)) || (rc = upload_vec(g.rgroups, d.groups))) return rc;
  // versions and rings start cleared: a plan is rebuilt whenever the step
  // counters may have gone back (the autotuner's restore), so no version
  // or step-end tag left from later steps survives into the new plan
  HIPC(g.rings.alloc(std::max<size_t>(d.ring_words, 4)));
  HIPC(hipMemset(g.rings.p, 0, std::max<size_t>(d.ring_words, 4) * sizeof(uint32_t)));
  HIPC(g.rver.alloc(2 * d.slabs.size()));
  HIPC(hipMemset(g.rver.p, 0, 2 * d.slabs.size() * sizeof(uint64_t)));
  g.r_ngroups = (uint32_t)d.groups.size();
  g.r_lds = d.lds_bytes;
  g.r_fine = fine;
  g.r_per = planes ? per : 0;
  if (s->vol_device) {
    if ((rc = side_stream(g))) return rc;
    HIPC(hipEventCreateWithFlags(&g.fork, hipEventDisableTiming));
    HIPC(hipEventCreateWithFlags(&g.join, hipEventDisableTiming));
  }
  g.resident = true;
  s->turn.plan = ResidentPlan{s->device, (uint32_t)d.groups.size(), (uint32_t)occ, (uint32_t)ncu};
  s->turn.stream = s->stream;
  if (!s->turn.event) HIPC(hipEventCreateWithFlags(&s->turn.event, hipEventDisableTiming));
  g_resident_gate.add(&s->turn);
  for (int p : g.points) s->ph[p].slab_T = 0;
  // the plan query reports a point's thickest slab
  for (const auto& r : d.slabs) s->ph[r.point].slab_T = std::max(s->ph[r.point].slab_T, r.T);
  return CVF_OK;
}

PointDev make_point_dev(const PointHost& P) {
  PointDev d;
  memset(&d, 0, sizeof d);
  d.seed = P.prm.seed;
  d.L = P.L;
  d.N = P.N;
  d.hL = P.L / 2;
  d.woff = P.woff;
  d.loff = P.loff;
  d.shell_off = P.shell_off;
  d.jeff_sign = P.thr.Jeff > 0 ? 1 : (P.thr.Jeff < 0 ? -1 : 0);
  d.vp = P.vp;
  memcpy(d.thr_sigma, P.thr.sigma, sizeof d.thr_sigma);
  memcpy(d.thr_eta, P.thr.eta, sizeof d.thr_eta);
  d.thr_sw[0] = P.thr.sw_hb;
  d.thr_sw[1] = P.thr.sw_s;
  return d;
}

BlockEnt make_entry(const PointHost& P, int point, uint32_t start) {
  BlockEnt e;
  e.point = point;
  e.start = start;
  e.L = P.L;
  e.N = P.N;
  e.woff = P.woff;
  e.loff = P.loff;
  e.seed_lo = (uint32_t)P.prm.seed;
  e.seed_hi = (uint32_t)(P.prm.seed >> 32);
  e.mL = make_fastdiv(P.L).m;
  e.mH = make_fastdiv(P.L / 2).m;
  e.mQ = make_fastdiv(P.L / 4).m;
  e.jeff_sign = P.thr.Jeff > 0 ? 1 : (P.thr.Jeff < 0 ? -1 : 0);
  e.thb_lo = (uint32_t)P.thr.sw_hb;
  e.thb_hi = (uint32_t)(P.thr.sw_hb >> 32);
  e.ts_lo = (uint32_t)P.thr.sw_s;
  e.ts_hi = (uint32_t)(P.thr.sw_s >> 32);
  const uint32_t LL = P.L * P.L;
  e.mLL = make_fastdiv(LL).m;
  e.mP8 = make_fastdiv(LL / 8).m;
  e.mP4 = make_fastdiv(LL / 4).m;
  e.mC = make_fastdiv((P.L / 4) * (P.L / 4)).m;
  e.T = 0;
  e.flags = P.prm.flag_chessboard ? 0u : kEntNoChess;
  e.pad[0] = e.pad[1] = 0;
  return e;
}

// LDS words of a fused launch for slabs of T planes: T + one plane per
// half-sweep of the chunk (worst-case halo) + one per side for the cubes;
// with the non-chessboard rule (no cubes) two planes per half-sweep.
uint32_t slab_lds_bytes(uint32_t L, uint32_t T, int chunk = kChunk, bool nc = false) {
  return (T + (nc ? 2 * chunk : chunk + 2)) * L * L * 4;
}

// Planes per slab: the requested count if it divides L and fits, else the
// thickest divisor of L up to kMaxSlab that fits in LDS and keeps the slab
// within max_cells cells, else the thinnest divisor that fits; 0 if none.
uint32_t choose_slab(uint32_t L, int requested, uint64_t max_cells, bool nc) {
  if (requested > 0 && L % (uint32_t)requested == 0 &&
      slab_lds_bytes(L, (uint32_t)requested, kChunk, nc) <= chunk_lds_limit())
    return (uint32_t)requested;
  uint32_t thinnest = 0;
  for (uint32_t T = kMaxSlab; T >= 1; --T)
    if (L % T == 0 && slab_lds_bytes(L, T, kChunk, nc) <= chunk_lds_limit()) {
      if ((uint64_t)T * L * L <= max_cells) return T;
      thinnest = T;
    }
  return thinnest;
}

// Automatic slab size: at most the handle's cells per CU (256 on MI355X).
// A fused launch lasts as long as its largest workgroup, so thick slabs
// (less halo work) are taken only while no slab outgrows the CUs' even
// share; small handles (one L=32 point) get one-plane slabs.
uint64_t auto_slab_cells(const cvf_sim* s) {
  uint64_t total = 0;
  for (const auto& P : s->ph) total += P.N;
  return std::max<uint64_t>(total / 256, 1);
}

// Block table over `count(P)` work items per point of `points`, `block`
// items per workgroup, padded to a multiple of the XCD count.
template <class F>
std::vector<BlockEnt> make_table(const std::vector<PointHost>& ph, const std::vector<int>& points,
                                 uint32_t block, F count) {
  std::vector<BlockEnt> t;
  for (int p : points) {
    const uint32_t n = count(ph[p]);
    for (uint32_t st = 0; st < n; st += block) t.push_back(make_entry(ph[p], p, st));
  }
  while (t.size() % kNumXcd) {
    BlockEnt pad;
    memset(&pad, 0, sizeof pad);
    pad.point = -1;
    t.push_back(pad);
  }
  return t;
}

template <class T>
int upload_vec(DevBuf<T>& buf, const std::vector<T>& v) {
  HIPC(buf.alloc(v.size()));
  HIPC(hipMemcpy(buf.p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
  return CVF_OK;
}

int upload_tables(cvf_sim* s) {
  std::vector<PointDev> pd;
  std::vector<float> dist;
  std::vector<int32_t> freq;
  for (int p = 0; p < s->npts; ++p) {
    auto& P = s->ph[p];
    P.shell_off = (uint32_t)dist.size();
    P.vp.nshell = (int32_t)P.dist.size();
    dist.insert(dist.end(), P.dist.begin(), P.dist.end());
    freq.insert(freq.end(), P.freq.begin(), P.freq.end());
    pd.push_back(make_point_dev(P));
  }
  if (s->dist.p == nullptr || s->dist.n < dist.size()) {
    s->drop_graphs();  // captured graphs hold the old table pointers
    HIPC(s->dist.alloc(std::max<size_t>(dist.size(), 64)));
    HIPC(s->freq.alloc(std::max<size_t>(freq.size(), 64)));
  }
  HIPC(hipMemcpy(s->dist.p, dist.data(), dist.size() * 4, hipMemcpyHostToDevice));
  HIPC(hipMemcpy(s->freq.p, freq.data(), freq.size() * 4, hipMemcpyHostToDevice));
  HIPC(hipMemcpy(s->pts.p, pd.data(), pd.size() * sizeof(PointDev), hipMemcpyHostToDevice));
  return CVF_OK;
}

uint32_t cells_sigma(const PointHost& P) { return P.N / 8; }  // quads of active cells
// cube quads; no cube moves without the chessboard (gpu_water3D.cu:1348)
uint32_t cells_eta(const PointHost& P) {
  return P.prm.flag_chessboard ? (P.L / 2) * (P.L / 4) * (P.L / 4) : 0;
}
uint32_t cells_all(const PointHost& P) { return P.N; }

int valid_block(int b) { return b == 64 || b == 128 || b == 256 || b == 512 || b == 1024; }

// the groups' step counters take the handle's step count
int upload_group_steps(cvf_sim* s) {
  std::vector<uint64_t> v(s->groups.size(), (uint64_t)s->steps);
  HIPC(hipMemcpy(s->cur_steps.p, v.data(), v.size() * 8, hipMemcpyHostToDevice));
  return CVF_OK;
}

// z-slabs of a set of points, and the dynamic LDS of their launches
struct SlabTable {
  std::vector<BlockEnt> ents;  // empty: some point's do not fit
  uint32_t lds = 0;            // for kChunk half-sweeps
  uint32_t lds_long = 0;       // for kMaxChunk; 0 if that does not fit
  uint32_t lds_eta = 0;        // for the eta sweep alone
  bool any_nc = false;
};
SlabTable slab_table(const cvf_sim* s, const std::vector<int>& points, int requested) {
  const uint64_t slab_cells = auto_slab_cells(s);
  SlabTable st;
  bool long_fits = true;
  for (int p : points) {
    const PointHost& P = s->ph[p];
    const bool nc = !P.prm.flag_chessboard;
    st.any_nc = st.any_nc || nc;
    const uint32_t T = choose_slab(P.L, requested, slab_cells, nc);
    if (!T) {
      SlabTable none;
      for (int i : points) none.any_nc = none.any_nc || !s->ph[i].prm.flag_chessboard;
      return none;
    }
    st.lds = std::max(st.lds, slab_lds_bytes(P.L, T, kChunk, nc));
    st.lds_long = std::max(st.lds_long, slab_lds_bytes(P.L, T, kMaxChunk, nc));
    st.lds_eta = std::max(st.lds_eta, slab_lds_bytes(P.L, T, 0));
    long_fits = long_fits && slab_lds_bytes(P.L, T, kMaxChunk, nc) <= chunk_lds_limit();
    for (uint32_t z0 = 0; z0 < P.L; z0 += T) {
      BlockEnt en = make_entry(P, p, z0);
      en.T = T;
      st.ents.push_back(en);
    }
  }
  if (!long_fits) st.lds_long = 0;
  return st;
}

// Tiles of a set of points: an axis of length d takes ceil(d / edge) tiles of
// even length, the last one shorter; half-sweeps per launch, workgroup size
// and modeled length of a Metropolis pass.
// (the points: how many there are of each L; nc: some run without the
// chessboard)
struct TilePoints {
  std::map<uint32_t, uint32_t> count;
  bool nc = false;
  void add(const PointHost& P) {
    ++count[P.L];
    nc = nc || !P.prm.flag_chessboard;
  }
};
struct TilePlan {
  uint32_t edge[3] = {0, 0, 0}, nk = 0, block = 0;
  double us = 0;  // 0: none
};
uint32_t even_edge(uint32_t edge, uint32_t d) {
  const uint32_t n = (d + edge - 1) / edge;
  return (d + n - 1) / n;
}

// Modeled times, us: what a pass costs besides its launches, a launch, a
// workgroup of 1024 threads (schedule, tables, window), a half-sweep per trip
// of the workgroup over its quads and per 256 quads on the CU (few: in the
// one-cell-per-lane form), a cube family likewise.
struct TileCost {
  double pass, launch, group, trip, per256, few_trip, few_per256, cube_trip, cube_per256;
};
// fitted to 170 measured shapes of one point of L = 32 .. 200, to 7 % rms, and
// the chosen shape ran within 2 % of the fastest measured one at every L; without
// the chessboard to 64 shapes of 1 .. 256 points of L = 8 .. 160, to 8 %
constexpr TileCost kCost = {0, 7.1, 4.9, 0.22, 0.21, 0, 0.34, 3.8, 2.8};
constexpr TileCost kCostNc = {14.5, 1.5, 3.0, 0.64, 0.53, 0.2, 0.78, 0, 0};

double sweep_us(const TileCost& c, double quads, double co, uint32_t block) {
  return c.trip * std::ceil(quads / block) + c.per256 * co * quads / 256;
}
double cubes_us(const TileCost& c, double quads, double co, uint32_t block) {
  return c.cube_trip * std::ceil(quads / block) + c.cube_per256 * co * quads / 256;
}
// workgroups of `block` threads and `lds` bytes, per_cu of them to a CU, that
// run together there
double together(double per_cu, uint32_t lds, uint32_t block) {
  return std::max(1.0, std::min({per_cu, std::floor(160 * 1024.0 / (lds + 3072)), std::floor(2048.0 / block)}));
}

// Modeled length of a pass (cube sweep and 12 half-sweeps) in us, 0 if the
// windows do not fit.
double tile_model(const TilePoints& points, const TilePlan& t, uint32_t ncu) {
  struct Tile {
    double edge[3], n;
  };
  std::vector<Tile> tiles;
  uint32_t lds = 0;
  double total = 0;
  for (const auto& lc : points.count) {
    const uint32_t d[3] = {lc.first / 2, lc.first / 2, lc.first};
    uint32_t c[3];
    Tile q;
    q.n = lc.second;
    for (int a = 0; a < 3; ++a) {
      c[a] = even_edge(t.edge[a], d[a]);
      q.edge[a] = c[a];
      q.n *= (d[a] + c[a] - 1) / c[a];
    }
    lds = std::max(lds, 16 * tile_window_quads(c[0], c[1], c[2], t.nk, false));
    if (points.nc) lds = std::max(lds, 16 * tile_window_quads(c[0], c[1], c[2], t.nk, true));
    total += q.n;
    tiles.push_back(q);
  }
  if (lds > tile_lds_limit()) return 0;
  // tiles of a CU, and how many of them run together
  const double per_cu = std::ceil(total / ncu);
  const double co = together(per_cu, lds, t.block);
  const auto box = [](const Tile& q, double more) {
    return (q.edge[0] + more) * (q.edge[1] + more) * (q.edge[2] + more);
  };
  const TileCost& cost = points.nc ? kCostNc : kCost;
  double us = cost.pass;
  for (uint32_t launch = 0; launch < 12 / t.nk; ++launch) {
    double work = 0;
    for (const Tile& q : tiles) {
      double x = cost.group * co * t.block / 1024;
      if (launch == 0 && !points.nc) x += 2 * cubes_us(cost, box(q, t.nk / 6.0 + 2) / 8, co, t.block);
      // a later half-sweep adds 1/6 layer (1/3) on average to each axis
      for (uint32_t k = 0; k < t.nk; ++k) {
        const double quads = box(q, (t.nk - 1 - k) / (points.nc ? 3.0 : 6.0)) / 2;
        x += 4 * quads <= t.block ? cost.few_trip + cost.few_per256 * co * quads / 256
                                  : sweep_us(cost, quads, co, t.block);
      }
      work += q.n * x;
    }
    us += cost.launch + std::ceil(per_cu / co) * work / total;
  }
  return us;
}

// The same for the slabs of `tab` (windows of at most lds bytes): planes
// without a halo in the plane, a z half-sweep adding one to each window (two
// without the chessboard).  0.87: measured against kCost for the chessboard
// (0.73 - 1.0 over 22 handles of 1 - 128 points of L = 16 .. 64); without it
// their half-sweeps, word by word, take 2.5 times as long (0.85 - 1.2 over 11).
double slab_model(const SlabTable& st, uint32_t nk, uint32_t block, uint32_t ncu) {
  const std::vector<BlockEnt>& tab = st.ents;
  const bool nc = st.any_nc;
  const uint32_t lds = nk == (uint32_t)kMaxChunk ? st.lds_long : st.lds;
  const double per_cu = std::ceil((double)tab.size() / ncu), co = together(per_cu, lds, block);
  double us = 0;
  for (uint32_t launch = 0; launch < 12 / nk; ++launch) {
    double work = 0;
    for (const BlockEnt& e : tab) {
      const double plane = e.L * e.L / 4.0;
      double x = kCost.group * co * block / 1024;
      if (launch == 0 && !nc) x += 2 * cubes_us(kCost, (e.T + 2 + nk / 3.0) * plane / 8, co, block);
      for (uint32_t k = 0; k < nk; ++k)
        x += (nc ? 2.5 : 1) * sweep_us(kCost, (e.T + (nk - 1 - k) * (nc ? 2 : 1) / 3.0) * plane / 2, co, block);
      work += x;
    }
    us += kCost.launch + std::ceil(per_cu / co) * work / (double)tab.size();
  }
  return nc ? us : 0.87 * us;
}

// The fastest modeled shape with t's launch length and workgroup size: every
// number of tiles along the axes of the largest point, boxes at most three
// times as long as thin.
TilePlan best_tiles(const TilePoints& points, uint32_t nk, uint32_t block, uint32_t ncu) {
  const uint32_t L = points.count.rbegin()->first;
  const auto edges = [](uint32_t d) {
    std::vector<uint32_t> e;
    for (uint32_t n = 1; n <= d; ++n) {
      const uint32_t c = (d + n - 1) / n;
      if (c <= std::min(32u, kMaxTile) && c >= std::min(3u, d) && (e.empty() || e.back() != c)) e.push_back(c);
    }
    return e;
  };
  TilePlan best;
  for (uint32_t ex : edges(L / 2))
    for (uint32_t ey : edges(L / 2))
      for (uint32_t ez : edges(L)) {
        if (ey > ex || std::max(ex, ez) > 3 * std::min(ey, ez) + 2) continue;
        TilePlan t;
        t.edge[0] = ex, t.edge[1] = ey, t.edge[2] = ez;
        t.nk = nk;
        t.block = block;
        t.us = tile_model(points, t, ncu);
        if (t.us > 0 && (best.us == 0 || t.us < best.us)) best = t;
      }
  return best;
}

// Fused launches can run on tiles: the reference schedule, no slab thickness
// asked for, and workgroups as the kernel needs.
bool tiles_possible(const cvf_sim* s, const cvf_tuning& t) {
  return s->sched == CVF_SCHED_REFERENCE && s->nm > 0 && t.fused != 0 && t.slab_planes == 0 &&
         t.block_chunk >= (int32_t)kTileMinBlock;
}

int cu_count(const cvf_sim* s, uint32_t& ncu) {
  int n = 0;
  HIPC(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, s->device));
  ncu = (uint32_t)std::max(n, 1);
  return CVF_OK;
}

// Tiles for the fused launches of `points` (us = 0: none) where slabs do not
// fit LDS (L > 64; L = 72 / 96 / 128 / 160 / 200 / 252: 27.1 / 33.2 / 47.6 / 75.6 /
// 142 / 268 us per step, unfused 44.9 / 49.9 / 67.2 / 104 / 162 / 304) or the
// models say that they take longer: thin slabs recompute as many planes as they
// own, and large ones are alone on a CU.  A step with a cluster sweep at L = 8 /
// 16 / 32 / 48 / 64: 31.1 / 30.6 / 34.3 / 37.8 / 43.2 us, slabs 32.6 / 30.9 / 36.2 /
// 49.4 / 57.8; 8 / 16 / 32 points of L = 48: 37 / 49 / 74, slabs 66 / 53 / 72;
// thick slabs of small lattices stay (128 points of L = 16: 22.7, tiles 31).
// Without the chessboard L = 8 / 16 / 32 / 64: 20.7 / 20.0 / 21.5 / 29.2 us, slabs
// 24.9 / 25.4 / 30.3 / 46.6; 128 points of L = 16: 39, slabs 30.8.
TilePlan fused_tiles(const cvf_sim* s, const cvf_tuning& t, const std::vector<int>& points, const SlabTable& slabs,
                     uint32_t ncu) {
  if (!tiles_possible(s, t)) return TilePlan();
  TilePoints count;
  for (int p : points) count.add(s->ph[p]);
  const bool whole = t.chunk_sweeps == kMaxChunk;
  TilePlan best = best_tiles(count, whole ? kMaxChunk : kChunk, (uint32_t)t.block_chunk, ncu);
  if (best.us == 0) best = best_tiles(count, kChunk, (uint32_t)t.block_chunk, ncu);
  // (without the chessboard a whole-pass slab launch is no faster than two)
  const bool whole_slabs = whole && slabs.lds_long && !slabs.any_nc;
  if (!slabs.ents.empty() &&
      slab_model(slabs, whole_slabs ? kMaxChunk : kChunk, (uint32_t)t.block_chunk, ncu) <= best.us)
    return TilePlan();
  return best;
}

int build_tiles(cvf_sim* s, Group& g, const SlabTable& slabs) {
  g.tiled = false;
  uint32_t ncu = 0;
  int rc = cu_count(s, ncu);
  if (rc) return rc;
  const TilePlan t = fused_tiles(s, s->tune, g.points, slabs, std::max(1u, ncu / (uint32_t)s->groups.size()));
  if (t.us == 0) return CVF_OK;
  std::vector<TileEnt> tab;
  uint32_t lds = 0, lds_long = 0;
  for (int p : g.points) {
    const PointHost& P = s->ph[p];
    const uint32_t hL = P.L / 2, d[3] = {hL, hL, P.L};
    uint32_t c[3];
    for (int a = 0; a < 3; ++a) c[a] = even_edge(t.edge[a], d[a]);
    const bool nc = !P.prm.flag_chessboard;
    lds = std::max(lds, 16 * tile_window_quads(c[0], c[1], c[2], kChunk, nc));
    lds_long = std::max(lds_long, 16 * tile_window_quads(c[0], c[1], c[2], kMaxChunk, nc));
    for (uint32_t z = 0; z < d[2]; z += c[2])
      for (uint32_t y = 0; y < d[1]; y += c[1])
        for (uint32_t x = 0; x < d[0]; x += c[0])
          tab.push_back(TileEnt{p, P.L, P.woff, (uint32_t)P.prm.seed, (uint32_t)(P.prm.seed >> 32), x, y, z,
                                std::min(c[0], d[0] - x), std::min(c[1], d[1] - y), std::min(c[2], d[2] - z),
                                nc ? 1u : 0u});
  }
  TileEnt pad;
  memset(&pad, 0, sizeof pad);
  pad.point = -1;
  while (tab.size() % kNumXcd) tab.push_back(pad);
  if (lds > tile_lds_limit()) return CVF_OK;
  if ((rc = upload_vec(g.tab_tile, tab))) return rc;
  g.nb_tile = (uint32_t)tab.size();
  g.chunk_lds = lds;
  g.chunk_lds_long = lds_long <= tile_lds_limit() ? lds_long : 0;
  g.fused = true;
  g.tiled = true;
  return CVF_OK;
}

// (Re)build the groups for the current tuning: points are dealt to groups
// largest-first onto the group with the fewest cells.
int build_groups(cvf_sim* s) {
  HIPC(hipDeviceSynchronize());
  g_resident_gate.remove(&s->turn);
  s->groups.clear();
  // the resident kernel takes every point in one group (its workgroups must
  // all be resident at once, one per CU at most)
  const int ng = s->tune.fused == 2 ? 1 : std::max(1, std::min(s->tune.streams, s->npts));
  for (int g = 0; g < ng; ++g) s->groups.emplace_back(new Group);
  std::vector<int> order(s->npts);
  for (int i = 0; i < s->npts; ++i) order[i] = i;
  std::stable_sort(order.begin(), order.end(),
                   [&](int a, int b) { return s->ph[a].N > s->ph[b].N; });
  for (int p : order) {
    Group* best = s->groups[0].get();
    for (auto& g : s->groups)
      if (g->cells < best->cells) best = g.get();
    best->points.push_back(p);
    best->cells += s->ph[p].N;
  }
  for (auto& g : s->groups) {
    std::sort(g->points.begin(), g->points.end());
    if (ng == 1) {
      g->stream = s->stream;
    } else {
      HIPC(hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking));
      g->own_stream = true;
    }
    HIPC(hipEventCreateWithFlags(&g->done, hipEventDisableTiming));
    const auto th = make_table(s->ph, g->points, (uint32_t)s->tune.block_sigma, cells_sigma);
    // k_eta runs four threads per cube quad: block_eta / 4 quads per workgroup
    const auto tc = make_table(s->ph, g->points, (uint32_t)s->tune.block_eta / 4, cells_eta);
    const auto tl = make_table(s->ph, g->points, (uint32_t)s->tune.block_cell, cells_all);
    int rc;
    if ((rc = upload_vec(g->tab_half, th)) || (rc = upload_vec(g->tab_cube, tc)) ||
        (rc = upload_vec(g->tab_cell, tl)))
      return rc;
    g->nb_half = (uint32_t)th.size();
    g->nb_cube = (uint32_t)tc.size();
    g->nb_cell = (uint32_t)tl.size();
    std::vector<int32_t> pl(g->points.begin(), g->points.end());
    if ((rc = upload_vec(g->plist, pl))) return rc;
    // fused path when every point's slab fits in LDS: the reference
    // schedule's eta sweep and half-sweeps, or the fast schedule's eta sweep
    g->fused = s->tune.fused != 0;  // (fused = 2: the resident kernel where it applies, else fused slabs)
    SlabTable slabs = slab_table(s, g->points, s->tune.slab_planes);
    std::vector<BlockEnt>& ts = slabs.ents;
    g->fused = g->fused && !ts.empty();
    g->chunk_lds = slabs.lds;
    g->chunk_lds_long = slabs.lds_long;
    g->chunk_lds_eta = slabs.lds_eta;
    g->any_nc = slabs.any_nc;
    g->sigma_cells = 0;
    for (int p : g->points) g->sigma_cells += s->ph[p].N;
    if ((rc = build_tiles(s, *g, slabs))) return rc;
    for (int p : g->points) {
      s->ph[p].group = (int32_t)(&g - &s->groups[0]);
      s->ph[p].slab_T = 0;
    }
    if (g->fused && !g->tiled)
      for (const BlockEnt& en : ts) s->ph[en.point].slab_T = en.T;
    if (g->fused && !g->tiled) {
      // largest slabs first (the kernel takes entries in launch order, and
      // each XCD's dispatcher hands out its share in that order)
      std::stable_sort(ts.begin(), ts.end(), [](const BlockEnt& a, const BlockEnt& b) {
        return (uint64_t)a.L * a.L * (a.T + 2) > (uint64_t)b.L * b.L * (b.T + 2);
      });
      while (ts.size() % kNumXcd) {
        BlockEnt pad;
        memset(&pad, 0, sizeof pad);
        pad.point = -1;
        ts.push_back(pad);
      }
      if ((rc = upload_vec(g->tab_slab, ts))) return rc;
      g->nb_slab = (uint32_t)ts.size();
    }
    if (s->tune.fused == 2 && (rc = build_resident(s, *g))) return rc;
  }
  HIPC(s->cur_steps.alloc(s->groups.size()));
  int rc0 = upload_group_steps(s);
  if (rc0) return rc0;
  std::vector<int> all(s->npts);
  for (int i = 0; i < s->npts; ++i) all[i] = i;
  if (!s->pinned.p) {  // the observables' table does not depend on the tuning
    const auto ta = make_table(s->ph, all, observe_span(s->total_cells), cells_all);
    int rc = upload_vec(s->tab_cell_all, ta);
    if (rc) return rc;
    s->nb_cell_all = (uint32_t)ta.size();
    for (const BlockEnt& en : ta) s->obs_point.push_back(en.point);
    std::vector<CappedEnt> tc;
    for (int p = 0; p < s->npts; ++p) {
      const PointHost& P = s->ph[p];
      if (P.prm.flag_chessboard) continue;
      tc.push_back(CappedEnt{p, P.L, P.woff, make_fastdiv(P.L / 2).m});
      s->capped_L = std::max(s->capped_L, P.L);
    }
    if (!tc.empty()) {
      if ((rc = upload_vec(s->tab_capped, tc))) return rc;
      HIPC(s->bonds.alloc(s->total_cells));
      s->n_capped = (uint32_t)tc.size();
    }
    static_assert(sizeof(ClusterSums) % 8 == 0 && sizeof(PointState) % 8 == 0 && sizeof(uint2) == 8, "8-byte words");
    const size_t n = (size_t)s->npts, ps_at = sizeof(ClusterSums) / 8, part_at = ps_at + n * (sizeof(PointState) / 8);
    HIPC(s->pinned.alloc(part_at + ta.size() + 1 + (n + 1) / 2));
    s->csums = reinterpret_cast<ClusterSums*>(s->pinned.p);
    s->obs_ps = reinterpret_cast<PointState*>(s->pinned.p + ps_at);
    s->obs_part = reinterpret_cast<uint2*>(s->pinned.p + part_at);
    s->obs_status = reinterpret_cast<uint32_t*>(s->pinned.p + part_at + ta.size());
    s->obs_capped = reinterpret_cast<uint32_t*>(s->pinned.p + part_at + ta.size() + 1);
  }
  HIPC(hipDeviceSynchronize());
  return CVF_OK;
}

// nsteps steps of resident group g in one launch (launch_resident's stepp,
// step_off and step_out).  A sequence of launches keeps the lattice before its
// first one (24 points of L = 32 with a cluster sweep, a launch per step: 0.9 us
// of 69 where every one does).
void run_resident(cvf_sim* s, const Group& g, hipStream_t st, const uint64_t* stepp, uint64_t step_off,
                  uint32_t nsteps, uint64_t* step_out) {
  s->resident_used = true;
  uint32_t* kept = stepp && step_off ? nullptr : s->words2.p;
  if (g.r_per)
    launch_plane(st, g.rgroups.p, g.r_ngroups, (uint32_t)s->tune.block_chunk, g.r_lds, g.rslabs.p, s->pts.p,
                 s->words.p, kept, g.rings.p, g.rver.p, stepp, step_off, nsteps, step_out, s->rstatus.p, g.r_per);
  else
    launch_resident(st, g.rgroups.p, g.r_ngroups, (uint32_t)s->tune.block_chunk, g.r_lds, g.rslabs.p, s->pts.p,
                    s->words.p, kept, g.rings.p, g.rver.p, stepp, step_off, nsteps, step_out, s->rstatus.p, g.r_fine,
                    s->sched == CVF_SCHED_FAST);
}

// A fused launch of half-sweeps k0 .. k0 + nk - 1 of group g from src to dst.
void launch_fused(cvf_sim* s, const Group& g, hipStream_t st, const uint64_t* stepp, uint32_t step_off,
                  const uint32_t* src, uint32_t* dst, uint32_t k0, uint32_t nk, int with_eta) {
  const uint32_t lds = nk == (uint32_t)kMaxChunk ? g.chunk_lds_long : g.chunk_lds;
  if (g.tiled)
    launch_tile(st, g.tab_tile.p, g.nb_tile, (uint32_t)s->tune.block_chunk, stepp, step_off, s->pts.p, src, dst, k0,
                nk, with_eta, lds, g.any_nc);
  else
    launch_chunk(st, Launch{g.tab_slab.p, g.nb_slab, (uint32_t)s->tune.block_chunk, stepp, step_off}, s->pts.p, src,
                 dst, k0, nk, with_eta, lds, g.any_nc);
}

struct Untimed {
  template <class F>
  void operator()(int, F&& f) const {
    f();
  }
};

// Lattice part of one MC step of group g (MonteCarlo_Step,
// gpu_water3D.cu:1346-1733): the step is the group's counter + step_off.
// `timed(class, launch)` wraps every launch (profiling) or just makes it.
// The fused launches ping-pong between the two word arrays: `par` says which
// one holds the state (1: words2) and is updated.  `variant` selects the
// step's other fused form: with the reference schedule, whole-pass launches
// (kMaxChunk half-sweeps each instead of kChunk); with the fast schedule, the
// eta sweep as one slab launch instead of one in-place launch per family.
template <class Timed>
void enqueue_lattice(cvf_sim* s, int gi, hipStream_t st, uint32_t step_off, Timed&& timed, int& par,
                     bool variant = false) {
  Group& g = *s->groups[gi];
  const uint64_t* stepp = s->cur_steps.p + gi;
  const Launch lh{g.tab_half.p, g.nb_half, (uint32_t)s->tune.block_sigma, stepp, step_off};
  const Launch lc{g.tab_cube.p, g.nb_cube, (uint32_t)s->tune.block_eta, stepp, step_off};
  const Launch ll{g.tab_cell.p, g.nb_cell, (uint32_t)s->tune.block_cell, stepp, step_off};
  if (g.resident) {
    // one step of the resident kernel, in place on `words`
    timed(CVF_KCLASS_RESIDENT, [&] { run_resident(s, g, st, stepp, step_off, 1, nullptr); });
  } else if (s->sched == CVF_SCHED_FAST) {
    // eta cube sweep, then n_metropolis x the two colour passes (in place,
    // on the array holding the state)
    uint32_t* cur = par ? s->words2.p : s->words.p;
    if (variant) {
      uint32_t* nxt = par ? s->words.p : s->words2.p;
      const Launch lz{g.tab_slab.p, g.nb_slab, (uint32_t)s->tune.block_chunk, stepp, step_off};
      timed(CVF_KCLASS_CHUNK, [&] { launch_chunk(st, lz, s->pts.p, cur, nxt, 0, 0, 1, g.chunk_lds_eta, false); });
      par ^= 1;
      cur = nxt;
    } else {
      for (int f = 0; f < 2 && g.nb_cube; ++f)
        timed(CVF_KCLASS_ETA, [&] { launch_eta(st, lc, s->pts.p, cur, f); });
    }
    for (int pass = 0; pass < 2 * s->nm; ++pass)
      timed(CVF_KCLASS_SIGMA, [&] { launch_sigma_f(st, lh, s->pts.p, cur, (uint32_t)pass); });
  } else if (g.fused && s->nm > 0) {
    // 12*n_metropolis half-sweeps in launches of kChunk (kMaxChunk in the variant form)
    const int len = variant ? kMaxChunk : kChunk;
    for (int c = 0; c < 12 * s->nm / len; ++c) {
      const uint32_t* src = par ? s->words2.p : s->words.p;
      uint32_t* dst = par ? s->words.p : s->words2.p;
      timed(CVF_KCLASS_CHUNK, [&] {
        launch_fused(s, g, st, stepp, step_off, src, dst, (uint32_t)(c * len), (uint32_t)len, c == 0);
      });
      par ^= 1;
    }
  } else {
    for (int f = 0; f < 2 && g.nb_cube; ++f)
      timed(CVF_KCLASS_ETA, [&] { launch_eta(st, lc, s->pts.p, s->words.p, f); });
    for (int sub = 0; sub < 12 * s->nm; ++sub)
      timed(CVF_KCLASS_SIGMA, [&] { launch_sigma(st, lh, s->pts.p, s->words.p, (uint32_t)sub); });
  }
  // Swendsen-Wang steps on the array holding the state
  uint32_t* cur = par ? s->words2.p : s->words.p;
  for (int jc = 0; jc < s->nc; ++jc) {
    timed(CVF_KCLASS_SW_LOCAL, [&] { launch_sw_local(st, ll, cur, s->parent.p, s->cov.p, (uint32_t)jc); });
    timed(CVF_KCLASS_SW_UNION, [&] { launch_sw_union(st, ll, s->parent.p, s->cov.p); });
    timed(CVF_KCLASS_SW_FLIP, [&] { launch_sw_flip(st, ll, cur, s->parent.p, (uint32_t)jc); });
  }
}

constexpr uint32_t kHistSpan = 4096;  // per-step histograms per copy back

// nsteps MC steps of group g: the lattice kernels of every step, then one
// kernel with the device volume moves of all of them (the chain never reads
// the lattice) that also moves the group's step counter on.  With rec, the
// sigma histogram of point s->rec_pt follows every step.
//
// The steps' variant forms (whole-pass launches with chunk_sweeps = 12; the
// fast schedule's slab eta sweep) can leave the state in words2; the kernels
// that read the lattice between steps (SW, the per-step histogram) take the
// array holding it, and the last step of a sequence takes its plain form
// when the variant would end there in words2: every sequence ends with the
// state in `words`.
// Without moves the volume chain stays where it is.
int enqueue_steps(cvf_sim* s, int gi, hipStream_t st, int nsteps, bool rec = false, bool moves = true) {
  Group& g = *s->groups[gi];
  const bool ok = g.fused && s->nm > 0;
  bool variant_ok = false;
  int flips = 0;  // word-array swaps of one variant step
  if (s->sched == CVF_SCHED_REFERENCE) {
    variant_ok = ok && s->tune.chunk_sweeps == kMaxChunk && g.chunk_lds_long != 0;
    flips = s->nm & 1;
  } else if (s->sched == CVF_SCHED_FAST) {
    variant_ok = ok && g.nb_cube != 0;
    flips = 1;
  }
  int par = 0;
  for (int i = 0; i < nsteps; ++i) {
    const bool variant = variant_ok && (i < nsteps - 1 || (par ^ flips) == 0);
    enqueue_lattice(s, gi, st, (uint32_t)i, Untimed{}, par, variant);
    if (rec) {
      const PointHost& P = s->ph[s->rec_pt];
      launch_sigma_hist_slot(st, (par ? s->words2.p : s->words.p) + P.woff, P.N, s->hist_series.p + 1,
                             i == nsteps - 1 ? s->rstatus.p : nullptr, s->hist_series.p, s->cur_steps.p + gi,
                             (uint32_t)i, s->hist_base.p, kHistSpan);
    }
  }
  launch_vol_chain(st, s->pts.p, g.plist.p, (int)g.points.size(), s->pst.p, s->cur_steps.p + gi,
                   (uint32_t)nsteps, s->dist.p, s->freq.p, s->precision, moves && s->vol_device);
  return CVF_OK;
}

// Group g runs whole sequences of steps in single resident launches: nothing
// reads the lattice between its steps.
bool resident_sequences(const cvf_sim* s, const Group& g) { return g.resident && s->nc == 0; }

// nsteps MC steps of a resident group (resident_sequences) from step s->steps
// on, as one resident launch on st.  One launch takes any number of steps, so
// no graph is captured for it: a captured sequence of fixed length cut a
// 10-step call into launches of 8 and 2 steps, each with its own staging and
// counter kernel (L = 32, 10 steps and a sample: 266 us; as one launch, with
// the sample in one kernel, 175).  The device volume chain of the same steps
// runs beside it on the group's second stream: it never reads the lattice,
// and takes the volume state only from its own last run.
int enqueue_resident(cvf_sim* s, int gi, hipStream_t st, int nsteps) {
  Group& g = *s->groups[gi];
  s->resident_used = true;
  if (s->vol_device) {
    HIPC(hipEventRecord(g.fork, st));
    HIPC(hipStreamWaitEvent(g.side, g.fork, 0));
    launch_vol_chain(g.side, s->pts.p, g.plist.p, (int)g.points.size(), s->pst.p, nullptr, (uint32_t)nsteps,
                     s->dist.p, s->freq.p, s->precision, 1);
    HIPC(hipEventRecord(g.join, g.side));
  }
  run_resident(s, g, st, nullptr, (uint64_t)s->steps, (uint32_t)nsteps, s->cur_steps.p + gi);
  if (s->vol_device) HIPC(hipStreamWaitEvent(st, g.join, 0));
  HIPC(hipGetLastError());
  return CVF_OK;
}

int capture(cvf_sim* s, int gi, int nsteps, hipGraph_t* g, hipGraphExec_t* ge, bool rec = false) {
  // (not the stream of resident launches, on which another handle's thread may
  // record an event)
  int rc = CVF_OK;
  if (s->groups[gi]->resident && (rc = side_stream(*s->groups[gi]))) return rc;
  hipStream_t st = s->groups[gi]->resident ? s->groups[gi]->side : s->groups[gi]->stream;
  HIPC(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  rc = enqueue_steps(s, gi, st, nsteps, rec);
  hipError_t e = hipStreamEndCapture(st, g);
  if (rc) return rc;
  if (e != hipSuccess) return fail(CVF_EDEVICE, "graph capture failed: %s", hipGetErrorString(e));
  HIPC(hipGraphInstantiate(ge, *g, nullptr, nullptr, 0));
  return CVF_OK;
}

// The MC step is a fixed launch sequence whose step index lives in device
// memory, so one captured graph replays any step.
int capture_step_graphs(cvf_sim* s) {
  for (size_t gi = 0; gi < s->groups.size(); ++gi) {
    Group& g = *s->groups[gi];
    if (!g.gexecs.empty()) continue;
    g.drop_graphs();
    std::vector<int> sizes = {s->tune.graph_steps};
    for (int p = 1; p < s->tune.graph_steps; p *= 2) sizes.push_back(p);
    std::sort(sizes.rbegin(), sizes.rend());
    for (int k : sizes) {
      hipGraph_t gr = nullptr;
      hipGraphExec_t ge = nullptr;
      const int rc = capture(s, (int)gi, k, &gr, &ge);
      g.gsteps.push_back(k);
      g.graphs.push_back(gr);
      g.gexecs.push_back(ge);
      if (rc) return rc;
    }
  }
  return CVF_OK;
}

// The recording sequences of group gi (same sizes as its plain ones).
int capture_rec_graphs(cvf_sim* s, int gi) {
  Group& g = *s->groups[gi];
  if (!g.rgexecs.empty()) return CVF_OK;
  for (int k : g.gsteps) {
    hipGraph_t gr = nullptr;
    hipGraphExec_t ge = nullptr;
    const int rc = capture(s, gi, k, &gr, &ge, true);
    g.rgraphs.push_back(gr);
    g.rgexecs.push_back(ge);
    if (rc) return rc;
  }
  return CVF_OK;
}

// group streams start after the work already on the main stream
int fork_groups(cvf_sim* s) {
  HIPC(hipEventRecord(s->start_ev, s->stream));
  for (auto& g : s->groups) HIPC(hipStreamWaitEvent(g->stream, s->start_ev, 0));
  return CVF_OK;
}

// the main stream continues after every group's work
int join_groups(cvf_sim* s) {
  for (auto& g : s->groups) {
    HIPC(hipEventRecord(g->done, g->stream));
    HIPC(hipStreamWaitEvent(s->stream, g->done, 0));
  }
  return CVF_OK;
}

void host_volume_moves(cvf_sim* s) {
  for (auto& P : s->ph) {
    double u2 = 0;
    const double trial = volume_trial(P.vol, P.vp, (uint64_t)s->steps, &u2);
    const double te =
        vdw_energy_fp64(trial, P.prm.r_cutoff, P.dist.data(), P.freq.data(), (int)P.dist.size());
    volume_accept(P.vol, P.vp, trial, te, u2);
  }
}

// The handle moves on by n steps.  The volume chain does not read the
// lattice: in host-volume mode the host advances it while the device runs
// the lattice steps just enqueued.
void host_moves(cvf_sim* s, int n) {
  for (int j = 0; j < n; ++j) {
    if (!s->vol_device) host_volume_moves(s);
    ++s->steps;
  }
}

int check_pt(cvf_sim* s, int32_t pt) {
  if (!s) return fail(CVF_EINVAL, "null handle");
  if (pt < 0 || pt >= s->npts) return fail(CVF_EINVAL, "state point %d out of range [0,%d)", pt, s->npts);
  return CVF_OK;
}

int check_tuning(const cvf_tuning& t) {
  if (t.streams < 1 || t.streams > 8) return fail(CVF_EINVAL, "streams must be in [1, 8]");
  if (!valid_block(t.block_sigma) || !valid_block(t.block_eta) || !valid_block(t.block_cell))
    return fail(CVF_EINVAL, "block sizes must be 64, 128, 256, 512 or 1024");
  if (t.graph_steps < 1 || t.graph_steps > 64) return fail(CVF_EINVAL, "graph_steps must be in [1, 64]");
  if (!valid_block(t.block_chunk)) return fail(CVF_EINVAL, "block_chunk must be a power of 2 in [64, 1024]");
  if (t.slab_planes < 0 || t.slab_planes > kMaxSlab)
    return fail(CVF_EINVAL, "slab_planes must be in [0, %d]", kMaxSlab);
  if (t.fused < 0 || t.fused > 2) return fail(CVF_EINVAL, "fused must be 0, 1 or 2");
  if (t.chunk_sweeps != 0 && t.chunk_sweeps != kChunk && t.chunk_sweeps != kMaxChunk)
    return fail(CVF_EINVAL, "chunk_sweeps must be 0, %d or %d", kChunk, kMaxChunk);
  return CVF_OK;
}

// (resident: with resident plans where they are the faster ones)
cvf_tuning default_tuning(const cvf_sim* s, bool resident = true) {
  cvf_tuning t;
  t.streams = 1;
  t.block_sigma = s->total_cells < (1u << 20) ? 64 : 256;
  t.block_eta = t.block_sigma;
  t.block_cell = 256;
  t.graph_steps = 16;
  t.fused = 1;
  t.slab_planes = 0;
  t.block_chunk = 512;
  // small handles are bound by per-launch cost: a whole Metropolis pass per
  // fused launch where the window fits (not with the non-chessboard rule,
  // whose 24-plane halo reserve costs more than the launch it saves)
  bool any_nc = false;
  for (const auto& P : s->ph) {
    any_nc = any_nc || !P.prm.flag_chessboard;
  }
  t.chunk_sweeps = s->total_cells < (1u << 20) && !any_nc ? kMaxChunk : kChunk;
  // tiles, where they are the faster fused launches, at the launch length and
  // workgroup size that their model gives the shortest pass
  uint32_t ncu = 0;
  if (tiles_possible(s, t) && cu_count(s, ncu) == CVF_OK) {
    std::vector<int> all(s->npts);
    for (int i = 0; i < s->npts; ++i) all[i] = i;
    const SlabTable slabs = slab_table(s, all, 0);
    if (fused_tiles(s, t, all, slabs, ncu).us > 0) {
      TilePoints count;
      for (int p : all) count.add(s->ph[p]);
      TilePlan best;
      for (uint32_t nk : {(uint32_t)kChunk, (uint32_t)kMaxChunk})
        for (uint32_t block : {512u, 1024u}) {
          const TilePlan p = best_tiles(count, nk, block, ncu);
          if (p.us > 0 && (best.us == 0 || p.us < best.us)) best = p;
        }
      t.chunk_sweeps = (int32_t)best.nk;
      t.block_chunk = (int32_t)best.block;
    }
  }
  if (!resident) return t;
  // One Metropolis sweep per step up to L = 64: the resident kernels.  One-plane
  // slabs while there are workgroups for the planes, one to four of them per CU:
  // 256 threads up to L = 16 and 512 up to L = 32, fewer where more share a CU
  // (one point of L = 16 / 32 / 48 / 64: 8.1 / 10.9 / 17.0 / 24.4 us per step, whole-pass
  // fused launches 18.4 / 20.9 / 32.4 / 38.2; two per CU, 16 points of L = 32 / 32 of
  // L = 16: 15.9 / 9.8, fused 29.2 / 19.6; three, 24 of L = 32 / 48 of L = 16: 21.3 /
  // 11.0, fused 39.2 / 23.2; four, 40 of L = 24 / 64 of L = 16: 19.3 / 11.7, fused 32.8
  // / 20.8).  Else thicker slabs, one workgroup per CU (32 points of L = 32 / 48, 96
  // of L = 16 / 32 / 48: 23.0 / 35 / 57 us, fused 35.1 / 73 / 136), from L = 12 on
  // (96 points of L = 12 18.9 and 21.8 us, 140 of L = 8 24.2 and 20.3).
  uint64_t planes = 0;
  uint32_t maxL = 0;
  for (const auto& P : s->ph) {
    planes += P.L;
    maxL = std::max(maxL, P.L);
  }
  // words of all CUs' LDS; windows hold ghost planes too
  const uint64_t room = cu_count(s, ncu) == CVF_OK ? (uint64_t)ncu * resident_lds_limit() / 4 : 0;
  const bool fits = s->total_cells <= room / 5 * 4;
  if (!any_nc && maxL <= 64 && s->sched == CVF_SCHED_REFERENCE && s->nm == 1) {
    const uint64_t per_cu = (planes + ncu - 1) / std::max(ncu, 1u);
    int block = 0;
    if (per_cu <= 1)
      block = maxL <= 16 ? 256 : maxL <= 32 ? 512 : 1024;
    else if (per_cu == 2 && maxL <= 40)
      block = maxL <= 16 ? 256 : 512;
    else if (per_cu == 3 && maxL <= 32)
      block = 256;
    else if (per_cu == 4 && maxL <= 24)
      block = maxL <= 16 ? 128 : 256;
    // with a cluster sweep, a launch per step, small lattices only (L = 8 / 16 /
    // 32: 26.2 / 28.5 / 32.6 us per step, tiles 32.7 / 33.8 / 35.0; 24 of L = 32
    // 72.9 and 77.8)
    const bool one_plane =
        block && (s->nc == 0 ? planes > ncu || s->total_cells < (1u << 20) : maxL <= 32 && per_cu <= 3);
    if (one_plane) {
      t.fused = 2;
      t.streams = (int32_t)per_cu;
      t.slab_planes = 1;
      t.block_chunk = block;
      t.graph_steps = s->nc == 0 ? 64 : 16;
    } else if (s->nc == 0 && maxL >= 12 && fits) {
      t.fused = 2;
      t.slab_planes = 0;
      t.block_chunk = maxL <= 24 ? 512 : 1024;
      t.graph_steps = 64;
    }
  }
  // the fast schedule's step of four phases with two exchanges between: the
  // resident kernel where it holds the points (one-plane slabs while there is
  // a workgroup per plane), up to L = 64, beyond which it has too few
  // workgroups (L = 8 / 16 / 32 / 48 / 64 / 80: 8.9 / 9.4 / 10.9 / 16.6 / 21.1 / 33.3 us per
  // step, the per-pass kernels 19.0 / 20.4 / 20.0 / 20.8 / 22.7 / 21.6; 32 points of
  // L = 32 17.7 and 28.0, 128 of L = 16 .. 48 58.0 and 69.4).  With a cluster
  // sweep, a launch per step, only small ones gain (L = 16 / 32 / 64: 29.3 / 31.2 /
  // 47.3 and 35.4 / 35.0 / 43.0).
  if (s->sched == CVF_SCHED_FAST && s->nm == 1) {
    const bool planes_fit = planes <= ncu, small = maxL <= 32 && s->total_cells < (1u << 21);
    if (s->nc == 0 ? maxL <= 64 && fits : maxL <= 32 && planes_fit) {
      t.fused = 2;
      t.slab_planes = planes_fit ? 1 : 0;
      t.block_chunk = small ? 512 : 1024;
      t.graph_steps = 64;
    }
  }
  return t;
}

// The steps since the aborted resident launch of this mark, again: from the
// lattice that it started from, by launches that wait for nothing, which are
// the handle's plan from now on.  (Its plan needs the card to itself, and
// another process has a part of it.)  The volume chain, which never reads the
// lattice, stands.  rec_base: the steps from there on are recorded again for
// point rec_pt.  The handle's stream has been synchronised.
int redo_steps(cvf_sim* s, uint32_t mark, int64_t rec_base = -1) {
  const int64_t end = s->steps;
  int64_t at = end - (int64_t)(((uint32_t)end + 1 - mark) & 0x7FFFFFFFu);
  HIPC(hipMemcpy(s->words.p, s->words2.p, s->total_cells * 4, hipMemcpyDeviceToDevice));
  s->tune = default_tuning(s, false);
  s->steps = at;
  int rc = build_groups(s);
  s->steps = end;
  if (rc) return rc;
  if (rec_base >= 0) {
    const size_t first = (size_t)(std::max(at, rec_base) - rec_base), n = (size_t)(end - rec_base);
    launch_zero_u32(s->stream, (uint32_t*)(s->hist_series.p + 1 + kHistWords * first), 2 * kHistWords * (n - first));
  }
  if ((rc = fork_groups(s))) return rc;
  while (at < end) {
    const int64_t to = at < rec_base ? std::min(rec_base, end) : end;
    const int n = (int)std::min<int64_t>(64, to - at);
    for (size_t gi = 0; gi < s->groups.size(); ++gi) {
      const bool rec = rec_base >= 0 && at >= rec_base && (int32_t)gi == s->ph[s->rec_pt].group;
      if ((rc = enqueue_steps(s, (int)gi, s->groups[gi]->stream, n, rec, false))) return rc;
    }
    at += n;
  }
  if ((rc = join_groups(s))) return rc;
  HIPC(hipGetLastError());
  HIPC(hipStreamSynchronize(s->stream));
  HIPC(hipMemset(s->rstatus.p, 0, 2 * sizeof(uint32_t)));
  HIPC(hipDeviceSynchronize());
  s->resident_used = false;
  s->obs_at = -1;
  return CVF_OK;
}

// A handle whose stream has been synchronised: steps that a resident launch
// could not finish are done again.  (*done: whether there were any.)
int settle(cvf_sim* s, int64_t rec_base = -1, bool* done = nullptr) {
  if (done) *done = false;
  if (!s->resident_used) return CVF_OK;
  uint32_t status[2];
  HIPC(hipMemcpy(status, s->rstatus.p, sizeof status, hipMemcpyDeviceToHost));
  if (!status[0]) return CVF_OK;
  if (done) *done = true;
  return redo_steps(s, status[1], rec_base);
}

int create_impl(const cvf_params* pts, int32_t n, cvf_sim** out) {
  if (!pts || !out || n <= 0) return fail(CVF_EINVAL, "bad arguments");
  *out = nullptr;
  for (int i = 0; i < n; ++i) {
    int rc = validate(pts[i]);
    if (rc) return rc;
    if (pts[i].n_metropolis != pts[0].n_metropolis || pts[i].n_cluster != pts[0].n_cluster ||
        pts[i].precision != pts[0].precision || pts[i].device_id != pts[0].device_id ||
        pts[i].volume_mode != pts[0].volume_mode || pts[i].schedule != pts[0].schedule)
      return fail(CVF_EINVAL, "state points of a batch must share the MC schedule, precision, "
                              "volume mode and device");
  }
  int ndev = 0;
  HIPC(hipGetDeviceCount(&ndev));
  if (pts[0].device_id < 0 || pts[0].device_id >= ndev)
    // the reference's message, typo included (gpu_water3D.cu:461-465)
    return fail(CVF_EINVAL, "Error: Tried to execute in GPU deive ID = %d\n\tTotal number of devices is %d",
                pts[0].device_id, ndev);
  HIPC(hipSetDevice(pts[0].device_id));
  std::unique_ptr<cvf_sim> s(new cvf_sim);
  s->device = pts[0].device_id;
  s->npts = n;
  s->nm = pts[0].n_metropolis;
  s->nc = pts[0].n_cluster;
  s->precision = pts[0].precision;
  s->sched = pts[0].schedule;
  s->vol_device = pts[0].volume_mode == CVF_VOLUME_DEVICE;
  HIPC(hipStreamCreateWithFlags(&s->stream, hipStreamNonBlocking));
  HIPC(hipEventCreateWithFlags(&s->start_ev, hipEventDisableTiming));
  size_t woff = 0;
  uint32_t maxL = 0;
  for (int i = 0; i < n; ++i) {
    PointHost P;
    P.prm = pts[i];
    P.L = (uint32_t)pts[i].L;
    P.N = P.L * P.L * P.L;
    woff = (woff + 63) & ~(size_t)63;  // 256-byte aligned point start
    P.woff = (uint32_t)woff;
    woff += P.N;
    P.thr = make_thresholds(P.prm.P, P.prm.T, P.prm.J_hb, P.prm.J_sig, P.prm.v_hb);
    shell_table((int)P.L, P.prm.r_cutoff, P.dist, P.freq);
    P.vp.seed = P.prm.seed;
    P.vp.L = (int32_t)P.L;
    P.vp.N = (int32_t)P.N;
    P.vp.T = P.prm.T;
    P.vp.P = P.prm.P;
    P.vp.r_cutoff = P.prm.r_cutoff;
    P.vp.nshell = (int32_t)P.dist.size();
    P.vp.beta = P.thr.beta;
    // volume chain start (gpu_water3D.cu:150, 481, 1128)
    P.vol.r_cell = 1.0001;
    P.vol.V = (double)(int)P.N * P.vol.r_cell * P.vol.r_cell * P.vol.r_cell;
    P.vol.E_vdw = vdw_energy_fp64(P.vol.r_cell, P.prm.r_cutoff, P.dist.data(), P.freq.data(),
                                  (int)P.dist.size());
    P.vol.accepted = 0;
    P.vol.pad = 0;
    maxL = std::max(maxL, P.L);
    s->ph.push_back(P);
  }
  s->total_cells = woff;
  size_t loff = 0;
  for (auto& P : s->ph) {
    P.loff = (uint32_t)loff;
    loff += 6 * (size_t)P.N;
  }
  s->total_nodes = loff;
  if (loff >= 0xFFFFFFFFull) return fail(CVF_ENOMEM, "batch too large for 32-bit node offsets");
  // device buffers
  HIPC(s->words.alloc(s->total_cells));
  HIPC(s->words2.alloc(s->total_cells));
  HIPC(s->parent.alloc(s->total_nodes));
  HIPC(hipMemset(s->parent.p, 0, s->total_nodes * 4));  // labels read as 0 before the first SW step
  HIPC(s->cov.alloc(s->total_cells));
  HIPC(s->pts.alloc(n));
  HIPC(s->pst.alloc(n));
  const uint32_t maxN = maxL * maxL * maxL;
  HIPC(s->csize.alloc(6 * (size_t)maxN));
  HIPC(s->slot.alloc(6 * (size_t)maxN));
  HIPC(s->cclusters.alloc(6 * (size_t)maxN));
  HIPC(s->cblock.alloc(compact_blocks(6 * maxN)));
  HIPC(s->cmom.alloc(4 * (size_t)compact_blocks(6 * maxN)));
  s->max_slots = 3 * maxL * maxL + 1;  // a cluster of >= 2L nodes: at most 6N/(2L)
  HIPC(s->cover.alloc((size_t)s->max_slots * 3 * ((maxL + 31) / 32)));
  HIPC(s->nslot_nperc.alloc(2));
  HIPC(s->rstatus.alloc(4));
  HIPC(hipMemset(s->rstatus.p, 0, 4 * sizeof(uint32_t)));
  int rc = upload_tables(s.get());
  if (rc) return rc;
  std::vector<PointState> st(n);
  for (int i = 0; i < n; ++i) {
    st[i].step = 0;
    st[i].vol = s->ph[i].vol;
  }
  HIPC(hipMemcpy(s->pst.p, st.data(), n * sizeof(PointState), hipMemcpyHostToDevice));
  s->tune = default_tuning(s.get());
  if ((rc = build_groups(s.get()))) return rc;
  // initial configurations
  std::vector<uint32_t> w;
  for (int i = 0; i < n; ++i) {
    init_words(s->ph[i], w);
    rc = upload_point_words(s.get(), i, w);
    if (rc) return rc;
  }
  HIPC(hipDeviceSynchronize());
  *out = s.release();
  return CVF_OK;
}

}  // namespace

extern "C" {

void cvf_params_default(cvf_params* p) {
  memset(p, 0, sizeof *p);
  p->L = 32;
  p->P = 0.45f;
  p->T = 0.815f;
  p->seed = 44648604ull;
  p->n_metropolis = 1;
  p->n_cluster = 0;
  p->r_cutoff = 6.0f;
  p->flag_config = 0;
  p->flag_chessboard = 1;
  p->device_id = 0;
  p->J_hb = 0.5f;
  p->J_sig = 0.08f;
  p->v_hb = 0.6f;
  p->precision = CVF_FP64;
  p->volume_mode = CVF_VOLUME_HOST;
}

int cvf_create(const cvf_params* p, cvf_sim** out) { return create_impl(p, 1, out); }

int cvf_create_batch(const cvf_params* pts, int32_t n, cvf_sim** out) {
  return create_impl(pts, n, out);
}

void cvf_destroy(cvf_sim* s) {
  if (!s) return;
  (void)hipSetDevice(s->device);
  (void)hipStreamSynchronize(s->stream);
  delete s;
}

const char* cvf_last_error(void) { return g_err.c_str(); }

int cvf_set_config(cvf_sim* s, int32_t pt, const uint8_t* sigma6N, const uint8_t* eta6N) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  if (!sigma6N || !eta6N) return fail(CVF_EINVAL, "null config buffer");
  HIPC(hipSetDevice(s->device));
  const PointHost& P = s->ph[pt];
  const size_t n6 = 6 * (size_t)P.N;
  if ((rc = reserve_config(s, n6))) return rc;
  uint8_t* dev = s->cfg_bytes.p;
  uint32_t* res = reinterpret_cast<uint32_t*>(dev + 2 * n6);
  std::vector<uint8_t> in;  // both arrays and the results' initial bits, of a small point
  if (P.N < kSmallConfig) {
    in.assign(2 * n6 + kConfigResults, 0xFF);
    memcpy(in.data(), sigma6N, n6);
    memcpy(in.data() + n6, eta6N, n6);
  }
  uint32_t out[3];
  for (;;) {
    if (!in.empty()) {
      HIPC(hipMemcpyAsync(dev, in.data(), in.size(), hipMemcpyHostToDevice, s->stream));
    } else {
      HIPC(hipMemcpyAsync(dev, sigma6N, n6, hipMemcpyHostToDevice, s->stream));
      HIPC(hipMemcpyAsync(dev + n6, eta6N, n6, hipMemcpyHostToDevice, s->stream));
      HIPC(hipMemsetAsync(res, 0xFF, kConfigResults, s->stream));
    }
    // words2 is free between steps (unless a resident launch was aborted): the
    // packed input, decoded into words
    launch_config_in(s->stream, dev, dev + n6, P.L, P.prm.flag_chessboard, s->words2.p + P.woff, s->words.p + P.woff,
                     res, res + 1, s->rstatus.p, res + 2);
    HIPC(hipGetLastError());
    HIPC(hipMemcpyAsync(out, res, sizeof out, hipMemcpyDeviceToHost, s->stream));
    HIPC(hipStreamSynchronize(s->stream));
    bool again = false;
    if (out[2] && (rc = settle(s, -1, &again))) return rc;
    if (!again) break;
  }
  if (out[0] != 0xFFFFFFFFu) {
    const uint32_t i = out[0] / 2;
    if (out[0] & 1u)
      return fail(CVF_ERANGE, "Unexpected value for active_bond (%d) appeared in line %u", eta6N[i], i % P.N);
    return fail(CVF_ERANGE, "Unexpected value for spin (%d) appeared in line %u", sigma6N[i], i % P.N);
  }
  s->obs_at = -1;
  return (int)(out[1] + 1u);  // counted from all ones; without the chessboard nothing is counted
}

int cvf_get_config(cvf_sim* s, int32_t pt, uint8_t* sigma6N, uint8_t* eta6N) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  HIPC(hipSetDevice(s->device));
  const PointHost& P = s->ph[pt];
  const size_t N = P.N, n6 = 6 * N;
  if (N < kSmallConfig) {
    HIPC(hipStreamSynchronize(s->stream));
    if ((rc = settle(s))) return rc;
    std::vector<uint32_t> w(N);
    HIPC(hipMemcpy(w.data(), s->words.p + P.woff, N * sizeof(uint32_t), hipMemcpyDeviceToHost));
    for (int a = 0; a < 6; ++a) {
      if (sigma6N)
        for (size_t c = 0; c < N; ++c) sigma6N[a * N + c] = (uint8_t)sigma_of(w[c], a);
      if (eta6N)
        for (size_t c = 0; c < N; ++c) eta6N[a * N + c] = (uint8_t)eta_of(w[c], a);
    }
    return CVF_OK;
  }
  if ((rc = reserve_config(s, n6))) return rc;
  bool again;
  do {
    launch_config_out(s->stream, s->words.p + P.woff, P.N, s->cfg_bytes.p, s->cfg_bytes.p + n6);
    HIPC(hipGetLastError());
    HIPC(hipStreamSynchronize(s->stream));
    if ((rc = settle(s, -1, &again))) return rc;
  } while (again);
  if (sigma6N) HIPC(hipMemcpy(sigma6N, s->cfg_bytes.p, n6, hipMemcpyDeviceToHost));
  if (eta6N) HIPC(hipMemcpy(eta6N, s->cfg_bytes.p + n6, n6, hipMemcpyDeviceToHost));
  return CVF_OK;
}

// n_steps MC steps as resident launches or graph launches; group rec_gi (if
// >= 0) replays its recording sequences.
int run_steps(cvf_sim* s, int64_t n_steps, int rec_gi) {
  if (rec_gi < 0 && s->groups.size() == 1 && resident_sequences(s, *s->groups[0])) {
    for (int64_t i = 0; i < n_steps;) {
      const int k = (int)std::min<int64_t>(s->tune.graph_steps, n_steps - i);
      {
        ResidentTurn turn;
        HIPC(turn.take(&s->turn));
        if (int rc = enqueue_resident(s, 0, s->stream, k)) return rc;
      }
      host_moves(s, k);
      i += k;
    }
    return CVF_OK;
  }
  int rc = capture_step_graphs(s);
  if (rc) return rc;
  if (s->nc > 0 && n_steps > 0) s->sw_labels = true;
  if (rec_gi >= 0 && (rc = capture_rec_graphs(s, rec_gi))) return rc;
  // one group's graphs go to the main stream itself
  const bool fork = s->groups.size() > 1;
  if (fork && (rc = fork_groups(s))) return rc;
  const std::vector<int>& sizes = s->groups[0]->gsteps;  // the same for every group
  for (int64_t i = 0; i < n_steps;) {
    size_t c = 0;
    while (sizes[c] > n_steps - i) ++c;  // the last size is 1
    {
      ResidentTurn turn;
      if (s->groups[0]->resident) HIPC(turn.take(&s->turn));
      for (size_t gi = 0; gi < s->groups.size(); ++gi) {
        Group& g = *s->groups[gi];
        if (g.resident) s->resident_used = true;
        HIPC(hipGraphLaunch((int)gi == rec_gi ? g.rgexecs[c] : g.gexecs[c], fork ? g.stream : s->stream));
      }
    }
    host_moves(s, sizes[c]);
    i += sizes[c];
  }
  return fork ? join_groups(s) : CVF_OK;
}

int cvf_step(cvf_sim* s, int64_t n_steps) {
  if (!s) return fail(CVF_EINVAL, "null handle");
  if (n_steps < 0) return fail(CVF_EINVAL, "negative step count");
  if (n_steps == 0) return CVF_OK;
  HIPC(hipSetDevice(s->device));
  return run_steps(s, n_steps, -1);
}

int cvf_sync(cvf_sim* s) {
  if (!s) return fail(CVF_EINVAL, "null handle");
  HIPC(hipSetDevice(s->device));
  HIPC(hipStreamSynchronize(s->stream));
  return settle(s);
}

// For the tests: the handle's next resident launch (of steps not yet enqueued)
// finds itself aborted, as one of its waits that timed out leaves it.
int cvf_abort_next_launch(cvf_sim* s) {
  if (!s->groups[0]->resident) return fail(CVF_EINVAL, "no resident plan");
  HIPC(hipSetDevice(s->device));
  HIPC(hipStreamSynchronize(s->stream));
  const uint32_t status[2] = {1u, launch_mark((uint64_t)s->steps)};
  HIPC(hipMemcpy(s->rstatus.p, status, sizeof status, hipMemcpyHostToDevice));
  return CVF_OK;
}

int cvf_get_volume(cvf_sim* s, int32_t pt, double* r_cell, double* V, double* E_vdw) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  HIPC(hipSetDevice(s->device));
  VolState v = s->ph[pt].vol;
  if (s->vol_device) {
    PointState st;
    HIPC(hipStreamSynchronize(s->stream));
    HIPC(hipMemcpy(&st, s->pst.p + pt, sizeof st, hipMemcpyDeviceToHost));
    v = st.vol;
  }
  if (r_cell) *r_cell = v.r_cell;
  if (V) *V = v.V;
  if (E_vdw) *E_vdw = v.E_vdw;
  return CVF_OK;
}

int cvf_observe(cvf_sim* s, int32_t pt, cvf_obs* o) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  if (!o) return fail(CVF_EINVAL, "null output");
  HIPC(hipSetDevice(s->device));
  while (s->obs_at != s->steps) {
    launch_observe(s->stream, s->tab_cell_all.p, s->nb_cell_all, s->words.p, observe_span(s->total_cells), s->pst.p,
                   s->rstatus.p, ObsOut{s->obs_part, s->obs_ps, s->obs_status}, s->bonds.p);
    if (s->n_capped)
      launch_capped_hb(s->stream, s->tab_capped.p, s->n_capped, s->capped_L, s->bonds.p, s->obs_capped);
    HIPC(hipGetLastError());
    HIPC(hipStreamSynchronize(s->stream));
    bool again = false;
    if (*s->obs_status && (rc = settle(s, -1, &again))) return rc;
    if (again) continue;
    s->obs_nhb2.assign(s->npts, 0);
    s->obs_nsig.assign(s->npts, 0);
    for (size_t b = 0; b < s->obs_point.size(); ++b)
      if (s->obs_point[b] >= 0) {
        s->obs_nhb2[s->obs_point[b]] += s->obs_part[b].x;
        s->obs_nsig[s->obs_point[b]] += s->obs_part[b].y;
      }
    s->obs_at = s->steps;
  }
  // the volume chain as of the same step
  const VolState& vol = s->vol_device ? s->obs_ps[pt].vol : s->ph[pt].vol;
  const double r_cell = vol.r_cell, E_vdw = vol.E_vdw;
  const PointHost& P = s->ph[pt];
  const int64_t nhb2 = P.prm.flag_chessboard ? s->obs_nhb2[pt] : (int64_t)s->obs_capped[pt];
  const int64_t nsig = s->obs_nsig[pt];
  // measure(), gpu_water3D.cu:2138-2152
  const double n_hb = 0.5 * (double)nhb2;
  double e = E_vdw + n_hb * (double)(-P.prm.J_hb);
  const double v = (double)(int)P.N * r_cell * r_cell * r_cell + n_hb * (double)P.prm.v_hb;
  e += (double)(-P.prm.J_sig) * (double)nsig;
  o->step = s->steps;
  o->E = e;
  o->H = e + (double)P.prm.P * v;
  o->V = v;
  o->n_hb = n_hb;
  o->m = (double)nsig / (1. * (double)P.N * 15.);
  o->r_cell = r_cell;
  o->E_vdw = E_vdw;
  o->nhb2 = nhb2;
  o->n_sigma = nsig;
  return CVF_OK;
}

int cvf_sigma_histogram(cvf_sim* s, int32_t pt, int64_t counts6[6]) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  if (!counts6) return fail(CVF_EINVAL, "null output");
  HIPC(hipSetDevice(s->device));
  const PointHost& P = s->ph[pt];
  if (!s->hist.p) HIPC(s->hist.alloc(1 + kHistWords));  // kept for the handle's life: called every step
  unsigned long long out[1 + kHistWords];
  bool again;
  do {
    again = false;
    launch_zero_u32(s->stream, (uint32_t*)s->hist.p, 2 * (1 + kHistWords));
    launch_sigma_hist(s->stream, s->words.p + P.woff, P.N, s->hist.p + 1, s->rstatus.p, s->hist.p);
    HIPC(hipMemcpyAsync(out, s->hist.p, sizeof out, hipMemcpyDeviceToHost, s->stream));
    HIPC(hipStreamSynchronize(s->stream));
    if (out[0] && (rc = settle(s, -1, &again))) return rc;
  } while (again);
  for (int i = 0; i < 6; ++i) {
    counts6[i] = 0;
    for (int r = 0; r < kHistReplicas; ++r) counts6[i] += (int64_t)out[1 + 6 * r + i];
  }
  return CVF_OK;
}

int cvf_step_histograms(cvf_sim* s, int32_t pt, int64_t n_steps, int64_t* counts) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  if (n_steps < 0) return fail(CVF_EINVAL, "negative step count");
  if (n_steps == 0) return CVF_OK;
  if (!counts) return fail(CVF_EINVAL, "null output");
  HIPC(hipSetDevice(s->device));
  if (!s->hist_series.p) HIPC(s->hist_series.alloc(1 + kHistWords * (size_t)kHistSpan));
  if (!s->hist_base.p) HIPC(s->hist_base.alloc(1));
  if (s->rec_pt != pt) {
    for (auto& g : s->groups) g->drop_rec_graphs();
    s->rec_pt = pt;
  }
  std::vector<unsigned long long> buf;
  for (int64_t i0 = 0; i0 < n_steps; i0 += kHistSpan) {
    const int64_t n = std::min<int64_t>(kHistSpan, n_steps - i0);
    // slots are counted from the step count before this span
    s->hist_base_host = (uint64_t)s->steps;
    HIPC(hipMemcpyAsync(s->hist_base.p, &s->hist_base_host, sizeof(uint64_t), hipMemcpyHostToDevice, s->stream));
    launch_zero_u32(s->stream, (uint32_t*)s->hist_series.p, 2 * (1 + kHistWords * (size_t)n));
    if ((rc = run_steps(s, n, s->ph[pt].group))) return rc;
    buf.resize(1 + kHistWords * (size_t)n);
    bool again;
    do {
      again = false;
      HIPC(hipMemcpyAsync(buf.data(), s->hist_series.p, buf.size() * sizeof(unsigned long long),
                          hipMemcpyDeviceToHost, s->stream));
      HIPC(hipStreamSynchronize(s->stream));
      if (buf[0] && (rc = settle(s, (int64_t)s->hist_base_host, &again))) return rc;
    } while (again);
    for (int64_t i = 0; i < n; ++i)
      for (int v = 0; v < 6; ++v) {
        int64_t c = 0;
        for (int r = 0; r < kHistReplicas; ++r) c += (int64_t)buf[1 + kHistWords * i + 6 * r + v];
        counts[6 * (i0 + i) + v] = c;
      }
  }
  return CVF_OK;
}

int cvf_get_labels(cvf_sim* s, int32_t pt, int32_t* labels6N) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  HIPC(hipSetDevice(s->device));
  HIPC(hipStreamSynchronize(s->stream));
  if ((rc = settle(s))) return rc;
  const PointHost& P = s->ph[pt];
  HIPC(hipMemcpy(labels6N, s->parent.p + P.loff, 6 * (size_t)P.N * 4, hipMemcpyDeviceToHost));
  return CVF_OK;
}

namespace {

// print_cluster_statistics (gpu_water3D.cu:2677-2721) on the cluster sizes
// indexed by label (0 where no cluster): float sums in ascending label
// order, int32 size*size with wrap-around.
void assemble_cluster_row(const int32_t* size, uint32_t n, int32_t n_perc, cvf_cstat* c) {
  int32_t largest = 0, second = 0, ncl = 0;
  float average = 0, average2 = 0;
  for (uint32_t i = 0; i < n; ++i) {
    const int32_t sz = size[i];
    if (sz == 0) continue;
    ++ncl;
    average += (float)sz;
    average2 += (float)(int32_t)((uint32_t)sz * (uint32_t)sz);
    if (sz > largest) {
      second = largest;
      largest = sz;
    } else if (sz > second) {
      second = sz;
    }
  }
  average /= (float)ncl;
  average2 /= (float)ncl;
  average2 -= average * average;
  c->largest = largest;
  c->second = second;
  c->n_perc = n_perc;
  c->n_clusters = ncl;
  c->mean = average;
  c->var = average2;
}

}  // namespace

int cvf_cluster_stats(cvf_sim* s, int32_t pt, cvf_cstat* c) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  if (!c) return fail(CVF_EINVAL, "null output");
  HIPC(hipSetDevice(s->device));
  const PointHost& P = s->ph[pt];
  const uint32_t nn = 6 * P.N, L = P.L;
  if (!s->sw_labels) {
    // no Swendsen-Wang step yet: every label is 0, one cluster of all 6N
    // nodes that covers every x (the row SOURCE/cluster.out shows)
    const int32_t all = (int32_t)nn;
    assemble_cluster_row(&all, 1, nn >= 2 * L ? 1 : 0, c);
    return CVF_OK;
  }
  const uint32_t* label = s->parent.p + P.loff;
  const uint32_t minsize = 2 * L, nw = (L + 31) / 32;
  uint32_t* nslot = s->nslot_nperc.p;
  bool again;
  do {
    again = false;
    launch_zero3_u32(s->stream, (uint32_t*)s->csize.p, nn, nslot, 2, s->cover.p, (size_t)s->max_slots * 3 * nw);
    launch_cluster_sizes(s->stream, label, nn, s->csize.p);
    // the clusters' counts, moments and slots, then the percolation test of
    // those that have a slot
    launch_compact_count(s->stream, label, s->csize.p, nn, s->cblock.p, s->cmom.p, minsize, s->slot.p, nslot,
                         s->max_slots);
    launch_perc_cover(s->stream, label, nn, L, s->csize.p, minsize, s->slot.p, nslot, s->cover.p, s->max_slots);
    launch_perc_count(s->stream, s->cover.p, nslot, L, s->max_slots, nslot + 1);
    launch_compact_scan(s->stream, s->cblock.p, nn, s->cmom.p, nslot, s->rstatus.p, s->csums);
    HIPC(hipGetLastError());
    HIPC(hipStreamSynchronize(s->stream));
    if (s->csums->aborted && (rc = settle(s, -1, &again))) return rc;
  } while (again);
  const ClusterSums& sums = *s->csums;
  const uint32_t np[2] = {sums.slots, sums.percolating}, ncl = sums.clusters;
  if (np[0] > s->max_slots) return fail(CVF_EDEVICE, "percolation slot overflow");
  if (ncl == 0 || ncl > nn) return fail(CVF_EDEVICE, "cluster compaction overflow");
  constexpr uint64_t kExact = 1ull << 24;  // every integer up to 2^24 is a float
  if (sums.sum <= kExact && sums.squares <= kExact) {
    // print_cluster_statistics (gpu_water3D.cu:2691-2718) adds the sizes and
    // their squares as floats in label order: with every partial sum an
    // integer up to 2^24 (and every size below 4097, so no int32 square
    // wraps) each addition is exact, and the sums are these integers
    float average = (float)sums.sum, average2 = (float)sums.squares;
    average /= (float)ncl;
    average2 /= (float)ncl;
    average2 -= average * average;
    c->largest = (int32_t)sums.largest;
    c->second = (int32_t)sums.second;
    c->n_perc = (int32_t)np[1];
    c->n_clusters = (int32_t)ncl;
    c->mean = average;
    c->var = average2;
    return CVF_OK;
  }
  // larger sums round: the host adds the sizes in label order
  launch_compact_write(s->stream, label, s->csize.p, nn, s->cblock.p, s->cclusters.p);
  std::vector<int32_t> size(ncl);
  HIPC(hipMemcpyAsync(size.data(), s->cclusters.p, (size_t)ncl * 4, hipMemcpyDeviceToHost, s->stream));
  HIPC(hipStreamSynchronize(s->stream));
  assemble_cluster_row(size.data(), ncl, (int32_t)np[1], c);
  return CVF_OK;
}

int cvf_get_shells(cvf_sim* s, int32_t pt, float* dist, int32_t* freq, int32_t cap, int32_t* nshell) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  const PointHost& P = s->ph[pt];
  if (nshell) *nshell = (int32_t)P.dist.size();
  const int32_t n = std::min<int32_t>(cap, (int32_t)P.dist.size());
  for (int32_t k = 0; k < n; ++k) {
    if (dist) dist[k] = P.dist[k];
    if (freq) freq[k] = P.freq[k];
  }
  return CVF_OK;
}

int cvf_set_shells(cvf_sim* s, int32_t pt, const float* dist, const int32_t* freq, int32_t nshell) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  if (nshell < 0 || (nshell > 0 && (!dist || !freq))) return fail(CVF_EINVAL, "bad shell table");
  HIPC(hipSetDevice(s->device));
  HIPC(hipStreamSynchronize(s->stream));
  PointHost& P = s->ph[pt];
  P.dist.assign(dist, dist + nshell);
  P.freq.assign(freq, freq + nshell);
  P.vol.E_vdw = vdw_energy_fp64(P.vol.r_cell, P.prm.r_cutoff, P.dist.data(), P.freq.data(), nshell);
  rc = upload_tables(s);
  if (rc) return rc;
  // device-side volume state follows the host one
  PointState st;
  HIPC(hipMemcpy(&st, s->pst.p + pt, sizeof st, hipMemcpyDeviceToHost));
  st.vol.E_vdw = vdw_energy_fp64(st.vol.r_cell, P.prm.r_cutoff, P.dist.data(), P.freq.data(), nshell);
  HIPC(hipMemcpy(s->pst.p + pt, &st, sizeof st, hipMemcpyHostToDevice));
  s->obs_at = -1;
  return CVF_OK;
}

int cvf_info(cvf_sim* s, int32_t pt, int32_t* n_points, int32_t* L, int64_t* steps) {
  if (!s) return fail(CVF_EINVAL, "null handle");
  if (n_points) *n_points = s->npts;
  if (steps) *steps = s->steps;
  if (L) {
    int rc = check_pt(s, pt);
    if (rc) return rc;
    *L = (int32_t)s->ph[pt].L;
  }
  return CVF_OK;
}

int cvf_get_stream(cvf_sim* s, void** stream) {
  if (!s || !stream) return fail(CVF_EINVAL, "null argument");
  *stream = (void*)s->stream;
  return CVF_OK;
}

int cvf_profile_steps(cvf_sim* s, int64_t n_steps, double* kernel_ms, int64_t* launches,
                      int32_t n_classes) {
  if (!s || n_steps < 0 || !kernel_ms || n_classes < CVF_KCLASS_COUNT)
    return fail(CVF_EINVAL, "bad arguments");
  HIPC(hipSetDevice(s->device));
  if (!s->vol_device && n_steps > 0)
    return fail(CVF_EUNSUPPORTED, "profiling needs the device volume mode");
  struct Rec {
    hipEvent_t a, b;
    int cls;
  };
  std::vector<Rec> recs;
  hipError_t err = hipSuccess;
  // each launch records its own start and end (hipExtLaunchKernelGGL); the
  // groups run concurrently on their streams, as in cvf_step
  auto timed = [&](int cls, auto&& fn) {
    Rec r{nullptr, nullptr, cls};
    if (err == hipSuccess) err = hipEventCreate(&r.a);
    if (err == hipSuccess) err = hipEventCreate(&r.b);
    if (err != hipSuccess) return;
    set_launch_timing(r.a, r.b);
    fn();
    set_launch_timing(nullptr, nullptr);
    recs.push_back(r);
  };
  ResidentTurn turn;
  if (s->groups[0]->resident) HIPC(turn.take(&s->turn));
  int rc = fork_groups(s);
  if (rc) return rc;
  if (s->nc > 0 && n_steps > 0) s->sw_labels = true;
  // a resident group without SW steps runs all n_steps in one launch, as in
  // its captured graphs (timed once, with one volume-chain launch)
  for (size_t gi = 0; gi < s->groups.size(); ++gi) {
    Group& g = *s->groups[gi];
    if (!g.resident || s->nc > 0 || n_steps == 0) continue;
    s->resident_used = true;
    timed(CVF_KCLASS_RESIDENT, [&] {
      run_resident(s, g, g.stream, s->cur_steps.p + gi, 0, (uint32_t)n_steps, nullptr);
    });
    timed(CVF_KCLASS_BEGIN, [&] {
      launch_vol_chain(g.stream, s->pts.p, g.plist.p, (int)g.points.size(), s->pst.p, s->cur_steps.p + gi,
                       (uint32_t)n_steps, s->dist.p, s->freq.p, s->precision, s->vol_device);
    });
  }
  for (int64_t i = 0; i < n_steps; ++i) {
    for (size_t gi = 0; gi < s->groups.size(); ++gi) {
      Group& g = *s->groups[gi];
      if (g.resident && s->nc == 0) continue;
      hipStream_t st = g.stream;
      int par = 0;
      enqueue_lattice(s, (int)gi, st, 0, timed, par);
      timed(CVF_KCLASS_BEGIN, [&] {
        launch_vol_chain(st, s->pts.p, g.plist.p, (int)g.points.size(), s->pst.p, s->cur_steps.p + gi, 1,
                         s->dist.p, s->freq.p, s->precision, s->vol_device);
      });
    }
    ++s->steps;
  }
  if (err != hipSuccess) return fail(CVF_EDEVICE, "event creation failed: %s", hipGetErrorString(err));
  if ((rc = join_groups(s))) return rc;
  HIPC(hipGetLastError());
  HIPC(hipStreamSynchronize(s->stream));
  std::vector<double> tot(CVF_KCLASS_COUNT, 0.0);
  std::vector<int64_t> cnt(CVF_KCLASS_COUNT, 0);
  for (auto& r : recs) {
    float ms = 0;
    HIPC(hipEventElapsedTime(&ms, r.a, r.b));
    tot[r.cls] += ms;
    cnt[r.cls] += 1;
  }
  for (auto& r : recs) {
    (void)hipEventDestroy(r.a);
    (void)hipEventDestroy(r.b);
  }
  for (int c = 0; c < CVF_KCLASS_COUNT; ++c) {
    kernel_ms[c] = cnt[c] ? tot[c] / (double)cnt[c] : 0.0;
    if (launches) launches[c] = cnt[c];
  }
  s->obs_at = -1;
  return settle(s);
}

int cvf_get_plan(cvf_sim* s, int32_t pt, int32_t* group, int32_t* slab_planes, int32_t* chunk_sweeps,
                 int32_t* kind) {
  int rc = check_pt(s, pt);
  if (rc) return rc;
  const PointHost& P = s->ph[pt];
  const Group& g = *s->groups[P.group];
  if (group) *group = P.group;
  if (kind) *kind = g.resident ? 2 : P.slab_T || g.tiled ? 1 : 0;
  if (g.resident) {
    if (slab_planes) *slab_planes = (int32_t)P.slab_T;
    if (chunk_sweeps) *chunk_sweeps = 0;
    return CVF_OK;
  }
  if (slab_planes) *slab_planes = (int32_t)P.slab_T;
  if (chunk_sweeps) {
    // half-sweeps per fused launch of the reference schedule: whole passes
    // only where every window of the group holds the wider halo
    const bool whole = s->sched == CVF_SCHED_REFERENCE && s->tune.chunk_sweeps == kMaxChunk &&
                       g.chunk_lds_long != 0;
    const bool none = (P.slab_T == 0 && !g.tiled) || s->nm == 0 || s->sched != CVF_SCHED_REFERENCE;
    *chunk_sweeps = none ? 0 : whole ? kMaxChunk : kChunk;
  }
  return CVF_OK;
}

int cvf_get_tuning(cvf_sim* s, cvf_tuning* t) {
  if (!s || !t) return fail(CVF_EINVAL, "null argument");
  *t = s->tune;
  return CVF_OK;
}

int cvf_set_tuning(cvf_sim* s, const cvf_tuning* t) {
  if (!s || !t) return fail(CVF_EINVAL, "null argument");
  int rc = check_tuning(*t);
  if (rc) return rc;
  HIPC(hipSetDevice(s->device));
  HIPC(hipStreamSynchronize(s->stream));
  if ((rc = settle(s))) return rc;
  s->tune = *t;
  return build_groups(s);
}

}  // extern "C"

namespace {

std::string tune_key(cvf_sim* s) {
  hipDeviceProp_t prop;
  std::string arch = hipGetDeviceProperties(&prop, s->device) == hipSuccess ? prop.gcnArchName : "?";
  std::vector<uint32_t> Ls;
  for (auto& P : s->ph) Ls.push_back(P.L);
  std::sort(Ls.begin(), Ls.end());
  std::string k = arch.substr(0, arch.find(':')) + "|";
  for (size_t i = 0; i < Ls.size();) {
    size_t j = i;
    while (j < Ls.size() && Ls[j] == Ls[i]) ++j;
    k += std::to_string(Ls[i]) + "x" + std::to_string(j - i) + ",";
    i = j;
  }
  // the non-chessboard rule changes the window halos and the default
  // launch length, so its points are part of the shape
  int n_nochess = 0;
  for (const auto& P : s->ph) n_nochess += !P.prm.flag_chessboard;
  k += "|nm" + std::to_string(s->nm) + "|nc" + std::to_string(s->nc) + "|ncb" + std::to_string(n_nochess) + "|p" +
       std::to_string(s->precision) + "|v" + std::to_string(s->vol_device) + "|s" + std::to_string(s->sched);
  return k;
}

// Some stream group can run whole-pass fused launches (chunk_sweeps = 12).
bool whole_passes_possible(const cvf_sim* s) {
  if (s->sched != CVF_SCHED_REFERENCE || s->nm <= 0) return false;
  for (const auto& g : s->groups)
    if (g->fused && g->chunk_lds_long != 0) return true;
  return false;
}

bool cache_lookup(const std::string& key, cvf_tuning* t) {
  const char* path = getenv("CVF_TUNE_CACHE");
  if (!path || !*path) return false;
  FILE* f = fopen(path, "r");
  if (!f) return false;
  char line[1024];
  bool found = false;
  while (fgets(line, sizeof line, f)) {
    char k[768];
    cvf_tuning c;
    if (sscanf(line, "%767s %d %d %d %d %d %d %d %d %d", k, &c.streams, &c.block_sigma, &c.block_eta,
               &c.block_cell, &c.graph_steps, &c.fused, &c.slab_planes, &c.block_chunk, &c.chunk_sweeps) == 10 &&
        key == k) {
      *t = c;
      found = true;
    }
  }
  fclose(f);
  return found;
}

void cache_store(const std::string& key, const cvf_tuning& c) {
  const char* path = getenv("CVF_TUNE_CACHE");
  if (!path || !*path) return;
  FILE* f = fopen(path, "a");
  if (!f) return;
  fprintf(f, "%s %d %d %d %d %d %d %d %d %d\n", key.c_str(), c.streams, c.block_sigma, c.block_eta,
          c.block_cell, c.graph_steps, c.fused, c.slab_planes, c.block_chunk, c.chunk_sweeps);
  fclose(f);
}

}  // namespace

extern "C" {

extern "C" int cvf_autotune(cvf_sim* s, int32_t steps_per_trial, cvf_tuning* chosen) {
  if (!s || steps_per_trial < 1) return fail(CVF_EINVAL, "bad arguments");
  HIPC(hipSetDevice(s->device));
  const std::string key = tune_key(s);
  cvf_tuning best = s->tune;
  int rc;
  if (cache_lookup(key, &best) && check_tuning(best) == CVF_OK) {
    if ((rc = cvf_set_tuning(s, &best))) return rc;
    if (chosen) *chosen = best;
    return CVF_OK;
  }
  // snapshot of everything a step changes
  HIPC(hipStreamSynchronize(s->stream));
  if ((rc = settle(s))) return rc;
  DevBuf<uint32_t> w0, l0;
  DevBuf<PointState> p0;
  HIPC(w0.alloc(s->total_cells));
  HIPC(l0.alloc(s->total_nodes));
  HIPC(p0.alloc(s->npts));
  HIPC(hipMemcpy(w0.p, s->words.p, s->total_cells * 4, hipMemcpyDeviceToDevice));
  HIPC(hipMemcpy(l0.p, s->parent.p, s->total_nodes * 4, hipMemcpyDeviceToDevice));
  HIPC(hipMemcpy(p0.p, s->pst.p, s->npts * sizeof(PointState), hipMemcpyDeviceToDevice));
  std::vector<VolState> hv;
  for (auto& P : s->ph) hv.push_back(P.vol);
  const int64_t steps0 = s->steps;
  const bool sw0 = s->sw_labels;
  // candidates
  std::vector<cvf_tuning> cand;
  const cvf_tuning base = default_tuning(s);
  cand.push_back(base);
  for (int streams : {1, 2, 4}) {
    if (streams > s->npts) continue;
    if (s->sched == CVF_SCHED_FAST) {
      // colour-pass workgroup sizes, the eta sweep per family or as one slab
      // launch (fused)
      for (int bs : {64, 128, 256, 512})
        for (int fused : {0, 1})
          for (int bc : {512, 1024}) {
            if (!fused && bc != 512) continue;
            cvf_tuning t = base;
            t.streams = streams;
            t.fused = fused;
            t.block_chunk = bc;
            t.slab_planes = 0;
            t.graph_steps = 16;
            t.chunk_sweeps = kChunk;  // no half-sweeps in fused launches here
            t.block_sigma = t.block_eta = bs;
            cand.push_back(t);
          }
      // the resident kernel, `streams` workgroups per CU
      if (streams <= 2)
        for (int bc : {512, 1024})
          for (int slab : {0, 1}) {
            cvf_tuning t = base;
            t.streams = streams;
            t.fused = 2;
            t.slab_planes = slab;
            t.block_chunk = bc;
            t.graph_steps = 64;
            t.chunk_sweeps = kChunk;
            cand.push_back(t);
          }
      continue;
    }
    for (int slab : {0, 8, 4, 2, 1})
      for (int bc : {256, 512, 1024})
        for (int len : {kChunk, kMaxChunk}) {
          // whole-pass launches only where the wider windows can fit
          if (len == kMaxChunk && slab == 8) continue;
          cvf_tuning t = base;
          t.streams = streams;
          t.fused = 1;
          t.slab_planes = slab;
          t.block_chunk = bc;
          t.chunk_sweeps = len;
          cand.push_back(t);
        }
    if (streams <= 2)
      for (int bc : {256, 512, 1024})
        for (int gs : {16, 64})
          for (int slab : {0, 1}) {
            // resident kernel: one stream group, `streams` workgroups per CU;
            // automatic slabs, or one-plane slabs (small or wide lattices)
            // at 512 and 1024 threads
            if (slab && bc == 256) continue;
            cvf_tuning t = base;
            t.streams = streams;
            t.fused = 2;
            t.slab_planes = slab;
            t.block_chunk = bc;
            t.graph_steps = gs;
            t.chunk_sweeps = kChunk;
            cand.push_back(t);
          }
    for (int bs : {64, 256}) {
      cvf_tuning t = base;
      t.streams = streams;
      t.fused = 0;
      t.chunk_sweeps = kChunk;
      t.block_sigma = t.block_eta = bs;
      cand.push_back(t);
    }
  }
  hipEvent_t a, b;
  HIPC(hipEventCreate(&a));
  HIPC(hipEventCreate(&b));
  double best_ms = 1e30;
  for (const auto& t : cand) {
    if ((rc = cvf_set_tuning(s, &t))) break;
    // a whole-pass candidate that no stream group can take launches exactly
    // as its 6-sweep twin: not timed, so the result names what runs
    if (t.fused && t.chunk_sweeps == kMaxChunk && !whole_passes_possible(s)) continue;
    if ((rc = cvf_step(s, 2))) break;
    // at least one replay of the candidate's longest step graph (shorter
    // trials would replay the same shorter graphs for every graph length);
    // candidates compare by time per step
    const int n = std::max<int>(steps_per_trial, t.graph_steps);
    HIPC(hipEventRecord(a, s->stream));
    if ((rc = cvf_step(s, n))) break;
    HIPC(hipEventRecord(b, s->stream));
    HIPC(hipEventSynchronize(b));
    float ms = 0;
    HIPC(hipEventElapsedTime(&ms, a, b));
    bool aborted = false;
    if ((rc = settle(s, -1, &aborted))) break;
    if (!aborted && (double)ms / n < best_ms) {
      best_ms = (double)ms / n;
      best = t;
    }
  }
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  // restore the snapshot and apply the winner
  HIPC(hipStreamSynchronize(s->stream));
  if (!rc) rc = settle(s);
  HIPC(hipMemcpy(s->words.p, w0.p, s->total_cells * 4, hipMemcpyDeviceToDevice));
  HIPC(hipMemcpy(s->parent.p, l0.p, s->total_nodes * 4, hipMemcpyDeviceToDevice));
  HIPC(hipMemcpy(s->pst.p, p0.p, s->npts * sizeof(PointState), hipMemcpyDeviceToDevice));
  for (size_t i = 0; i < s->ph.size(); ++i) s->ph[i].vol = hv[i];
  s->steps = steps0;
  s->sw_labels = sw0;
  s->obs_at = -1;
  if (rc) return rc;
  if ((rc = upload_group_steps(s))) return rc;
  if ((rc = cvf_set_tuning(s, &best))) return rc;
  cache_store(key, best);
  if (chosen) *chosen = best;
  return CVF_OK;
}

int cvf_vdw_energy(int32_t device_id, int32_t L, const float* dist, const int32_t* freq,
                   int32_t nshell, float r_cutoff, const double* r, int32_t n_r, int32_t precision,
                   double* energy) {
  if (L < 2 || nshell <= 0 || n_r <= 0 || !dist || !freq || !r || !energy)
    return fail(CVF_EINVAL, "bad arguments");
  if (precision != CVF_FP64 && precision != CVF_FP32_COMPENSATED)
    return fail(CVF_EINVAL, "unknown precision");
  HIPC(hipSetDevice(device_id));
  const int N = L * L * L;  // f_k = (count_k/2) * N
  DevBuf<float> d;
  DevBuf<int32_t> f;
  DevBuf<double> dr, de;
  HIPC(d.alloc(nshell));
  HIPC(f.alloc(nshell));
  HIPC(dr.alloc(n_r));
  HIPC(de.alloc(n_r));
  HIPC(hipMemcpy(d.p, dist, nshell * 4, hipMemcpyHostToDevice));
  HIPC(hipMemcpy(f.p, freq, nshell * 4, hipMemcpyHostToDevice));
  HIPC(hipMemcpy(dr.p, r, n_r * 8, hipMemcpyHostToDevice));
  launch_vdw_eval(nullptr, d.p, f.p, nshell, r_cutoff, N, dr.p, n_r, precision, de.p);
  HIPC(hipGetLastError());
  HIPC(hipMemcpy(energy, de.p, n_r * 8, hipMemcpyDeviceToHost));
  return CVF_OK;
}

int cvf_vdw_pair_energy(int32_t device_id, int32_t L, float r_cutoff, const double* r, int32_t n_r,
                        int32_t precision, double* energy) {
  if (L < 2 || L > kMaxL || n_r <= 0 || !r || !energy || !(r_cutoff > 0.f))
    return fail(CVF_EINVAL, "bad arguments");
  if (precision != CVF_FP64 && precision != CVF_FP32_COMPENSATED) return fail(CVF_EINVAL, "unknown precision");
  HIPC(hipSetDevice(device_id));
  const uint32_t nb = vdw_pair_blocks(L);
  DevBuf<double> dr, part;
  HIPC(dr.alloc(n_r));
  HIPC(part.alloc((size_t)nb * n_r));
  HIPC(hipMemcpy(dr.p, r, n_r * 8, hipMemcpyHostToDevice));
  launch_vdw_pairs(nullptr, L, r_cutoff, dr.p, n_r, precision, part.p);
  HIPC(hipGetLastError());
  std::vector<double> h((size_t)nb * n_r);
  HIPC(hipMemcpy(h.data(), part.p, h.size() * 8, hipMemcpyDeviceToHost));
  for (int32_t k = 0; k < n_r; ++k) {
    double t = 0;
    for (uint32_t b = 0; b < nb; ++b) t += h[(size_t)k * nb + b];
    energy[k] = 0.5 * t;  // every pair was counted from both ends
  }
  return CVF_OK;
}

}  // extern "C"

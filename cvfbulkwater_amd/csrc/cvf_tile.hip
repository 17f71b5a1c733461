// Tile kernel: the fused Metropolis launch of cvf_kernels.hip's slab kernel
// (optional eta cube sweep, then nk consecutive sigma half-sweeps on a window
// staged in LDS) on boxes that are short along all three axes.
//
// A point is folded over its quadrants: quad (X, Y, Z), X, Y < L/2, is the
// four cells (X + a L/2, Y + b L/2, Z), which share a Philox block and move
// together.  A workgroup takes the core box of Tx x Ty x Tz quads and the halo
// that its result depends on, runs every phase on the part of the window that
// later phases still need, and writes its core to the other word array.
// Halo cells are recomputed, with the site-keyed random numbers that their
// own tile uses, so the result is that of the unfused kernels.
//
// The halo is found from the launch's own schedule, walking it backwards:
// a + (-) half-sweep along an axis adds one layer on the upper (lower) side,
// and only when the outermost layer moves in it (its parity); without the
// chessboard, whose moves also write the facing cell's bond count, the layer
// beyond the other end counts likewise.  The cube sweep adds one layer on every
// side.  That is about half a layer per side for six
// half-sweeps, where a slab of T full planes recomputes whole planes: an
// L = 32 point of a 16-point handle has 2-plane slabs whose windows hold 4-5
// planes, and above L = 64 no slab's window fits LDS at all.
//
// Window coordinates are not wrapped: position w along x stands for X =
// (origin + w), and slots (a', b') of its quad hold the cells X + a' L/2, Y +
// b' L/2 with periodic X, Y.  Neighbours are then always the next quad, same
// slot; only the draws of a quad whose X (Y) lies an odd number of half
// lattices away have their words exchanged between the halves.  A window
// longer than the lattice holds copies of cells, each computed from its own
// copies of its neighbours.
//
// What bounds it: the phases, serial in a workgroup; one costs about what the
// random numbers of its quads take to issue (L = 160, 16^3 quads of 1024
// threads: 7100-7700 clocks for 2600 quads, some 600 per wave and trip on a
// SIMD that runs four of them) and the window's loads take less than one phase.
// A step at L = 160 is 75.6 us, of which the unfused kernels' fourteen launches
// took 104.

#include "cvf_device.h"
#include "cvf_kernels.h"

#include <atomic>

#include <hip/hip_ext.h>

namespace cvf {

namespace {

// Canonical coordinate of a window position, and the halves' exchange (0 or
// `bit`).
__device__ __forceinline__ uint32_t fold(int v, int period, uint32_t bit, uint32_t& sw) {
  int k = 0;
  while (v < 0) v += period, ++k;
  while (v >= period) v -= period, ++k;
  sw = (k & 1) ? bit : 0u;
  return (uint32_t)v;
}

// Words (by canonical half) of a quad or a draw in slot order, sw = the
// exchange: slot h holds half h ^ sw.
__device__ __forceinline__ void swap_by(uint32_t (&v)[4], uint32_t sw) {
  const bool s2 = sw & 2u, s1 = sw & 1u;
  uint32_t t[4];
#pragma unroll
  for (int h = 0; h < 4; ++h) t[h] = s2 ? v[h ^ 2] : v[h];
#pragma unroll
  for (int h = 0; h < 4; ++h) v[h] = s1 ? t[h ^ 1] : t[h];
}
__device__ __forceinline__ U4 draw_swap(U4 r, uint32_t sw) {
  if (__ballot(sw)) {
    uint32_t v[4] = {r.x, r.y, r.z, r.w};
    swap_by(v, sw);
    r = U4{v[0], v[1], v[2], v[3]};
  }
  return r;
}

constexpr uint32_t kFoldMask = 0x0FFFFFFFu;  // site bits of a folded coordinate; the exchange is above them

}  // namespace

// kAnyNc: the launch may hold non-chessboard points (compiled out otherwise)
template <bool kAnyNc>
__global__ __launch_bounds__(1024) void k_tile(const TileEnt* __restrict__ tab, uint32_t ntiles,
                                                const uint64_t* __restrict__ stepp, uint32_t step_off,
                                                const PointDev* __restrict__ pts, const uint32_t* __restrict__ src,
                                                uint32_t* __restrict__ dst, uint32_t k0, uint32_t nk, int with_eta) {
  extern __shared__ __align__(16) uint32_t win[];
  __shared__ uint32_t thr_s[33];
  __shared__ uint64_t thr_e[9];
  __shared__ uint64_t etab[9];
  // per axis and window position: its share of the quad's site (of its cube's
  // index), the exchange in the top bits
  __shared__ uint32_t site_t[3][kMaxTileWin], cube_t[3][kMaxTileWin];
  __shared__ uint32_t magic[kMaxTileWin + 1];  // fast-division multipliers
  // each XCD takes a contiguous range of the table: neighbouring tiles share
  // halos, and an XCD its L2
  const TileEnt e = tab[(blockIdx.x % kNumXcd) * (ntiles / kNumXcd) + blockIdx.x / kNumXcd];
  if (e.point < 0) return;
  const uint32_t tid = threadIdx.x, nt = blockDim.x;
  const PointDev& P = pts[e.point];
  if (tid < 33) thr_s[tid] = sigma_thr32(P.thr_sigma[tid]);
  if (tid < 9) {
    thr_e[tid] = P.thr_eta[tid];
    etab[tid] = eta_table_entry(tid);
  }
  if (tid <= kMaxTileWin) magic[tid] = tid <= 1 ? 0u : 0xFFFFFFFFu / tid + 1u;
  const uint64_t step = *stepp + step_off;
  const uint64_t seed = ((uint64_t)e.seed_hi << 32) | e.seed_lo;
  // the launch's half-sweeps in lanes 0 .. nk - 1 of every wavefront (arm | kept
  // parity << 3), so that no wavefront waits for another's draws
  uint32_t sch;
  {
    const U4 r = draw(seed, kStSched, 0, step, k0 + (tid & 63u));
    sch = uniform_int(r.x, 6) | (((r.y >> 31) ? 0u : 1u) << 3);
  }
  const auto entry = [&](uint32_t k) { return (uint32_t)__builtin_amdgcn_readlane((int)sch, (int)k); };
  const int L = (int)e.L, hL = L / 2;
  const int org[3] = {(int)e.x0, (int)e.y0, (int)e.z0};
  const bool nc = kAnyNc && e.nc != 0;
  // the box valid after the last half-sweep, and walking back the boxes
  // before: bit k of grow_lo, grow_hi says that half-sweep k adds a layer
  // below, above
  int lo[3] = {0, 0, 0}, hi[3] = {(int)e.tx, (int)e.ty, (int)e.tz};
  uint32_t grow_lo = 0, grow_hi = 0;
  for (int k = (int)nk - 1; k >= 0; --k) {
    const uint32_t s = entry((uint32_t)k), arm = s & 7u, q = s >> 3, down = arm & 1u;
#pragma unroll
    for (int a = 0; a < 3; ++a)
      if (a == (int)(arm >> 1)) {
        // the cell at the arm's end of the box faces one outside, if it moves;
        // without the chessboard the cell before the other end, if it moves,
        // changes the counter of the box's first one
        const bool end = ((uint32_t)(org[a] + (down ? lo[a] : hi[a] - 1)) & 1u) == q;
        const bool start = nc && ((uint32_t)(org[a] + (down ? hi[a] : lo[a] - 1)) & 1u) == q;
        if (down ? end : start) grow_lo |= 1u << k, --lo[a];
        if (down ? start : end) grow_hi |= 1u << k, ++hi[a];
      }
  }
  const bool cubes = with_eta && !nc;
  const int ext = cubes ? 1 : 0;
  int wo[3], wn[3];  // window origin relative to the core, window size
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    wo[a] = lo[a] - ext;
    wn[a] = hi[a] + ext - wo[a];
  }
  const uint32_t nx = (uint32_t)wn[0], ny = (uint32_t)wn[1], nz = (uint32_t)wn[2];
  const uint32_t sy = 4 * nx, sz = 4 * nx * ny;  // words per step along y and z
  if (tid >= 64 && tid < kTileMinBlock) {
    const uint32_t a = (tid - 64) / kMaxTileWin, i = (tid - 64) % kMaxTileWin;
    uint32_t sw = 0;
    if (a == 0 && i < nx) {
      const uint32_t c = fold(org[0] + wo[0] + (int)i, hL, 2u, sw);
      site_t[0][i] = c | sw << 28;
      cube_t[0][i] = c / 2 | sw << 28;
    } else if (a == 1 && i < ny) {
      const uint32_t c = fold(org[1] + wo[1] + (int)i, hL, 1u, sw);
      site_t[1][i] = c * (uint32_t)L | sw << 28;
      cube_t[1][i] = c / 2 * (uint32_t)hL | sw << 28;
    } else if (a == 2 && i < nz) {
      const uint32_t c = fold(org[2] + wo[2] + (int)i, L, 0u, sw);
      site_t[2][i] = c * (uint32_t)(L * L);
      cube_t[2][i] = c * (uint32_t)(hL * hL);
    }
  }
  __syncthreads();
  const auto div_of = [&](uint32_t d) { return FastDiv{d, uni(magic[d])}; };
  // the window word of item (ix, iy, iz) of the box at window position f with
  // steps m, and its site (cube index) with the exchange above it
  const auto place = [&](const uint32_t (*t)[kMaxTileWin], const uint32_t (&f)[3], uint32_t mx, uint32_t my,
                         uint32_t mz, uint32_t ix, uint32_t iy, uint32_t iz, uint32_t& w) {
    const uint32_t wx = f[0] + mx * ix, wy = f[1] + my * iy, wz = f[2] + mz * iz;
    w = 4 * wx + sy * wy + sz * wz;
    return t[0][wx] + t[1][wy] + t[2][wz];
  };
  {
    // stage the window, a quad's four words per lane (more loads in flight per
    // lane were slower: with 1 / 2 / 4 / 8 quads a lane, L = 160 ran at 75.5 /
    // 77.9 / 85.7 / 98.7 us per step)
    const uint32_t n = nx * ny * nz, oy = (uint32_t)hL * (uint32_t)L, ox = (uint32_t)hL;
    const FastDiv dx = div_of(nx), dy = div_of(ny);
    const uint32_t* S = src + e.woff;
    for (uint32_t i = tid; i < n; i += nt) {
      const uint32_t r = fdiv(i, dx), wx = i - r * nx, wz = fdiv(r, dy), wy = r - wz * ny;
      const uint32_t c = site_t[0][wx] + site_t[1][wy] + site_t[2][wz], sw = c >> 28;
      const uint32_t* s = S + (c & kFoldMask);
      uint32_t v[4] = {s[0], s[oy], s[ox], s[ox + oy]};
      if (__ballot(sw)) swap_by(v, sw);
      quad_store(win, 4 * i, v);
    }
  }
  __syncthreads();
  if (cubes) {
    for (int fam = 0; fam < 2; ++fam) {
      // origins of the family's parity whose cubes hold a cell of the box
      uint32_t f[3], cnt[3];
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const int l = lo[a] - (((org[a] + lo[a]) & 1) != fam);
        f[a] = (uint32_t)(l - wo[a]);
        cnt[a] = (uint32_t)(hi[a] - l + 1) / 2;
      }
      const uint32_t n = cnt[0] * cnt[1] * cnt[2];
      const FastDiv dx = div_of(cnt[0]), dy = div_of(cnt[1]);
      const auto item = [&](uint32_t i, uint32_t& w0) {
        const uint32_t r = fdiv(i, dx), iz = fdiv(r, dy);
        return place(cube_t, f, 2, 2, 2, i - r * cnt[0], r - iz * cnt[1], iz, w0);
      };
      const PhiloxFixed pf = phase_draws(seed, kStEta, step, 0);
      if (4 * n <= nt) {
        // few items: one cube per lane
        if (tid < 4 * n) {
          uint32_t w0, w[8];
          const uint32_t h = tid & 3u, c = item(tid >> 2, w0);
          const U4 r = draw_site(c & kFoldMask, pf);
          w0 += h;
#pragma unroll
          for (int b = 0; b < 8; ++b) w[b] = win[w0 + ((b & 1) ? 4 : 0) + ((b & 2) ? sy : 0) + ((b & 4) ? sz : 0)];
          eta_cube_move(w, thr_e, etab, pick4(r, h ^ (c >> 28)), [&](int b, uint32_t v) {
            win[w0 + ((b & 1) ? 4 : 0) + ((b & 2) ? sy : 0) + ((b & 4) ? sz : 0)] = v;
          });
        }
      } else {
        for (uint32_t i = tid; i < n; i += nt) {
          uint32_t w0, v[8][4];
          const uint32_t c = item(i, w0);
#pragma unroll
          for (int b = 0; b < 8; ++b)
            quad_load(win, w0 + ((b & 1) ? 4 : 0) + ((b & 2) ? sy : 0) + ((b & 4) ? sz : 0), v[b]);
          const U4 r = draw_swap(draw_site(c & kFoldMask, pf), c >> 28);
#pragma unroll
          for (int h = 0; h < 4; ++h) {
            const uint32_t rw = h == 0 ? r.x : h == 1 ? r.y : h == 2 ? r.z : r.w;
            uint32_t w[8];
#pragma unroll
            for (int b = 0; b < 8; ++b) w[b] = v[b][h];
            eta_cube_move(w, thr_e, etab, rw, [&](int b, uint32_t nv) { v[b][h] = nv; });
          }
#pragma unroll
          for (int b = 0; b < 8; ++b)
            quad_store(win, w0 + ((b & 1) ? 4 : 0) + ((b & 2) ? sy : 0) + ((b & 4) ? sz : 0), v[b]);
        }
      }
      __syncthreads();
    }
  }
  for (uint32_t k = 0; k < nk; ++k) {
    const uint32_t sk = entry(k), q = sk >> 3;
    const int arm = (int)(sk & 7u), ax = arm >> 1;
    uint32_t f[3], cnt[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      int first = lo[a], end = hi[a];
      if (a == ax) {
        // without the chessboard every pair within the box before, else the
        // cells of the box after
        if (nc) {
          if (arm & 1)
            ++first;
          else
            --end;
        }
        lo[a] += (int)((grow_lo >> k) & 1u);
        hi[a] -= (int)((grow_hi >> k) & 1u);
        if (!nc) first = lo[a], end = hi[a];
        // the layers of the kept parity
        first += ((uint32_t)(org[a] + first) & 1u) != q;
      }
      f[a] = (uint32_t)(first - wo[a]);
      cnt[a] = (uint32_t)(a == ax ? (end - first + 1) / 2 : end - first);
    }
    const uint32_t n = cnt[0] * cnt[1] * cnt[2];
    const uint32_t mx = ax == 0 ? 2u : 1u, my = ax == 1 ? 2u : 1u, mz = ax == 2 ? 2u : 1u;
    const uint32_t st = ax == 0 ? 4u : ax == 1 ? sy : sz, dn = (arm & 1) ? 0u - st : st;
    const FastDiv dx = div_of(cnt[0]), dy = div_of(cnt[1]);
    const auto item = [&](uint32_t i, uint32_t& w0) {
      const uint32_t r = fdiv(i, dx), iz = fdiv(r, dy);
      return place(site_t, f, mx, my, mz, i - r * cnt[0], r - iz * cnt[1], iz, w0);
    };
    const PhiloxFixed pf = phase_draws(seed, kStSigma, step, k0 + k);
    if (4 * n <= nt) {
      // few items: one cell per lane
      if (tid < 4 * n) {
        uint32_t w0;
        const uint32_t h = tid & 3u, c = item(tid >> 2, w0);
        const uint32_t w = win[w0 + h], wf = win[w0 + dn + h];
        const U4 r = draw_site(c & kFoldMask, pf);
        const uint32_t rw = pick4(r, h ^ (c >> 28));
        if (nc) {
          uint32_t v = w, vf = wf;
          sigma_cell_nc(v, vf, thr_s, arm, rw);
          win[w0 + h] = v;
          win[w0 + dn + h] = vf;
        } else {
          win[w0 + h] = sigma_cell(w, wf, thr_s, arm, rw);
        }
      }
    } else {
      for (uint32_t i = tid; i < n; i += nt) {
        uint32_t w0, w[4], wf[4];
        const uint32_t c = item(i, w0);
        quad_load(win, w0, w);
        quad_load(win, w0 + dn, wf);
        const U4 r = draw_swap(draw_site(c & kFoldMask, pf), c >> 28);
        if (nc) {
          sigma_cell_nc(w[0], wf[0], thr_s, arm, r.x);
          sigma_cell_nc(w[1], wf[1], thr_s, arm, r.y);
          sigma_cell_nc(w[2], wf[2], thr_s, arm, r.z);
          sigma_cell_nc(w[3], wf[3], thr_s, arm, r.w);
          quad_store(win, w0 + dn, wf);
        } else {
          sigma_quad_regs(w, wf, thr_s, arm, r);
        }
        quad_store(win, w0, w);
      }
    }
    __syncthreads();
  }
  {
    // the core to the other array (its positions are within the half lattice,
    // so no halves are exchanged)
    const uint32_t tx = e.tx, ty = e.ty, n = tx * ty * e.tz, oy = (uint32_t)hL * (uint32_t)L, ox = (uint32_t)hL;
    const FastDiv dx = div_of(tx), dy = div_of(ty);
    uint32_t* D = dst + e.woff + e.x0 + (uint32_t)L * (e.y0 + (uint32_t)L * e.z0);
    const uint32_t c0 = 4u * ((uint32_t)(-wo[0]) + nx * ((uint32_t)(-wo[1]) + ny * (uint32_t)(-wo[2])));
    for (uint32_t i = tid; i < n; i += nt) {
      const uint32_t r = fdiv(i, dx), ix = i - r * tx, iz = fdiv(r, dy), iy = r - iz * ty;
      uint32_t v[4];
      quad_load(win, c0 + 4 * (ix + nx * (iy + ny * iz)), v);
      uint32_t* d = D + ix + (uint32_t)L * (iy + (uint32_t)L * iz);
      d[0] = v[0];
      d[oy] = v[1];
      d[ox] = v[2];
      d[ox + oy] = v[3];
    }
  }
}

uint32_t tile_window_quads(uint32_t tx, uint32_t ty, uint32_t tz, uint32_t nk, bool nc) {
  // every half-sweep can add a layer to one axis (two without the chessboard,
  // which has no cubes): the largest window over how they may fall on the
  // three
  const uint32_t e = nc ? 0u : 2u, g = nc ? 2u : 1u;
  uint32_t most = 0;
  for (uint32_t a = 0; a <= nk; ++a)
    for (uint32_t b = 0; a + b <= nk; ++b)
      most = std::max(most, (tx + e + g * a) * (ty + e + g * b) * (tz + e + g * (nk - a - b)));
  return most;
}

namespace {
template <bool kAnyNc>
void launch_tile_t(hipStream_t st, const TileEnt* tab, uint32_t ntiles, uint32_t block, const uint64_t* stepp,
                   uint32_t step_off, const PointDev* pts, const uint32_t* src, uint32_t* dst, uint32_t k0,
                   uint32_t nk, int with_eta, uint32_t lds_bytes) {
  // the dynamic-LDS limit is a per-device function attribute
  static std::atomic<uint64_t> attr_set{0};
  int dev = 0;
  (void)hipGetDevice(&dev);
  const uint64_t bit = 1ull << (dev & 63);
  if (!(attr_set.load(std::memory_order_acquire) & bit)) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_tile<kAnyNc>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)tile_lds_limit());
    attr_set.fetch_or(bit, std::memory_order_acq_rel);
  }
  hipEvent_t t0, t1;
  get_launch_timing(&t0, &t1);
  if (t0)
    hipExtLaunchKernelGGL(k_tile<kAnyNc>, dim3(ntiles), dim3(block), lds_bytes, st, t0, t1, 0, tab, ntiles, stepp,
                          step_off, pts, src, dst, k0, nk, with_eta);
  else
    hipLaunchKernelGGL(k_tile<kAnyNc>, dim3(ntiles), dim3(block), lds_bytes, st, tab, ntiles, stepp, step_off, pts,
                       src, dst, k0, nk, with_eta);
}
}  // namespace

void launch_tile(hipStream_t st, const TileEnt* tab, uint32_t ntiles, uint32_t block, const uint64_t* stepp,
                 uint32_t step_off, const PointDev* pts, const uint32_t* src, uint32_t* dst, uint32_t k0, uint32_t nk,
                 int with_eta, uint32_t lds_bytes, bool any_nc) {
  (any_nc ? launch_tile_t<true> : launch_tile_t<false>)(st, tab, ntiles, block, stepp, step_off, pts, src, dst, k0, nk,
                                                        with_eta, lds_bytes);
}

}  // namespace cvf

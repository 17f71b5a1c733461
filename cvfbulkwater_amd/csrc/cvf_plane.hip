// Resident Metropolis kernel for one-plane slabs: one workgroup per plane of a
// point, which holds the plane and ghost copies of its two neighbours in LDS
// for a whole sequence of MC steps of the reference schedule.  Window layout,
// rings, tags, versions and the rules for what is published when are those of
// cvf_resident.hip; this kernel is for the small handles, whose phases are a
// few waves each and nothing but latency.
//
// A wave that is alone on its SIMD issues an instruction about every eight
// clocks, so a phase lasts as long as the instructions on one lane's way: the
// general kernel's took 1830 clocks for the 72 cells of a plane of L = 12, with
// its slab's fields, the item's place and its Philox block all on that way.
// Here
//   * the moves of a batch of half-sweeps (all twelve, where LDS holds them)
//     are made ahead by all the workgroup's lanes at once, a quad of one
//     half-sweep each: a record of its window word, its facing word and its
//     four random words.  A phase only reads its record, the two cells and
//     the threshold;
//   * the schedule is drawn for four steps at a time, in the lanes of every
//     wave, so that no wave waits for another's;
//   * z half-sweeps in which the plane rests are skipped, barrier included;
//   * the step-end plane is published from the registers of the step's last
//     moving phase, the cells which rest in it alongside, and the next step's
//     schedule, first records and cube draws are made while the neighbours'
//     planes are on the way.
// L = 12 / 16 / 24 / 32 / 48: 7.2 / 7.4 / 9.4 / 10.3 / 16.5 us per step of a long run, the
// general kernel 13.7 / 13.6 / 15.8 / 15.8 / 22.3; of 18050 clocks at L = 12, 740 a phase
// in the plane, 3500 from a step's start to its neighbours' planes, 2800 the cubes.
// The moves of all twelve half-sweeps are made at once up to L = 32 (512 threads),
// of six from L = 48 on: as a workgroup's share of LDS holds them.
#include "cvf_device.h"
#include "cvf_kernels.h"
#include "cvf_ring.h"

#include <atomic>

#include <hip/hip_ext.h>

namespace cvf {

namespace {

// a where the mask m is set, else b (masks are all ones or zero)
__device__ __forceinline__ uint32_t pick(uint32_t m, uint32_t a, uint32_t b) {
  uint32_t r;
  asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "v"(m), "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ uint32_t ones(bool b) { return b ? ~0u : 0u; }

// x of lane `from` (a value of each lane's own); y pushed to lane `to`
__device__ __forceinline__ uint32_t lane_read(uint32_t x, uint32_t from) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(4 * from), (int)x);
}
__device__ __forceinline__ uint32_t lane_push(uint32_t y, uint32_t to) {
  return (uint32_t)__builtin_amdgcn_ds_permute((int)(4 * to), (int)y);
}

}  // namespace

// per: half-sweeps per batch of records (a divisor of 12); dynamic LDS: three
// planes of L^2 words, then the batch's records (plane_lds_bytes)
__global__ __launch_bounds__(1024) void k_plane(const RGroupEnt* __restrict__ grp, const RSlab* __restrict__ slabs,
                                                 const PointDev* __restrict__ pts, uint32_t* __restrict__ words,
                                                 uint32_t* __restrict__ kept, uint32_t* __restrict__ rings,
                                                 uint64_t* __restrict__ ver,
                                                 const uint64_t* __restrict__ stepp, uint64_t step_off,
                                                 uint32_t nsteps, uint64_t* __restrict__ step_out,
                                                 uint32_t* __restrict__ status, uint32_t per) {
  extern __shared__ __align__(16) uint32_t lds[];  // the plane below, the plane, the plane above; records
  __shared__ uint32_t thr_s[33];
  __shared__ uint64_t thr_e[9], etab[9];
  __shared__ uint32_t abort_s;
  const uint32_t tid = threadIdx.x, nt = blockDim.x, lane = tid & 63u, h = tid & 3u;
  const uint32_t me = grp[blockIdx.x].first, flag = status[0];
  const RSlab S = slabs[me];
  const uint32_t L = S.L, hL = L / 2, qL = L / 4, LL = L * L, Q4 = LL / 4, Q8 = LL / 8, z0 = S.z0, par = z0 & 1u;
  const uint64_t seed = ((uint64_t)S.seed_hi << 32) | S.seed_lo;
  const FastDiv dH{hL, S.mH}, dQ{qL, S.mQ}, dP8{Q8, S.mP8};
  uint4* rec_r = reinterpret_cast<uint4*>(lds + 3 * LL);  // a record's random words ...
  uint32_t* rec_a = lds + 3 * LL + 4 * 2 * per * Q8;      // ... and window words: the quad's | the facing quad's << 16,
                                                          // whose low bits are the exchange of its halves
  if (tid < 33) thr_s[tid] = sigma_thr32(pts[S.point].thr_sigma[tid]);
  if (tid < 9) {
    thr_e[tid] = pts[S.point].thr_eta[tid];
    etab[tid] = eta_table_entry(tid);
  }
  if (tid == 0) abort_s = 0;
  const uint64_t step0 = (stepp ? *stepp : 0) + step_off;
  for (uint32_t i = tid; i < 3 * Q4; i += nt) {
    const uint32_t p = fdiv(i, FastDiv{Q4, S.mP4}), r = i - p * Q4, y = fdiv(r, dH), x = r - y * hL;
    const uint32_t zp = z0 + L - 1 + p, z = zp >= 2 * L ? zp - 2 * L : zp >= L ? zp - L : zp;
    const uint32_t* s = words + S.woff + z * LL + x + L * y;
    reinterpret_cast<uint4*>(lds)[i] = make_uint4(s[0], s[hL * L], s[hL], s[hL * L + hL]);
  }
  __syncthreads();
  const auto store_plane = [&](uint32_t* to) {
    for (uint32_t i = tid; i < Q4; i += nt) {
      const uint32_t y = fdiv(i, dH), x = i - y * hL;
      const uint4 v = reinterpret_cast<const uint4*>(lds + LL)[i];
      uint32_t* d = to + S.woff + z0 * LL + x + L * y;
      d[0] = v.x;
      d[hL * L] = v.y;
      d[hL] = v.z;
      d[hL * L + hL] = v.w;
    }
  };
  // (not as it is staged: the next loads would wait for these stores)
  if (kept) {
    // (the same in all threads: no workgroup of this launch was waited for in
    // vain before its mark was there)
    if (!keeps_start(flag, status, step0)) return;
    store_plane(kept);
  }
  leave_mark(kept, flag, status, step0);
  if (step_out && blockIdx.x == 0 && tid == 0) *step_out = step0 + nsteps;
  bool aborted = false;
  // lane 16 j + k: half-sweep k of the j-th of four steps, k | arm << 4 |
  // parity << 7 | rd << 8 | wr << 12 (rd, wr: ring slots, as in
  // cvf_resident.hip); moves: those that move this plane
  uint32_t sch = 0;
  uint64_t moves = 0, zmoves = 0;
  for (uint32_t si = 0; si < nsteps; ++si) {
    const uint64_t step = step0 + si;
    const uint32_t half = (uint32_t)(step & 1u) * kRingHalf, tag = end_tag(step), seg = 16 * (si & 3u);
    const uint64_t tw = (uint64_t)tag << 32;
    // the neighbours' planes at the end of the last step: first loads out,
    // checked below
    const uint32_t prev = (uint32_t)((step - 1) & 1u) * kRingHalf + kEndSlot;
    const uint64_t* hi = reinterpret_cast<const uint64_t*>(rings + S.ring_hi + prev * LL);
    const uint64_t* lo = reinterpret_cast<const uint64_t*>(rings + S.ring_lo + prev * LL);
    if (seg == 0) {
      const uint32_t k = lane & 15u;
      const U4 r = draw(seed, kStSched, 0, step + (lane >> 4), k);
      const uint32_t arm = uniform_int(r.x, 6), q = (r.y >> 31) ? 0u : 1u;
      const bool in = k < 12;
      const uint64_t up = __ballot(in && arm == 4 && q == par), dn = __ballot(in && arm == 5 && q == par);
      const uint64_t ab = __ballot(in && arm == 5 && q != par), bl = __ballot(in && arm == 4 && q != par);
      zmoves = up | dn;
      moves = __ballot(in && arm < 4) | zmoves;
      const uint64_t mine = 0xFFFFull << (lane & 48u), bit = 1ull << lane;
      const uint64_t before = mine & (bit - 1), after = mine & ~(bit | (bit - 1));
      uint32_t rd = 0, wr = 0;
      if (in && arm >= 4 && q == par) {
        const uint64_t other = arm == 4 ? ab : bl, self = arm == 4 ? up : dn;
        if (other & before) rd = 64 - (uint32_t)__builtin_clzll(other & before) - (lane & 48u);
        const uint64_t ra = other & after, ua = self & after;
        if (ra && (!ua || __builtin_ctzll(ra) < __builtin_ctzll(ua))) wr = 1;
      }
      sch = k | (arm << 4) | (q << 7) | (rd << 8) | (wr << 12);
    }
    const uint32_t mask = (uint32_t)(moves >> seg) & 0xFFFu, zmask = (uint32_t)(zmoves >> seg) & 0xFFFu;
    const auto entry = [&](uint32_t k) { return (uint32_t)__builtin_amdgcn_readlane((int)sch, (int)(seg + k)); };
    // The records of the moving half-sweeps from first to first + per - 1, in
    // units of L^2/8 quads: one for an in-plane half-sweep, two for z.
    const auto make_records = [&](uint32_t first) {
      const uint32_t m = mask >> first & ((1u << per) - 1), zm = zmask >> first & ((1u << per) - 1);
      // lane r: the entry of unit r, second halves marked
      const uint32_t k = lane - first;
      const uint32_t e = lane_read(sch, seg + lane);
      const bool moving = k < per && (m >> k & 1u), zk = moving && (zm >> k & 1u);
      const uint32_t below = k < per ? (1u << k) - 1 : 0u;
      const uint32_t at = (uint32_t)(popc32(m & below) + popc32(zm & below));
      const uint32_t u1 = lane_push(e, moving ? at : 63u), u2 = lane_push(e | 1u << 31, zk ? at + 1 : 63u);
      const uint32_t units = (uint32_t)(popc32(m) + popc32(zm));
      // (a lane that nothing was pushed to reads zero)
      const uint32_t unit = lane < 63 ? u1 | u2 : 0u;
      for (uint32_t i = tid; __ballot(i < units * Q8); i += nt) {
        const uint32_t r = min(fdiv(i, dP8), 62u), u = i - r * Q8, v = lane_read(unit, r);
        const uint32_t arm = v >> 4 & 7u, q = v >> 7 & 1u;
        const uint32_t alongx = ones(arm < 2), alongy = ones((arm & 6u) == 2), z = ones(arm >= 4);
        const uint32_t w = u + (v >> 31 ? Q8 : 0u);  // (z: the quad)
        const uint32_t yq = fdiv(u, dQ), yh = fdiv(w, dH);
        const uint32_t x = pick(alongx, 2 * (u - yq * qL) + q, w - yh * hL);
        const uint32_t y = pick(alongx, yq, pick(alongy, 2 * yh + q, yh));
        const uint32_t a = LL + 4 * (x + hL * y);
        const uint32_t st = pick(alongx, 4u, pick(alongy, 4 * hL, LL)), dn = ones(arm & 1u);
        const uint32_t wrap = ~z & ones(pick(alongx, x, y) == (dn ? 0u : hL - 1));
        // the facing quad: one step up or down, across the edge hL - 1 steps
        // back with the halves along the axis exchanged
        const uint32_t d = pick(wrap, (hL - 1) * st, st), neg = wrap ^ dn;
        const uint32_t f = a + ((d ^ neg) - neg) + (wrap & pick(alongx, 2u, 1u));
        const U4 rnd = draw(seed, kStSigma, x + L * y + LL * z0, step, v & 15u);
        if (i < units * Q8) {
          rec_a[i] = a | f << 16;
          rec_r[i] = make_uint4(rnd.x, rnd.y, rnd.z, rnd.w);
        }
      }
    };
    make_records(0);
    uint64_t gv[4];
    const uint64_t* gs[4];
    if (si > 0) {
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        const uint32_t i = min(tid + u * nt, 2 * LL - 1);
        gs[u] = i < LL ? hi + i : lo + (i - LL);
        gv[u] = ring_load64(gs[u]);
      }
    }
    // cubes: cube c of item it, families 0 and 1, one with the plane below
    // (origin there) and one with the plane above
    const PhiloxFixed pfe = phase_draws(seed, kStEta, step, 0);
    const uint32_t zb = z0 ? z0 - 1 : L - 1;
    const auto cube_word = [&](uint32_t p, uint32_t fam) {
      const uint32_t it = p >> 2, jj = fdiv(it, dQ), ii = it - jj * qL;
      const U4 r = draw_site(ii + hL * jj + (LL / 4) * (fam == par ? z0 : zb), pfe);
      const uint32_t c1 = ones(p & 1u), c2 = ones(p & 2u);
      return pick(c2, pick(c1, r.w, r.z), pick(c1, r.y, r.x));
    };
    const auto cube = [&](uint32_t p, uint32_t fam, uint32_t rw) {
      const uint32_t it = p >> 2, jj = fdiv(it, dQ), ii = it - jj * qL;
      const uint32_t B = fam == par ? LL : 0u;
      eta_cube_one_q(lds, B, B + LL, thr_e, etab, hL, 2 * ii + fam, 2 * jj + fam, p & 3u, rw);
    };
    const uint32_t rc0 = cube_word(tid, 0), rc1 = cube_word(tid, 1);
    if (si > 0) {
      const uint32_t ptag = end_tag(step - 1);
      bool ok = wait_tags(gs, ptag, gv, status);
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        const uint32_t i = tid + u * nt;
        if (i < 2 * LL) lds[i < LL ? 2 * LL + i : i - LL] = (uint32_t)gv[u];
      }
      for (uint32_t i0 = tid + 4 * nt; i0 < 2 * LL; i0 += 4 * nt) {
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
          const uint32_t i = min(i0 + u * nt, 2 * LL - 1);
          gs[u] = i < LL ? hi + i : lo + (i - LL);
          gv[u] = ring_load64(gs[u]);
        }
        ok = wait_tags(gs, ptag, gv, status) && ok;
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
          const uint32_t i = i0 + u * nt;
          if (i < 2 * LL) lds[i < LL ? 2 * LL + i : i - LL] = (uint32_t)gv[u];
        }
      }
      if (__ballot(!ok)) abort_s = 1;
    }
    __syncthreads();
    // (read by every wave before the next barrier, and not written before it:
    // the same in all)
    if (abort_s) {
      aborted = true;
      break;
    }
    // A lane's first move of the phase whose records start at b: window words,
    // proposal and acceptance word.  Read a phase ahead.
    uint32_t cw, fw, sp, ra;
    const uint32_t tq = min(tid >> 2, 2 * Q8 - 1);  // (a phase has room for 2 Q8 records)
    const auto fetch = [&](uint32_t b) {
      const uint32_t a = rec_a[b + tq], rw = reinterpret_cast<const uint32_t*>(rec_r + b + tq)[h];
      cw = (a & 0xFFFFu) + h;
      fw = (a >> 16) ^ h;
      split_word(rw, 6, sp, ra);
    };
    // ---------------------------------------------------------- cube sweep
    for (uint32_t p = tid; p < LL / 4; p += nt) cube(p, 0, p == tid ? rc0 : cube_word(p, 0));
    __syncthreads();
    fetch(0);
    for (uint32_t p = tid; p < LL / 4; p += nt) cube(p, 1, p == tid ? rc1 : cube_word(p, 1));
    __syncthreads();
    // --------------------------------------------------------- half-sweeps
    uint64_t* end = reinterpret_cast<uint64_t*>(rings + S.ring + (half + kEndSlot) * LL);
    const bool last_step = si + 1 == nsteps;
    for (uint32_t first = 0; first < 12; first += per) {
      if (first) {
        // (the batch before is done with its records: its last barrier)
        make_records(first);
        __syncthreads();
        fetch(0);
      }
      uint32_t base = 0;  // the phase's first record
      for (uint32_t left = mask >> first & ((1u << per) - 1); left; left &= left - 1) {
        const uint32_t k = first + (uint32_t)__builtin_ctz(left), e = entry(k);
        const uint32_t arm = e >> 4 & 7u;
        const bool z = arm >= 4, last = (mask >> k) == 1;
        const uint32_t items = z ? LL : LL / 2, at = base;
        base += z ? 2 * Q8 : Q8;
        const auto moved = [&](uint32_t w, uint32_t n, uint32_t to, uint32_t acc) {
          const uint32_t sa = sigma_of(w, (int)arm);
          const uint32_t t = thr_s[sigma_thr_index(w, n, (int)arm, sa, to)];
          return to != sa && acc < t ? (w & ~(7u << (3 * arm))) | (to << (3 * arm)) : w;
        };
        if (!z && !last) {
          const uint32_t c = cw, to = sp, acc = ra;
          uint32_t w = 0, n = 0;
          if (tid < items) w = lds[c], n = lds[fw];
          fetch(left & (left - 1) ? base : 0u);
          if (tid < items) lds[c] = moved(w, n, to, acc);
          for (uint32_t p = tid + nt; p < items; p += nt) {
            const uint32_t a = rec_a[at + (p >> 2)], rw = reinterpret_cast<const uint32_t*>(rec_r + at)[p];
            const uint32_t o = (a & 0xFFFFu) + h;
            lds[o] = sigma_cell(lds[o], lds[(a >> 16) ^ h], thr_s, (int)arm, rw);
          }
          __syncthreads();
          continue;
        }
        // the neighbour's plane as of its half-sweep rd - 1 (0: the ghost)
        const uint32_t rd = e >> 8 & 15u;
        const uint64_t* RG =
            z && rd ? reinterpret_cast<const uint64_t*>(
                          arm == 4 ? rings + S.ring_hi + (half + ring_slot(rd - 1)) * LL
                                   : rings + S.ring_lo + (2 * kRingHalf + half + ring_slot(rd - 1)) * LL)
                    : nullptr;
        uint64_t* RW = z && (e >> 12 & 1u)
                           ? reinterpret_cast<uint64_t*>(
                                 rings + S.ring + ((arm == 4 ? 2 * kRingHalf : 0u) + half + ring_slot(k)) * LL)
                           : nullptr;
        const bool ab = abort_s;
        bool ok = true;
        for (uint32_t p = tid; p < items; p += nt) {
          if (p != tid) {
            const uint32_t a = rec_a[at + (p >> 2)], rw = reinterpret_cast<const uint32_t*>(rec_r + at)[p];
            cw = (a & 0xFFFFu) + h;
            fw = (a >> 16) ^ h;
            split_word(rw, 6, sp, ra);
          }
          const uint32_t o = cw - LL, w = lds[cw];
          uint32_t n;
          if (RG) {
            const uint64_t* const src[1] = {RG + o};
            uint64_t v[1] = {ring_load64(src[0])};
            ok = wait_tags(src, tag, v, status) && ok;
            n = (uint32_t)v[0];
          } else {
            n = lds[fw];
          }
          const uint32_t nw = moved(w, n, sp, ra);
          lds[cw] = nw;
          if (ab || !ok) continue;
          if (RW) ring_store64(RW + o, tw | nw);
          if (last) {
            // the step's last moving phase: its cells, and in the plane
            // those of the other parity, are final
            ring_store64(end + o, tw | nw);
            if (!z) {
              const uint32_t d = arm < 2 ? 4u : 4 * hL, other = cw + ((e >> 7 & 1u) ? 0u - d : d);
              ring_store64(end + (other - LL), tw | lds[other]);
            }
          }
        }
        if (RG && __ballot(!ok)) abort_s = 1;
        fetch(left & (left - 1) ? base : 0u);
        __syncthreads();
      }
    }
    if (!mask)  // no half-sweep moves the plane
      for (uint32_t i = tid; i < LL; i += nt) ring_store64(end + i, tw | lds[LL + i]);
    if (last_step) {
      ring_stores_done();
      __syncthreads();
      if (tid == 0 && !abort_s) {
        __hip_atomic_store(ver + 2 * me, end_version(step), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(ver + 2 * me + 1, end_version(step), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  // the neighbours have read their windows long before they published their
  // last step's version: only then this plane is overwritten in `words`
  if (!aborted && nsteps > 0 && tid == 0) {
    const uint64_t want = end_version(step0 + nsteps - 1);
    if (!wait_version(ver + 2 * S.above, want, status) || !wait_version(ver + 2 * S.below + 1, want, status))
      abort_s = 1;
  }
  __syncthreads();
  if (abort_s) return;  // after the last barrier
  store_plane(words);
}

uint32_t plane_lds_bytes(uint32_t L, uint32_t per) { return 4 * 3 * L * L + 20 * 2 * per * (L * L / 8); }

namespace {
void set_plane_attribute() {
  // the dynamic-LDS limit is a per-device function attribute
  static std::atomic<uint64_t> attr_set{0};
  int dev = 0;
  (void)hipGetDevice(&dev);
  const uint64_t bit = 1ull << (dev & 63);
  if (!(attr_set.load(std::memory_order_acquire) & bit)) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_plane), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)resident_lds_limit());
    attr_set.fetch_or(bit, std::memory_order_acq_rel);
  }
}
}  // namespace

hipError_t plane_occupancy(int* per_cu, uint32_t block, uint32_t lds_bytes) {
  set_plane_attribute();
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, k_plane, (int)block, (size_t)lds_bytes);
}

void launch_plane(hipStream_t st, const RGroupEnt* grp, uint32_t ngroups, uint32_t block, uint32_t lds_bytes,
                  const RSlab* slabs, const PointDev* pts, uint32_t* words, uint32_t* kept, uint32_t* rings,
                  uint64_t* ver, const uint64_t* stepp, uint64_t step_off, uint32_t nsteps, uint64_t* step_out, uint32_t* status,
                  uint32_t per) {
  set_plane_attribute();
  hipEvent_t t0, t1;
  get_launch_timing(&t0, &t1);
  if (t0)
    hipExtLaunchKernelGGL(k_plane, dim3(ngroups), dim3(block), lds_bytes, st, t0, t1, 0, grp, slabs, pts, words, kept,
                          rings, ver, stepp, step_off, nsteps, step_out, status, per);
  else
    hipLaunchKernelGGL(k_plane, dim3(ngroups), dim3(block), lds_bytes, st, grp, slabs, pts, words, kept, rings, ver,
                       stepp, step_off, nsteps, step_out, status, per);
}

}  // namespace cvf

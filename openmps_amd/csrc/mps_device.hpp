// Device-side helpers shared by the particle, PPE and CG kernels.
//
// All FP64 arithmetic here must round exactly as the reference's host code:
// the library is compiled with -ffp-contract=off, and every expression keeps
// the association order of the reference source it cites.
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

namespace mps {

// Particle::W, Particle.hpp:71-75
__device__ __forceinline__ double weight(double r, double re) {
  return ((0 < r) && (r < re)) ? (re / r - 1) : 0;
}

// Slot k of particle i in the neighbour layout: per slice of 64 particles,
// groups of four consecutive slots of one particle (16 bytes), the 64
// particles' groups side by side; kstride (slots per particle) is a
// multiple of 4.  The search stores and the walks load a whole group at once.
__host__ __device__ __forceinline__ size_t nbr_slot(uint32_t i, uint32_t k, uint32_t kstride) {
  return ((static_cast<size_t>(i >> 6) * (kstride >> 2) + (k >> 2)) * 64 + (i & 63u)) * 4 + (k & 3u);
}

// SPP ghost particle, Computer.hpp:657-693.  (sx, sz) is sum W(|dx|) dx over
// the r_e-filtered neighbours; the ghost exists when nWithoutSpp_i < n0 and
// the centroid offset exceeds DBL_EPSILON.
__device__ __forceinline__ bool ghost_pos(double xi, double zi, double sx, double sz, double nws_i,
                                          double n0, double re, double& gx, double& gz) {
  sx /= n0;
  sz /= n0;
  if (!(nws_i < n0)) return false;
  const double rg = sqrt(sx * sx + sz * sz);
  if (!(rg > DBL_EPSILON)) return false;
  const double wspp = n0 - nws_i;
  const double rspp = re / (wspp + 1);
  gx = xi - (rspp / rg) * sx;
  gz = zi - (rspp / rg) * sz;
  return true;
}

// Walks particle i's m-entry neighbour list in list order, four neighbours (one
// group of slots) at a time: use(j, f, in) gets the group's ids, load(j) of each
// (the gathered fields, as a T) and which of them are in the list (the last
// group's rest holds particle i itself).
//
// `use` computes all four neighbours' terms first, without branches, and then
// adds those that count in list order.  A term is a chain of a dozen to thirty
// dependent FP64 instructions (square root, division): behind a branch per
// neighbour, which some lane of a wavefront nearly always takes, the four
// chains run one after the other; without it they overlap.  The next group's
// ids and fields are loaded before the current group's arithmetic.  (Density
// and acceleration pass, bound by FP64 issue: 2k particles 23 -> 16 us, 131k 46
// -> 37, 1.05M 215 -> 180.)
//
// What is loaded ahead at a list's end is thrown away: the first group's again, or
// TIGHT, the particle's own, which costs nothing where gathers miss the caches (a
// shuffled order) and a few registers.
template <class T, bool TIGHT = false, class Load, class Use>
__device__ __forceinline__ void walk_list(uint32_t i, uint32_t m, const uint32_t* __restrict__ ids, uint32_t kmax,
                                          Load load, Use use) {
  if (m == 0) return;
  auto group = [&](uint32_t q, uint32_t j[4]) {
    const uint4 g = *reinterpret_cast<const uint4*>(ids + nbr_slot(i, !TIGHT || q < m ? q : 0u, kmax));
    j[0] = (!TIGHT || q < m) ? g.x : i;
    j[1] = (q + 1 < m) ? g.y : i;
    j[2] = (q + 2 < m) ? g.z : i;
    j[3] = (q + 3 < m) ? g.w : i;
  };
  uint32_t j[4], jn[4];
  T f[4];
  group(0, j);
  group(TIGHT || m > 4 ? 4u : 0u, jn);
#pragma unroll
  for (int v = 0; v < 4; v++) f[v] = load(j[v]);
  for (uint32_t q = 0; q < m; q += 4) {
    T fn[4];
    uint32_t j2[4];
#pragma unroll
    for (int v = 0; v < 4; v++) fn[v] = load(jn[v]);
    group(TIGHT || q + 8 < m ? q + 8 : 0u, j2);
    bool in[4];
#pragma unroll
    for (int v = 0; v < 4; v++) in[v] = q + v < m;
    use(j, f, in);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      j[v] = jn[v];
      jn[v] = j2[v];
      f[v] = fn[v];
    }
  }
}

// walk_list without loads ahead: a third fewer registers, and none thrown away at the
// list's end; the wavefronts that a compute unit then holds hide the loads once there
// are enough of them (from about 100k particles on; k_density).
template <class T, class Load, class Use>
__device__ __forceinline__ void walk_plain(uint32_t i, uint32_t m, const uint32_t* __restrict__ ids, uint32_t kmax,
                                           Load load, Use use) {
  for (uint32_t q = 0; q < m; q += 4) {
    const uint4 g = *reinterpret_cast<const uint4*>(ids + nbr_slot(i, q, kmax));
    const uint32_t j[4] = {g.x, (q + 1 < m) ? g.y : i, (q + 2 < m) ? g.z : i, (q + 3 < m) ? g.w : i};
    T f[4];
#pragma unroll
    for (int v = 0; v < 4; v++) f[v] = load(j[v]);
    bool in[4];
#pragma unroll
    for (int v = 0; v < 4; v++) in[v] = q + v < m;
    use(j, f, in);
  }
}

// walk_list with the same number of groups for every lane of the wavefront (mw: the
// longest list; m may be 0), so that `use` may work across lanes.
template <class T, class Load, class Use>
__device__ __forceinline__ void walk_uniform(uint32_t i, uint32_t m, uint32_t mw, const uint32_t* __restrict__ ids,
                                             uint32_t kmax, Load load, Use use) {
  auto group = [&](uint32_t q, uint32_t j[4]) {
    const uint4 g = *reinterpret_cast<const uint4*>(ids + nbr_slot(i, q < m ? q : 0u, kmax));
    j[0] = (q < m) ? g.x : i;
    j[1] = (q + 1 < m) ? g.y : i;
    j[2] = (q + 2 < m) ? g.z : i;
    j[3] = (q + 3 < m) ? g.w : i;
  };
  uint32_t j[4], jn[4];
  T f[4];
  group(0, j);
  group(4, jn);
#pragma unroll
  for (int v = 0; v < 4; v++) f[v] = load(j[v]);
  for (uint32_t q = 0; q < mw; q += 4) {
    T fn[4];
    uint32_t j2[4];
#pragma unroll
    for (int v = 0; v < 4; v++) fn[v] = load(jn[v]);
    group(q + 8, j2);
    bool in[4];
#pragma unroll
    for (int v = 0; v < 4; v++) in[v] = q + v < m;
    use(j, f, in);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      j[v] = jn[v];
      jn[v] = j2[v];
      f[v] = fn[v];
    }
  }
}

// The walk of a pass whose expensive terms only count for the nearer neighbours
// (r < r_e, while the list reaches r_lap): far(j, p, f1, in, e) gets four
// neighbours' positions p (pos) and fields f1 (load1), adds the terms of all of them
// and sets e[v] for the nearer ones; near(p, f2, e) gets those with the fields
// f2 (load2) and adds their terms, in list order.
//
// NEAR: a lane first collects its nearer neighbours in its column of `queue`
// (LDS, kNearQueue slots, [slot][thread]), then computes their terms, so that a
// wavefront goes through the expensive instructions as often as its lanes have
// near neighbours (about 14 times, for r_e = 2.1 and r_lap = 3.1) and not once
// per list entry (37): gradient of 1.05M particles 147 -> 97 us, density and
// count pass 153 -> 137; 131k 32 -> 19 and 33 -> 25.  Otherwise (the radii are
// alike and nearly every neighbour is near: collecting would only add a pass;
// 6k particles at r_e = r_lap = 2.4: gradient 9.9, count 12.1 us) the terms are
// computed on the way.  The line (near_pays): near neighbours below three
// quarters of the list.
constexpr uint32_t kNearQueue = 24;
inline bool near_pays(double re, double rl) { return re * re < 0.75 * rl * rl; }
template <bool NEAR, int THREADS, class F1, class F2, class Pos, class Load1, class Load2, class Far, class Near>
__device__ __forceinline__ void walk_near(uint32_t i, uint32_t m, const uint32_t* __restrict__ ids, uint32_t kmax,
                                          Pos pos, uint32_t (*queue)[THREADS], Load1 load1,
                                          Load2 load2, Far far, Near near) {
  if (m == 0) return;
  auto group = [&](uint32_t q, uint32_t j[4]) {
    const uint4 g = *reinterpret_cast<const uint4*>(ids + nbr_slot(i, q, kmax));
    j[0] = g.x;
    j[1] = (q + 1 < m) ? g.y : i;
    j[2] = (q + 2 < m) ? g.z : i;
    j[3] = (q + 3 < m) ? g.w : i;
  };
  uint32_t j[4], jn[4];
  double2 p[4], pn[4];
  F1 f[4], fn[4];
  F2 g[4], gn[4];
  group(0, j);
  group(m > 4 ? 4u : 0u, jn);
#pragma unroll
  for (int v = 0; v < 4; v++) {
    p[v] = pos(j[v]);
    f[v] = load1(j[v]);
    if (!NEAR) g[v] = load2(j[v]);
  }
  uint32_t q = 0;
  do {
    uint32_t found = 0;
    for (; q < m && (!NEAR || found + 4 <= kNearQueue); q += 4) {
      uint32_t j2[4];
#pragma unroll
      for (int v = 0; v < 4; v++) {
        pn[v] = pos(jn[v]);
        fn[v] = load1(jn[v]);
        if (!NEAR) gn[v] = load2(jn[v]);
      }
      group(q + 8 < m ? q + 8 : 0u, j2);
      bool in[4], e[4];
#pragma unroll
      for (int v = 0; v < 4; v++) in[v] = q + v < m;
      far(j, p, f, in, e);
      if (NEAR) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
          queue[found][threadIdx.x] = j[v];  // (overwritten by the next near one if it is not)
          found += e[v] ? 1u : 0u;
        }
      } else {
        near(p, g, e);
      }
#pragma unroll
      for (int v = 0; v < 4; v++) {
        j[v] = jn[v];
        jn[v] = j2[v];
        p[v] = pn[v];
        f[v] = fn[v];
        if (!NEAR) g[v] = gn[v];
      }
    }
    if (NEAR)
      for (uint32_t k = 0; k < found; k += 4) {
        double2 pk[4];
        F2 gk[4];
        bool e[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
          e[v] = k + v < found;
          const uint32_t jk = e[v] ? queue[k + v < kNearQueue ? k + v : 0u][threadIdx.x] : i;
          pk[v] = pos(jk);
          gk[v] = load2(jk);
        }
        near(pk, gk, e);
      }
  } while (NEAR && q < m);
}

// XCD-aware block order: hardware hands consecutive workgroups to the 8 XCDs
// round-robin; remapping makes each XCD walk one contiguous range of
// particles, so gathered neighbour data stays in that XCD's L2.
__device__ __forceinline__ unsigned xcd_block(unsigned b, unsigned nb) {
  const unsigned per = nb / 8u;
  if (per == 0u || b >= per * 8u) return b;
  return (b % 8u) * per + b / 8u;
}

// Wavefront (64-lane) butterflies without the LDS crossbar: each step pairs lane
// l with lane l ^ 32, 16, 8, 4, 2, 1 in turn.  The first two swap halves and
// rows (permlane swaps); 8 is a rotation of the 16-lane row; after it the
// values repeat every 8 lanes, so a rotation by 4 pairs as l ^ 4 does; 2 and 1
// are quad permutations.  Sums are those of the __shfl_xor butterflies bit
// for bit (each step adds the same two values) in 190 instead of 480 cycles.
// Every lane of the wavefront must be active.
template <int CTRL>
__device__ __forceinline__ unsigned dpp_u32(unsigned v) {
  return static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(v));
  const unsigned lo = dpp_u32<CTRL>(static_cast<unsigned>(b)), hi = dpp_u32<CTRL>(static_cast<unsigned>(b >> 32));
  return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}
constexpr int kRowRor8 = 0x128, kRowRor4 = 0x124, kQuad2301 = 0x4E, kQuad1032 = 0xB1;
struct PairU32 {
  unsigned a, b;  // a lane's own and its partner's value, in the same order on both
};
__device__ __forceinline__ PairU32 pair32(unsigned v) {
  const auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return PairU32{s[0], s[1]};
}
__device__ __forceinline__ PairU32 pair16(unsigned v) {
  const auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return PairU32{s[0], s[1]};
}
__device__ __forceinline__ double join_f64(unsigned lo, unsigned hi) {
  return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}
__device__ __forceinline__ double wave_sum(double v) {
  const auto halves = [](double x, auto pair) {
    const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(x));
    const PairU32 l = pair(static_cast<unsigned>(b)), h = pair(static_cast<unsigned>(b >> 32));
    return join_f64(l.a, h.a) + join_f64(l.b, h.b);
  };
  v = halves(v, pair32);
  v = halves(v, pair16);
  v += dpp_f64<kRowRor8>(v);
  v += dpp_f64<kRowRor4>(v);
  v += dpp_f64<kQuad2301>(v);
  v += dpp_f64<kQuad1032>(v);
  return v;
}
template <class Op>
__device__ __forceinline__ unsigned wave_fold_u32(unsigned v, Op op) {
  PairU32 p = pair32(v);
  v = op(p.a, p.b);
  p = pair16(v);
  v = op(p.a, p.b);
  v = op(v, dpp_u32<kRowRor8>(v));
  v = op(v, dpp_u32<kRowRor4>(v));
  v = op(v, dpp_u32<kQuad2301>(v));
  return op(v, dpp_u32<kQuad1032>(v));
}
__device__ __forceinline__ unsigned wave_min_u32(unsigned v) {
  return wave_fold_u32(v, [](unsigned a, unsigned b) { return b < a ? b : a; });
}
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
  return wave_fold_u32(v, [](unsigned a, unsigned b) { return b > a ? b : a; });
}

// Adds the sum of v over the block (THREADS threads, every one calls it) to
// *total: one atomic a block.  One a wavefront, 16k of them to one address at
// 1.05M particles, took a third of the passes that count: the search 237 -> 151
// us, the density and count pass 230 -> 153.
template <int THREADS>
__device__ __forceinline__ void block_count(uint32_t v, unsigned long long* total) {
  __shared__ unsigned part[THREADS / 64];
  const unsigned w = wave_fold_u32(v, [](unsigned a, unsigned b) { return a + b; });
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned long long t = 0;
    for (int k = 0; k < THREADS / 64; k++) t += part[k];
    if (t > 0) atomicAdd(total, t);
  }
}

// Deterministic block sum of one double per thread (blockDim.x == NT):
// fixed wavefront butterflies, then the NT/64 wavefront sums in order.
template <int NT>
__device__ __forceinline__ double block_sum(double v, double* lds) {
  v = wave_sum(v);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) lds[wv] = v;
  __syncthreads();
  double s = lds[0];
#pragma unroll
  for (int k = 1; k < NT / 64; k++) s += lds[k];
  __syncthreads();
  return s;
}

// Sum of `count` partials in a fixed order that every block reproduces
// identically (thread t takes t, t+NT, ...; then block_sum).
template <int NT>
__device__ __forceinline__ double reduce_partials(const double* part, int count, double* lds) {
  double s = 0;
  for (int k = threadIdx.x; k < count; k += NT) s += part[k];
  return block_sum<NT>(s, lds);
}

// Block sums of two values per thread at once (lds: 2 * NT / 64 entries),
// in the order of block_sum.
template <int NT>
__device__ __forceinline__ void block_sum2(double a, double b, double* lds, double& sa, double& sb) {
  a = wave_sum(a);
  b = wave_sum(b);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) {
    lds[wv] = a;
    lds[NT / 64 + wv] = b;
  }
  __syncthreads();
  sa = lds[0];
  sb = lds[NT / 64];
#pragma unroll
  for (int k = 1; k < NT / 64; k++) {
    sa += lds[k];
    sb += lds[NT / 64 + k];
  }
  __syncthreads();
}

// What the learned warm start's feature pass gathers of a neighbour, one
// 32-byte record (one cache line access where four arrays cost four): the
// position (x = NaN for dummy particles, which no r^2 < r_lap^2 test
// accepts), the pressure p_prev and the residual r0 = b - A p_prev.
struct __attribute__((aligned(32))) FeatRec {
  double x, z, p, r0;
};

// The feature scales from the reduced sums out[0] = |r0|^2, out[2] = sum p^2,
// out[3] = sum diag^2, out[4] = alive count (one thread): out[6..9] =
// |r0|^2, 1/s_p, 1/s_r and s_d = s_r / RMS(diag) over the alive rows, with
// s_v = RMS(v); zero where a scale is zero or no row is alive.
__device__ __forceinline__ void feat_scales(double* out) {
  const double rr = out[0], pp = out[2], dd = out[3], na = out[4];
  double inv_sp = 0, inv_sr = 0, sd = 0;
  if (na > 0) {
    const double s_r = sqrt(rr / na), s_p = sqrt(pp / na), drms = sqrt(dd / na);
    inv_sp = s_p > 0 ? 1.0 / s_p : 0.0;
    inv_sr = s_r > 0 ? 1.0 / s_r : 0.0;
    sd = (drms > 0 && s_r > 0) ? s_r / drms : 0.0;
  }
  out[6] = rr;
  out[7] = inv_sp;
  out[8] = inv_sr;
  out[9] = sd;
}

}  // namespace mps

// Batched neighbour-list traversal shared by the pair kernels.
#pragma once

#include <type_traits>

#include "common.hpp"

namespace sophia {

// Fields of one neighbour j of particle i, gathered before any of them is
// used; dx, dy, dz = x_i - x_j.
template <typename R>
struct Nb {
  double dx, dy, dz, m, rho, pres, h;
  R ux, uy, uz, temp, grx, gry, grz;
  double rref, por;
  int pt;
  int j;  // the neighbour's index, for fields a few kernels read on condition
};

// Particle i's side of the differences: FP64 position, or its pos4 record.
struct NbOrigin {
  double x, y, z;
  float4 p4;
};

// REL (FP32 fields only): the differences come from the pos4 records (one
// 16 B gather, error below 2^-21 of the grid spacing) instead of three FP64
// gathers, for stages that use them in FP32.  Otherwise FP64 differences.
template <bool REL, typename R>
__device__ inline Nb<R> load_nb(const SphView<R>& v, int j, const NbOrigin& o) {
  Nb<R> q;
  if constexpr (REL && std::is_same<R, float>::value) {
    const float3 d = rel_diff(o.p4, v.pos4[j], v.pgrid, v.pmask);
    q.dx = d.x; q.dy = d.y; q.dz = d.z;
  } else {
    pdiff(v, o.x, o.y, o.z, j, q.dx, q.dy, q.dz);
  }
  q.m = v.m[j]; q.rho = v.rho[j]; q.pres = v.pres[j]; q.h = v.h[j];
  q.ux = v.ux[j]; q.uy = v.uy[j]; q.uz = v.uz[j]; q.temp = v.temp[j]; q.rref = v.rho_ref[j];
  q.grx = v.grx[j]; q.gry = v.gry[j]; q.grz = v.grz[j]; q.por = v.por[j];
  q.pt = v.ptype[j];
  q.j = j;
  return q;
}

// Lanes per particle of the pair kernels.  With one lane a particle's ~81
// neighbours are ~20 dependent batches, which only other waves hide, and small
// runs have few (4,200 particles are 66 waves on 1024 SIMDs).  With G lanes
// lane g takes the quads g, g + G, ... of the list and the lanes' sums meet in
// a butterfly (group_sum): the order of a sum changes, not its terms.
template <int G>
__device__ inline int pair_particle() { return particle_index() / G; }
template <int G>
__device__ inline int pair_sub() { return (int)threadIdx.x & (G - 1); }

// One rule for all of them, by the whole step (us, with 1 / 2 / 4 / 8 lanes), since
// the kernels of a step differ by a few per cent either way: ISPH with one Jacobi
// sweep, mixed, 627 / 478 / 432 / 410 at 5,200 particles, 718 / 619 / 590 / 587 at 37,000,
// 782 / 643 / 642 / 636 at 51,000, 833 / 704 / 697 / 716 at 70,000, 860 / 778 / 780 / 791 at
// 92,000, 1492 / 1342 / 1412 / 1566 at 276,000, 4937 / 4647 / 4562 / 4767 at 1.16 M; FP64
// 871 / 766 / 734 / 731 at 51,000, 1115 / 852 / 814 / 834 at 70,000, 1179 / 989 / 938 / 949
// at 92,000, 2179 / 1890 / 1930 / 2109 at 276,000.  WCSPH and the 2D step lie the same
// way; the rule is within 2 % of the best but at 92,000 in FP64 (5 %).
inline int pair_lanes(int n) { return n >= 90000 ? 2 : (n >= 40000 ? 4 : 8); }

// f(lanes as an integral constant, grid) for n particles
template <class F>
inline int pair_launch(int n, int lanes, F&& f) {
  if (n <= 0) return 0;
  switch (lanes) {
    case 1: f(std::integral_constant<int, 1>{}, grid_xcd(n)); break;
    case 2: f(std::integral_constant<int, 2>{}, grid_xcd(n * 2)); break;
    case 4: f(std::integral_constant<int, 4>{}, grid_xcd(n * 4)); break;
    default: f(std::integral_constant<int, 8>{}, grid_xcd(n * 8)); break;
  }
  HIP_TRY(hipGetLastError());
  return 0;
}
template <class F>
inline int pair_launch(int n, F&& f) {
  // two lanes per particle stay within an int: 2^30 particles do not fit the
  // device's memory
  return pair_launch(n, pair_lanes(n), static_cast<F&&>(f));
}

// The list in batches of four, in list order, in two phases: the fields of
// all four neighbours are gathered (straight-line code, so every load of the
// batch is in flight together), then f(q, on) runs per neighbour; the next
// batch's indices are loaded before this batch is consumed.  Loads of fields
// a body never reads are dropped by the compiler.  Slots past the count
// repeat the last entry with on = false; bodies add `on ? term : 0` (a
// select: exact, and NaN-safe for the unused slots).  With G lanes each visits
// every G-th quad, and the caller sums over the lanes.
template <bool REL = false, int G = 1, typename R, class F>
__device__ inline void for_nbrs4(const SphView<R>& v, int i, bool eps_rule, F&& f) {
  const int cnt = min(v.nbr_cnt[i], v.nbr_cap);
  if (cnt <= 0) return;
  const size_t n = (size_t)v.n;
  NbOrigin o;
  if constexpr (REL && std::is_same<R, float>::value) {
    o.p4 = v.pos4[i];
  } else {
    o.x = v.x[i]; o.y = v.y[i]; o.z = v.z[i];
  }
  const int last4 = (cnt - 1) & ~3;
  const int k0 = G == 1 ? 0 : 4 * pair_sub<G>();
  uint4 en4 = *(const uint4*)(v.nbr + nbr_slot(min(k0, last4), i, (int)n));
  for (int k = k0; k < cnt; k += 4 * G) {
    const uint32_t en[4] = {en4.x, en4.y, en4.z, en4.w};
    uint32_t e[4];
#pragma unroll
    for (int u = 0; u < 4; u++) e[u] = en[u];
    Nb<R> q[4];
#pragma unroll
    for (int u = 0; u < 4; u++) q[u] = load_nb<REL>(v, (int)(e[u] & ~kNbrFlag), o);
    en4 = *(const uint4*)(v.nbr + nbr_slot(min(k + 4 * G, last4), i, (int)n));
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const bool on = (k + u < cnt) && !(eps_rule && (e[u] & kNbrFlag));
      f(q[u], on);
    }
  }
}

// One neighbour from the packed records: the members of Nb that the
// FP64-geometry pair sums read (h and the velocities only with VEL).
template <typename R>
struct NbP {
  double dx, dy, dz, m, vol, pres;
  R ux, uy, uz, temp, h;
  int pt;
  int j;
  double S;  // flux-wall sum (mixed path with VEL; otherwise flux_s[j])
};

// The list in batches of four like for_nbrs4, reading the packed records
// pk = {x, y, z, m} and pk2 = {V, p}, then with VEL pkv = {ux, uy, uz, T}
// and pkh = {h, p_type}, else p_type: four or three gathers per neighbour in
// place of twelve or seven.  With VEL on the mixed path pk, pkb = {V, p,
// u, T} and pkc = {S, h, p_type}: three.  dx = x_i - x_j (minimum image on periodic axes),
// the same bits as pdiff.
template <bool VEL, int G = 1, typename R, class F>
__device__ inline void for_nbrs4_pk(const SphView<R>& v, int i, bool eps_rule, F&& f) {
  const int cnt = min(v.nbr_cnt[i], v.nbr_cap);
  if (cnt <= 0) return;
  const int n = v.n;
  const double4 pi = v.pk[i];
  const int last4 = (cnt - 1) & ~3;
  const int k0 = G == 1 ? 0 : 4 * pair_sub<G>();
  uint4 en4 = *(const uint4*)(v.nbr + nbr_slot(min(k0, last4), i, n));
  for (int k = k0; k < cnt; k += 4 * G) {
    const uint32_t en[4] = {en4.x, en4.y, en4.z, en4.w};
    NbP<R> q[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = (int)(en[u] & ~kNbrFlag);
      const double4 a = v.pk[j];
      q[u].dx = pi.x - a.x;
      q[u].dy = pi.y - a.y;
      q[u].dz = pi.z - a.z;
      q[u].m = a.w;
      if constexpr (VEL && std::is_same<R, float>::value) {
        // mixed path: two more records, {V, p, u, T} and {S, h, p_type}
        const PkB b = v.pkb[j];
        const PkC c = v.pkc[j];
        q[u].vol = b.vol; q[u].pres = b.p;
        q[u].ux = b.ux; q[u].uy = b.uy; q[u].uz = b.uz; q[u].temp = b.temp;
        q[u].S = c.S; q[u].h = c.h; q[u].pt = c.pt;
        q[u].j = j;
        continue;
      }
      const double2 b = v.pk2[j];
      q[u].vol = b.x;
      q[u].pres = b.y;
      if constexpr (VEL) {
        const auto w = v.pkv[j];
        const HRec<R> hr = v.pkh[j];
        q[u].ux = w.x; q[u].uy = w.y; q[u].uz = w.z; q[u].temp = w.w;
        q[u].h = hr.h;
        q[u].pt = hr.pt;
      } else {
        q[u].pt = v.ptype[j];
      }
      q[u].j = j;
    }
    en4 = *(const uint4*)(v.nbr + nbr_slot(min(k + 4 * G, last4), i, n));
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const bool on = (k + u < cnt) && !(eps_rule && (en[u] & kNbrFlag));
      if (v.pmask) {
        if (v.pmask & 1) q[u].dx = per_wrap(q[u].dx, v.plx);
        if (v.pmask & 2) q[u].dy = per_wrap(q[u].dy, v.ply);
        if (v.pmask & 4) q[u].dz = per_wrap(q[u].dz, v.plz);
      }
      f(q[u], on);
    }
  }
}

// One neighbour from the 32 B records (FP32 pair kernels): the members of Nb
// those kernels read, the differences from the position records.
struct NbR {
  float dx, dy, dz, vol, aux;
  float ux, uy, uz, temp;
  int pt;
  int j;
  bool flag;  // the entry's eps-rule flag (kNbrFlag), for kernels that apply it themselves
};

// The list in batches of four like for_nbrs4<true>, reading r32 (and with
// VEL pkv = {ux, uy, uz, T}): one or two gathers per neighbour in place of
// four to eight, the same values.
template <bool VEL, int G = 1, class F>
__device__ inline void for_nbrs4_r32(const SphView<float>& v, int i, bool eps_rule, F&& f) {
  const int cnt = min(v.nbr_cnt[i], v.nbr_cap);
  if (cnt <= 0) return;
  const int n = v.n;
  const float4 pi4 = v.pos4[i];
  const int last4 = (cnt - 1) & ~3;
  const int k0 = G == 1 ? 0 : 4 * pair_sub<G>();
  uint4 en4 = *(const uint4*)(v.nbr + nbr_slot(min(k0, last4), i, n));
  for (int k = k0; k < cnt; k += 4 * G) {
    const uint32_t en[4] = {en4.x, en4.y, en4.z, en4.w};
    NbR q[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int j = (int)(en[u] & ~kNbrFlag);
      const Rec32 a = v.r32[j];
      const float3 d = rel_diff(pi4, a.p, v.pgrid, v.pmask);
      q[u].dx = d.x; q[u].dy = d.y; q[u].dz = d.z;
      q[u].vol = a.vol; q[u].aux = a.aux; q[u].pt = a.pt;
      if constexpr (VEL) {
        const float4 w = v.pkv[j];
        q[u].ux = w.x; q[u].uy = w.y; q[u].uz = w.z; q[u].temp = w.w;
      }
      q[u].j = j;
      q[u].flag = (en[u] & kNbrFlag) != 0;
    }
    en4 = *(const uint4*)(v.nbr + nbr_slot(min(k + 4 * G, last4), i, n));
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const bool on = (k + u < cnt) && !(eps_rule && (en[u] & kNbrFlag));
      f(q[u], on);
    }
  }
}

// V = m / rho of a neighbour, from its record where there is one
template <typename R>
__device__ inline double nb_vol(const Nb<R>& q) { return q.m / q.rho; }
template <typename R>
__device__ inline double nb_vol(const NbP<R>& q) { return q.vol; }
__device__ inline float nb_vol(const NbR& q) { return q.vol; }

}  // namespace sophia

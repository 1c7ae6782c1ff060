// LDS-staged traversal of the mixed operator's window format (kFmtWin).
//
// A tile of consecutive rows (cell-sorted particles) needs the columns of the
// cells around its own cells.  In the extended key e = x + 1 + (NI + 2)(y + NJ z),
// x = -1 .. NI, the cells of the tile are a range [ea, eb], and the planes
// e = ea - 1 .. eb + 1 hold every column: plane e is the nine (dz, dy) cells
// around (x, y, z), in the order of the neighbour list, periodic axes
// wrapped.  win_stage copies the planes' particles of a vector into LDS in that order,
// so the window of a row in cell e is the planes e - 1, e, e + 1: one
// contiguous LDS range, and a column is the window's base plus the 11-bit slot
// of its entry.  Against run offsets (a u8 from the first particle of one of nine
// x-runs) this takes the eight compares and selects per entry that find the
// run out of the inner loop, and it works across a periodic wrap.
//
// Bound: the operator stream from HBM (4 B per entry) plus 28 B per row; the
// staging reads about 11 values per row from L2.
#pragma once

#include "ppe.hpp"

namespace sophia {

constexpr int kWinThreads = 256;
constexpr int kWinCells = 256;  // staged cells per tile
constexpr int kWinPlanes = kWinCells / 9;
// staged values per tile: a 256-row tile of the 1 mm columns takes about 2800;
// with the tables it is 19.5 KB in FP32, eight blocks per CU
constexpr int kWinCap = 4096;  // the coarse correction's table leaves no room for more
static_assert(kWinMax < kWinCap, "a single row's window always fits");

// Where the cells of a tile's planes go: cell c = 9 p + r, cell r of the p-th
// planned plane, holds the slots [pre[c], pre[c + 1]) of the staged copy.
struct WinPlan {
  int pre[kWinCells + 1];
  int start[kWinCells];  // cellval of the cell
  int wsum[kWinThreads / 64];
  // a tile with gaps (kWinGaps): its planes, and each row's first
  int plane[kWinPlanes];
  int cut;
  uint8_t first[kWinThreads];
};
constexpr int kWinGaps = INT32_MIN;
template <typename XT>
struct WinStage {
  XT x[kWinCap];
  WinPlan p;
};

template <class O>
__device__ inline int win_ekey(const O& o, uint32_t key) {
  const int t = (int)(key / (uint32_t)o.NI);
  return (int)(key - (uint32_t)t * (uint32_t)o.NI) + 1 + (o.NI + 2) * t;
}

// inclusive sum or maximum over the block's threads; w takes one word per wave
template <bool MAX>
__device__ inline int win_scan(int v, int* w) {
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  for (int off = 1; off < 64; off <<= 1) {
    const int u = __shfl_up(v, off);
    if (lane >= off) v = MAX ? max(v, u) : v + u;
  }
  if (lane == 63) w[wave] = v;
  __syncthreads();
  for (int k = 0; k < kWinThreads / 64 - 1; k++) {
    const int u = w[k];
    if (k < wave) v = MAX ? max(v, u) : v + u;
  }
  __syncthreads();  // w may be written again
  return v;
}

// The particles of planned cell c, the r-th of the plane around extended key e, and
// S.start[c] from `cellval`.
template <class O, class CV>
__device__ inline int win_cell_len(const O& o, int e, int r, int c, WinPlan& S, CV&& cellval) {
  const int row = e / (o.NI + 2);
  int x = e - (o.NI + 2) * row - 1, z = row / o.NJ;
  int y = row - o.NJ * z;
  y += r % 3 - 1;
  z += r / 3 - 1;
  int first = -1, len = 0;  // outside the grid: no particles
  if (cell_in(o.pmask, 2, z, o.NK) && cell_in(o.pmask, 1, y, o.NJ) && cell_in(o.pmask, 0, x, o.NI)) {
    const int k = x + o.NI * (y + o.NJ * z);
    first = (int)o.cell_off[k];
    len = (int)o.cell_off[k + 1] - first;
  }
  S.start[c] = cellval(x, y, z, first);
  return len;
}

// A plan for a range whose cells lie too far apart, or hold too much, for one run
// of planes: the planes around its rows' cells alone, side by side, each once
// (walls and other particles that are not rows need none: a range without rows is
// done at once).  Returns the end of the rows that fit.  (Halving the range until
// its run of planes fits, walls and empty cells included, took 85 us a pass for a
// film of two layers on sparse walls, 278 k particles, in place of 17.2; 37.5 / 21.6
// for a column of 144 k rows under walls three times its height; 29.0 / 11.7 for one
// of 64 k rows in a domain sixteen times as wide.)
template <class O, class CV>
__device__ int win_plan_gaps(const O& o, int i0, int i1, WinPlan& S, int* ncells, CV&& cellval) {
  const int t = (int)threadIdx.x, i = i0 + t;
  int e = -1;
  if (i < i1 && o.row[i] != 0) {
    const uint32_t key = o.keys[i];
    if (key < (uint32_t)o.ncell) e = win_ekey(o, key);
  }
  // keys ascend: the row before this one has the largest key so far
  const int emax = win_scan<true>(e, S.wsum);
  const int up = __shfl_up(emax, 1);
  if ((t & 63) == 63) S.wsum[t >> 6] = emax;
  if (t == 0) S.cut = i1;
  __syncthreads();
  const int prev = t == 0 ? -1 : ((t & 63) == 0 ? S.wsum[(t >> 6) - 1] : up);
  __syncthreads();
  const int add = e < 0 ? 0 : (prev < 0 ? 3 : min(e - prev, 3));
  const int p = win_scan<false>(add, S.wsum);  // planes up to this row's e + 1
  if (e >= 0 && p > kWinPlanes) atomicMin(&S.cut, i);
  if (e >= 0 && p <= kWinPlanes) {
    if (add > 0) S.plane[p - 1] = e + 1;
    if (add > 1) S.plane[p - 2] = e;
    if (add > 2) S.plane[p - 3] = e - 1;
    S.first[t] = (uint8_t)(p - 3);
  } else {
    S.first[t] = 0;
  }
  // planes in use: those of the last row that fits
  int np = win_scan<true>(e >= 0 && p <= kWinPlanes ? p : 0, S.wsum);
  if (t == kWinThreads - 1) S.wsum[0] = np;
  __syncthreads();
  np = S.wsum[0];
  __syncthreads();
  if (np == 0) return i1;  // no rows
  const int len = t < 9 * np ? win_cell_len(o, S.plane[t / 9], t % 9, t, S, static_cast<CV&&>(cellval)) : 0;
  const int pre = win_scan<false>(len, S.wsum);
  S.pre[t + 1] = pre;
  if (t == 0) S.pre[0] = 0;
  __syncthreads();
  while (np >= 3 && S.pre[9 * np] > kWinCap) np--;
  // np < 3: a particle whose window does not fit (no row of an assembled operator)
  *ncells = np >= 3 ? 9 * np : 0;
  if (e >= 0 && p > max(np, 3)) atomicMin(&S.cut, i);
  __syncthreads();
  return S.cut;
}

// The block plans the row range [i0, i1), or as much of it from i0 on as fits, and
// returns the planned end m (all threads alike); *e0 is the extended key of row i0,
// or kWinGaps (win_first), and *cells the planned cells, 0 when there is nothing to
// stage: no rows, or a row whose window does not fit (no row of an assembled
// operator).  `cellval(x, y, z, first)` is kept per cell in S.start; first is -1 for
// places outside the grid.
template <class O, class CV>
__device__ int win_plan(const O& o, int i0, int i1, WinPlan& S, int* e0, int* ncells, CV&& cellval) {
  const int t = (int)threadIdx.x, lane = t & 63;
  const uint32_t ka = o.keys[i0], kb = o.keys[i1 - 1];
  *e0 = kWinGaps;
  *ncells = 0;
  __syncthreads();  // the previous tile is done with S
  if (ka >= (uint32_t)o.ncell) return i1;  // past the last cell
  const int ea = win_ekey(o, ka);
  const int cells = kb < (uint32_t)o.ncell ? 9 * (win_ekey(o, kb) - ea + 3) : kWinCells + 1;
  if (cells <= kWinCells) {
    const int len = t < cells ? win_cell_len(o, ea - 1 + t / 9, t % 9, t, S, cellval) : 0;
    int inc = len;
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(inc, off);
      if (lane >= off) inc += v;
    }
    if (lane == 63) S.wsum[t >> 6] = inc;
    __syncthreads();
    int add = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kWinThreads / 64; w++) {
      const int v = S.wsum[w];
      add += w < (t >> 6) ? v : 0;
      total += v;
    }
    if (total <= kWinCap) {
      S.pre[t + 1] = inc + add;
      if (t == 0) S.pre[0] = 0;
      __syncthreads();
      *e0 = ea;
      *ncells = cells;
      return i1;
    }
    __syncthreads();  // S.wsum is read
  }
  return win_plan_gaps(o, i0, i1, S, ncells, static_cast<CV&&>(cellval));
}

// first planned cell of the window of row i, whose cell key is `key`, of the tile
// planned from row s0 on
template <class O>
__device__ inline int win_first(const O& o, const WinPlan& S, int e0, int s0, int i, uint32_t key) {
  return e0 == kWinGaps ? 9 * S.first[i - s0] : 9 * (win_ekey(o, key) - e0);
}

// win_plan, then the values: `val(cellval, l, c)` is that of the l-th particle of
// planned cell c
template <typename XT, class CV, class F>
__device__ int win_stage(const PpeOp& o, int i0, int i1, WinStage<XT>& S, int* e0, CV&& cellval, F&& val) {
  int cells;
  const int m = win_plan(o, i0, i1, S.p, e0, &cells, static_cast<CV&&>(cellval));
  if (cells == 0) return m;
  // half a wave per cell (about 23 particles), four cells in flight
  const int h = (int)threadIdx.x >> 5, l0 = (int)threadIdx.x & 31;
  for (int c = h; c < cells; c += 32) {
    XT v[4];
    int at[4], n[4], st[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int cc = c + 8 * u;
      at[u] = cc < cells ? S.p.pre[cc] : 0;
      n[u] = cc < cells ? S.p.pre[cc + 1] - at[u] : 0;
      st[u] = l0 < n[u] ? S.p.start[cc] : 0;
      if (l0 < n[u]) v[u] = val(st[u], l0, cc);
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      if (l0 < n[u]) S.x[at[u] + l0] = v[u];
      for (int l = l0 + 32; l < n[u]; l += 32) S.x[at[u] + l] = val(st[u], l, c + 8 * u);
    }
  }
  __syncthreads();
  return m;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <bool NT>
__device__ __forceinline__ u32x4 ldq(const u32x4* p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}

// What a lane has in hand of its row before the tile is staged: the row's
// first two quads travel while the block stages.  G = 1 (operators streamed from
// HBM, win_group) loads past the caches, so that x stays in L2: 83.3 -> 78.5 us at
// 1.16 M rows, 69.4 -> 64.4 us for the 10^6-row box.  Two quads in flight: one 92,
// three 90, four 96 us (registers spill at eight waves).
constexpr int kWinQ = 2;
template <int G>
struct WinHead {
  int i, row, cnt, anc;
  u32x4 w[kWinQ];
  __device__ void load(const PpeOp& o, int ii, int sub) {
    i = ii;
    row = o.row[i];
    const int meta = o.ccnt[i];
    cnt = meta & 0xFFFF;
    anc = (meta >> 16) << 23;
    const u32x4* hp = reinterpret_cast<const u32x4*>(o.hi) + i;
#pragma unroll
    for (int u = 0; u < kWinQ; u++) w[u] = ldq<G == 1>(hp + (size_t)min(sub + u * G, o.nq - 1) * (size_t)o.n);
  }
};

// The head of a pass that only asks whether the row is one.
struct WinRow {
  int row;
};

// f(i, base, lead, head(i), cell) for every row of this block's share, by G
// lanes each: base is the LDS slot of row i's window, cell the planned cell that
// holds the row, lead marks the first of its lanes, and head(i) has run before
// the tile was staged (cellval and val as in win_stage).  (Leaving out the
// staging of tiles without rows, behind a barrier vote, costs every tile more
// than the walls' tiles save: 78.4 -> 85.2 us at 1.16 M rows.)
template <int G, typename XT, class H, class CV, class VL, class F>
__device__ __forceinline__ void win_rows(const PpeOp& o, WinStage<XT>& S, H&& head, CV&& cellval, VL&& val, F&& f) {
  constexpr int TR = kWinThreads / G;
  const int per = (int)gridDim.x >> 3;
  const int chunk = ((((o.n + 7) >> 3) + 63) >> 6) << 6;  // rows per XCD, as xcd_rows
  const int lo = (int)(blockIdx.x & 7) * chunk, hi = min(o.n, lo + chunk);
  const int t = (int)threadIdx.x, tr = t / G;
  for (int i0 = lo + (int)(blockIdx.x >> 3) * TR; i0 < hi; i0 += per * TR) {
    const int i1 = min(i0 + TR, hi);
    for (int s0 = i0; s0 < i1;) {
      int e0;
      auto hd = head(min(s0 + tr, i1 - 1));
      const int m = win_stage(o, s0, i1, S, &e0, cellval, val);
      const int i = s0 + tr;
      if (i < m) {
        // particles that no cell or plan holds are not rows: any slot will do
        const uint32_t key = o.keys[i];
        const int c = key < (uint32_t)o.ncell ? win_first(o, S.p, e0, s0, i, key) : 0;
        const int cw = min(max(c, 0), kWinCells - 27);
        f(i, S.p.pre[cw], (t & (G - 1)) == 0, hd, cw + 13);
      }
      s0 = m;
    }
  }
}

// This lane's share of sum_j hi_ij x_j over the stored columns of row i (quads
// sub, sub + G, ...); xw is the row's window.  Padding entries need no mask:
// they are a value on the row's own column that the inner diagonal takes up.
// Two quads are consumed while the next two are in flight.
template <int G>
__device__ __forceinline__ float win_row_sum(const PpeOp& o, WinHead<G>& h, const float* xw) {
  constexpr int Q = kWinQ;
  const int nq = (h.cnt + 3) >> 2, last = nq - 1;
  const int sub = (int)threadIdx.x & (G - 1);
  float s = 0.f;
  const u32x4* hp = reinterpret_cast<const u32x4*>(o.hi) + h.i;
  const size_t n = (size_t)o.n;
  // quads past the row's last were read ahead of its count: slot 0, unused
#pragma unroll
  for (int u = 0; u < Q; u++)
    if (sub + u * G >= nq) h.w[u] = 0u;
  for (int q = sub; q < nq; q += Q * G) {
    u32x4 c[Q];
    float xv[Q][4];
#pragma unroll
    for (int u = 0; u < Q; u++) {
      c[u] = h.w[u];
#pragma unroll
      for (int k = 0; k < 4; k++) xv[u][k] = xw[c[u][k] & (uint32_t)kWinMax];
    }
#pragma unroll
    for (int u = 0; u < Q; u++) h.w[u] = ldq<G == 1>(hp + (size_t)min(q + (Q + u) * G, last) * n);
#pragma unroll
    for (int u = 0; u < Q; u++)
      if (q + u * G < nq) {
#pragma unroll
        for (int k = 0; k < 4; k++) s += win_val(c[u][k], h.anc) * xv[u][k];
      }
  }
  return s;
}

// the same with hi + lo in FP64
template <int G>
__device__ __forceinline__ double win_row_sum_full(const PpeOp& o, int i, const double* xw) {
  const int meta = o.ccnt[i];
  const int nq = ((meta & 0xFFFF) + 3) >> 2, last = nq - 1;
  const int anc = (meta >> 16) << 23;
  const int sub = (int)threadIdx.x & (G - 1);
  double s = 0;
  if (sub >= nq) return s;
  const uint4* hp = reinterpret_cast<const uint4*>(o.hi) + i;
  const float4* lp = reinterpret_cast<const float4*>(o.lo) + i;
  const size_t n = (size_t)o.n;
  uint4 w = hp[(size_t)sub * n];
  float4 l = lp[(size_t)sub * n];
  for (int q = sub; q < nq; q += G) {
    const uint32_t c[4] = {w.x, w.y, w.z, w.w};
    const float lv[4] = {l.x, l.y, l.z, l.w};
    double xv[4];
#pragma unroll
    for (int u = 0; u < 4; u++) xv[u] = xw[c[u] & (uint32_t)kWinMax];
    w = hp[(size_t)min(q + G, last) * n];
    l = lp[(size_t)min(q + G, last) * n];
#pragma unroll
    for (int u = 0; u < 4; u++) s += ((double)win_val(c[u], anc) + (double)lv[u]) * xv[u];
  }
  return s;
}

// Lanes per row of the window-staged passes.  One lane walks about 20 quads in
// turn, which hides behind other waves only when there are many: at 4,200 /
// 92,000 / 276,000 / 1,160,000 rows the inner product takes 14.7 / 15.3 / 27.2 /
// 78.5 us with one lane, 8.2 / 10.5 / 22.7 / 86 with two and 7.1 / 11.2 / 26 / 110
// with four (a tile has 256 / G rows, so more lanes stage more per row).  One lane
// pays where the words come from HBM, past the 256 MB last-level cache (us per
// BiCGStab iteration, one lane past the caches / two through them):
//   columns, 494 k / 616 k / 806 k / 1.16 M particles  125 / 158 / 211 / 311 MB
//                                      106 / 87, 127 / 102, 148 / 128, 196 / 203
//   h = 1.0 dx, 616 k particles                58 MB   140 / 100
//   h = 1.6 dx, 616 k and 1.16 M         277, 546 MB   199 / 174, 335 / 311
//   boxes, 512 k / 729 k / 1 M      164 / 233 / 320 MB  96 / 94, 149 / 127, 161 / 189
constexpr int64_t kWinStream = 290000000;  // bytes of words
constexpr int kWinTwo = 40000;
inline int win_group(int n, int64_t nnz) { return 4 * nnz > kWinStream ? 1 : (n >= kWinTwo ? 2 : 4); }

}  // namespace sophia

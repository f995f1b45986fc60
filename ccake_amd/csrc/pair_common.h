// Shared device helpers of the pair kernels (smoothing, gradients,
// diffusion, neighbour counts, pair export).  A wave's 64 lanes own 64
// consecutive particles of the cell-sorted order (a "tile").  The tile's
// bounding box selects, row by row, the contiguous run of cells within the
// interaction radius; every lane then walks the candidates in the same order,
// so the candidate index is wave-uniform and candidate records are fetched
// with scalar loads into SGPRs instead of being staged through LDS.
#pragma once
#include "ccake_internal.h"
#include <climits>
#include <type_traits>

namespace ccake {

// Wave reductions and scans over data-parallel moves (row shifts by 1, 2, 4
// and 8 lanes, then the last lane of a row of 16 to the next row and of the
// lower half to the upper): six dependent steps of a few cycles each, where
// a shuffle through LDS takes over a hundred.  The setup of a pair walk is a
// chain of them, which is most of a small event's pass.  Lane 63 ends with
// the whole wave's result.  The host emulation build uses the shuffles.
#ifndef CCAKE_HOST_EMU
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_move(int ident, int v)
{
  return __builtin_amdgcn_update_dpp(ident, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double ident, double v)
{
  const long long i = __double_as_longlong(ident), b = __double_as_longlong(v);
  const int lo = dpp_move<CTRL, ROWS>((int)i, (int)b), hi = dpp_move<CTRL, ROWS>((int)(i >> 32), (int)(b >> 32));
  return __hiloint2double(hi, lo);
}
// inclusive scan of `op` with identity `ident`
template <class T, class Op>
__device__ __forceinline__ T wave_scan(T v, T ident, Op&& op)
{
  v = op(v, dpp_move<0x111, 0xf>(ident, v));   // row_shr:1
  v = op(v, dpp_move<0x112, 0xf>(ident, v));
  v = op(v, dpp_move<0x114, 0xf>(ident, v));
  v = op(v, dpp_move<0x118, 0xf>(ident, v));
  v = op(v, dpp_move<0x142, 0xa>(ident, v));   // row_bcast:15 into rows 1 and 3
  v = op(v, dpp_move<0x143, 0xc>(ident, v));   // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ int last_lane(int v) { return __builtin_amdgcn_readlane(v, kWave - 1); }
__device__ __forceinline__ double last_lane(double v)
{
  const long long b = __double_as_longlong(v);
  return __hiloint2double(__builtin_amdgcn_readlane((int)(b >> 32), kWave - 1),
                          __builtin_amdgcn_readlane((int)b, kWave - 1));
}
#else
template <class T, class Op>
__device__ __forceinline__ T wave_scan(T v, T ident, Op&& op)
{
  const int lane = threadIdx.x & (kWave - 1);
  for (int o = 1; o < kWave; o <<= 1) {
    const T y = __shfl_up(v, o);
    if (lane >= o) v = op(v, y);
  }
  return v;
}
template <class T>
__device__ __forceinline__ T last_lane(T v) { return __shfl(v, kWave - 1); }
#endif
// wave-uniform results
__device__ __forceinline__ double wave_min_d(double v)
{
  return last_lane(wave_scan(v, (double)INFINITY, [](double a, double b) { return fmin(a, b); }));
}
__device__ __forceinline__ double wave_max_d(double v)
{
  return last_lane(wave_scan(v, -(double)INFINITY, [](double a, double b) { return fmax(a, b); }));
}
__device__ __forceinline__ int wave_incl_scan_i(int v)
{
  return wave_scan(v, 0, [](int a, int b) { return a + b; });
}
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ double uni(double v)
{
  union { double d; int i[2]; } u;
  u.d = v;
  u.i[0] = __builtin_amdgcn_readfirstlane(u.i[0]);
  u.i[1] = __builtin_amdgcn_readfirstlane(u.i[1]);
  return u.d;
}
__device__ __forceinline__ int cell_of(double x, double lo, double inv, int nc)
{
  int c = (int)floor((x - lo) * inv);
  return c < 0 ? 0 : (c >= nc ? nc - 1 : c);
}

// Pair predicate of the build contract: fl(fl(dx*dx) + fl(dy*dy)) <= rc2,
// evaluated without FMA contraction so that it rounds exactly like the
// CPU oracle.
__device__ __forceinline__ double dist2_nocontract(double dx, double dy)
{
  #pragma clang fp contract(off)
  const double a = dx * dx;
  const double b = dy * dy;
  return a + b;
}

// Segment of a tile: lanes whose particle sits in cell row `row`.
struct Seg {
  int row;
  double xmn, xmx, ymn, ymx;
};

// The event that owns key row `row` (wave-uniform): 0 for a single event,
// else a binary search over the batch's first rows.  Kernels then read that
// event's grid through a reference (scalar loads): a by-value copy selected
// between two sources cost the gradient walk 12 VGPRs and 64 bytes of
// scratch per lane (one wave less per SIMD).
__device__ __forceinline__ int event_index(const Grid* __restrict__ gp, const Grid& g0, int row)
{
  if (g0.nev <= 1) return 0;
  int lo = 0, hi = g0.nev - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (gp[mid].row0 <= row) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Walk the candidate spans of one tile segment.  `body(j)` is called with a
// wave-uniform sorted index j for every candidate in range of the segment's
// bounding box (rows ascending, cells ascending within a row).
template <class Body>
__device__ __forceinline__ void for_spans(const Grid& g, const int32_t* __restrict__ cell_off,
                                          const Seg& s, double rcs, Body&& body)
{
  const int ry0 = uni(cell_of(s.ymn - rcs, g.lo[1], g.inv_cell, g.nc[1]));
  const int ry1 = uni(cell_of(s.ymx + rcs, g.lo[1], g.inv_cell, g.nc[1]));
  for (int ry = ry0; ry <= ry1; ++ry) {
    const double ylo = g.lo[1] + ry * g.cell, yhi = ylo + g.cell;
    const double dy = fmax(0.0, fmax(ylo - s.ymx, s.ymn - yhi));
    if (dy > rcs) continue;
    const double hw = sqrt(fmax(rcs * rcs - dy * dy, 0.0));
    const int cx0 = cell_of(s.xmn - hw, g.lo[0], g.inv_cellx, g.nc[0]);
    const int cx1 = cell_of(s.xmx + hw, g.lo[0], g.inv_cellx, g.nc[0]);
    const int kr = (g.row0 + ry) * g.stride;
    const int beg = uni(cell_off[kr + cx0]);
    const int end = uni(cell_off[kr + cx1 + 1]);
    for (int j = beg; j < end; ++j) body(j);
  }
}

// Workgroups are dispatched round-robin over the chip's 8 XCDs, each with
// its own L2.  Remap the workgroup index so that every XCD walks one
// contiguous range of tiles (neighbouring tiles share most candidates).
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_tile(int bid, int nblk)
{
  const int x = bid % kXcds, r = bid / kXcds;
  const int per = nblk / kXcds, rem = nblk % kXcds;
  return x * per + (x < rem ? x : rem) + r;
}

// Hot pair kernels split a tile's flattened candidate list into `nslices`
// slices, each walked by one wave (the waves of one workgroup, or workgroups
// of one wave), so the work units are small enough to spread evenly over the
// chip's SIMDs even when there are few tiles.  Every wave of a tile computes
// the same segments and spans (wave-uniform values).

// Candidate run of cell row ry0 + r for a segment: [b, e) in sorted order
// (empty when r >= nrow or the row is out of reach).  Evaluated per lane.
__device__ __forceinline__ void row_run(const Grid& g, const int32_t* __restrict__ cell_off, const Seg& s,
                                        double rcs, int ry0, int nrow, int r, int& b, int& e)
{
  b = e = 0;
  if (r >= nrow) return;
  const int ry = ry0 + r;
  const double ylo = g.lo[1] + ry * g.cell, yhi = ylo + g.cell;
  const double dy = fmax(0.0, fmax(ylo - s.ymx, s.ymn - yhi));
  if (dy > rcs) return;
  const double hw = sqrt(fmax(rcs * rcs - dy * dy, 0.0));
  const int cx0 = cell_of(s.xmn - hw, g.lo[0], g.inv_cellx, g.nc[0]);
  const int cx1 = cell_of(s.xmx + hw, g.lo[0], g.inv_cellx, g.nc[0]);
  const int kr = (g.row0 + ry) * g.stride;
  b = cell_off[kr + cx0];
  e = cell_off[kr + cx1 + 1];
}

// The candidates of one slice of a segment that can be in range, in order,
// 64 cell rows' worth (the rows are resolved lane-parallel, lane r holding
// row r's run, so their cell offsets arrive with one vector load).  The
// slice's flattened list is taken in batches of 64, a candidate per lane:
// the lanes find their candidates' sorted indices, load their positions and
// keep those no farther than the cutoff from the segment's bounding box.  At
// the ends of the runs, which follow the cutoff disc only to a cell row, that
// drops one candidate in five (188,250 particles) at a 64th of the cost of
// meeting it in the walk, where it would still wait for its record.  The
// positions of a batch are requested before the one in hand is walked; they
// also bring the records' lines into the L2, which the walk's scalar loads
// would go past one by one.
struct RunCursor {
  // lane r: the flattened index of row r's first candidate, its sorted index, the run's length
  int first, run, len;
  int t, hi, step;                // wave-uniform: flattened index of the next batch's first candidate, the slice's
                                  // end, and how far apart its candidates are (1, or the number of slices)
  const double* pos;              // records with x, y in front
  int stride;
  const Seg* seg;
  double far2;                    // square of the cutoff with a margin for rounding
  uint64_t mask = 0;              // lanes of the batch in hand that are still to visit
  int j = 0;                      // their sorted indices
  bool ahead = false;             // a batch is requested: jn, vn, xn, yn
  int jn = 0;
  bool vn = false;
  double xn = 0.0, yn = 0.0;

  __device__ __forceinline__ void request()
  {
    ahead = t < hi;
    if (!ahead) return;
    const int q = t + step * (int)(threadIdx.x & (kWave - 1));
    vn = q < hi;
    jn = 0;
    for (uint64_t m = __ballot(len > 0 && first < t + kWave * step && first + len > t); m; m &= m - 1) {
      const int r = __builtin_ctzll(m);
      const int f = __builtin_amdgcn_readlane(first, r), l = __builtin_amdgcn_readlane(len, r);
      const int s = __builtin_amdgcn_readlane(run, r);
      if (q >= f && q < f + l) jn = s + q - f;
    }
    xn = pos[(size_t)jn * stride];
    yn = pos[(size_t)jn * stride + 1];
    t += kWave * step;
  }
  // the next candidate's sorted index (wave-uniform), -1 after the last
  __device__ __forceinline__ int next()
  {
    while (mask == 0) {
      if (!ahead) return -1;
      const double bx = fmax(fmax(seg->xmn - xn, xn - seg->xmx), 0.0);
      const double by = fmax(fmax(seg->ymn - yn, yn - seg->ymx), 0.0);
      mask = __ballot(vn && bx * bx + by * by <= far2);
      j = jn;
      request();
    }
    const int l = __builtin_ctzll(mask);
    mask &= mask - 1;
    return __builtin_amdgcn_readlane(j, l);
  }
};

// Slice `slice` of `nslices` of a segment's flattened candidate list (rows
// ascending, cells ascending within a row): every nslices-th candidate, so
// that the slices have equal shares of every row.  (Contiguous slices have
// equal shares of the list, but the first and the last have more of it out of
// range, and they are always the same SIMDs' waves: gradients of
// 188,250 particles 987 us contiguous, 965 dealt out.)
// KEEP: contiguous all the same (keep_order).  body(cursor) once per 64 cell
// rows that hold some of the slice.  Called with every lane of the wave
// active; body runs on every lane (wave-uniform control flow): a lane outside
// the segment stands at kFarAway, where every candidate's weight is 0.
template <int STRIDE, bool KEEP, class Body>
__device__ __forceinline__ void for_spans_slice(const Grid& g, const int32_t* __restrict__ cell_off,
                                                const double* __restrict__ cand, const Seg& s, double rc2, double rcs,
                                                int slice, int nslices, Body&& body)
{
  const int lane = threadIdx.x & (kWave - 1);
  const int ry0 = uni(cell_of(s.ymn - rcs, g.lo[1], g.inv_cell, g.nc[1]));
  const int ry1 = uni(cell_of(s.ymx + rcs, g.lo[1], g.inv_cell, g.nc[1]));
  const int nrow = ry1 - ry0 + 1;
  int b, e;
  row_run(g, cell_off, s, rcs, ry0, nrow, lane, b, e);
  int incl = wave_incl_scan_i(e - b);
  int tot = last_lane(incl);
  int lo = 0, hi = INT_MAX;
  if (KEEP) {
    for (int r0 = kWave; r0 < nrow; r0 += kWave) {     // more than 64 rows: rare
      int b2, e2;
      row_run(g, cell_off, s, rcs, ry0, nrow, r0 + lane, b2, e2);
      tot += last_lane(wave_incl_scan_i(e2 - b2));
    }
    lo = (int)(((long long)tot * slice) / nslices);
    hi = (int)(((long long)tot * (slice + 1)) / nslices);
  }
  int base = 0;
  for (int r0 = 0; r0 < nrow && base < hi; r0 += kWave) {
    if (r0 > 0) {
      row_run(g, cell_off, s, rcs, ry0, nrow, r0 + lane, b, e);
      incl = wave_incl_scan_i(e - b);
    }
    const int end = base + last_lane(incl);
    RunCursor c;
    c.run = b;
    c.len = e - b;
    c.first = base + incl - c.len;
    c.t = KEEP ? (lo > base ? lo : base) : base + slice;
    c.hi = hi < end ? hi : end;
    c.step = KEEP ? 1 : nslices;
    c.pos = cand;
    c.stride = STRIDE;
    c.seg = &s;
    c.far2 = rc2 * (1.0 + 1e-9);
    c.request();
    body(c);
    base = end;
  }
}

// Number of slices per tile for `ntiles` tiles on `simds` SIMDs: the
// smallest that gives near-whole rounds of single-wave work units and at
// least about four waves per SIMD (to hide load latency), at most 16.  An event
// is created with that count (ccake_event_pair_slices), and its buffer of partial
// sums sized for it.
inline int choose_slices(int ntiles, int simds)
{
  int best = 1;
  double best_score = -1.0;
  for (int s = 1; s <= 16; ++s) {
    const double w = (double)ntiles * s / (simds > 0 ? simds : 1);
    const double rounds = w <= 1.0 ? 1.0 : __builtin_ceil(w);
    const double score = (w / rounds) * (w < 4.0 ? w / 4.0 : 1.0);
    if (score > best_score + 1e-9) { best_score = score; best = s; }
  }
  return best;
}

// The gradient walk's waves are longer: 4 once they fill the SIMDs (188,250
// particles, 2,942 tiles: 965 us with 4, 974 with 8; 182,355 in six events:
// 349 against 369; 40,401 particles, 632 tiles: 96 us with 4, 89 with 8).
inline int grad_tile_waves(int waves, int ntiles, int simds) { return waves == 8 && ntiles >= simds ? 4 : waves; }

// An event (or batch) of at most a wave per SIMD (for_segments).
inline bool small_event(const ccake_event* ev, int ntiles) { return 8 * ntiles <= ev->dev->simds; }
// A small event or batch in FP64 whose freeze-out hypersurface is recorded
// (keep_order) has an order and a form of its pair sums of its own, kKeep, that
// of the hypersurfaces recorded so far: their divE column is the reciprocal of a
// difference, so another rounding of the sums moves its worst entries by 1e-11
// to 2e-9 after the 300 steps to freeze-out (10 events of 5,000 to 7,650
// particles), and they are compared entry by entry.  Events beyond that size
// have the common form.  While the waves do not fill the chip a pass is the
// latency of its setup and loads, and the shorter arithmetic gains little:
// smoothing and gradients of 7,650 particles take 31 and 48 us in this form,
// 30 and 40 in the other with 8 waves per tile.  The size is the one the event was
// created with: a batch stays with its form while its events retire.
inline bool keep_order(const ccake_event* ev)
{
  return ev->snaps && small_event(ev, (ev->n + kTile - 1) / kTile);
}
constexpr int kKeepSmoothWaves = 8, kKeepGradWaves = 4;

// Per-slice partial sums: part[(slice * nacc + f) * npad + k] for sorted
// position k (every tile lane, k < ntiles * 64 <= npad, has a slot).
constexpr int kMaxAcc = 17;
constexpr int kMaxSlices = 16;

// Hold values at this point of the program: what uses them is not scheduled
// above it, and the loads that made them are not sunk below it.
__device__ __forceinline__ void pin_vector(double& a, double& b)
{
#ifndef CCAKE_HOST_EMU
  asm volatile("" : "+v"(a), "+v"(b));
#endif
}
template <int NR>
__device__ __forceinline__ void pin_scalar(const double (&r)[NR])
{
#ifndef CCAKE_HOST_EMU
  __builtin_amdgcn_sched_barrier(0);
  #pragma unroll
  for (int q = 0; q < NR; ++q) asm volatile("" :: "s"(r[q]));
#endif
}

// One step of walk_records: the record `cur` is evaluated while the one at
// sorted index n is requested.  A wait on scalar loads covers every one in
// flight (they can return out of order), so the wait for `cur` is taken by its
// offsets, before the request (pin_vector), and the wait for `nxt` falls after
// the whole of this step's arithmetic (pin_scalar: the compiler would otherwise
// move its loads to their use in the next step).
template <int NR, int STRIDE, class Body>
__device__ __forceinline__ void walk_step(const double (&cur)[NR], double (&nxt)[NR], const double* __restrict__ cand,
                                          int n, double xi, double yi, Body&& body)
{
  double dx = xi - cur[0], dy = yi - cur[1];
  pin_vector(dx, dy);
  __builtin_amdgcn_sched_barrier(0);
  #pragma unroll
  for (int q = 0; q < NR; ++q) nxt[q] = cand[(size_t)n * STRIDE + q];
  __builtin_amdgcn_sched_barrier(0);
  body(cur, dx, dy, dist2_nocontract(dx, dy));
  pin_scalar<NR>(nxt);
}

// Walk the candidates of a cursor, their records in scalar registers, the next
// one requested ahead into the other of two register sets: with one set and a
// copy, the loads of a record cannot be issued before the last use of the one
// it replaces, and every candidate waits for its own loads.  body(c, dx, dy,
// r2) adds one candidate's terms.  IN_RANGE: only on the lanes that have it in
// range, one record after the other (for_tile_sums).
template <int NR, int STRIDE, bool IN_RANGE, class Body>
__device__ __forceinline__ void walk_records(const double* __restrict__ cand, double xi, double yi, double rc2,
                                             RunCursor& cur, Body&& body)
{
  if (IN_RANGE) {
    for (int j = cur.next(); j >= 0; j = cur.next()) {
      const double* c = cand + (size_t)j * STRIDE;
      const double dx = xi - c[0], dy = yi - c[1], r2 = dist2_nocontract(dx, dy);
      if (r2 <= rc2) body(c, dx, dy, r2);
    }
    return;
  }
  double a[NR], b[NR];
  int n = cur.next();             // the next record's index; past the last the one before stays (in bounds, unused)
  if (n < 0) return;
  #pragma unroll
  for (int q = 0; q < NR; ++q) a[q] = cand[(size_t)n * STRIDE + q];
  for (;;) {
    int j = cur.next();
    if (j >= 0) n = j;
    walk_step<NR, STRIDE>(a, b, cand, n, xi, yi, body);
    if (j < 0) break;
    j = cur.next();
    if (j >= 0) n = j;
    walk_step<NR, STRIDE>(b, a, cand, n, xi, yi, body);
    if (j < 0) break;
  }
}

// The sums acc[NACC] of a tile's walk.  walk(in_range) adds every candidate's
// terms to them: on every lane at first, the weight being 0 where the candidate
// is out of range.  0 times NaN or infinity is not 0, though, and a tile can
// hold targets that such a candidate has nothing to do with (out of its range,
// another event's); so where a sum is not finite, the walk is done again with
// each candidate's terms added by the lanes that have it in range alone.
// (Masking every candidate of every walk: 188,250 particles, smoothing 610 ->
// 649 us, gradients 965 -> 1,051; 7,650: 30 -> 37 and 50 -> 70.)
template <int NACC, class Walk>
__device__ __forceinline__ void for_tile_sums(double (&acc)[NACC], Walk&& walk)
{
  #pragma unroll
  for (int q = 0; q < NACC; ++q) acc[q] = 0.0;
  walk(std::false_type());
  double z = 0.0;                  // stays 0 while every sum is finite
  #pragma unroll
  for (int q = 0; q < NACC; ++q) z = fma(acc[q], 0.0, z);
  if (__ballot(z != 0.0) == 0ull) return;
  #pragma unroll
  for (int q = 0; q < NACC; ++q) acc[q] = 0.0;
  walk(std::true_type());
}

// q = r/h and 1/q from r^2: the hardware reciprocal square root
// (v_rsq_f64) of q^2 refined by one Newton step y <- y (3 - x y^2) / 2,
// relative error about 1e-14, which the pair sums tolerate.  1e-300 is added
// to q^2 so that coincident particles get q = 1e-150 (0 to rounding)
// instead of 0 * inf.  The pair predicate never uses it.
__device__ __forceinline__ void q_and_inverse(double r2, double hinv2, double& q, double& iq)
{
  const double x = fma(r2, hinv2, 1e-300);
  const double y = __builtin_amdgcn_rsq(x);
  const double hx = 0.5 * x;
  const double e = fma(-(hx * y), y, 1.5);
  iq = y * e;
  q = x * iq;
}

// Cubic spline in branch-free form (src/kernel.cpp:34-48 and 73-118, D = 2),
// with t = max(2 - q, 0) and u = max(1 - q, 0):
//   W      = norm2 * (t^3 - 4 u^3)       [4 - 6q^2 + 3q^3 for q < 1, since
//                                         norm / norm2 = 4; (2 - q)^3 for
//                                         1 <= q < 2; 0 beyond]
//   grad W = C * rel * (t^2 - 4 u^2) / q [4 - 3q for q < 1; (2 - q)^2 / q
//                                         for 1 <= q < 2; 0 beyond], with
//   C = kgrad / h^4 = -kgrad2 / (2 h^4), kgrad = -15/(14 pi), kgrad2 = 15/(7 pi).
// Non-neighbours weigh exactly 0 and the self pair (q = 0 to rounding)
// weighs W(0) and has zero gradient, so the pair loops need no selects.
__device__ __forceinline__ double spline_w(double q)
{
  const double t = fmax(2.0 - q, 0.0), u = fmax(1.0 - q, 0.0);
  return fma(-4.0, u * u * u, t * t * t);
}
__device__ __forceinline__ double spline_g(double q, double iq)
{
  const double t = fmax(2.0 - q, 0.0), u = fmax(1.0 - q, 0.0);
  return fma(-4.0, u * u, t * t) * iq;
}

// The same kernel arithmetic in fewer instructions, from r^2 and 1/h:
//   x = r^2 + 1e-300, y = v_rsq_f64(x), f = x y, e = 3 - f y (2 to the
//   instruction's error): f e = 2 r and y e = 2 / r
// is the Newton step of q_and_inverse without its two halvings, and with
//   t = clamp(1 - r / 2h), u = clamp(1 - r / h)   (to [0, 1], one instruction each)
// spline_g(q, 1/q) = 2 h (t^2 - u^2) (2 / r) and
// spline_w(q) = 8 (t^3 - (k u)^3), k = 2^(-1/3): the clamps make the cut at
// 2h and the switch at h.  The walks apply the factors 2 h and 8 once per
// particle.  A lane whose position is kFarAway weighs every candidate exactly 0
// (r^2 = 1e200 stays finite).
constexpr double kFarAway = 1e100;
constexpr double kSplineW = 8.0;                     // spline_w / spline_w8
__device__ __forceinline__ double clamp01(double v) { return fmin(fmax(v, 0.0), 1.0); }
// FORM of a walk: kExact with the arithmetic above; kKeep with that of
// q_and_inverse, spline_w and spline_g (keep_order); kSingle without the
// Newton step (pair_precision 1): y and f as they are, so r and 1/r instead of
// 2 r and 2 / r, with v_rsq_f64's relative error (5.2e-8 at most, 1.0e-8
// rms over 4M arguments: less than one rounding to single precision),
// everything else in FP64.  Single-precision arithmetic would not be faster: it
// issues at the FP64 rate here.  188,250 particles: smoothing 615 -> 580 us,
// gradients 970 -> 915 us (pair terms in FP32 with compensated sums: 548 and 990).
// The constants m4h and m2h (mk2h) are then twice as large, and the gradient's
// final factor.  kRoot: kSingle with r from v_sqrt_f64 where 1/r is not needed
// (many_neighbours): two instructions fewer, 188,250 particles 547 us.
// kSmall: kExact with the rows of a tile as one segment where that reaches less
// (for_segments), for events whose waves do not fill the SIMDs.
enum Form { kExact, kKeep, kSingle, kSmall, kRoot };
// kRoot's rule.  v_sqrt_f64 is as exact as v_rsq_f64 (2.7e-8 and 8.4e-9), but
// with its other errors the densities' are no longer the gradients', and where a
// lattice has few distances (v - v_a) grad W / sigma loses by that: a stage at 402
// neighbours has grad v off by 7.8e-9 instead of 5.4e-10.  They average out over
// many, and then what is left, the errors' mean with the weight that a pair's r
// has in a density or a gradient, is taken out by the constants: -3.3e-9 for
// v_sqrt_f64 (-3.1e-9 to -3.5e-9 for h from 0.1 to 1), 3.3e-9 for v_rsq_f64
// (2.5e-9 to 4.0e-9), as measured.  2,141 to 10,343 neighbours: sigma off by 1.9e-10
// to 1.3e-9 (kSingle 5.2e-9 to 6.9e-9), grad p 4.6e-10 to 2.1e-9 (6.3e-9 to 8.9e-9),
// grad v 4.8e-10 to 2.2e-9 (4.5e-10 to 2.2e-9).  So above 2,000, where smoothing is
// most of a step besides: 751,500 particles (10,326 neighbours) 7.6 -> 7.1 ms (8.0 in
// FP64, 7.2 with FP32 terms), gradients 12.2 (13.0; 12.6).  An event alone: a
// batch's mean says little of its events.
constexpr double kSqrtMean = -3.3e-9, kRsqMean = 3.3e-9;
constexpr int kManyNeighbours = 2000;
// 2 r of a pair; ir2 receives 2 / r (kSingle: r and 1 / r)
template <int FORM>
__device__ __forceinline__ double twice_r(double r2, double& ir2)
{
  const double x = r2 + 1e-300;
  const double y = __builtin_amdgcn_rsq(x);
  const double f = x * y;
  if (FORM == kSingle) {
    ir2 = y;
    return f;
  }
  const double e = fma(-f, y, 3.0);
  ir2 = y * e;
  return f * e;
}
// (t^2 - u^2) * 2 / r; m4h = -1 / (4 h), m2h = -1 / (2 h) (kSingle: twice those, and half the result)
template <int FORM = kExact>
__device__ __forceinline__ double spline_g2(double r2, double m4h, double m2h)
{
  double ir2;
  const double d = twice_r<FORM>(r2, ir2);
  const double t = clamp01(fma(d, m4h, 1.0)), u = clamp01(fma(d, m2h, 1.0));
  return fma(-u, u, t * t) * ir2;
}
// t^3 - (k u)^3
constexpr double kSplineK = 0.79370052598409973738;  // 2^(-1/3)
template <int FORM = kExact>
__device__ __forceinline__ double spline_w8(double r2, double m4h, double mk2h)
{
  double ir2, d;
  if (FORM == kRoot) d = __builtin_amdgcn_sqrt(r2);
  else d = twice_r<FORM>(r2, ir2);
  const double t = clamp01(fma(d, m4h, 1.0)), u = clamp01(fma(d, mk2h, kSplineK));
  return fma(-(u * u), u, (t * t) * t);
}

// The lanes' bounding box (wave-uniform).
__device__ __forceinline__ Seg box_of(int row, bool in, double xi, double yi)
{
  Seg s;
  s.row = row;
  s.xmn = wave_min_d(in ? xi : INFINITY);
  s.xmx = wave_max_d(in ? xi : -INFINITY);
  s.ymn = wave_min_d(in ? yi : INFINITY);
  s.ymx = wave_max_d(in ? yi : -INFINITY);
  return s;
}

// Iterate over the row segments of the tile owned by this wave.  `fn(seg,
// in_seg)` runs once per segment with in_seg true on the lanes of the segment.
// Sorted positions have ascending key rows, so a segment is a run of lanes.
// With rc > 0 (kSmall) the rows of a tile are one segment where that reaches less: when
// the area within rc of the tile's box is smaller than the rows' areas
// together (a tile of short rows, which its rows' walks would cover row by row
// with some of the lanes each).  A tile of two long rows is the end of one and
// the start of the next, far apart, and stays two segments, as do the rows of
// two events.  2,601 particles in rows of 51: smoothing 25 -> 18 us, gradients
// 28 -> 20; 30,300 in rows of 174, where few tiles hold more than two: 50 -> 52
// and 69 -> 71, for the boxes.  So only while 8 waves a tile fill no more than
// the SIMDs (small_event).
template <class Fn>
__device__ __forceinline__ void for_segments(const Grid* __restrict__ gp, const Grid& g0, double rc, bool act, int myrow,
                                             double xi, double yi, Fn&& fn)
{
  uint64_t todo = __ballot(act);
  bool whole = false;
  if (rc > 0.0 && todo) {
    const int l0 = __builtin_ctzll(todo), l1 = kWave - 1 - __builtin_clzll(todo);
    const int first = __builtin_amdgcn_readlane(myrow, l0), last = __builtin_amdgcn_readlane(myrow, l1);
    if (first != last && event_index(gp, g0, first) == event_index(gp, g0, last)) {
      double apart = 0.0;
      for (uint64_t t = todo; t;) {
        const int r = __builtin_amdgcn_readlane(myrow, __builtin_ctzll(t));
        const bool in = act && myrow == r;
        const Seg s = box_of(r, in, xi, yi);
        apart += (s.xmx - s.xmn + 2.0 * rc) * (s.ymx - s.ymn + 2.0 * rc);
        t &= ~__ballot(in);
      }
      const Seg s = box_of(first, act, xi, yi);
      whole = (s.xmx - s.xmn + 2.0 * rc) * (s.ymx - s.ymn + 2.0 * rc) < apart;
    }
  }
  while (todo) {
    const int r = __builtin_amdgcn_readlane(myrow, __builtin_ctzll(todo));
    const bool in = act && (whole || myrow == r);
    const Seg s = box_of(r, in, xi, yi);
    fn(s, in);
    todo &= ~__ballot(in);
  }
}

}  // namespace ccake

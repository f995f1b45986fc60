// The 3+1D Milne path (tau, x, y, eta_s; D = 3) on gfx950: the stages whose
// geometry or data layout differ from 2+1D.  The EoS inversion, the
// transport coefficients, the smoothing sum pass, the freeze-out status
// machine and the reductions are the 2+1D kernels (they are per particle and
// do not depend on D).
//
//   gamma and v          EoM_default::update_velocity (src/eom_default.cpp:17-38):
//                        gamma = sqrt(1 - u_cov . u), u_cov = (-u^x, -u^y, -tau^2 u^eta)
//   neighbour build      SystemState::reset_neighbour_list (src/system_state.cpp:650-719):
//                        isotropic radius 2 hT in (x, y, eta) (also with the factorized
//                        kernel, 689); cubic cells, key rows over (eta, y) cell pairs
//   smoothing            smooth_all_particle_fields / calculate_intial_sigma
//                        (src/sph_workstation.cpp:494-640) with SPHkernel<3>
//                        (src/kernel.cpp:10-118), or the factorized kernel
//                        W_2D(r_perp, hT) W_1D(|d eta|, hEta) (129-170, chosen at 502)
//   gradients            smooth_all_particle_gradients (796-986), D = 3, with the
//                        factorized gradKernel branch (843)
//   equations of motion  EoM_default::evaluate_time_derivatives (src/eom_default.cpp:211-869)
//                        and calculate_MRF_shear (882-1412) with the tau^2 metric factors
//                        and the delta_{i eta} terms (include/milne.hpp:85-107, 415-530,
//                        1093-1108), diffusion off
//   RK update            Evolver::step_rk (src/evolver.cpp:363-484), three positions and
//                        three velocity components
//
// The pair kernels are owner-computes without atomics, as in 2+1D, but in three
// dimensions a tile of 64 targets reaches 3.4 times the volume of one target's
// cutoff sphere (100,007 particles, 734 neighbours each), so at most 29 % of
// its lanes would have a pair.  A tile is 16 cell-sorted targets (43 %): lane l
// has target l % 16 and, of every four candidates, candidate l / 16.  A
// workgroup of W waves shares a tile's candidates and adds its sums in LDS.
// A tile segment is the set of targets in one (y, eta) cell row; the cell
// rows within reach of its bounding box are walked as x runs.
#include "pair_common.h"
#include <type_traits>

namespace ccake {

// ---------------------------------------------------------------------------
// Phase 02 with the (x, y, eta) bounding-box partials (six per workgroup).
__device__ __forceinline__ void gamma_v3(double* __restrict__ F, int npad, int i, double t2)
{
  auto col = [&](int c) -> double& { return F[(size_t)c * npad + i]; };
  const double ux = col(CCAKE_F_UX), uy = col(CCAKE_F_UY), ue = col(CCAKE_F_UETA);
  // milne::contract(u_cov, u), u_cov = (-u^x, -u^y, -tau^2 u^eta)
  double c = 0.0;
  c += (-ux) * ux;
  c += (-uy) * uy;
  c += (ue * -t2) * ue;
  const double g = sqrt(1.0 - c);
  col(CCAKE_F_GAMMA) = g;
  col(CCAKE_F_VX) = ux / g;
  col(CCAKE_F_VY) = uy / g;
  col(CCAKE_F_VETA) = ue / g;
}

__global__ __launch_bounds__(256) void k3_stage_begin(double* __restrict__ F, int npad, int n,
                                                      double* __restrict__ bbox_part, int do_gamma, double t2)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double mn[3] = { INFINITY, INFINITY, INFINITY }, mx[3] = { -INFINITY, -INFINITY, -INFINITY };
  if (i < n) {
    if (do_gamma) gamma_v3(F, npad, i, t2);
    const double r[3] = { F[(size_t)CCAKE_F_X * npad + i], F[(size_t)CCAKE_F_Y * npad + i],
                          F[(size_t)CCAKE_F_ETA * npad + i] };
    for (int d = 0; d < 3; ++d) mn[d] = mx[d] = r[d];
  }
  for (int o = 32; o > 0; o >>= 1)
    for (int d = 0; d < 3; ++d) { mn[d] = fmin(mn[d], __shfl_xor(mn[d], o)); mx[d] = fmax(mx[d], __shfl_xor(mx[d], o)); }
  __shared__ double s[4][6];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (l == 0) for (int d = 0; d < 3; ++d) { s[w][2 * d] = mn[d]; s[w][2 * d + 1] = mx[d]; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < 4; ++k)
      for (int d = 0; d < 3; ++d) { mn[d] = fmin(mn[d], s[k][2 * d]); mx[d] = fmax(mx[d], s[k][2 * d + 1]); }
    double* b = bbox_part + 6 * blockIdx.x;
    for (int d = 0; d < 3; ++d) { b[2 * d] = mn[d]; b[2 * d + 1] = mx[d]; }
  }
}

// A stage that keeps the cell sort: gamma, v and the smoothing record of
// particle perm[k] at sorted position k, and the stage's pair count cleared.
__global__ __launch_bounds__(256) void k3_stage_gather(double* __restrict__ F, int npad, int n,
                                                       const int32_t* __restrict__ perm, double* __restrict__ cand,
                                                       unsigned long long* __restrict__ pair_count, double t2)
{
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k == 0) pair_count[0] = 0ull;
  if (k >= n) return;
  const int i = perm[k];
  gamma_v3(F, npad, i, t2);
  smooth_record3(F, npad, i, cand + (size_t)k * kCandS);
}

// ---------------------------------------------------------------------------
// The pair predicate of the build contract in 3D:
// fl(fl(fl(dx*dx) + fl(dy*dy)) + fl(dz*dz)) <= rc2, no FMA contraction.
__device__ __forceinline__ double dist2_3(double dx, double dy, double dz)
{
  #pragma clang fp contract(off)
  const double a = dx * dx;
  const double b = dy * dy;
  const double c = dz * dz;
  return (a + b) + c;
}
__device__ __forceinline__ double dist2_perp(double dx, double dy)
{
  #pragma clang fp contract(off)
  const double a = dx * dx;
  const double b = dy * dy;
  return a + b;
}

struct Seg3 {
  int row;
  double mn[3], mx[3];
};

// The (y, eta) cell-row segments of the tile owned by this wave (runs of
// lanes: sorted positions have ascending key rows).
template <class Fn>
__device__ __forceinline__ void for_segments3(bool act, int myrow, const double* r, Fn&& fn)
{
  uint64_t todo = __ballot(act);
  while (todo) {
    Seg3 s;
    s.row = __builtin_amdgcn_readlane(myrow, __builtin_ctzll(todo));
    const bool in = act && myrow == s.row;
    #pragma unroll
    for (int d = 0; d < 3; ++d) {
      s.mn[d] = wave_min_d(in ? r[d] : INFINITY);
      s.mx[d] = wave_max_d(in ? r[d] : -INFINITY);
    }
    fn(s, in);
    todo &= ~__ballot(in);
  }
}

// Candidate run of flattened cell row r (y fastest) of a segment: [b, e)
// in sorted order, empty when r >= nrow or the row is out of reach.
__device__ __forceinline__ void row_run3(const Grid& g, const int32_t* __restrict__ cell_off, const Seg3& s,
                                         double rcs, int ry0, int nry, int rz0, int nrow, int r, int& b, int& e)
{
  b = e = 0;
  if (r >= nrow) return;
  const int ry = ry0 + r % nry, rz = rz0 + r / nry;
  const double ylo = g.lo[1] + ry * g.cell, yhi = ylo + g.cell;
  const double zlo = g.lo[2] + rz * g.cell, zhi = zlo + g.cell;
  const double dy = fmax(0.0, fmax(ylo - s.mx[1], s.mn[1] - yhi));
  const double dz = fmax(0.0, fmax(zlo - s.mx[2], s.mn[2] - zhi));
  const double d2 = dy * dy + dz * dz;
  if (d2 > rcs * rcs) return;
  const double hw = sqrt(fmax(rcs * rcs - d2, 0.0));
  const int cx0 = cell_of(s.mn[0] - hw, g.lo[0], g.inv_cellx, g.nc[0]);
  const int cx1 = cell_of(s.mx[0] + hw, g.lo[0], g.inv_cellx, g.nc[0]);
  const int kr = (rz * g.nc[1] + ry) * g.stride;
  b = cell_off[kr + cx0];
  e = cell_off[kr + cx1 + 1];
}

__device__ __forceinline__ void row_range3(const Grid& g, const Seg3& s, double rcs, int& ry0, int& nry, int& rz0,
                                           int& nrow)
{
  ry0 = uni(cell_of(s.mn[1] - rcs, g.lo[1], g.inv_cell, g.nc[1]));
  const int ry1 = uni(cell_of(s.mx[1] + rcs, g.lo[1], g.inv_cell, g.nc[1]));
  rz0 = uni(cell_of(s.mn[2] - rcs, g.lo[2], g.inv_cell, g.nc[2]));
  const int rz1 = uni(cell_of(s.mx[2] + rcs, g.lo[2], g.inv_cell, g.nc[2]));
  nry = ry1 - ry0 + 1;
  nrow = nry * (rz1 - rz0 + 1);
}

constexpr int kTile3 = 16;                            // targets of a tile
constexpr int kGroups3 = kWave / kTile3;              // candidates of a step
constexpr int kAhead3 = 4;                            // steps worked between two looks at the list
constexpr int kList3 = kWave + kGroups3 * kAhead3;    // entries of a wave's list

// What one lane of a wave wrote to LDS is there for the others.
__device__ __forceinline__ void wave_sync()
{
#ifdef CCAKE_HOST_EMU
  (void)__ballot(1);
#else
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#endif
}

// Wave `slice` of a tile's W waves walks its share of a segment's candidates
// (every W-th of the flattened list).  The list is taken in batches of 64, a
// candidate per lane, as RunCursor does in 2+1D: the lanes find their
// candidates' sorted indices, read NP doubles of their records, and those
// within the cutoff of the segment's bounding box are put into the wave's
// list in LDS: read(j, c) reads candidate j's entry (c[0..2] its position),
// put(e, c, j) writes it at e, move(from, to) moves one entry.  work(e,
// steps) does `steps` steps of four candidates from entry e on: kAhead3 at a
// time while the list holds as many, one at a time at the end, where
// pad(e) fills up the last four.  The next batch is read while a list is
// worked.
template <int W, int NP, class Read, class Put, class Move, class Pad, class Work>
__device__ __forceinline__ void walk_tile3(const Grid& g, const int32_t* __restrict__ cell_off, const Seg3& seg,
                                           double rc2, double rcs, int slice, Read&& read, Put&& put, Move&& move,
                                           Pad&& pad, Work&& work)
{
  const int lane = threadIdx.x & (kWave - 1);
  const double far2 = rc2 * (1.0 + 1e-9);             // margin for rounding
  int ry0, nry, rz0, nrow;
  row_range3(g, seg, rcs, ry0, nry, rz0, nrow);
  int fill = 0, base = 0;
  for (int r0 = 0; r0 < nrow; r0 += kWave) {
    int run, e;
    row_run3(g, cell_off, seg, rcs, ry0, nry, rz0, nrow, r0 + lane, run, e);
    const int len = e - run, incl = wave_incl_scan_i(len), first = base + incl - len;
    const int end = base + last_lane(incl);
    int t = base + slice, jn = 0;
    bool vn = false;
    double next[NP];
    auto request = [&]() -> bool {
      if (t >= end) return false;
      const int q = t + W * lane;
      vn = q < end;
      jn = 0;
      for (uint64_t m = __ballot(len > 0 && first < t + kWave * W && first + len > t); m; m &= m - 1) {
        const int r = __builtin_ctzll(m);
        const int f = __builtin_amdgcn_readlane(first, r), l = __builtin_amdgcn_readlane(len, r);
        const int s = __builtin_amdgcn_readlane(run, r);
        if (q >= f && q < f + l) jn = s + q - f;
      }
      read(jn, next);
      t += kWave * W;
      return true;
    };
    bool more = request();
    while (more) {
      double c[NP];
      #pragma unroll
      for (int q = 0; q < NP; ++q) c[q] = next[q];
      const int j = jn;
      double d2 = 0.0;
      #pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double x = fmax(fmax(seg.mn[d] - c[d], c[d] - seg.mx[d]), 0.0);
        d2 += x * x;
      }
      const bool keep = vn && d2 <= far2;
      const uint64_t mask = __ballot(keep);
      more = request();
      if (keep) put(fill + __popcll(mask & ((1ull << lane) - 1)), c, j);
      fill += __popcll(mask);
      wave_sync();
      int done = 0;
      for (; fill - done >= kGroups3 * kAhead3; done += kGroups3 * kAhead3) work(done, std::integral_constant<int, kAhead3>());
      if (done) {
        wave_sync();
        fill -= done;
        if (lane < fill) move(done + lane, lane);
        wave_sync();
      }
    }
    base = end;
  }
  if (fill) {
    const int whole = (fill + kGroups3 - 1) / kGroups3 * kGroups3;
    if (lane >= fill && lane < whole) pad(lane);
    wave_sync();
    for (int e = 0; e < whole; e += kGroups3) work(e, std::integral_constant<int, 1>());
    wave_sync();
  }
}

// Every candidate of a segment, one at a time (the export walk).
template <class Body>
__device__ __forceinline__ void for_spans3(const Grid& g, const int32_t* __restrict__ cell_off, const Seg3& s,
                                           double rcs, Body&& body)
{
  int ry0, nry, rz0, nrow;
  row_range3(g, s, rcs, ry0, nry, rz0, nrow);
  for (int r = 0; r < nrow; ++r) {
    int b, e;
    row_run3(g, cell_off, s, rcs, ry0, nry, rz0, nrow, r, b, e);
    b = uni(b); e = uni(e);
    for (int j = b; j < e; ++j) body(j);
  }
}

// Kernel constants of a 3+1D event.  Isotropic: W = norm2 w(q),
// grad W = C rel g(q) with q = r / hT (SPHkernel<3>: norm2 = 1/(4 pi hT^3),
// C = kgrad / hT^5 = -3/(4 pi hT^5)).  Factorized: W = norm2 w(q_perp) w(q_eta)
// (norm2 = 5/(14 pi hT^2) * 1/(6 hEta)), and with C = kgrad_2D / hT^4 *
// 1/(6 hEta) the gradient is C (rel_x g_perp w_eta, rel_y g_perp w_eta,
// kfac w_perp rel_eta g_eta), kfac = (5/(14 pi hT^2)) (-1/(2 hEta^3)) / C.
struct Kern3 {
  double norm2, C, kfac;
};
static Kern3 kern3(const ccake_params& p)
{
  Kern3 k;
  const double h = p.hT, he = p.hEta;
  if (p.factorized_kernel) {
    const double n2 = 5.0 / (14.0 * kPi) / (h * h), n1 = (1.0 / 6.0) / he;
    const double C2 = -15.0 / (14.0 * kPi) / pow(h, 4), C1 = -0.5 / pow(he, 3);
    k.norm2 = n2 * n1;
    k.C = C2 * n1;
    k.kfac = n2 * C1 / k.C;
  } else {
    k.norm2 = 1.0 / (4.0 * kPi) / pow(h, 3);
    k.C = -3.0 / (4.0 * kPi) / pow(h, 5);
    k.kfac = 1.0;
  }
  return k;
}

// The tile and the target of this lane.
struct Target3 {
  int tile, slice, i, group, k;      // k: sorted position
  bool act;
};
__device__ __forceinline__ Target3 target3(int n)
{
  Target3 t;
  const int lane = threadIdx.x & (kWave - 1);
  t.tile = xcd_tile(blockIdx.x, gridDim.x);
  t.slice = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);   // wave-uniform
  t.i = lane % kTile3;
  t.group = lane / kTile3;
  const int k = t.tile * kTile3 + t.i;
  t.act = k < n;
  t.k = t.act ? k : 0;
  return t;
}

// ---------------------------------------------------------------------------
// Smoothing, pair part: MODE 0 sigma_lab, s, B, S, Q and the neighbour count
// (6 sums); MODE 1 sigma_lab and the count (initial sigma); MODE 2 the count
// alone, written as btrack, and the pair total.  The sums go to `part` as
// those of a single slice, so k_smooth_sum reads them.
// Bound: the FP64 vector unit, 29 instructions per step of four candidates, and
// the list's reads from LDS (32 of its cycles a step, four SIMDs a CU).  A
// smoothing pass of 100,007 particles (73 M pairs): 363 us with 64 targets a
// tile and records in scalar registers, 212 us now.  MODE 2 the same way: the
// count walked one candidate at a time took 1.7 ms.  The register budget keeps the
// 5 waves per SIMD (4 in the other modes) that the walk has without its repeat for
// sums that are not finite (for_tile_sums).
template <int MODE, bool FACT, int W>
__global__ __launch_bounds__(kWave * W) __attribute__((amdgpu_waves_per_eu((MODE == 0 && !FACT) ? 5 : 4))) void k3_smooth_tile(const double* __restrict__ cand,
                                                            const int32_t* __restrict__ skey,
                                                            const int32_t* __restrict__ cell_off,
                                                            const Grid* __restrict__ gridp, int n, double rc2,
                                                            double rcs, double hinv, double heinv,
                                                            double* __restrict__ part, int npad,
                                                            const int32_t* __restrict__ perm,
                                                            int32_t* __restrict__ btrack,
                                                            unsigned long long* __restrict__ pair_total)
{
  constexpr int NACC = MODE == 0 ? 6 : (MODE == 1 ? 2 : 1);   // the count last
  constexpr int NP = MODE == 0 ? 8 : 4;
  __shared__ alignas(16) double list[W][kList3 * NP];
  static_assert(kList3 * NP >= NACC * kWave, "the lists are reused for the sums");
  const Grid& g = *gridp;
  const Target3 t = target3(n);
  const double* me = cand + (size_t)t.k * kCandS;
  const double r[3] = { me[0], me[1], me[2] };
  const int myrow = t.act ? skey[t.k] / g.stride : INT_MAX;
  const double m4h = -0.25 * hinv, mk2h = -0.5 * hinv * kSplineK;
  double* mine = list[t.slice];

  double acc[5];
  int cnt;
  for_tile_sums<5>(acc, [&](auto in_range) {
    cnt = 0;
    for_segments3(t.act, myrow, r, [&](const Seg3& seg, bool in) {
      const double xs = in ? r[0] : kFarAway;
      walk_tile3<W, NP>(g, cell_off, seg, rc2, rcs, t.slice,
        [&](int j, double (&c)[NP]) {
          #pragma unroll
          for (int q = 0; q < NP; ++q) c[q] = cand[(size_t)j * kCandS + q];
        },
        [&](int e, const double (&c)[NP], int) {
          #pragma unroll
          for (int q = 0; q < NP; ++q) mine[e * NP + q] = c[q];
        },
        [&](int from, int to) {
          #pragma unroll
          for (int q = 0; q < NP; ++q) mine[to * NP + q] = mine[from * NP + q];
        },
        [&](int e) {
          mine[e * NP] = -kFarAway;
          #pragma unroll
          for (int q = 1; q < NP; ++q) mine[e * NP + q] = 0.0;
        },
        [&](int e0, auto steps) {
          auto one = [&](int u) {
            const double* c = mine + (e0 + kGroups3 * u + t.group) * NP;
            const double dx = xs - c[0], dy = r[1] - c[1], dz = r[2] - c[2];
            const double r2 = dist2_3(dx, dy, dz);
            const bool nb = r2 <= rc2;
            cnt += nb ? 1 : 0;
            if (MODE == 2 || (decltype(in_range)::value && !nb)) return;
            double w;
            if (FACT) {
              double qp, iqp, qe, iqe;
              q_and_inverse(dist2_perp(dx, dy), hinv * hinv, qp, iqp);
              q_and_inverse(dz * dz, heinv * heinv, qe, iqe);
              w = nb ? spline_w(qp) * spline_w(qe) : 0.0;
            } else {
              w = spline_w8(r2, m4h, mk2h);
            }
            acc[0] += c[3] * w;
            if (MODE == 0) {
              #pragma unroll
              for (int q = 1; q < 5; ++q) acc[q] += c[MODE == 0 ? 3 + q : 0] * w;
            }
          };
          if (decltype(in_range)::value) {
            #pragma unroll 1
            for (int u = 0; u < decltype(steps)::value; ++u) one(u);
          } else {
            #pragma unroll
            for (int u = 0; u < decltype(steps)::value; ++u) one(u);
          }
        });
    });
  });
  // the four groups of the W waves, in order
  #pragma unroll
  for (int q = 0; q < NACC - 1; ++q) mine[q * kWave + (threadIdx.x & (kWave - 1))] = FACT ? acc[q] : kSplineW * acc[q];
  mine[(NACC - 1) * kWave + (threadIdx.x & (kWave - 1))] = (double)cnt;
  __syncthreads();
  unsigned long long tot = 0;
  for (int o = threadIdx.x; o < NACC * kTile3; o += kWave * W) {
    const int q = o / kTile3, i = o % kTile3;
    double s = 0.0;
    #pragma unroll
    for (int w = 0; w < W; ++w)
      #pragma unroll
      for (int h = 0; h < kGroups3; ++h) s += list[w][q * kWave + h * kTile3 + i];
    const int k = t.tile * kTile3 + i;
    if (MODE == 2) {
      if (k < n) {
        // without the particle itself (counted unless its position is not finite)
        const double* c = cand + (size_t)k * kCandS;
        const int nb = (int)s - (dist2_3(c[0] - c[0], c[1] - c[1], c[2] - c[2]) <= rc2 ? 1 : 0);
        const int id = perm[k];
        tot = nb;
        if (btrack[id] != -1) btrack[id] = nb;
      }
    } else {
      // columns sigma_lab, count, s, B, S, Q
      const int col = q == 0 ? 0 : (q == NACC - 1 ? 1 : q + 1);
      part[(size_t)col * npad + k] = s;
    }
  }
  if (MODE == 2 && pair_total && threadIdx.x < kWave) {
    for (int o = 32; o > 0; o >>= 1) tot += __shfl_xor(tot, o);
    if (threadIdx.x == 0) atomicAdd(pair_total, tot);
  }
}

// The pair rows (parity export) at the row offsets.
__global__ __launch_bounds__(64) void k3_export(const double* __restrict__ cand, const int32_t* __restrict__ skey,
                                                const int32_t* __restrict__ perm, const int32_t* __restrict__ cell_off,
                                                const Grid* __restrict__ gridp, int n, double rc2, double rcs,
                                                const int64_t* __restrict__ row_off, int32_t* __restrict__ out_i,
                                                int32_t* __restrict__ out_j)
{
  const Grid& g = *gridp;
  const int lane = threadIdx.x;
  const int k = blockIdx.x * kTile + lane;
  const bool act = k < n;
  const int kk = act ? k : 0;
  const double* me = cand + (size_t)kk * kCandS;
  const double r[3] = { me[0], me[1], me[2] };
  const int myrow = act ? skey[kk] / g.stride : INT_MAX;
  const int id = act ? perm[kk] : 0;
  int64_t wpos = act ? row_off[id] : 0;
  for_segments3(act, myrow, r, [&](const Seg3& seg, bool in) {
    for_spans3(g, cell_off, seg, rcs, [&](int j) {
      const double* c = cand + (size_t)j * kCandS;
      const double r2 = dist2_3(r[0] - c[0], r[1] - c[1], r[2] - c[2]);
      if (in && (r2 <= rc2) && (j != k)) { out_i[wpos] = id; out_j[wpos] = perm[j]; ++wpos; }
    });
  });
}

// ---------------------------------------------------------------------------
// Gradients.  Of a candidate's record the kernel sums, per target and with
// w_d = m_b d_d W_ab / C, the 3 x 16 products w_d f_j of the fields f_j =
// (p/sl^2, e, Pi/sl^2, v (3), pi^{0i}/sl^2 (3), pi^{ij}/sl^2 (6), 1): a matrix
// product of 16 targets by 16 fields over the candidates, which is what
// v_mfma_f64_16x16x4 does four candidates at a time.  39 of the 48 are needed
// (v_a is constant over b, so (w . v_a) pi^{0i} is a sum of them).
// FP64 matrix instructions run at the vector unit's rate (65 cycles, against 39
// vector instructions of 4), but each lane then needs one field of one
// candidate, one coalesced load a step, where lanes of four candidates
// would each read a whole record of 19 values; and the sums take 24 registers.
// Bound: the FP64 unit, 24 vector instructions and three matrix instructions
// (300 cycles) a step.  Gradients of 100,007 particles: 890 us with 64 targets a
// tile, vector sums and a sum pass over the slices, 390 us now.
typedef double Sums3 __attribute__((vector_size(4 * sizeof(double))));   // targets group + 4 r, field lane % 16
__device__ __forceinline__ void outer3(const double (&w)[3], double f, Sums3 (&acc)[3])
{
#ifdef CCAKE_HOST_EMU
  __shared__ double s[8][4][kWave];
  const int lane = threadIdx.x % kWave;
  auto& mine = s[threadIdx.x / kWave];
  for (int d = 0; d < 3; ++d) mine[d][lane] = w[d];
  mine[3][lane] = f;
  wave_sync();
  for (int d = 0; d < 3; ++d)
    for (int r = 0; r < 4; ++r)
      for (int k = 0; k < kGroups3; ++k)
        acc[d][r] += mine[d][lane / kTile3 + 4 * r + kTile3 * k] * mine[3][lane % kTile3 + kTile3 * k];
  wave_sync();
#else
  #pragma unroll
  for (int d = 0; d < 3; ++d) acc[d] = __builtin_amdgcn_mfma_f64_16x16x4f64(w[d], f, acc[d], 0, 0, 0);
#endif
}

// The same on the targets that have the candidate in range (`nb`, of this lane's
// target and candidate), and for_tile_sums for these sums.
__device__ __forceinline__ void outer3_in_range(const double (&w)[3], double f, bool nb, Sums3 (&acc)[3])
{
  const int lane = threadIdx.x & (kWave - 1);
  #pragma unroll 1
  for (int k = 0; k < kGroups3; ++k) {
    const double fk = __shfl(f, lane % kTile3 + kTile3 * k);
    #pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int from = lane / kTile3 + 4 * r + kTile3 * k;
      const int has = __shfl((int)nb, from);
      #pragma unroll
      for (int d = 0; d < 3; ++d) {
        const double wd = __shfl(w[d], from);
        if (has) acc[d][r] += wd * fk;
      }
    }
  }
}
template <class Walk>
__device__ __forceinline__ void for_tile_sums(Sums3 (&acc)[3], Walk&& walk)
{
  const Sums3 none = { 0.0, 0.0, 0.0, 0.0 };
  acc[0] = acc[1] = acc[2] = none;
  walk(std::false_type());
  double z = 0.0;
  #pragma unroll
  for (int q = 0; q < 12; ++q) z = fma(acc[q / 4][q % 4], 0.0, z);
  if (__ballot(z != 0.0) == 0ull) return;
  acc[0] = acc[1] = acc[2] = none;
  walk(std::true_type());
}

// The register budget: 4 waves per SIMD, as without the repeat (which would
// take 160 registers and leave 3).
template <bool SHEAR, bool FACT, int W>
__global__ __launch_bounds__(kWave * W) __attribute__((amdgpu_waves_per_eu(4))) void k3_grad_tile(const double* __restrict__ cand,
                                                          const int32_t* __restrict__ skey,
                                                          const int32_t* __restrict__ cell_off,
                                                          const Grid* __restrict__ gridp, int n, double rc2,
                                                          double rcs, double hinv, double heinv, double kfac, double C,
                                                          const int32_t* __restrict__ perm, int npad,
                                                          double* __restrict__ F)
{
  constexpr int NSUM = 3 * 16 * kTile3;               // a wave's sums: [direction][field][target]
  constexpr int NP = 4;                               // x, y, eta, m
  static_assert(NSUM >= kList3 * (NP + 1), "the lists are reused for the sums");
  __shared__ alignas(16) double buf[W][NSUM];
  const Grid& g = *gridp;
  const Target3 t = target3(n);
  const int lane = threadIdx.x & (kWave - 1);
  const double* me = cand + (size_t)t.k * kCandG3;
  const double r[3] = { me[0], me[1], me[2] };
  const int myrow = t.act ? skey[t.k] / g.stride : INT_MAX;
  const double m4h = -0.25 * hinv, m2h = -0.5 * hinv;
  double* pos = buf[t.slice];
  long long* off = reinterpret_cast<long long*>(buf[t.slice] + kList3 * NP);   // a record's first field
  const double* fields = cand + 4 + t.i;

  Sums3 acc[3];
  for_tile_sums(acc, [&](auto in_range) {
    for_segments3(t.act, myrow, r, [&](const Seg3& seg, bool in) {
      const double xs = in ? r[0] : kFarAway;
      walk_tile3<W, NP>(g, cell_off, seg, rc2, rcs, t.slice,
        [&](int j, double (&c)[NP]) {
          #pragma unroll
          for (int q = 0; q < NP; ++q) c[q] = cand[(size_t)j * kCandG3 + q];
        },
        [&](int e, const double (&c)[NP], int j) {
          #pragma unroll
          for (int q = 0; q < NP; ++q) pos[e * NP + q] = c[q];
          off[e] = (long long)j * kCandG3;
        },
        [&](int from, int to) {
          #pragma unroll
          for (int q = 0; q < NP; ++q) pos[to * NP + q] = pos[from * NP + q];
          off[to] = off[from];
        },
        [&](int e) {
          pos[e * NP] = -kFarAway;
          #pragma unroll
          for (int q = 1; q < NP; ++q) pos[e * NP + q] = 0.0;
          off[e] = off[0];
        },
        [&](int e0, auto steps) {
          constexpr int U = decltype(steps)::value;
          auto one = [&](int u, double f) {
            const double* c = pos + (e0 + kGroups3 * u + t.group) * NP;
            const double dx = xs - c[0], dy = r[1] - c[1], dz = r[2] - c[2];
            double w[3];
            if (FACT) {
              double qp, iqp, qe, iqe;
              q_and_inverse(dist2_perp(dx, dy), hinv * hinv, qp, iqp);
              q_and_inverse(dz * dz, heinv * heinv, qe, iqe);
              const double m = dist2_3(dx, dy, dz) <= rc2 ? c[3] : 0.0;
              const double gp = m * spline_g(qp, iqp) * spline_w(qe);
              w[0] = gp * dx; w[1] = gp * dy;
              w[2] = m * kfac * spline_w(qp) * spline_g(qe, iqe) * dz;
            } else {
              const double gm = c[3] * spline_g2(fma(dx, dx, fma(dy, dy, dz * dz)), m4h, m2h);
              w[0] = gm * dx; w[1] = gm * dy; w[2] = gm * dz;
            }
            if (decltype(in_range)::value) outer3_in_range(w, f, dist2_3(dx, dy, dz) <= rc2, acc);
            else outer3(w, f, acc);
          };
          if (decltype(in_range)::value) {
            #pragma unroll 1
            for (int u = 0; u < U; ++u) one(u, fields[off[e0 + kGroups3 * u + t.group]]);
            return;
          }
          double f[U];
          #pragma unroll
          for (int u = 0; u < U; ++u) f[u] = fields[off[e0 + kGroups3 * u + t.group]];
          #pragma unroll
          for (int u = 0; u < U; ++u) one(u, f[u]);
        });
    });
  });
  #pragma unroll
  for (int d = 0; d < 3; ++d)
    #pragma unroll
    for (int q = 0; q < 4; ++q) buf[t.slice][(d * 16 + lane % 16) * kTile3 + lane / 16 + 4 * q] = acc[d][q];
  __syncthreads();
  if (W > 1) {
    for (int o = threadIdx.x; o < NSUM; o += kWave * W) {
      double s = buf[0][o];
      #pragma unroll
      for (int w = 1; w < W; ++w) s += buf[w][o];
      buf[0][o] = s;
    }
    __syncthreads();
  }
  // the owner terms, a thread per target and direction, by particle id
  const int i = threadIdx.x % kTile3, d = threadIdx.x / kTile3, k = t.tile * kTile3 + i;
  if (d >= 3 || k >= n) return;
  const double scale = FACT ? C : C * (2.0 / hinv);   // spline_g = 2 h spline_g2
  auto sum = [&](int dir, int field) { return scale * buf[0][(dir * 16 + field) * kTile3 + i]; };
  const double* own = cand + (size_t)k * kCandG3;
  const int id = perm[k];
  auto put = [&](int c, double v) { F[(size_t)c * npad + id] = v; };
  const double sla = own[20], isla = 1.0 / sla;
  const double s1 = sum(d, 15);                       // sum w_d
  put(CCAKE_F_GRADP0 + d, sla * (sum(d, 0) + own[4] * s1));
  put(CCAKE_F_GRADE0 + d, (sum(d, 1) - own[5] * s1) * isla);
  put(CCAKE_F_GRADBULK0 + d, sla * (sum(d, 2) + own[6] * s1));
  #pragma unroll
  for (int e = 0; e < 3; ++e) put(CCAKE_F_GRADV0 + 3 * d + e, (sum(d, 3 + e) - own[7 + e] * s1) * isla);
  double gs = 0.0, ds = 0.0;
  if (SHEAR) {
    double cv = 0.0, c0 = 0.0, ci = 0.0, oi = 0.0;
    #pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double s = sum(a, 15);
      cv += s * own[7 + a];                           // sum w . v_a
      c0 += sum(a, 6 + d) * own[7 + a];               // sum (w . v_a) pi^{0d}
      // pi^{da}: (xx, xy, x eta, yy, y eta, eta eta)
      const int q = d < a ? d : a, p = 9 + q * (5 - q) / 2 + (d < a ? a : d);
      ci += sum(a, p);
      oi += own[4 + p] * s;
    }
    gs = sla * (c0 + own[10 + d] * cv);
    ds = sla * (ci + oi);
  }
  put(CCAKE_F_GRADSHEAR0 + d, gs);
  put(CCAKE_F_DIVSHEAR0 + d, ds);
}

// ---------------------------------------------------------------------------
// Equations of motion, D = 3 (diffusion off).  Milne helpers
// (include/milne.hpp): a D-vector is lowered by (-1, -1, -tau^2) and raised by
// (-1, -1, -1/tau^2); Matrix<4,4>::make_covariant(slot) flips slots 1, 2 and
// multiplies slot 3 by -tau^2; Matrix<D,D>::make_contravariant(0) flips rows
// 0, 1 and multiplies row 2 by -1/tau^2.
struct Col3 {
  double* F; int npad; int i;
  __device__ __forceinline__ double& operator()(int c) const { return F[(size_t)c * npad + i]; }
};

__device__ __forceinline__ void mat4_cov(double M[4][4], int slot, double t2)
{
  if (slot == 0) {
    #pragma unroll
    for (int j = 0; j < 4; ++j) { M[1][j] = -M[1][j]; M[2][j] = -M[2][j]; M[3][j] *= -t2; }
  } else {
    #pragma unroll
    for (int i = 0; i < 4; ++i) { M[i][1] = -M[i][1]; M[i][2] = -M[i][2]; M[i][3] *= -t2; }
  }
}

// milne::inverse of a 3x3 matrix (cofactors over the rule-of-Sarrus determinant).
__device__ __forceinline__ void inverse3(const double A[3][3], double R[3][3])
{
  const double det = A[0][0] * A[1][1] * A[2][2] + A[0][1] * A[1][2] * A[2][0] + A[0][2] * A[1][0] * A[2][1]
                   - A[0][2] * A[1][1] * A[2][0] - A[0][1] * A[1][0] * A[2][2] - A[0][0] * A[1][2] * A[2][1];
  R[0][0] = (A[1][1] * A[2][2] - A[1][2] * A[2][1]) / det;
  R[0][1] = (A[0][2] * A[2][1] - A[0][1] * A[2][2]) / det;
  R[0][2] = (A[0][1] * A[1][2] - A[0][2] * A[1][1]) / det;
  R[1][0] = (A[1][2] * A[2][0] - A[1][0] * A[2][2]) / det;
  R[1][1] = (A[0][0] * A[2][2] - A[0][2] * A[2][0]) / det;
  R[1][2] = (A[0][2] * A[1][0] - A[0][0] * A[1][2]) / det;
  R[2][0] = (A[1][0] * A[2][1] - A[1][1] * A[2][0]) / det;
  R[2][1] = (A[0][1] * A[2][0] - A[0][0] * A[2][1]) / det;
  R[2][2] = (A[0][0] * A[1][1] - A[0][1] * A[1][0]) / det;
}

template <bool SHEAR>
__device__ __forceinline__ void eom_d3(const Col3& col, double t, double use_vort, double du_dt[3], double* d_s,
                                       double dN[3], double* d_b, double dshv[5], double* theta_out,
                                       double* snu_out, double* dez_out)
{
  const double t2 = t * t;
  const double cmd[4] = { 1.0, -1.0, -1.0, -1.0 / t / t };   // get_contra_metric_diagonal<3>
  const double dl[3] = { 0.0, 0.0, 1.0 };                     // delta_i_eta<3>
  const double gamma = col(CCAKE_F_GAMMA), sigma = col(CCAKE_F_SIGMA), bulk = col(CCAKE_F_BULK);
  const double T = col(CCAKE_F_T), w = col(CCAKE_F_W), s = col(CCAKE_F_S);
  const double dwds = col(CCAKE_F_DWDS);
  const double mu[3] = { col(CCAKE_F_MUB), col(CCAKE_F_MUS), col(CCAKE_F_MUQ) };
  const double rho[3] = { col(CCAKE_F_RHOB), col(CCAKE_F_RHOS), col(CCAKE_F_RHOQ) };
  const double dwdr[3] = { col(CCAKE_F_DWDB), col(CCAKE_F_DWDS_S), col(CCAKE_F_DWDQ) };
  const double zeta = col(CCAKE_F_ZETA_PI), tau_Pi = col(CCAKE_F_TAU_BULK);
  const double delta_PiPi = col(CCAKE_F_DELTA_BB), lambda_Pipi = col(CCAKE_F_LAMBDA_BPI);
  const double phi1 = col(CCAKE_F_PHI1), phi3 = col(CCAKE_F_PHI3);

  const double u[3] = { col(CCAKE_F_UX), col(CCAKE_F_UY), col(CCAKE_F_UETA) };
  const double v[3] = { col(CCAKE_F_VX), col(CCAKE_F_VY), col(CCAKE_F_VETA) };
  const double uc[3] = { -u[0], -u[1], u[2] * -t2 };            // u_cov (also the fixed-size u_cov)
  double gradV[3][3], divV = 0.0;
  #pragma unroll
  for (int a = 0; a < 3; ++a) {
    divV += col(CCAKE_F_GRADV0 + 4 * a);
    #pragma unroll
    for (int b = 0; b < 3; ++b) gradV[a][b] = col(CCAKE_F_GRADV0 + 3 * a + b);
  }
  const double gf = dl[2] * u[2] * u[2] * t / gamma;          // geometric_factor
  const double expf = gf + gamma / t + gamma * divV;
  double S[4][4], H[4][4], C[4][4];
  #pragma unroll
  for (int a = 0; a < 4; ++a)
    #pragma unroll
    for (int b = 0; b < 4; ++b) S[a][b] = col(CCAKE_F_SHV0 + 4 * a + b);
  #pragma unroll
  for (int a = 0; a < 4; ++a)
    #pragma unroll
    for (int b = 0; b < 4; ++b) H[a][b] = S[a][b];
  mat4_cov(H, 1, t2);
  #pragma unroll
  for (int a = 0; a < 4; ++a)
    #pragma unroll
    for (int b = 0; b < 4; ++b) C[a][b] = H[a][b];
  mat4_cov(C, 0, t2);
  double shv_shvcov = 0.0;
  #pragma unroll
  for (int a = 0; a < 4; ++a)
    #pragma unroll
    for (int b = 0; b < 4; ++b) shv_shvcov += S[a][b] * C[a][b];

  // ---------------- calculate_MRF_shear (src/eom_default.cpp:882-1412) ----------------
  double M_snu[3] = { 0, 0, 0 }, F_snu = 0.0;
  double F_0i[3] = { 0, 0, 0 }, M_0i[3][3] = { { 0 } };
  double F_es[2][3] = { { 0 } }, M_es[2][3][3] = { { { 0 } } };
  if (SHEAR) {
    const double eta_pi = col(CCAKE_F_ETA_PI), tau_pi = col(CCAKE_F_TAU_PI);
    const double delta_pipi = col(CCAKE_F_DELTA_PIPI), lambda_piPi = col(CCAKE_F_LAMBDA_PIB);
    const double phi6 = col(CCAKE_F_PHI6), phi7 = col(CCAKE_F_PHI7), tau_pipi = col(CCAKE_F_TAU_PIPI);
    double guj[3][3], gu0[3];
    #pragma unroll
    for (int a = 0; a < 3; ++a)
      #pragma unroll
      for (int b = 0; b < 3; ++b) {
        double x = gamma * gradV[a][b];
        #pragma unroll
        for (int k = 0; k < 3; ++k) x += -gamma * u[b] * uc[k] * gradV[a][k];
        guj[a][b] = x;
      }
    #pragma unroll
    for (int a = 0; a < 3; ++a) {
      double c = 0.0;
      #pragma unroll
      for (int b = 0; b < 3; ++b) c += guj[a][b] * uc[b];
      gu0[a] = -1. * c / gamma;
    }
    const double gu0c[3] = { -gu0[0], -gu0[1], gu0[2] * (-1.0 / t2) };
    double cg[3][3];                                            // contra_grad_uj
    #pragma unroll
    for (int b = 0; b < 3; ++b) { cg[0][b] = -guj[0][b]; cg[1][b] = -guj[1][b]; cg[2][b] = guj[2][b] * (-1.0 / t2); }
    double guv[3] = { 0, 0, 0 };                                // contract(grad_uj, v, FirstIndex)
    #pragma unroll
    for (int b = 0; b < 3; ++b)
      #pragma unroll
      for (int a = 0; a < 3; ++a) guv[b] += guj[a][b] * v[a];
    double gu0v = 0.0;
    #pragma unroll
    for (int a = 0; a < 3; ++a) gu0v += gu0[a] * v[a];
    double vgs[3] = { 0, 0, 0 }, gugs[3] = { 0, 0, 0 }, sgui[3] = { 0, 0, 0 }, vsgu[3] = { 0, 0, 0 };
    #pragma unroll
    for (int a = 0; a < 3; ++a) {
      #pragma unroll
      for (int b = 0; b < 3; ++b) vgs[a] += guv[b] * H[a + 1][b + 1];
      vgs[a] += gu0v * H[a + 1][0];
      #pragma unroll
      for (int b = 0; b < 3; ++b) gugs[a] += cg[a][b] * H[0][b + 1];
      gugs[a] += cmd[a + 1] * gu0[a] * H[0][0];
      #pragma unroll
      for (int b = 0; b < 3; ++b) sgui[a] += S[b + 1][0] * guj[b][a] + S[b + 1][a + 1] * gu0[b];
      #pragma unroll
      for (int b = 0; b < 3; ++b) vsgu[a] += v[b] * S[0][0] * guj[b][a] + v[b] * S[0][a + 1] * gu0[b];
    }
    double sgu = 0.0;                                           // shv_grad_u
    #pragma unroll
    for (int a = 0; a < 3; ++a) {
      #pragma unroll
      for (int b = 0; b < 3; ++b) sgu += (H[a + 1][b + 1] - v[a] * H[0][b + 1]) * guj[a][b];
      sgu += (H[a + 1][0] - v[a] * H[0][0]) * gu0[a];
    }
    double sl0l[3] = { 0, 0, 0 };
    #pragma unroll
    for (int a = 0; a < 3; ++a)
      #pragma unroll
      for (int b = 0; b < 4; ++b) sl0l[a] += (S[0][b] * H[a + 1][b] + S[a + 1][b] * H[0][b]) / 2.;
    const double uD = u[2];
    #pragma unroll
    for (int a = 0; a < 3; ++a) {
      double Fsig = -(guv[a] - gu0c[a]) / 2. + u[a] * gamma * (gf + gamma / t + gamma * divV) / 3.
                  - gamma * gf * u[a] / 2.;
      double FD = gamma * (u[a] * H[0][0] + gamma * H[a + 1][0]) * gf + t * uD * S[3][a + 1] * dl[a];
      double Fds = -(vgs[a] - gugs[a] - 4. * gamma * u[a] * sgu / 3. - sgui[a] + vsgu[a]) / 4.
                 + (H[a + 1][0] - gamma * gamma * H[a + 1][0] - gamma * u[a] * H[0][0] + S[0][a + 1]
                    + 4. * u[a] * gamma * H[0][0] / 3.) * gf / 4.
                 + (gamma * cmd[a + 1] * H[0][3] * dl[a] / t + gamma * S[3][0] * dl[a] / t
                    + 4. * gamma * u[a] * (gamma * H[3][3] / t) / 3.) / 4.
                 - S[0][a + 1] * (gamma / t + gf + gamma * divV) / 3.;
      double Fdo = -(vgs[a] - gugs[a] + sgui[a] - vsgu[a]) / 4.
                 + (H[a + 1][0] - gamma * gamma * H[a + 1][0] - gamma * u[a] * H[0][0] - S[0][a + 1]) * gf / 4.
                 + (gamma * cmd[a + 1] * H[0][3] * dl[a] / t - gamma * S[3][0] * dl[a] / t) / 4.;
      const double Fdd = S[a + 1][0] * expf;
      double Msig[3], MD[3], Mds[3], Mdo[3], Mdd[3];
      #pragma unroll
      for (int b = 0; b < 3; ++b) {
        Msig[b] = u[a] * uc[b] / (2. * 3.);
        MD[b] = gamma * u[a] * (H[0][b + 1] - H[0][0] * uc[b] / gamma)
              + gamma * gamma * (H[a + 1][b + 1] - H[a + 1][0] * uc[b] / gamma);
        Mds[b] = (H[a + 1][b + 1] - H[a + 1][0] * uc[b] / gamma - gamma * gamma * H[a + 1][b + 1]
                  - gamma * u[a] * H[0][b + 1] + uc[b] * gamma * H[a + 1][0] + uc[b] * u[a] * H[0][0]
                  + 4. * gamma * u[a] * (H[0][b + 1] - H[0][0] * uc[b] / gamma) / 3.
                  + (-S[0][a + 1] + 4. * S[0][a + 1] / 3.) * uc[b] / gamma) / 4.;
        Mdo[b] = (H[a + 1][b + 1] - H[a + 1][0] * uc[b] / gamma - gamma * gamma * H[a + 1][b + 1]
                  - gamma * u[a] * H[0][b + 1] + uc[b] * gamma * H[a + 1][0] + uc[b] * u[a] * H[0][0]
                  + S[0][a + 1] * uc[b] / gamma) / 4.;
        Mdd[b] = -S[a + 1][0] * uc[b] / gamma;
      }
      Msig[a] += (1. - gamma * gamma) / 2.;
      Mdo[a] += -S[0][0] / 4.;
      Mds[a] += +S[0][0] / 4.;
      // metric-only terms
      Fsig += dl[a] * (-(-uD * t - uD / t + gamma * uD * uD * t + 2. * gamma * gamma * uD / t) / 2.);
      FD += dl[a] * (uD * S[0][0] / t + gamma * S[3][0] / t);
      Fds += (t * uD * dl[a] * cmd[a + 1] * H[0][0] + uD * H[a + 1][3] * gamma / t / 4. + H[a + 1][3] * t * uD
              + S[0][0] * dl[a] * uD / t + t * uD * uD * (gamma * H[a + 1][0] + u[a] * H[0][0])
              + 2. * gamma * uD * (gamma * H[a + 1][3] + u[a] * S[0][3]) / t) / 4.
           + gamma * u[a] * (H[3][0] * uD * t + uD * H[0][3] / t) / 3.;
      Fdo += (t * uD * dl[a] * cmd[a + 1] * H[0][0] + uD * H[a + 1][3] * gamma / t - H[3][a + 1] * t * uD
              - S[0][0] * dl[a] * uD / t + t * uD * uD * (gamma * H[a + 1][0] + u[a] * H[0][0])
              + 2. * gamma * uD * (gamma * H[a + 1][3] + u[a] * S[0][3]) / t) / 4.;
      F_0i[a] = (-S[a + 1][0] - tau_pi * FD - delta_pipi * Fdd + 2. * tau_pi * Fdo * use_vort - tau_pipi * Fds
                 + (2. * eta_pi + lambda_piPi * bulk) * Fsig + phi6 * bulk * S[a + 1][0]
                 + phi7 * (sl0l[a] + gamma * u[a] * shv_shvcov / 3.)) / (tau_pi * gamma);
      #pragma unroll
      for (int b = 0; b < 3; ++b)
        M_0i[a][b] = (-tau_pi * MD[b] - delta_pipi * Mdd[b] + 2. * tau_pi * Mdo[b] * use_vort - tau_pipi * Mds[b]
                      + (2. * eta_pi + lambda_piPi * bulk) * Msig[b]) / (tau_pi * gamma);
    }
    // shv_nabla_u = pi^{ij} nabla_i u_j
    #pragma unroll
    for (int a = 0; a < 3; ++a) {
      M_snu[a] = H[0][a + 1] - H[0][0] * uc[a] / gamma;
      #pragma unroll
      for (int b = 0; b < 3; ++b) F_snu += (H[a + 1][b + 1] - v[a] * H[0][b + 1]) * guj[a][b];
      F_snu += (H[a + 1][0] - v[a] * H[0][0]) * gu0[a];
    }
    F_snu += +H[3][3] * gamma / t + H[0][0] * gf + (t * H[3][0] + H[0][3] / t) * u[2] * dl[2];

    // extensive-shear MRFs, components (a, b) = (0,0), (0,1), (0,2), (1,1), (1,2)
    const double tilde_delta = delta_pipi - tau_pi;
    #pragma unroll
    for (int a = 0; a < 2; ++a) {
      double FDm[3] = { 0, 0, 0 }, Fsm[3] = { 0, 0, 0 }, Fdl[3] = { 0, 0, 0 }, Fdom[3] = { 0, 0, 0 },
             Fdsm[3] = { 0, 0, 0 };
      double MDm[3][3] = { { 0 } }, Msm[3][3] = { { 0 } }, Mdl[3][3] = { { 0 } }, Mdom[3][3] = { { 0 } },
             Mdsm[3][3] = { { 0 } };
      double sls[3] = { 0, 0, 0 };
      #pragma unroll
      for (int b = a; b < 3; ++b) {
        double gugj = 0.0, sgu2 = 0.0, vsg = 0.0;
        #pragma unroll
        for (int k = 0; k < 3; ++k) {
          gugj += cg[a][k] * H[b + 1][k + 1] + cg[b][k] * H[a + 1][k + 1];
          sgu2 += S[k + 1][a + 1] * guj[k][b] + S[k + 1][b + 1] * guj[k][a];
          vsg += v[k] * S[0][a + 1] * guj[k][b] + v[k] * S[0][b + 1] * guj[k][a];
        }
        #pragma unroll
        for (int k = 0; k < 4; ++k) sls[b] += (S[a + 1][k] * H[b + 1][k] + S[b + 1][k] * H[a + 1][k]) / 2.;
        FDm[b] = gamma * gf * (u[a] * H[b + 1][0] + u[b] * H[a + 1][0]);
        Fsm[b] = cg[a][b] / 2. + cg[b][a] / 2. + u[a] * u[b] * expf / 3.;
        Fdl[b] = S[a + 1][b + 1] * expf;
        const double metric_terms =
            t * u[2] * (cmd[a + 1] * H[b + 1][0] * dl[a] + cmd[b + 1] * H[a + 1][0] * dl[b])
          + gamma * (cmd[a + 1] * H[b + 1][3] * dl[a] + cmd[b + 1] * H[a + 1][3] * dl[b]) / t
          + u[2] * u[2] * t * (u[a] * H[b + 1][0] + u[b] * H[a + 1][0])
          + 2. * gamma * u[2] * (u[a] * H[b + 1][3] + u[b] * H[a + 1][3]) / t;
        Fdom[b] = -(-gugj + sgu2 - vsg) / 4.
                + (-u[a] * gamma * H[b + 1][0] - u[b] * gamma * H[a + 1][0]) * gf / 4.
                + (metric_terms - gamma * (S[3][a + 1] * dl[b] + S[3][b + 1] * dl[a]) / t
                   - u[2] * (S[0][a + 1] * dl[b] + S[0][b + 1] * dl[a]) / t) / 4.;
        Fdsm[b] = -(-gugj - sgu2 + vsg - 4. * (u[a] * u[b]) * sgu / 3.) / 4.
                + (-u[a] * gamma * H[b + 1][0] - u[b] * gamma * H[a + 1][0] + 4. * u[a] * u[b] * H[0][0] / 3.) * gf / 4.
                + (metric_terms + gamma * (S[3][a + 1] * dl[b] + S[3][b + 1] * dl[a]) / t
                   + u[2] * (S[0][a + 1] * dl[b] + S[0][b + 1] * dl[a]) / t
                   + 4. * u[a] * u[b] * (H[3][0] * u[2] * t + gamma * H[3][3] / t + u[2] * H[0][3] / t) / 3.) / 4.
                - S[a + 1][b + 1] * (gamma / t + gf + gamma * divV) / 3.;
        #pragma unroll
        for (int k = 0; k < 3; ++k) {
          MDm[b][k] = gamma * (u[a] * H[b + 1][k + 1] - u[a] * H[b + 1][0] * uc[k] / gamma
                               + u[b] * H[a + 1][k + 1] - u[b] * H[a + 1][0] * uc[k] / gamma);
          Msm[b][k] = -u[a] * u[b] * uc[k] / (3. * gamma);
          Mdl[b][k] = -S[a + 1][b + 1] * uc[k] / gamma;
          Mdom[b][k] = (-u[a] * H[b + 1][k + 1] * gamma - u[b] * H[a + 1][k + 1] * gamma
                        + uc[k] * u[a] * H[b + 1][0] + uc[k] * u[b] * H[a + 1][0]) / 4.;
          Mdsm[b][k] = (-u[a] * H[b + 1][k + 1] * gamma - u[b] * H[a + 1][k + 1] * gamma
                        + uc[k] * u[a] * H[b + 1][0] + uc[k] * u[b] * H[a + 1][0]
                        + 4. * u[a] * u[b] * (H[0][k + 1] - H[0][0] * uc[k] / gamma) / 3.
                        + 4. * S[a + 1][b + 1] * uc[k] / 3. / gamma) / 4.;
        }
        Mdsm[b][a] += S[0][b + 1] / 4.;
        Mdom[b][a] += -S[0][b + 1] / 4.;
        Msm[b][a] += -gamma * u[b] / 2.;
      }
      #pragma unroll
      for (int b = a; b < 3; ++b) {
        Msm[b][b] += -gamma * u[a] / 2.;
        Mdsm[b][b] += S[0][a + 1] / 4.;
        Mdom[b][b] += -S[0][a + 1] / 4.;
      }
      #pragma unroll
      for (int k = 0; k < 3; ++k) {
        Msm[a][k] += cmd[a + 1] * uc[k] / (gamma * 3.);
        Mdsm[a][k] += -cmd[a + 1] * (H[0][k + 1] - H[0][0] * uc[k] / gamma) / 3.;
      }
      const double ueta = u[2];
      FDm[2] += gamma * S[3][a + 1] / t + ueta * S[0][a + 1] / t;
      Fsm[a] += -cmd[a + 1] * expf / 3.;
      Fsm[2] += -u[a] * ueta * ueta * t / 2. - u[a] * ueta * gamma / t;
      Fdsm[a] += -cmd[a + 1] * sgu / 3. - cmd[a + 1] * H[0][0] * gf / 3.
                 - cmd[a + 1] * (H[3][0] * u[2] * t + gamma * H[3][3] / t + u[2] * H[0][3] / t) / 3.;
      #pragma unroll
      for (int b = a; b < 3; ++b) {
        F_es[a][b] = (-S[a + 1][b + 1] - tilde_delta * Fdl[b] - tau_pi * FDm[b] + 2. * tau_pi * Fdom[b] * use_vort
                      - tau_pipi * Fdsm[b] + (2. * eta_pi + lambda_piPi * bulk) * Fsm[b] + phi6 * bulk * S[a + 1][b + 1]
                      + phi7 * (sls[b] + u[a] * u[b] * shv_shvcov / 3.)) / (sigma * tau_pi * gamma);
        #pragma unroll
        for (int k = 0; k < 3; ++k)
          M_es[a][b][k] = (-tau_pi * MDm[b][k] - tilde_delta * Mdl[b][k] + 2. * tau_pi * Mdom[b][k] * use_vort
                           - tau_pipi * Mdsm[b][k] + (2. * eta_pi + lambda_piPi * bulk) * Msm[b][k])
                        / (sigma * tau_pi * gamma);
      }
      F_es[a][a] += phi7 * (-cmd[a + 1] * shv_shvcov) / (3. * tau_pi * gamma * sigma);
    }
  }

  // ---------------- fill_auxiliary_variables (230-362) ----------------
  const double zeta_tilde = zeta + (delta_PiPi - tau_Pi) * bulk;
  double M_eb[3], M_S[3];
  #pragma unroll
  for (int a = 0; a < 3; ++a) {
    M_eb[a] = (zeta_tilde * uc[a] / gamma) / (sigma * gamma * tau_Pi);
    M_S[a] = (bulk * uc[a] / gamma) / (sigma * gamma * T);
  }
  double R_S[3];
  #pragma unroll
  for (int c = 0; c < 3; ++c) R_S[c] = -mu[c] / T;
  double F_eb = -(zeta_tilde * (gamma * divV + gamma / t + gf) + bulk - phi1 * bulk * bulk) / (sigma * gamma * tau_Pi);
  double F_S = (-bulk * (gamma * divV + gamma / t + gf)) / (sigma * gamma * T);
  if (SHEAR) {
    F_S += F_snu / (sigma * gamma * T);
    F_eb += -(lambda_Pipi * F_snu - phi3 * shv_shvcov) / (sigma * gamma * tau_Pi);
    #pragma unroll
    for (int a = 0; a < 3; ++a) {
      M_eb[a] += -lambda_Pipi * M_snu[a] / (sigma * gamma * tau_Pi);
      M_S[a] += M_snu[a] / (sigma * gamma * T);
    }
  }

  // ---------------- compute_charge_derivative (369-453), diffusion off ----------------
  // R_N = gamma sigma I, F_N = 0 (no sources), M_N = 0: dN/dt = 0.

  // ---------------- compute_velocity_derivative (459-618) ----------------
  const double gP[3] = { -col(CCAKE_F_GRADP0), -col(CCAKE_F_GRADP0 + 1), col(CCAKE_F_GRADP0 + 2) * (-1.0 / t2) };
  const double gB[3] = { -col(CCAKE_F_GRADBULK0), -col(CCAKE_F_GRADBULK0 + 1),
                         col(CCAKE_F_GRADBULK0 + 2) * (-1.0 / t2) };
  const double rdw = rho[0] * dwdr[0] + rho[1] * dwdr[1] + rho[2] * dwdr[2];
  double M_w[3], R_w[3];
  #pragma unroll
  for (int a = 0; a < 3; ++a) M_w[a] = (s * dwds / gamma + rdw / gamma) * uc[a] / gamma + sigma * dwds * M_S[a];
  #pragma unroll
  for (int c = 0; c < 3; ++c) R_w[c] = sigma * dwdr[c] + sigma * dwds * R_S[c];
  (void)R_w;   // R_u R_N^{-1} multiplies M_N = 0 and F_N = 0 without diffusion
  double F_S_ex = F_S;
  const double F_w = -(s * dwds / gamma + rdw / gamma) * (gf + gamma / t + gamma * divV) + sigma * dwds * F_S_ex;
  const double F_bulk = sigma * F_eb - bulk * (gamma * divV + gamma / t + gf) / gamma;
  double M_u[3][3], F_u[3];
  #pragma unroll
  for (int a = 0; a < 3; ++a) {
    #pragma unroll
    for (int b = 0; b < 3; ++b) M_u[a][b] = u[a] * gamma * (M_eb[b] + M_w[b]) - u[a] * uc[b] * (w + bulk) / gamma;
    M_u[a][a] += gamma * (w + bulk);
  }
  #pragma unroll
  for (int a = 0; a < 3; ++a)
    F_u[a] = (gP[a] + gB[a]) - gamma * (F_w + F_bulk) * u[a] - (w + bulk) * (gamma * divV + gamma / t + gf) * u[a]
           - 2. * (w + bulk) * gamma * u[2] * dl[a] / t;
  if (SHEAR) {
    #pragma unroll
    for (int a = 0; a < 3; ++a) {
      F_u[a] += -S[a + 1][0] / t - 2. * dl[a] * S[0][3] / t - col(CCAKE_F_DIVSHEAR0 + a) + col(CCAKE_F_GRADSHEAR0 + a)
              - F_0i[a];
      #pragma unroll
      for (int b = 0; b < 3; ++b) M_u[a][b] += M_0i[a][b];
    }
  }
  double MI[3][3];
  inverse3(M_u, MI);
  #pragma unroll
  for (int a = 0; a < 3; ++a) {
    double x = 0.0;
    #pragma unroll
    for (int b = 0; b < 3; ++b) x += MI[a][b] * (F_u[b] + 0.0);
    du_dt[a] = x;
  }

  // ---------------- compute_derivatives (623-825) ----------------
  dN[0] = dN[1] = dN[2] = 0.0;
  double c1 = 0.0, c2 = 0.0, c3 = 0.0, ucdu = 0.0;
  #pragma unroll
  for (int a = 0; a < 3; ++a) {
    c1 += M_S[a] * du_dt[a];
    c2 += M_eb[a] * du_dt[a];
    c3 += M_snu[a] * du_dt[a];
    ucdu += uc[a] * du_dt[a];
  }
  const double rs = R_S[0] * dN[0] + R_S[1] * dN[1] + R_S[2] * dN[2];
  *d_s = c1 + F_S + rs;
  *d_b = c2 + F_eb + 0.0;
  *snu_out = c3 + F_snu;
  *theta_out = -1. * ucdu / gamma + gamma * divV + gamma / t + gf;
  if (SHEAR) {
    int q = 0;
    #pragma unroll
    for (int a = 0; a < 2; ++a)
      #pragma unroll
      for (int b = a; b < 3; ++b) {
        double m = 0.0;
        #pragma unroll
        for (int c = 0; c < 3; ++c) m += M_es[a][b][c] * du_dt[c];
        dshv[q++] = m + F_es[a][b];
      }
  }
  // ---------------- compute_Ez_derivative (828-862) ----------------
  const double p = col(CCAKE_F_P), e = col(CCAKE_F_E);
  *dez_out = ((e + p + bulk) * u[2] * u[2] + (p + bulk) / t2 + S[3][3]) * col(CCAKE_F_MASS_S) * t2
             / col(CCAKE_F_SIGMA_LAB);
}

__device__ __forceinline__ void cache_state3(const Col3& col)
{
  for (int q = 0; q < 5; ++q) col(P_C_SHV0 + q) = col(CCAKE_F_EXT_SHV0 + q);
  col(P_C_UX) = col(CCAKE_F_UX); col(P_C_UY) = col(CCAKE_F_UY); col(P_C_UETA) = col(CCAKE_F_UETA);
  col(P_C_X) = col(CCAKE_F_X); col(P_C_Y) = col(CCAKE_F_Y); col(P_C_ETA) = col(CCAKE_F_ETA);
  col(P_C_S) = col(CCAKE_F_EXT_S); col(P_C_BULK) = col(CCAKE_F_EXT_BULK);
  col(P_C_B) = col(CCAKE_F_EXT_B); col(P_C_SS) = col(CCAKE_F_EXT_SS); col(P_C_Q) = col(CCAKE_F_EXT_Q);
  col(P_C_EZ) = col(CCAKE_F_EZ);
}

// y = y0 + dt f with the negative-entropy rule (Evolver::step_rk,
// src/evolver.cpp:363-484), from the derivatives stored in F.
__device__ __forceinline__ void rk_update3(const Col3& col, int freeze, double dt, int32_t* __restrict__ err)
{
  double es = col(P_C_S) + dt * col(CCAKE_F_DEXT_S);
  if (es < 0.0 && freeze > 3) es = 1.e-3;
  else if (es < 0.0) atomicOr(err, DE_NEG_ENTROPY);
  col(CCAKE_F_EXT_S) = es;
  col(CCAKE_F_EXT_BULK) = col(P_C_BULK) + dt * col(CCAKE_F_DEXT_BULK);
  col(CCAKE_F_EXT_B) = col(P_C_B) + dt * col(CCAKE_F_DEXT_B);
  col(CCAKE_F_EXT_SS) = col(P_C_SS) + dt * col(CCAKE_F_DEXT_SS);
  col(CCAKE_F_EXT_Q) = col(P_C_Q) + dt * col(CCAKE_F_DEXT_Q);
  col(CCAKE_F_EZ) = col(P_C_EZ) + dt * col(CCAKE_F_DEZ);
  col(CCAKE_F_X) = col(P_C_X) + dt * col(CCAKE_F_VX);
  col(CCAKE_F_Y) = col(P_C_Y) + dt * col(CCAKE_F_VY);
  col(CCAKE_F_ETA) = col(P_C_ETA) + dt * col(CCAKE_F_VETA);
  col(CCAKE_F_UX) = col(P_C_UX) + dt * col(CCAKE_F_DUDT0 + 0);
  col(CCAKE_F_UY) = col(P_C_UY) + dt * col(CCAKE_F_DUDT0 + 1);
  col(CCAKE_F_UETA) = col(P_C_UETA) + dt * col(CCAKE_F_DUDT0 + 2);
  for (int q = 0; q < 5; ++q) col(CCAKE_F_EXT_SHV0 + q) = col(P_C_SHV0 + q) + dt * col(CCAKE_F_DEXT_SHV0 + q);
}

// RK: 0 derivatives only, 1 and the RK update, 2 the RK cache first, then
// the update (the first stage of a step).
template <bool SHEAR>
__global__ __launch_bounds__(256) void k3_eom(double* __restrict__ F, int npad, int n,
                                              const int32_t* __restrict__ freeze, double t, double use_vort,
                                              double dt, int32_t* __restrict__ err, int rk)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Col3 col{ F, npad, i };
  double du[3], ds, dN[3], db, dshv[5] = { 0, 0, 0, 0, 0 }, theta, snu, dez;
  eom_d3<SHEAR>(col, t, use_vort, du, &ds, dN, &db, dshv, &theta, &snu, &dez);
  for (int a = 0; a < 3; ++a) col(CCAKE_F_DUDT0 + a) = du[a];
  col(CCAKE_F_DEXT_S) = ds;
  col(CCAKE_F_DEXT_B) = dN[0]; col(CCAKE_F_DEXT_SS) = dN[1]; col(CCAKE_F_DEXT_Q) = dN[2];
  col(CCAKE_F_DEXT_BULK) = db;
  if (SHEAR) for (int q = 0; q < 5; ++q) col(CCAKE_F_DEXT_SHV0 + q) = dshv[q];
  col(CCAKE_F_THETA) = theta;
  col(CCAKE_F_SHV_NABLA_U) = snu;
  col(CCAKE_F_DEZ) = dez;
  if (rk == 0) return;
  if (rk == 2) cache_state3(col);
  rk_update3(col, freeze[i], dt, err);
}

__global__ __launch_bounds__(256) void k3_rk(double* __restrict__ F, int npad, int n,
                                             const int32_t* __restrict__ freeze, double dt, int32_t* __restrict__ err)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  rk_update3(Col3{ F, npad, i }, freeze[i], dt, err);
}

__global__ __launch_bounds__(256) void k3_cache(double* __restrict__ F, int npad, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  cache_state3(Col3{ F, npad, i });
}

// ---------------------------------------------------------------------------
// Launchers.
int launch3_stage_begin(ccake_event* ev, int do_gamma)
{
  const int n = ev->n;
  hipLaunchKernelGGL(k3_stage_begin, dim3((n + 255) / 256), dim3(256), 0, ev->stream, ev->F, ev->npad, n, ev->bbox,
                     do_gamma, ev->t * ev->t);
  return hipGetLastError() == hipSuccess ? 0 : CCAKE_ERR_HIP;
}

int launch3_stage_gather(ccake_event* ev)
{
  const int n = ev->n;
  hipLaunchKernelGGL(k3_stage_gather, dim3((n + 255) / 256), dim3(256), 0, ev->stream, ev->F, ev->npad, n, ev->perm,
                     ev->cand_s, (unsigned long long*)ev->pair_count, ev->t * ev->t);
  return hipGetLastError() == hipSuccess ? 0 : CCAKE_ERR_HIP;
}

double smooth_norm2_event(const ccake_event* ev)
{
  if (ev->p.dim == 3) return kern3(ev->p).norm2;
  return smooth_norm2(ev->p.hT);
}

// Waves per tile: the event's slices, as far as there are variants.
static int tile3_waves(const ccake_event* ev)
{
  const int w = pair_waves(ev);
  return w >= 4 ? 4 : (w >= 2 ? 2 : 1);
}

int launch3_smooth_pairs(ccake_event* ev, int mode, bool count_pairs)
{
  const int n = ev->n;
  ev->smooth_sum_slices = 1;
  const double rc = 2.0 * ev->p.hT;
  const double hinv = 1.0 / ev->p.hT, heinv = ev->p.hEta > 0.0 ? 1.0 / ev->p.hEta : 0.0;
  unsigned long long* pc = mode == 2 && count_pairs ? (unsigned long long*)ev->pair_count : nullptr;
  auto go = [&](auto kern, int W) {
    hipLaunchKernelGGL(kern, dim3((n + kTile3 - 1) / kTile3), dim3(kWave * W), 0, ev->stream, ev->cand_s, ev->skey,
                       ev->cell_off, ev->grid, n, rc * rc, search_radius(ev), hinv, heinv, ev->part, ev->npad, ev->perm,
                       ev->I + (size_t)CCAKE_I_BTRACK * ev->npad, pc);
  };
  auto waves = [&](auto w) {
    constexpr int W = decltype(w)::value;
    if (mode == 2) go(k3_smooth_tile<2, false, W>, W);
    else if (ev->p.factorized_kernel) {
      if (mode == 0) go(k3_smooth_tile<0, true, W>, W); else go(k3_smooth_tile<1, true, W>, W);
    } else {
      if (mode == 0) go(k3_smooth_tile<0, false, W>, W); else go(k3_smooth_tile<1, false, W>, W);
    }
  };
  const int W = tile3_waves(ev);
  if (W == 4) waves(std::integral_constant<int, 4>());
  else if (W == 2) waves(std::integral_constant<int, 2>());
  else waves(std::integral_constant<int, 1>());
  return hipGetLastError() == hipSuccess ? 0 : CCAKE_ERR_HIP;
}

int launch3_export_pairs(ccake_event* ev, int32_t* pi, int32_t* pj, size_t cap, size_t* n_out)
{
  const int n = ev->n;
  hipStream_t st = ev->stream;
  std::vector<int32_t> saved_bt(n), cnt(n);
  int32_t* bt = ev->I + (size_t)CCAKE_I_BTRACK * ev->npad;
  CCAKE_HIP(hipMemcpyAsync(saved_bt.data(), bt, n * sizeof(int32_t), hipMemcpyDeviceToHost, st));
  CCAKE_HIP(hipMemsetAsync(bt, 0, n * sizeof(int32_t), st));
  const int rc_count = launch3_smooth_pairs(ev, 2, false);
  if (rc_count) { (void)hipStreamSynchronize(st); return rc_count; }
  CCAKE_HIP(hipMemcpyAsync(cnt.data(), bt, n * sizeof(int32_t), hipMemcpyDeviceToHost, st));
  CCAKE_HIP(hipStreamSynchronize(st));
  CCAKE_HIP(hipMemcpyAsync(bt, saved_bt.data(), n * sizeof(int32_t), hipMemcpyHostToDevice, st));
  CCAKE_HIP(hipStreamSynchronize(st));
  std::vector<int64_t> off(n + 1, 0);
  for (int i = 0; i < n; ++i) off[i + 1] = off[i] + cnt[i];
  const size_t total = (size_t)off[n];
  *n_out = total;
  if (total > cap) return CCAKE_ERR_CAPACITY;
  struct DevBuf {
    void* p = nullptr;
    ~DevBuf() { if (p) (void)hipFree(p); }
  } b_off, b_i, b_j;
  CCAKE_HIP(hipMalloc(&b_off.p, (n + 1) * sizeof(int64_t)));
  CCAKE_HIP(hipMalloc(&b_i.p, (total + 1) * sizeof(int32_t)));
  CCAKE_HIP(hipMalloc(&b_j.p, (total + 1) * sizeof(int32_t)));
  int64_t* d_off = static_cast<int64_t*>(b_off.p);
  int32_t* d_i = static_cast<int32_t*>(b_i.p);
  int32_t* d_j = static_cast<int32_t*>(b_j.p);
  CCAKE_HIP(hipMemcpyAsync(d_off, off.data(), (n + 1) * sizeof(int64_t), hipMemcpyHostToDevice, st));
  const double rc = 2.0 * ev->p.hT;
  hipLaunchKernelGGL(k3_export, dim3((n + kTile - 1) / kTile), dim3(kTile), 0, st, ev->cand_s, ev->skey, ev->perm,
                     ev->cell_off, ev->grid, n, rc * rc, search_radius(ev), d_off, d_i, d_j);
  const hipError_t le = hipGetLastError();
  if (le != hipSuccess) { (void)hipStreamSynchronize(st); return hip_fail(le, "k3_export"); }
  CCAKE_HIP(hipMemcpyAsync(pi, d_i, total * sizeof(int32_t), hipMemcpyDeviceToHost, st));
  CCAKE_HIP(hipMemcpyAsync(pj, d_j, total * sizeof(int32_t), hipMemcpyDeviceToHost, st));
  CCAKE_HIP(hipStreamSynchronize(st));
  for (int i = 0; i < n; ++i) std::sort(pj + off[i], pj + off[i + 1]);
  return 0;
}

int launch3_grad(ccake_event* ev)
{
  const int n = ev->n;
  const double rc = 2.0 * ev->p.hT;
  const double hinv = 1.0 / ev->p.hT, heinv = ev->p.hEta > 0.0 ? 1.0 / ev->p.hEta : 0.0;
  const Kern3 K = kern3(ev->p);
  auto go = [&](auto kern, int W) {
    hipLaunchKernelGGL(kern, dim3((n + kTile3 - 1) / kTile3), dim3(kWave * W), 0, ev->stream, ev->cand_g, ev->skey,
                       ev->cell_off, ev->grid, n, rc * rc, search_radius(ev), hinv, heinv, K.kfac, K.C, ev->perm, ev->npad,
                       ev->F);
  };
  auto waves = [&](auto w) {
    constexpr int W = decltype(w)::value;
    if (ev->p.using_shear) {
      if (ev->p.factorized_kernel) go(k3_grad_tile<true, true, W>, W); else go(k3_grad_tile<true, false, W>, W);
    } else {
      if (ev->p.factorized_kernel) go(k3_grad_tile<false, true, W>, W); else go(k3_grad_tile<false, false, W>, W);
    }
  };
  const int W = tile3_waves(ev);
  if (W == 4) waves(std::integral_constant<int, 4>());
  else if (W == 2) waves(std::integral_constant<int, 2>());
  else waves(std::integral_constant<int, 1>());
  return hipGetLastError() == hipSuccess ? 0 : CCAKE_ERR_HIP;
}

int launch3_eom(ccake_event* ev, int fuse_rk, double dt)
{
  const int n = ev->n;
  const dim3 g((n + 255) / 256), b(256);
  const int32_t* fz = ev->I + (size_t)CCAKE_I_FREEZE * ev->npad;
  const double uv = ev->p.using_vorticity ? 1.0 : 0.0;
  if (ev->p.using_shear)
    hipLaunchKernelGGL(k3_eom<true>, g, b, 0, ev->stream, ev->F, ev->npad, n, fz, ev->t, uv, dt, ev->err, fuse_rk);
  else
    hipLaunchKernelGGL(k3_eom<false>, g, b, 0, ev->stream, ev->F, ev->npad, n, fz, ev->t, uv, dt, ev->err, fuse_rk);
  return hipGetLastError() == hipSuccess ? 0 : CCAKE_ERR_HIP;
}

int launch3_rk(ccake_event* ev, double dt)
{
  const int n = ev->n;
  hipLaunchKernelGGL(k3_rk, dim3((n + 255) / 256), dim3(256), 0, ev->stream, ev->F, ev->npad, n,
                     ev->I + (size_t)CCAKE_I_FREEZE * ev->npad, dt, ev->err);
  return hipGetLastError() == hipSuccess ? 0 : CCAKE_ERR_HIP;
}

int launch3_cache(ccake_event* ev)
{
  const int n = ev->n;
  hipLaunchKernelGGL(k3_cache, dim3((n + 255) / 256), dim3(256), 0, ev->stream, ev->F, ev->npad, n);
  return hipGetLastError() == hipSuccess ? 0 : CCAKE_ERR_HIP;
}

}  // namespace ccake

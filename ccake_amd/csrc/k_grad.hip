// Gradient pair kernels on gfx950 (owner computes, no atomics).
// Replaces SPHWorkstation::smooth_all_particle_gradients
// (src/sph_workstation.cpp:796-986), D = 2, diffusion terms off.
//
// With K_ab = m_b sl_a grad W_ab the reference sums, per neighbour b,
//   gradP    += (p_b/sl_b^2 + p_a/sl_a^2) K_ab
//   gradE    += (m_b/sl_a)(e_b - e_a) grad W_ab
//   gradBulk += (Pi_b/sl_b^2 + Pi_a/sl_a^2) K_ab
//   gradV_ij += (m_b/sl_a)(v_b^j - v_a^j) d_i W_ab
//   gradshear+= (K_ab . v_a)(pi^{0i}_b/sl_b^2 + pi^{0i}_a/sl_a^2)
//   divshear_j += sum_i K_ab,i (pi^{ji}_b/sl_b^2 + pi^{ji}_a/sl_a^2).
// Every owner-side factor is constant over b, so the kernel accumulates
// only neighbour-side sums of w = m_b grad W_ab (17 accumulators) and
// applies the owner terms once at the end.
#include "pair_common.h"
#include "grad_sum.h"
#include <type_traits>

namespace ccake {

// The walk of one (tile, slice) unit: slice `slice` of `nslices` of the
// tile's candidates, one wave; fin(acc) receives the neighbour-side sums of
// m_b grad W / C, summed as spline_g2 m_b rel and scaled by its 2 h at the end.
// BULK false: the event's bulk pressure is zero on every particle (zeta = 0
// and no initial bulk, checked at initialize), so the grad Pi sums are the
// exact zeros the full walk would give and are not accumulated.
// Bound: the FP64 vector unit (80 % busy), 39 instructions per candidate and
// wave: the 20 sums, 5 for the offsets and r^2, 14 for the kernel.  FP64
// matrix instructions run in the same unit at the same rate (16x16x4: 65
// cycles, a vector instruction 4), so the sums stay on the vector side.
// 188,250 particles (479M pairs): 1.30 ms per launch with 50 instructions
// and no request ahead, 0.96 ms now.
template <bool SHEAR, bool BULK, int FORM, class Fin>
__device__ __forceinline__ void grad_walk(const double* __restrict__ cand, const int32_t* __restrict__ skey,
                                          const int32_t* __restrict__ cell_off, const Grid* __restrict__ gridp,
                                          int n, double rc2, double rcs, double hinv2, double m4h, double m2h, int tile, int slice,
                                          int nslices, Fin&& fin)
{
  constexpr bool KEEP = FORM == kKeep;
  const Grid& g0 = *gridp;
  const int lane = threadIdx.x & (kWave - 1);
  const int k = tile * kTile + lane;
  const bool act = k < n;
  const int kk = act ? k : 0;
  const double* me = cand + (size_t)kk * kCandG;
  const double xa = me[0], ya = me[1];
  const int myrow = act ? skey[kk] / g0.stride : INT_MAX;

  // the 12 sums of grad_nacc<false>, then pi^{0x} w (2), pi^{0y} w (2) and
  // the two of pi^{ij} w_i; KEEP: the sums of grad_nacc<SHEAR> themselves
  constexpr int NW = SHEAR ? (KEEP ? 17 : 18) : 12;
  const double vax = me[6], vay = me[7];
  double acc[NW];
  for_tile_sums<NW>(acc, [&](auto in_range) {
    for_segments(gridp, g0, FORM == kSmall ? rcs : 0.0, act, myrow, xa, ya, [&](const Seg& seg, bool in) {
      const Grid& g = gridp[event_index(gridp, g0, seg.row)];
      const double xs = in ? xa : kFarAway;      // lanes of other cell rows sit this segment's walk out
      for_spans_slice<kCandG, KEEP>(g, cell_off, cand, seg, rc2, rcs, slice, nslices, [&](RunCursor& cur) {
        constexpr int NR = SHEAR ? 13 : 8;
        walk_records<NR, kCandG, decltype(in_range)::value>(cand, xs, ya, rc2, cur,
                                 [&](const double* c, double dx, double dy, double r2) {
          double gm;
          if (KEEP) {
            double q, iq;
            q_and_inverse(r2, hinv2, q, iq);
            gm = c[2] * spline_g(q, iq);
          } else {
            gm = c[2] * spline_g2<FORM>(r2, m4h, m2h);
          }
          const double wx = gm * dx, wy = gm * dy;
          acc[0] += wx; acc[1] += wy;                    // sum m_b grad W
          acc[2] += c[3] * wx; acc[3] += c[3] * wy;      // p_b / sl_b^2
          acc[4] += c[4] * wx; acc[5] += c[4] * wy;      // e_b
          if (BULK) { acc[6] += c[5] * wx; acc[7] += c[5] * wy; }   // Pi_b / sl_b^2
          acc[8] += c[6] * wx; acc[9] += c[7] * wx;      // v_b d_x W
          acc[10] += c[6] * wy; acc[11] += c[7] * wy;    // v_b d_y W
          if (SHEAR && KEEP) {
            const double cv = wx * vax + wy * vay;
            acc[SHEAR ? 12 : 0] += cv;
            acc[SHEAR ? 13 : 0] += cv * c[SHEAR ? 8 : 0]; acc[SHEAR ? 14 : 0] += cv * c[SHEAR ? 9 : 0];
            acc[SHEAR ? 15 : 0] += wx * c[SHEAR ? 10 : 0] + wy * c[SHEAR ? 11 : 0];
            acc[SHEAR ? 16 : 0] += wx * c[SHEAR ? 11 : 0] + wy * c[SHEAR ? 12 : 0];
          } else if (SHEAR) {
            acc[SHEAR ? 12 : 0] += c[SHEAR ? 8 : 0] * wx; acc[SHEAR ? 13 : 0] += c[SHEAR ? 8 : 0] * wy;
            acc[SHEAR ? 14 : 0] += c[SHEAR ? 9 : 0] * wx; acc[SHEAR ? 15 : 0] += c[SHEAR ? 9 : 0] * wy;
            acc[SHEAR ? 16 : 0] += c[SHEAR ? 10 : 0] * wx; acc[SHEAR ? 16 : 0] += c[SHEAR ? 11 : 0] * wy;
            acc[NW - 1] += c[SHEAR ? 11 : 0] * wx; acc[NW - 1] += c[SHEAR ? 12 : 0] * wy;
          }
        });
      });
    });
  });
  if (!KEEP) {
    const double h2 = FORM == kSingle ? -4.0 * m2h / hinv2 : -1.0 / m2h;   // kSingle: 4 h, over 1/r's mean error
    #pragma unroll
    for (int q = 0; q < NW; ++q) acc[q] *= h2;
  }
  if (SHEAR && !KEEP) {
    // w . v_a and (w . v_a) pi^{0i}_b / sl_b^2, v_a being constant over b
    const double out[17] = { acc[0], acc[1], acc[2], acc[3], acc[4], acc[5], acc[6], acc[7], acc[8], acc[9], acc[10],
                             acc[11], vax * acc[0] + vay * acc[1],
                             vax * acc[SHEAR ? 12 : 0] + vay * acc[SHEAR ? 13 : 0],
                             vax * acc[SHEAR ? 14 : 0] + vay * acc[SHEAR ? 15 : 0],
                             acc[SHEAR ? 16 : 0], acc[NW - 1] };
    fin(out);
  } else {
    fin(acc);
  }
}

// Pair part: one single-wave workgroup per (tile, slice) unit walks its
// slice of the tile's candidates and stores the slice's neighbour-side sums;
// k_grad_sum adds the slices in slice order and applies the owner terms.
template <bool SHEAR, bool BULK, int FORM = kExact>
__global__ __launch_bounds__(kWave) void k_grad_slice(const double* __restrict__ cand,
                                                      const int32_t* __restrict__ skey,
                                                      const int32_t* __restrict__ cell_off,
                                                      const Grid* __restrict__ gridp, int n,
                                                      double rc2, double rcs, double hinv2, double m4h, double m2h, int nslices,
                                                      double* __restrict__ part, int npad)
{
  constexpr int NACC = grad_nacc<SHEAR>();
  const int unit = xcd_tile(blockIdx.x, gridDim.x);
  const int tile = unit / nslices;
  const int slice = unit - tile * nslices;
  grad_walk<SHEAR, BULK, FORM>(cand, skey, cell_off, gridp, n, rc2, rcs, hinv2, m4h, m2h, tile, slice, nslices,
                         [&](const double* acc) {
    double* p = part + (size_t)slice * NACC * npad + tile * kTile + threadIdx.x;
    for (int q = 0; q < NACC; ++q) p[(size_t)q * npad] = acc[q];
  });
}

// The same walk with the W slices of a tile in one workgroup of W waves
// (wave w walks slice w): the slices' sums are added in slice order in LDS
// and stored as the sums of a single slice, so the sum pass reads NACC
// values per particle instead of W * NACC and no partial sum of a slice
// goes through HBM.
template <bool SHEAR, bool BULK, int W, int FORM = kExact>
__global__ __launch_bounds__(kWave * W) void k_grad_tile(const double* __restrict__ cand,
                                                         const int32_t* __restrict__ skey,
                                                         const int32_t* __restrict__ cell_off,
                                                         const Grid* __restrict__ gridp, int n,
                                                         double rc2, double rcs, double hinv2, double m4h, double m2h,
                                                         double* __restrict__ part, int npad)
{
  // the sums go through LDS in two halves: 18 KB a tile of 4 waves instead of
  // 35, so that LDS does not hold the CU below its 6 waves per SIMD
  constexpr int NACC = grad_nacc<SHEAR>(), HALF = (NACC + 1) / 2;
  __shared__ double red[W][HALF][kWave];
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int slice = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);   // wave-uniform
  const int lane = threadIdx.x & (kWave - 1);
  grad_walk<SHEAR, BULK, FORM>(cand, skey, cell_off, gridp, n, rc2, rcs, hinv2, m4h, m2h, tile, slice, W,
                               [&](const double* acc) {
    #pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h) __syncthreads();                    // the first half has been read
      #pragma unroll
      for (int q = 0; q < HALF; ++q)
        if (h * HALF + q < NACC) red[slice][q][lane] = acc[h * HALF + q < NACC ? h * HALF + q : 0];
      __syncthreads();
      const int nq = NACC - h * HALF < HALF ? NACC - h * HALF : HALF;
      for (int t = threadIdx.x; t < nq * kWave; t += kWave * W) {
        const int q = t / kWave, l = t - q * kWave;
        double s = 0.0;
        #pragma unroll
        for (int w = 0; w < W; ++w) s += red[w][q][l];
        part[(size_t)(h * HALF + q) * npad + tile * kTile + l] = s;
      }
    }
  });
}

// Sum pass: the slices' sums in slice order, scaled by C = kgrad / h^4,
// then the owner terms, written by particle id (grad_sum_into).  S is the
// slice count, so every load of a particle is in flight at once.
template <bool SHEAR, int S>
__global__ __launch_bounds__(256) void k_grad_sum(const double* __restrict__ cand,
                                                  const int32_t* __restrict__ perm, int n, double C,
                                                  const double* __restrict__ part, int npad,
                                                  double* __restrict__ F)
{
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  grad_sum_into<SHEAR, S>(cand, k, perm[k], C, part, S, npad, F);
}

int launch_grad_pairs(ccake_event* ev)
{
  const int n = ev->n_live;          // sorted positions of the live events' particles
  const double h = ev->p.hT;
  const double rc = 2.0 * h;
  const bool single = ev->p.pair_precision == 1;
  const double hinv2 = 1.0 / (h * h), mean = ev->many_neighbours ? kRsqMean : 0.0;
  const double m4h = (single ? -0.5 / (1.0 + mean) : -0.25) / h, m2h = 2.0 * m4h;
  const int ntiles = (n + kTile - 1) / kTile;
  const double rcs = search_radius(ev);
  const int W = grad_tile_waves(lds_slices(ev), ntiles, ev->dev->simds);
  if (W) {
    // the tile's slices reduced in LDS: the sum pass sees one slice
    ev->grad_sum_slices = 1;
    auto go = [&](auto kern, int nw) {
      hipLaunchKernelGGL(kern, dim3(ntiles), dim3(kWave * nw), 0, ev->stream, ev->cand_g, ev->skey, ev->cell_off,
                         ev->grid, n, rc * rc, rcs, hinv2, m4h, m2h, ev->part, ev->npad);
    };
    auto form = [&](auto w, auto f) {
      constexpr int V = decltype(w)::value, FM = decltype(f)::value;
      const bool sh = ev->p.using_shear, bu = !ev->no_bulk;
      if (sh) { if (bu) go(k_grad_tile<true, true, V, FM>, V); else go(k_grad_tile<true, false, V, FM>, V); }
      else { if (bu) go(k_grad_tile<false, true, V, FM>, V); else go(k_grad_tile<false, false, V, FM>, V); }
    };
    const std::integral_constant<int, 8> w8;
    const std::integral_constant<int, 4> w4;
    if (single && W == 8) form(w8, std::integral_constant<int, kSingle>());
    else if (single) form(w4, std::integral_constant<int, kSingle>());
    else if (W >= 2 * kKeepGradWaves && keep_order(ev))
      form(std::integral_constant<int, kKeepGradWaves>(), std::integral_constant<int, kKeep>());
    else if (W == 8 && small_event(ev, ntiles)) form(w8, std::integral_constant<int, kSmall>());
    else if (W == 8) form(w8, std::integral_constant<int, kExact>());
    else form(w4, std::integral_constant<int, kExact>());
    return hipGetLastError() == hipSuccess ? 0 : CCAKE_ERR_HIP;
  }
  ev->grad_sum_slices = ev->nslices;
  const dim3 grid(ntiles * ev->nslices), blk(kWave);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, blk, 0, ev->stream, ev->cand_g, ev->skey, ev->cell_off, ev->grid, n, rc * rc,
                       rcs, hinv2, m4h, m2h, ev->nslices, ev->part, ev->npad);
  };
  auto form = [&](auto f) {
    constexpr int FM = decltype(f)::value;
    const bool bu = !ev->no_bulk;
    if (ev->p.using_shear) { if (bu) go(k_grad_slice<true, true, FM>); else go(k_grad_slice<true, false, FM>); }
    else { if (bu) go(k_grad_slice<false, true, FM>); else go(k_grad_slice<false, false, FM>); }
  };
  if (single) form(std::integral_constant<int, kSingle>()); else form(std::integral_constant<int, kExact>());
  return hipGetLastError() == hipSuccess ? 0 : CCAKE_ERR_HIP;
}

template <bool SHEAR, int S = 1>
static int grad_sum_dispatch(ccake_event* ev, double C)
{
  if constexpr (S > kMaxSlices) {
    set_error("slice count out of range");
    return CCAKE_ERR_INVALID;
  } else {
    if (ev->grad_sum_slices != S) return grad_sum_dispatch<SHEAR, S + 1>(ev, C);
    const int n = ev->n_live;
    hipLaunchKernelGGL((k_grad_sum<SHEAR, S>), dim3((n + 255) / 256), dim3(256), 0, ev->stream, ev->cand_g,
                       ev->perm, n, C, ev->part, ev->npad, ev->F);
    return 0;
  }
}

double grad_sum_scale(double h) { return -0.5 * (15.0 / (7.0 * kPi)) / pow(h, 4); }   // kgrad / h^4

int launch_grad_sum(ccake_event* ev)
{
  const double C = grad_sum_scale(ev->p.hT);
  const int rc = ev->p.using_shear ? grad_sum_dispatch<true>(ev, C) : grad_sum_dispatch<false>(ev, C);
  if (rc) return rc;
  return hipGetLastError() == hipSuccess ? 0 : CCAKE_ERR_HIP;
}

int launch_grad(ccake_event* ev)
{
  if (ev->p.dim == 3) return launch3_grad(ev);
  int rc = launch_grad_pairs(ev);
  return rc ? rc : launch_grad_sum(ev);
}

}  // namespace ccake

// mosaic.hip -- the mosaic / A-projection gridder (replaces mosaic_grid_jit,
// core/imaging/imaging_utils/mosaic_grid.py:306-486).
//
// Each sample is convolved with a non-separable, oversampled complex
// convolution function (already multiplied by the field's phase gradient)
// chosen by its baseline, channel and polarisation, over a support that the
// same three indices choose.  The samples come binned by a plan whose
// support is at least max_support = max(weight_support): every footprint
// then lies inside the tiles the plan records the sample in, and the plan's
// own bounds test keeps every sample that the reference's test (u_centre +-
// max_support inside the grid, mosaic_grid.py:379-383) keeps.  That test is
// applied here as records are staged, with max_support reduced from the
// table on the device.
//
// One workgroup per work unit, as many wavefronts as polarisations.  The
// unit's tile, all its polarisations, is accumulated in LDS.  Where the
// polarisations share their convolution functions (cf_pol_map equal, the
// usual case) each wavefront takes a band of the tile's rows and all
// polarisations: a tap's address, cell and kernel value serve them all, and a
// record costs a wavefront something only where it reaches its band (1.7 of 4
// bands on average for 9 taps in a tile of 32).  Otherwise each takes its own
// polarisation of the whole tile.
// Records are staged 64 at a time, one per lane (FP64 position, kernel
// offsets, convolution-function base and supports, weighted data), every
// wavefront for itself and in registers; then they are taken one after
// another, the lanes over the taps, with the record's values broadcast from
// the lane that staged it.  A tap reads its complex kernel value from global
// memory (read-only, shared by every unit of the same baseline group, so it
// stays in L2; by phase, see k_mosaic_phases) and adds kernel * data into its
// tile cell: the taps of one record are distinct cells and no other
// wavefront touches them, so no atomics.  The tile then goes to HBM once,
// split bins adding theirs with atomics.
//
// What bounds it: the wavefronts' instructions (vector units busy 75% of the
// time).  One wavefront per polarisation throughout, records staged through
// LDS and a flush that divided per cell took 5.08 ms for 6.45 M samples x 4
// polarisations on 32 planes of 2048^2 in FP32, this 3.57 ms; the planes
// alone take 0.95 ms to write.  FP64, 8 channels: 3.51 -> 2.51 ms; 1
// polarisation: 1.50 -> 1.19 ms; 4 convolution functions per record: 5.90 ->
// 5.85 ms (FP64 4.89 -> 3.36).
//
// The taps of a record that count (inside the band or tile and inside the
// convolution function) form a rectangle, which staging works out once per
// record.  The wavefronts then walk only that rectangle: a tap is a quotient
// by the rectangle's width and two 24-bit multiply-adds from wave-uniform
// bases, with no bounds tests, and taps outside (most of a record near an
// edge) cost nothing.
//
// The kernel sum of a record (the reference's `norm`, over all its taps)
// depends only on its convolution function and the kernel offsets of its
// first tap, so it is tabulated per call, summed in the reference's order
// (v outer, u inner, in FP64), and each wavefront adds its primary
// records' share of the sum of weights as it stages them: weight * Re(norm)
// for the PSF, weight * Re(norm^2) for data (mosaic_grid.py:470-484).
#include "tile_common.h"

namespace av {

constexpr int kMosaicStage = 64;
// units per XCD group: a tile's channels are consecutive units, so a group
// of 64 keeps a tile's units (and the samples they share) on one XCD's L2
constexpr uint32_t kMosaicGroup = 64;
// kernel values are copied by phase for this many samples or more, and at most so
// many values a sample (see launch_mosaic)
constexpr int64_t kPhaseSamples = 3 << 14, kPhaseValues = 32;

template <typename R>
struct MosaicArgs {
  const R *vis, *weight;
  const int32_t *cf_baseline_map, *cf_chan_map, *cf_pol_map;
  const R *cfpg;  // complex [ncb][ncc][ncp][cu][cv]
  const int32_t *weight_support;  // [ncb][ncc][ncp][2]
  int n_baseline, ncb, ncc, ncp, cu_n, cv_n, ov_u, ov_v;
  R *grid;
  // kernel sums [ncb * ncc * ncp][ndu][ndv] (re, im), for first-tap kernel
  // offsets cu_n / 2 + du_lo + du and cv_n / 2 + dv_lo + dv
  const double *norms;
  int du_lo, ndu, dv_lo, ndv;
  const int *max_support = nullptr;  // max(weight_support), one value on the device
  // how the gridder reads the kernel values: by phase (see k_mosaic_phases)
  // or in the caller's order; elements between taps along u and along v
  const R *taps = nullptr;
  int by_phase = 0, tap_u = 0, tap_v = 0;
  int64_t tap_cf = 0;       // elements per convolution function
  int phase_u = 0, phase_v = 0;  // elements between phases along u and v
  int taps_u = 0, taps_v = 0;    // taps of a phase, one less in phases past last_u (last_v)
  int last_u = 0, last_v = 0;
};

// The convolution functions by phase: [cf][cfu mod ov_u][cfv mod ov_v]
// [cfu / ov_u][cfv / ov_v], zeros where the last tap of a phase is past the
// table.  A record's taps are one phase: in the caller's order they lie ov_v
// elements apart along v and ov_u * cv_n along u, so the 64 lanes of a load
// touched 64 cache lines and the gridder waited on the vector L1, one line a
// cycle; by phase they are rows of consecutive elements, about 6 lines a
// load.  The copy is one pass over the table, made where the samples are worth it
// (launch_mosaic).
template <typename R>
__global__ __launch_bounds__(256) void k_mosaic_phases(MosaicArgs<R> A, int64_t total, R *out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int64_t cf = i / A.tap_cf;
  const int e = (int)(i - cf * A.tap_cf);
  const int fu = e / A.phase_u, eu = e - fu * A.phase_u;
  const int fv = eu / A.phase_v, t = eu - fv * A.phase_v;
  const int tu = t / A.tap_u, tv = t - tu * A.tap_u;
  const int cfu = tu * A.ov_u + fu, cfv = tv * A.ov_v + fv;
  Cplx2<R> v{(R)0, (R)0};
  if (cfu < A.cu_n && cfv < A.cv_n)
    v = ((const Cplx2<R> *)A.cfpg)[(size_t)cf * A.cu_n * A.cv_n + (size_t)cfu * A.cv_n + cfv];
  ((Cplx2<R> *)out)[i] = v;
}

// max(weight_support): the reference's max_support_center
// (mosaic_grid.py:345), by one workgroup of 256 threads
__global__ __launch_bounds__(256) void k_mosaic_max_support(const int32_t *ws, int n, int *out) {
  __shared__ int red[4];
  int m = INT_MIN;
  for (int i = threadIdx.x; i < n; i += 256) m = max(m, ws[i]);
  for (int off = 32; off >= 1; off >>= 1) m = max(m, __shfl_xor(m, off));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) *out = max(max(red[0], red[1]), max(red[2], red[3]));
}

// floor(x / d) for d > 0
__device__ inline int floor_div(int x, int d) { return x >= 0 ? x / d : -((-x + d - 1) / d); }

// The kernel-sum table: one thread per (convolution function, first-tap
// offsets), summing the in-range taps as the reference does.
template <typename R>
__global__ __launch_bounds__(256) void k_mosaic_norms(MosaicArgs<R> A, int ncf) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t per = (int64_t)A.ndu * A.ndv;
  if (i >= per * ncf) return;
  const int b = (int)(i / per), rem = (int)(i - (int64_t)b * per);
  const int du = rem / A.ndv, dv = rem - du * A.ndv;
  const int cfu0 = A.cu_n / 2 + A.du_lo + du, cfv0 = A.cv_n / 2 + A.dv_lo + dv;
  const int su = A.weight_support[2 * b], sv = A.weight_support[2 * b + 1];
  const int scu = su / 2, scv = sv / 2;
  const Cplx2<R> *cf = (const Cplx2<R> *)A.cfpg + (size_t)b * A.cu_n * A.cv_n;
  double nre = 0.0, nim = 0.0;
  for (int iv = -scv; iv < sv - scv; ++iv) {
    const int cfv = A.ov_v * iv + cfv0;
    for (int iu = -scu; iu < su - scu; ++iu) {
      const int cfu = A.ov_u * iu + cfu0;
      if (cfu < 0 || cfu >= A.cu_n || cfv < 0 || cfv >= A.cv_n) continue;
      const Cplx2<R> c = cf[(size_t)cfu * A.cv_n + cfv];
      nre = nre + (double)c.re;
      nim = nim + (double)c.im;
    }
  }
  ((double2 *)A.norms)[i] = make_double2(nre, nim);
}

// A value of lane k (uniform over the wavefront) in every lane.
__device__ inline int lane_value(int v, int k) { return __builtin_amdgcn_readlane(v, k); }
__device__ inline float lane_value(float v, int k) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), k));
}
__device__ inline double lane_value(double v, int k) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, k);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), k);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

// Tap t of a record's rectangle: its cell in `at`, its kernel value's offset
// from the record's first returned, unsigned: no sign extension before the
// 64-bit address.
template <typename R>
__device__ inline uint32_t tap_of(int t, int w, float rw, int cell0, int tile_v,
                                  const MosaicArgs<R> &A, int &at) {
  const int q = (int)((float)t * rw);
  const int p = t - (int)__umul24(q, w);
  at = cell0 + (int)__umul24(q, tile_v) + p;
  return (uint32_t)__umul24(q, A.tap_u) + (uint32_t)__umul24(p, A.tap_v);
}

// Polarisations of a tile cell that lie side by side in LDS: 16 bytes of
// them, so that a lane reads and writes them at once and neighbouring lanes
// hit neighbouring banks.
template <typename R, int NPOL>
struct alignas(sizeof(Cplx2<R>) * (NPOL < 16 / (int)sizeof(Cplx2<R>) ? NPOL
                                                                     : 16 / (int)sizeof(Cplx2<R>)))
    MosaicCell {
  static constexpr int kPols =
      NPOL < 16 / (int)sizeof(Cplx2<R>) ? NPOL : 16 / (int)sizeof(Cplx2<R>);
  Cplx2<R> v[kPols];
};

// Record k of a staged batch: its rectangle, and tap `lane`'s cell and kernel
// value.  A lane past the last tap loads the last one: every lane loads, so
// the wait for one record's values does not have to include the next's.
template <typename R>
struct MosaicTap {
  int n, at;
  Cplx2<R> c;
  __device__ inline void load(int k, int lane, int pn, int pw, int pcfoff, int pcell0, float prw,
                              const MosaicArgs<R> &A, int tile_v) {
    n = lane_value(pn, k);
    const Cplx2<R> *cf = (const Cplx2<R> *)A.taps + lane_value(pcfoff, k);
    c = cf[tap_of(min(lane, n - 1), lane_value(pw, k), lane_value(prw, k), lane_value(pcell0, k),
                  tile_v, A, at)];
  }
};

template <typename R, int NPOL>
__global__ __launch_bounds__(64 * NPOL) void k_mosaic_grid(PlanDev P, MosaicArgs<R> A, int psf,
                                                           int accumulate) {
  extern __shared__ __align__(16) char smem[];
  using Cell = MosaicCell<R, NPOL>;
  constexpr int kPols = Cell::kPols, kParts = NPOL / kPols;
  const int TV = P.tile_v, cells = P.tile_u * TV;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wp = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t u = xcd_grouped_block(blockIdx.x, kMosaicGroup);
  const uint32_t n_units = P.gunit_start[P.n_bins];
  if (u >= n_units) return;
  const uint4 unit = P.gunits[u];
  const uint32_t b = unit.x, first = unit.y, cnt = unit.z, fl = unit.w;
  uint32_t tile_i;
  int ic;
  bin_parts(P, (uint32_t)b, tile_i, ic);
  const uint32_t tu_i = tile_i / (uint32_t)P.ntv;
  const int u0 = (int)tu_i * P.tile_u, v0 = (int)(tile_i - tu_i * (uint32_t)P.ntv) * TV;
  const uint32_t prim_end = P.bin_start[b] + P.cnt_prim[b];
  R *gplane = A.grid + (size_t)ic * NPOL * P.n_u * P.n_v * 2;
  const size_t pstride = (size_t)P.n_u * P.n_v * 2;
  const int ncf = A.ncb * A.ncc * A.ncp;
  // this wavefront's rows of the tile, [s0, s1): it clears and flushes them,
  // and with one convolution function for all polarisations it grids them
  // alone, so no wavefront waits for another.  With several (by_pol) it grids
  // its own polarisation's cells of all rows, [r0, r1).
  const int rows = (P.tile_u + NPOL - 1) / NPOL;
  const int s0 = min(wp * rows, P.tile_u), s1 = min(s0 + rows, P.tile_u);
  const int pm = A.cf_pol_map[wp];
  bool by_pol = false;
#pragma unroll
  for (int p = 1; p < NPOL; ++p) by_pol |= A.cf_pol_map[p] != A.cf_pol_map[0];
  const int r0 = by_pol ? 0 : s0, r1 = by_pol ? P.tile_u : s1;
  Cell *tile = (Cell *)smem;  // [part][u][v]

  if (cnt > 0)
    for (int i = s0 * TV + lane; i < s1 * TV; i += 64)
#pragma unroll
      for (int a = 0; a < kParts; ++a) tile[a * cells + i] = Cell{};
  if (by_pol) __syncthreads();  // the same for every wavefront
  double swl = 0.0;  // this lane's records' sum of weights, polarisation wp
  const int ccu = A.cu_n / 2, ccv = A.cv_n / 2;
  const int cfsize = (int)A.tap_cf;  // the host bounds ncf * cfsize below 2^31
  const int msup = *A.max_support;
  constexpr unsigned kAll = (1u << NPOL) - 1;
  // the product first, then the cell, as the reference adds them
  const auto add_to = [](Cplx2<R> &cell, const Cplx2<R> &c, R dre, R dim) {
    cell.re += fma(c.re, dre, -(c.im * dim));
    cell.im += fma(c.re, dim, c.im * dre);
  };
  const auto add_pols = [&](int at, const Cplx2<R> &c, const R *dre, const R *dim,
                            unsigned pols) {
    if (by_pol) {
      add_to(tile[(wp / kPols) * cells + at].v[wp % kPols], c, dre[0], dim[0]);
      return;
    }
#pragma unroll
    for (int a = 0; a < kParts; ++a) {
      Cell &cell = tile[a * cells + at];
      Cell v = cell;
#pragma unroll
      for (int p = 0; p < kPols; ++p)
        if (pols >> (a * kPols + p) & 1) add_to(v.v[p], c, dre[a * kPols + p], dim[a * kPols + p]);
      cell = v;
    }
  };

  for (uint32_t base = first; base < first + cnt; base += kMosaicStage) {
    // ---- stage: lane l forms record base + l's rectangle in this
    // wavefront's rows and its weighted data, and keeps them in its
    // registers.  Tap t of the n = h * w taps that count (0: nothing to
    // add here) is row q = t / w, column p = t - q * w; its kernel value
    // is element cfoff + q * tap_u + p * tap_v of the kernel values, its
    // cell is cell0 + q * tile_v + p, and rw is 1 / w rounded up:
    // (int)(t * rw) = t / w for t < 2^16.
    int pn = 0, pw = 1, pcfoff = 0, pcell0 = 0;
    float prw = 1.0f;
    unsigned plive = 0;  // polarisations with data to add
    R pdre[NPOL] = {}, pdim[NPOL] = {};
    const uint32_t r = base + lane;
    if (r < first + cnt) {
      const uint32_t item = P.rec[3 * (size_t)r];
      const uint32_t geo = P.rec[3 * (size_t)r + 1];
      int au, ou, avv, ovv;
      unpack_geo(geo, au, ou, avv, ovv);
      const int64_t row = (int64_t)(item / (uint32_t)P.n_chan);
      const int ch = (int)(item - (uint32_t)row * (uint32_t)P.n_chan);
      R w[NPOL];
#pragma unroll
      for (int p = 0; p < NPOL; ++p) w[p] = A.weight[(size_t)item * NPOL + p];
      if (!psf) {
#pragma unroll
        for (int p = 0; p < NPOL; ++p) {
          pdre[p] = A.vis[((size_t)item * NPOL + p) * 2];
          pdim[p] = A.vis[((size_t)item * NPOL + p) * 2 + 1];
        }
      }
      // a 32-bit remainder: row < 2^32, as item = row * n_chan + ch is 32-bit
      const int cfb = A.cf_baseline_map[(uint32_t)row % (uint32_t)A.n_baseline];
      const int cfc = A.cf_chan_map[ch];
      const int idx = (cfb * A.ncc + cfc) * A.ncp + pm;
      // the reference's offsets at this call's oversampling, from the
      // same FP64 positions the plan binned (mosaic_grid.py:376-386)
      const double uu = P.uvw[row * 3] * P.gscale_u[ch] + (double)(P.n_u / 2);
      const double vv = P.uvw[row * 3 + 1] * P.gscale_v[ch] + (double)(P.n_v / 2);
      const int cu = au, cv = avv;
      const int gcu = u0 + cu, gcv = v0 + cv;
      // the reference's bounds test (mosaic_grid.py:379-383), written
      // without sums that could overflow for any table value
      const bool inside = gcu >= msup && P.n_u - gcu > msup && gcv >= msup && P.n_v - gcv > msup;
      const int cfu0 = (int)floor(((double)gcu - uu) * (double)A.ov_u + 0.5) + ccu;
      const int cfv0 = (int)floor(((double)gcv - vv) * (double)A.ov_v + 0.5) + ccv;
      const bool cf_ok = idx >= 0 && idx < ncf;
      const int idc = cf_ok ? idx : 0;  // in-bounds reads whatever the maps hold
      const int wsu = A.weight_support[2 * idc], wsv = A.weight_support[2 * idc + 1];
      // mosaic_grid.py:412: skip NaN or exactly-zero data (and, here,
      // convolution functions outside the table)
      if (inside && cf_ok) {
#pragma unroll
        for (int p = 0; p < NPOL; ++p) {
          pdre[p] = psf ? w[p] : pdre[p] * w[p];
          pdim[p] = psf ? (R)0 : pdim[p] * w[p];
          if (!(isnan(pdre[p]) || isnan(pdim[p])) && !(pdre[p] == (R)0 && pdim[p] == (R)0))
            plive |= 1u << p;
        }
        if (by_pol) {
          plive &= 1u << wp;
#pragma unroll
          for (int p = 1; p < NPOL; ++p) {
            pdre[0] = wp == p ? pdre[p] : pdre[0];
            pdim[0] = wp == p ? pdim[p] : pdim[0];
          }
        }
        if (r < prim_end && plive >> wp & 1) {
          const int du = min(max(cfu0 - ccu - A.du_lo, 0), A.ndu - 1);
          const int dv = min(max(cfv0 - ccv - A.dv_lo, 0), A.ndv - 1);
          const double2 nm = ((const double2 *)A.norms)[((size_t)idc * A.ndu + du) * A.ndv + dv];
          R wt = w[0];
#pragma unroll
          for (int p = 1; p < NPOL; ++p) wt = wp == p ? w[p] : wt;
          const double wd = (double)wt;
          swl += psf ? wd * nm.x : wd * (nm.x * nm.x - nm.y * nm.y);
        }
        // taps iu in [-wsu / 2, wsu - wsu / 2) whose kernel row
        // ov_u * iu + cfu0 lies in [0, cu_n) and whose cell cu + iu lies
        // in this wavefront's rows; the same along v and the tile
        const int scu = wsu / 2, scv = wsv / 2;
        const int qu = floor_div(cfu0, A.ov_u), qv = floor_div(cfv0, A.ov_v);
        const int iu_lo = max(max(-scu, -qu), r0 - cu);
        // the record's phase, and the last tap of that phase
        const int fu = cfu0 - qu * A.ov_u, fv = cfv0 - qv * A.ov_v;
        const int tu = A.taps_u - 1 - (fu > A.last_u), tv = A.taps_v - 1 - (fv > A.last_v);
        const int iu_hi = min(min(wsu - scu - 1, tu - qu), r1 - 1 - cu);
        const int iv_lo = max(max(-scv, -qv), -cv);
        const int iv_hi = min(min(wsv - scv - 1, tv - qv), TV - 1 - cv);
        if (plive && iu_hi >= iu_lo && iv_hi >= iv_lo) {
          pw = iv_hi - iv_lo + 1;
          pn = (iu_hi - iu_lo + 1) * pw;
          pcfoff = idx * cfsize +
                   (A.by_phase ? fu * A.phase_u + fv * A.phase_v + (qu + iu_lo) * A.tap_u +
                                     qv + iv_lo
                               : (A.ov_u * iu_lo + cfu0) * A.cv_n + A.ov_v * iv_lo + cfv0);
          pcell0 = (cu + iu_lo) * TV + cv + iv_lo;
          prw = (1.0f / (float)pw) * (1.0f + 0x1p-20f);
        }
      }
    }
    // ---- the records with taps here, one after another; lanes over the
    // taps, v fastest.  A record's kernel values are loaded while the one
    // before it is added, two records of registers taking turns.
    uint64_t live = __ballot(pn > 0);
    const uint64_t part = __ballot(pn > 0 && plive != kAll);  // not every polarisation
    const auto add = [&](const MosaicTap<R> &m, int k) {
      R dre[NPOL], dim[NPOL];
#pragma unroll
      for (int p = 0; p < NPOL; ++p) {
        dre[p] = lane_value(pdre[p], k);
        dim[p] = lane_value(pdim[p], k);
      }
      const unsigned pols =
          !by_pol && part >> k & 1 ? (unsigned)lane_value((int)plive, k) : kAll;
      if (pols == kAll) {
        if (lane < m.n) add_pols(m.at, m.c, dre, dim, kAll);
      } else {
        if (lane < m.n) add_pols(m.at, m.c, dre, dim, pols);
      }
      if (m.n > 64) {
        const int w = lane_value(pw, k), cell0 = lane_value(pcell0, k);
        const float rw = lane_value(prw, k);
        const Cplx2<R> *cf = (const Cplx2<R> *)A.taps + lane_value(pcfoff, k);
        for (int t = lane + 64; t < m.n; t += 64) {
          int at;
          const uint32_t off = tap_of(t, w, rw, cell0, TV, A, at);
          add_pols(at, cf[off], dre, dim, pols);
        }
      }
    };
    MosaicTap<R> ta, tb;
    int ka = 0, kb = 0;
    if (live) {
      ka = __builtin_ctzll(live);
      ta.load(ka, lane, pn, pw, pcfoff, pcell0, prw, A, TV);
    }
    while (live) {
      live &= live - 1;
      // with no record left, the last is loaded once more and not added
      kb = live ? __builtin_ctzll(live) : ka;
      tb.load(kb, lane, pn, pw, pcfoff, pcell0, prw, A, TV);
      add(ta, ka);
      if (!live) break;
      live &= live - 1;
      ka = live ? __builtin_ctzll(live) : kb;
      ta.load(ka, lane, pn, pw, pcfoff, pcell0, prw, A, TV);
      add(tb, kb);
    }
  }
  if (by_pol) __syncthreads();
  // ---- flush these rows of the tile (cells outside the grid dropped); a
  // lane's row and column step along, 64 cells at a time
  const bool multi = (fl & kUnitMulti) != 0;
  int row = lane / TV, col = lane - row * TV;
  row += s0;
  const int step_u = 64 / TV, step_v = 64 - step_u * TV;
  for (int i = s0 * TV + lane; i < s1 * TV; i += 64) {
    const int gu = u0 + row, gv = v0 + col;
    if (gu < P.n_u && gv < P.n_v) {
      R *dst = gplane + ((size_t)gu * P.n_v + gv) * 2;
#pragma unroll
      for (int a = 0; a < kParts; ++a) {
        const Cell val = cnt > 0 ? tile[a * cells + i] : Cell{};
#pragma unroll
        for (int p = 0; p < kPols; ++p, dst += pstride) {
          if (multi) {
            if (val.v[p].re != (R)0) atomicAdd(dst, val.v[p].re);
            if (val.v[p].im != (R)0) atomicAdd(dst + 1, val.v[p].im);
          } else if (accumulate) {
            dst[0] += val.v[p].re;
            dst[1] += val.v[p].im;
          } else {
            dst[0] = val.v[p].re;
            dst[1] = val.v[p].im;
          }
        }
      }
    }
    row += step_u;
    col += step_v;
    if (col >= TV) {
      col -= TV;
      ++row;
    }
  }
  for (int off = 32; off >= 1; off >>= 1) swl += __shfl_xor(swl, off);
  if (lane == 0) P.upart[(size_t)u * 4 + wp] = swl;
}

template <typename R, int NPOL>
static int launch_mosaic(av_plan *plan, MosaicArgs<R> A, double *sumwt, int mode,
                         hipStream_t s) {
  PlanDev &d = plan->d;
  const size_t lds = (size_t)d.tile_u * d.tile_v * NPOL * sizeof(Cplx2<R>);
  const DeviceProps &prop = device_props();
  if (prop.error) return hip_fail(prop.error, "av_mosaic_grid: device properties");
  if (lds > prop.lds_per_block)
    return fail(AV_ERR_UNSUPPORTED, "av_mosaic_grid: tile too large for LDS (" +
                                        std::to_string(lds) + " bytes)");
  {
    const int rc = ensure_lds_limit<k_mosaic_grid<R, NPOL>>((int)lds,
                                                            "av_mosaic_grid: hipFuncSetAttribute");
    if (rc) return rc;
  }
  const bool accumulate = (mode & AV_GRID_ACCUMULATE) != 0;
  if (!accumulate) {
    const int rc = prepare_grid(d, nullptr, A.grid, NPOL, sizeof(R) == 8, sumwt, s);
    if (rc) return rc;
  }
  // the kernel-sum table, in stream-ordered memory freed after the gridder
  // (first-tap offsets: floor(x * ov + 0.5) for x in (-1/2, 1/2], within
  // [-ov / 2 - 1, ov / 2 + 1])
  const int64_t ncf = (int64_t)A.ncb * A.ncc * A.ncp;
  if (ncf * A.cu_n * A.cv_n >= (int64_t)1 << 31)
    return fail(AV_ERR_UNSUPPORTED, "av_mosaic_grid: convolution functions of 2^31 elements or more");
  if ((int64_t)A.ov_u * A.cv_n >= 1 << 24 || A.ov_v >= 1 << 24)
    return fail(AV_ERR_UNSUPPORTED, "av_mosaic_grid: ov_u * cv_n must be below 2^24");
  if (d.tile_u * d.tile_v > 1 << 16)
    return fail(AV_ERR_UNSUPPORTED, "av_mosaic_grid: tile of more than 2^16 cells");
  A.du_lo = -(A.ov_u / 2) - 1;
  A.ndu = A.ov_u + 3;
  A.dv_lo = -(A.ov_v / 2) - 1;
  A.ndv = A.ov_v + 3;
  const int64_t entries = ncf * A.ndu * A.ndv;
  // The kernel values by phase where the samples are worth the pass over the
  // table and it has room: else the caller's order is read.  By phase and in
  // order, FP32: 8 k samples x 2 polarisations on 4 planes of 1024^2 and 0.1 M
  // kernel values 88 and 80 us, 10.8 M 216 and 102; 97 k and 4.8 M 267 and 231, 1.6
  // M at oversampling 32 204 and 232; 403 k and 0.1 M 328 and 339, 10.8 M 510 and
  // 471 (FP64 810 and 866), 1.6 M at oversampling 32 323 and 586; 65 k samples on
  // 32 planes of 768^2 and 0.1 M 168 and 183.
  const int64_t tu = ((int64_t)A.cu_n + A.ov_u - 1) / A.ov_u;
  const int64_t tv = ((int64_t)A.cv_n + A.ov_v - 1) / A.ov_v;
  A.taps_u = (int)tu;
  A.taps_v = (int)tv;
  A.last_u = (int)(A.cu_n - 1 - (tu - 1) * A.ov_u);
  A.last_v = (int)(A.cv_n - 1 - (tv - 1) * A.ov_v);
  const int64_t pad_u = tu * A.ov_u, pad_v = tv * A.ov_v;
  const bool phases = d.n_items >= kPhaseSamples &&
                      ncf * A.cu_n * A.cv_n <= kPhaseValues * d.n_items &&
                      pad_v < ((int64_t)1 << 31) / pad_u &&
                      pad_u * pad_v < ((int64_t)1 << 31) / ncf;
  const int64_t pad = phases ? ncf * pad_u * pad_v : 0;
  // one stream-ordered block: the kernel sums, max(weight_support), then the
  // kernel values by phase
  const size_t head = (size_t)entries * 2 * sizeof(double) + 16;
  void *norms = nullptr;
  hipError_t me = hipMallocAsync(&norms, head + (size_t)pad * sizeof(Cplx2<R>), s);
  A.by_phase = phases;
  if (me != hipSuccess && phases) {
    (void)hipGetLastError();
    A.by_phase = 0;
    me = hipMallocAsync(&norms, head, s);
  }
  if (me != hipSuccess) return hip_fail(me, "av_mosaic_grid: hipMallocAsync");
  A.norms = (const double *)norms;
  int *msup = (int *)((char *)norms + (size_t)entries * 2 * sizeof(double));
  A.max_support = msup;
  if (A.by_phase) {
    R *taps = (R *)((char *)norms + head);
    A.taps = taps;
    A.tap_u = (int)tv;
    A.tap_v = 1;
    A.phase_v = (int)(tu * tv);
    A.phase_u = (int)(A.ov_v * tu * tv);
    A.tap_cf = pad_u * pad_v;
    hipLaunchKernelGGL((k_mosaic_phases<R>), dim3((unsigned)((pad + 255) / 256)), dim3(256), 0, s,
                       A, pad, taps);
  } else {
    A.taps = A.cfpg;
    A.tap_u = A.ov_u * A.cv_n;
    A.tap_v = A.ov_v;
    A.tap_cf = (int64_t)A.cu_n * A.cv_n;
  }
  hipLaunchKernelGGL((k_mosaic_norms<R>), dim3((unsigned)((entries + 255) / 256)), dim3(256), 0, s,
                     A, (int)ncf);
  int rc = hipGetLastError() == hipSuccess ? AV_OK : fail(AV_ERR_HIP, "k_mosaic_norms launch");
  if (rc == AV_OK) {
    hipLaunchKernelGGL(k_mosaic_max_support, dim3(1), dim3(256), 0, s, A.weight_support,
                       (int)(2 * ncf), msup);
    if (hipGetLastError() != hipSuccess) rc = fail(AV_ERR_HIP, "k_mosaic_max_support launch");
  }
  if (rc == AV_OK) {
    hipLaunchKernelGGL((k_mosaic_grid<R, NPOL>),
                       dim3((unsigned)xcd_grouped_grid(d.max_gunits, kMosaicGroup)),
                       dim3(64 * NPOL), lds, s, d, A, (mode & AV_GRID_PSF) ? 1 : 0,
                       accumulate ? 1 : 0);
    if (hipGetLastError() != hipSuccess) rc = fail(AV_ERR_HIP, "k_mosaic_grid launch");
  }
  const hipError_t fe = hipFreeAsync(norms, s);
  if (rc) return rc;
  if (fe != hipSuccess) return hip_fail(fe, "av_mosaic_grid: hipFreeAsync");
  return reduce_sumwt(d, NPOL, sumwt, s);
}

template <typename R>
static int mosaic_by_pol(av_plan *plan, MosaicArgs<R> A, int npol, double *sumwt, int mode,
                         hipStream_t s) {
  switch (npol) {
    case 1: return launch_mosaic<R, 1>(plan, A, sumwt, mode, s);
    case 2: return launch_mosaic<R, 2>(plan, A, sumwt, mode, s);
    case 4: return launch_mosaic<R, 4>(plan, A, sumwt, mode, s);
    default: return fail(AV_ERR_UNSUPPORTED, "av_mosaic_grid: npol must be 1, 2 or 4");
  }
}

}  // namespace av

using namespace av;

extern "C" int av_mosaic_grid(av_plan *plan, const void *vis, const void *weight, int32_t n_pol,
                              int32_t n_baseline, const int32_t *cf_baseline_map,
                              const int32_t *cf_chan_map, const int32_t *cf_pol_map,
                              const void *cfpg, int32_t ncb, int32_t ncc, int32_t ncp,
                              int32_t cu_n,
                              int32_t cv_n, const int32_t *weight_support, int32_t ov_u,
                              int32_t ov_v, void *grid, double *sumwt, int32_t dtype,
                              int32_t mode, void *stream) {
  if (!plan || !weight || !cf_baseline_map || !cf_chan_map || !cf_pol_map || !cfpg ||
      !weight_support || !grid || !sumwt)
    return fail(AV_ERR_INVALID, "av_mosaic_grid: NULL argument");
  const bool psf = (mode & AV_GRID_PSF) != 0;
  if (!psf && !vis) return fail(AV_ERR_INVALID, "av_mosaic_grid: vis is NULL");
  if (mode & ~(AV_GRID_PSF | AV_GRID_ACCUMULATE))
    return fail(AV_ERR_UNSUPPORTED, "av_mosaic_grid: mode takes AV_GRID_PSF and "
                                    "AV_GRID_ACCUMULATE only");
  const PlanDev &d = plan->d;
  if (!d.uvw) return fail(AV_ERR_INVALID, "av_mosaic_grid: plan has no uvw (av_plan_set_uvw)");
  if (d.row_channels || d.geometry != AV_GEOM_REFERENCE || d.conjugate)
    return fail(AV_ERR_UNSUPPORTED, "av_mosaic_grid: needs an AV_GEOM_REFERENCE plan "
                                    "without row channels");
  if (n_baseline < 1 || d.n_rows % n_baseline != 0)
    return fail(AV_ERR_INVALID, "av_mosaic_grid: n_baseline must divide the plan's rows");
  if (ncb < 1 || ncc < 1 || ncp < 1 || cu_n < 1 || cv_n < 1 || ov_u < 1 || ov_v < 1)
    return fail(AV_ERR_INVALID, "av_mosaic_grid: bad convolution-function shape");
  hipStream_t s = (hipStream_t)stream;
  if (dtype == AV_F32) {
    MosaicArgs<float> A{(const float *)vis, (const float *)weight, cf_baseline_map, cf_chan_map,
                        cf_pol_map, (const float *)cfpg, weight_support, n_baseline, ncb, ncc,
                        ncp, cu_n, cv_n, ov_u, ov_v, (float *)grid, nullptr, 0, 0, 0, 0};
    return mosaic_by_pol<float>(plan, A, n_pol, sumwt, mode, s);
  }
  if (dtype == AV_F64) {
    MosaicArgs<double> A{(const double *)vis, (const double *)weight, cf_baseline_map,
                         cf_chan_map, cf_pol_map, (const double *)cfpg, weight_support,
                         n_baseline, ncb, ncc, ncp, cu_n, cv_n, ov_u, ov_v, (double *)grid,
                         nullptr, 0, 0, 0, 0};
    return mosaic_by_pol<double>(plan, A, n_pol, sumwt, mode, s);
  }
  return fail(AV_ERR_INVALID, "av_mosaic_grid: dtype must be AV_F32 or AV_F64");
}

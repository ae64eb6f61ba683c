// plan.hip -- binning of samples into (uv tile, image channel) bins.
//
// A sample is one (row, channel) pair with all its polarisations.  Its grid
// centre (standard_grid.py:322-352) and degrid centre
// (standard_degrid.py:435-462) are computed once, in FP64, here.  The sample
// is recorded in the bin of its anchor tile ("primary" record, carrying both
// geometries) and, for gridding, in every other tile its support footprint
// overlaps ("duplicate" records), so that each tile of the grid is produced
// by exactly one owner with no halo exchange.  Within a bin, primary records
// come first.  Bins are ordered tile-major, channel-minor, so neighbouring
// channels of the same rows are processed close together in time; where rows
// carry their own channel, channels share no samples, and bins are ordered
// channel-major instead: the units at work at one time then gather from few
// channels' samples, and a block of rows counts and places its records in one
// stretch of bins (96 planes of 512 x 512 with 20 million samples, supports 9,
// 7 and 5: FP32 gridders 715, 628 and 608 us channel-minor, 449, 419 and 416
// channel-major; binning 432, 407 and 426 -> 347, 326 and 341, and 314, 300
// and 304 with the block's own channel constants at hand).
//
// Binning is a counting sort.  The counts come from chunks (one channel, a
// range of rows) gathered in LDS when a channel's tiles fit there, else from
// global atomics (very many tiles).  The records are then written with one
// cursor per bin, the samples taken in order so that the records a
// wavefront writes land in neighbouring bins.  When rows carry their own
// channel, blocks of consecutive rows count and place their records through
// per-tile counters and cursors in LDS instead (row-block binning).  Validity bitmasks are channel-major: bit (chan, row) is
// bit row % 64 of word chan * ceil(n_rows / 64) + row / 64 (chan 0 when
// every row carries its own channel).
#include <algorithm>

#include "tile_common.h"

namespace av {

struct ItemGeo {
  int64_t row;
  int chan, ic;
  bool gvalid, dvalid;
  int iu, iv, ou, ov;  // grid centre and kernel offsets
  int lu, lv, fu, fv;  // degrid centre and kernel offsets
};

// The per-channel constants of the geometry: loaded once per channel where
// a loop visits many rows of one channel (the chunked binning passes),
// instead of once per sample behind the sample's own loads.
struct ChanGeo {
  int chan, ic, ch;  // channel, image channel, channel the tables are read at
  bool ok;           // both in range
  double freq, gsu, gsv;
};

__device__ inline ChanGeo chan_geo(const PlanDev &P, int chan) {
  ChanGeo c;
  c.chan = chan;
  c.ok = chan >= 0 && chan < P.n_chan;
  c.ch = c.ok ? chan : 0;
  c.ic = P.chan_map[c.ch];
  c.ok = c.ok && c.ic >= 0 && c.ic < P.n_img_chan;
  c.freq = P.freq[c.ch];
  c.gsu = P.gscale_u[c.ch];
  c.gsv = P.gscale_v[c.ch];
  return c;
}

// Geometry of the sample of row `row` at channel c, whose u and v are uu
// and vv.
__device__ inline void sample_geometry_at(const PlanDev &P, int64_t row, const ChanGeo &c,
                                          double uu, double vv, ItemGeo &g) {
  g.row = row;
  g.chan = c.chan;
  g.ic = c.ic;
  const bool chan_ok = c.ok;
  const int sc = P.support / 2;
  g.dvalid = degrid_geometry(uu, vv, c.freq, P.dscale_u, P.dscale_v, P.doff_u, P.doff_v,
                             P.n_u, P.n_v, P.support, P.ov, g.lu, g.lv, g.fu, g.fv) &&
             chan_ok;
  if (P.geometry == AV_GEOM_DEGRID) {
    g.gvalid = g.dvalid;
    g.iu = g.lu;
    g.iv = g.lv;
    g.ou = g.fu;
    g.ov = g.fv;
  } else {
    g.gvalid = grid_geometry(uu, vv, c.gsu, c.gsv, P.n_u, P.n_v, sc, P.ov, g.iu, g.iv, g.ou,
                             g.ov) &&
               chan_ok;
    if (P.conjugate) {
      // the second scatter of do_imaging_weight (standard_grid.py:330-340,
      // 389-425): the conjugate centre int(-u + N/2 + 0.5), the sample's own
      // kernel offsets and bounds test, no degrid record
      g.dvalid = false;
      if (g.gvalid) {
        const double u = uu * c.gsu, v = vv * c.gsv;
        g.iu = (int)(-u + (double)(P.n_u / 2) + 0.5);
        g.iv = (int)(-v + (double)(P.n_v / 2) + 0.5);
      }
    }
  }
}

// Geometry of the sample of row `row` at channel `chan` (the row's own
// channel when rows carry one).
__device__ inline void sample_geometry(const PlanDev &P, int64_t row, int chan, ItemGeo &g) {
  const ChanGeo c = chan_geo(P, P.row_chan ? P.row_chan[row] : chan);
  sample_geometry_at(P, row, c, P.uvw[row * 3 + 0], P.uvw[row * 3 + 1], g);
}

__device__ inline int64_t bin_of(const PlanDev &P, int tu, int tv, int ic) {
  return bin_number(P, (int64_t)tu * P.ntv + tv, ic);
}

// One channel's constants into the plan.
__device__ inline void setup_channel(const PlanDev &P, const double *freq,
                                     const int32_t *chan_map, int c) {
  double f = freq[c];
  P.freq[c] = f;
  // numpy: -(freq_chan * delta_lm[0] * n_uv[0]) / c   (standard_grid.py:298-299)
  P.gscale_u[c] = -(f * P.cell_u * (double)P.n_u) / kLightSpeed;
  P.gscale_v[c] = -(f * P.cell_v * (double)P.n_v) / kLightSpeed;
  int m;
  if (chan_map)
    m = chan_map[c];
  else
    m = (P.n_img_chan == P.n_chan) ? c : 0;
  P.chan_map[c] = m;
}

__global__ void k_chan_setup(PlanDev P, const double *freq, const int32_t *chan_map) {
  int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < P.n_chan) setup_channel(P, freq, chan_map, c);
}

// Records of one sample.  A grid-valid sample gets a primary record in the
// tile of its grid centre (carrying the degrid geometry too when the two
// centres are within one pixel, which is always the case for the reference
// transforms) and a duplicate in every other tile its footprint overlaps.
// A degrid-valid sample whose degrid centre is elsewhere (a caller-supplied
// degrid transform) gets its own primary record in the tile of that centre.
struct RecPlan {
  bool gprim, dsep;        // grid-primary record, separate degrid record
  bool share;              // grid-primary record also carries degrid geometry
  int tu, tv, du_t, dv_t;  // grid anchor tile, degrid anchor tile
  int tu0, tu1, tv0, tv1;  // tiles overlapped by the grid footprint
};

__device__ inline int tile_u_of(const PlanDev &P, int x) {
  return (int)__umulhi((uint32_t)x, P.tile_u_mul);
}
__device__ inline int tile_v_of(const PlanDev &P, int x) {
  return (int)__umulhi((uint32_t)x, P.tile_v_mul);
}

__device__ inline RecPlan record_plan(const PlanDev &P, const ItemGeo &g) {
  RecPlan r;
  const int sc = P.support / 2;
  r.gprim = g.gvalid;
  r.share = g.gvalid && g.dvalid && abs(g.lu - g.iu) <= 1 && abs(g.lv - g.iv) <= 1;
  r.dsep = g.dvalid && !r.share;
  r.tu = r.tv = r.du_t = r.dv_t = 0;
  r.tu0 = r.tu1 = r.tv0 = r.tv1 = 0;
  if (g.gvalid) {
    // tile numbers by multiply-high of positions clamped into [0, n) (n <
    // 2^24): a valid footprint lies inside the grid, a conjugate one may
    // reach past an edge, whose cells are dropped
    r.tu = tile_u_of(P, min(max(g.iu, 0), P.n_u - 1));
    r.tv = tile_v_of(P, min(max(g.iv, 0), P.n_v - 1));
    r.tu0 = tile_u_of(P, max(g.iu - sc, 0));
    r.tu1 = tile_u_of(P, min(g.iu + P.support - sc - 1, P.n_u - 1));
    r.tv0 = tile_v_of(P, max(g.iv - sc, 0));
    r.tv1 = tile_v_of(P, min(g.iv + P.support - sc - 1, P.n_v - 1));
  }
  if (r.dsep) {
    r.du_t = tile_u_of(P, g.lu);
    r.dv_t = tile_v_of(P, g.lv);
  }
  return r;
}

__device__ inline int64_t item_index(const PlanDev &P, int64_t row, int chan) {
  return P.row_chan ? row : row * P.n_chan + chan;
}

// The validity bits of a wavefront's 64 consecutive rows of one channel
// (rows from a multiple of 64): one mask word, written by lane 0.
__device__ inline void write_masks(const PlanDev &P, int64_t row, int chan, bool gvalid,
                                   bool dvalid) {
  const unsigned long long gm = __ballot(gvalid), dm = __ballot(dvalid);
  const int64_t first = row - __lane_id();
  if (__lane_id() == 0 && first < P.n_rows) {
    const int64_t w = (P.row_chan ? 0 : (int64_t)chan * P.mask_words_per_chan) + first / 64;
    P.gmask[w] = gm;
    P.dmask[w] = dm;
  }
}

// The records of one sample counted straight into the global bins.
__device__ inline void count_global(const PlanDev &P, const ItemGeo &g, const RecPlan &rp) {
  if (rp.gprim) {
    const int64_t pb = bin_of(P, rp.tu, rp.tv, g.ic);
    atomicAdd(&P.cnt_prim[pb], 1u);
    atomicAdd(&P.cnt_all[pb], 1u);
    for (int a = rp.tu0; a <= rp.tu1; ++a)
      for (int b = rp.tv0; b <= rp.tv1; ++b)
        if (a != rp.tu || b != rp.tv) atomicAdd(&P.cnt_all[bin_of(P, a, b, g.ic)], 1u);
  }
  if (rp.dsep) {
    const int64_t db = bin_of(P, rp.du_t, rp.dv_t, g.ic);
    atomicAdd(&P.cnt_prim[db], 1u);
    atomicAdd(&P.cnt_all[db], 1u);
  }
}

// Global-atomic binning, pass 1: count records per bin.  Threads walk the
// (channel, row) space with rows padded to a multiple of 64 per channel.
__global__ __launch_bounds__(256) void k_count(PlanDev P) {
  const int64_t rows_pad = P.mask_words_per_chan * 64;
  const int nch = P.row_chan ? 1 : P.n_chan;
  const int64_t total = rows_pad * nch;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;  // a multiple of 64
  for (int64_t it = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; it < total; it += stride) {
    const int chan = (int)(it / rows_pad);
    const int64_t row = it - (int64_t)chan * rows_pad;
    ItemGeo g;
    g.gvalid = g.dvalid = false;
    if (row < P.n_rows) sample_geometry(P, row, chan, g);
    write_masks(P, row, chan, g.gvalid, g.dvalid);
    if (!(g.gvalid || g.dvalid)) continue;
    count_global(P, g, record_plan(P, g));
  }
}

// One store per record: 12 bytes for a primary record, 8 for a duplicate
// (degrid units cover the primary records of a bin only, so a duplicate's
// degrid word is never read).
__device__ inline void write_records(const PlanDev &P, const ItemGeo &g, const RecPlan &rp,
                                     int64_t item, uint32_t slot, int a, int b, bool primary) {
  const int u0 = a * P.tile_u, v0 = b * P.tile_v;
  uint32_t *dst = P.rec + 3 * (size_t)slot;
  const uint32_t gg = pack_geo(g.iu - u0, g.ou, g.iv - v0, g.ov);
  if (primary) {
    const uint32_t dg = rp.share ? pack_geo(g.lu - u0, g.fu, g.lv - v0, g.fv) : kInvalidGeo;
    *(RecWords *)dst = RecWords{(uint32_t)item, gg, dg};
  } else {
    *(RecGridWords *)dst = RecGridWords{(uint32_t)item, gg};
  }
}

__device__ inline void write_degrid_record(const PlanDev &P, const ItemGeo &g, const RecPlan &rp,
                                           int64_t item, uint32_t slot) {
  const int u0 = rp.du_t * P.tile_u, v0 = rp.dv_t * P.tile_v;
  *(RecWords *)(P.rec + 3 * (size_t)slot) =
      RecWords{(uint32_t)item, kInvalidGeo, pack_geo(g.lu - u0, g.fu, g.lv - v0, g.fv)};
}

// The records of one sample, their slots taken from the global bin cursors.
__device__ inline void scatter_global(const PlanDev &P, const ItemGeo &g, const RecPlan &rp,
                                      int64_t item) {
  if (rp.gprim) {
    const uint32_t slot = atomicAdd(&P.cur_prim[bin_of(P, rp.tu, rp.tv, g.ic)], 1u);
    write_records(P, g, rp, item, slot, rp.tu, rp.tv, true);
    for (int a = rp.tu0; a <= rp.tu1; ++a)
      for (int b = rp.tv0; b <= rp.tv1; ++b)
        if (a != rp.tu || b != rp.tv) {
          const uint32_t s2 = atomicAdd(&P.cur_dup[bin_of(P, a, b, g.ic)], 1u);
          write_records(P, g, rp, item, s2, a, b, false);
        }
  }
  if (rp.dsep) {
    const uint32_t slot = atomicAdd(&P.cur_prim[bin_of(P, rp.du_t, rp.dv_t, g.ic)], 1u);
    write_degrid_record(P, g, rp, item, slot);
  }
}

// Binning pass 2: write the records, taking slots from the bins' cursors.
// Threads walk the samples in order, so a wavefront covers the channels of
// one or a few rows: their bins are neighbours (bins are channel-minor) and
// so are the records they write.
__global__ __launch_bounds__(256) void k_scatter(PlanDev P) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t item = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; item < P.n_items;
       item += stride) {
    int64_t row = item;
    int chan = 0;
    if (!P.row_chan) {  // samples number below 2^32: a 32-bit division
      const uint32_t r32 = (uint32_t)item / (uint32_t)P.n_chan;
      row = r32;
      chan = (int)((uint32_t)item - r32 * (uint32_t)P.n_chan);
    }
    ItemGeo g;
    sample_geometry(P, row, chan, g);
    if (!(g.gvalid || g.dvalid)) continue;
    scatter_global(P, g, record_plan(P, g), item);
  }
}

// ---- chunked binning ------------------------------------------------------
// A chunk is rows [r0, r0 + rows_per_chunk) of one channel.  Per tile it
// counts primaries (chunk_hist) and duplicates (chunk_dup), 32 bits each.

// Chunked pass 1: per-tile counts of one chunk, gathered in LDS.  The
// workgroup first forms its channels' constants (every chunk of a channel
// writes the same values), so no launch of their own precedes this one.  A
// wavefront takes 64 consecutive rows of one channel at a time.
template <bool ALL>
__global__ __launch_bounds__(kChunkThreads) void k_count_chunks(PlanDev P, const double *freq,
                                                                const int32_t *chan_map) {
  extern __shared__ uint32_t h[];  // [n_tiles] primaries, then [n_tiles] duplicates
  const int64_t w = blockIdx.x;
  const int chan0 = ALL ? 0 : (int)(w / P.chunks_per_chan);
  const int64_t r0 = (w - (int64_t)chan0 * P.chunks_per_chan) * P.rows_per_chunk;
  const int ntiles = P.ntu * P.ntv;
  uint32_t *hd = h + ntiles;
  if (ALL) {
    for (int c = threadIdx.x; c < P.n_chan; c += blockDim.x) setup_channel(P, freq, chan_map, c);
  } else if (threadIdx.x == 0) {
    setup_channel(P, freq, chan_map, chan0);
  }
  for (int i = threadIdx.x; i < 2 * ntiles; i += blockDim.x) h[i] = 0u;
  __syncthreads();
  const int nch = ALL ? P.n_chan : 1;
  const uint32_t groups = (uint32_t)P.rows_per_chunk / 64u;  // 64-row groups of the chunk
  const uint32_t waves = blockDim.x / 64u;
  int chan = chan0;
  uint32_t grp = threadIdx.x / 64u;
  while (grp >= groups) {
    grp -= groups;
    ++chan;
  }
  ChanGeo cg = chan_geo(P, min(chan, P.n_chan - 1));
  while (chan < chan0 + nch) {
    const int64_t row = r0 + grp * 64u + __lane_id();
    ItemGeo g;
    g.gvalid = g.dvalid = false;
    if (row < P.n_rows) sample_geometry_at(P, row, cg, P.uvw[row * 3 + 0], P.uvw[row * 3 + 1], g);
    write_masks(P, row, chan, g.gvalid, g.dvalid);
    if (g.gvalid || g.dvalid) {
      const RecPlan rp = record_plan(P, g);
      if (rp.gprim) {
        atomicAdd(&h[rp.tu * P.ntv + rp.tv], 1u);
        for (int a = rp.tu0; a <= rp.tu1; ++a)
          for (int b = rp.tv0; b <= rp.tv1; ++b)
            if (a != rp.tu || b != rp.tv) atomicAdd(&hd[a * P.ntv + b], 1u);
      }
      if (rp.dsep) atomicAdd(&h[rp.du_t * P.ntv + rp.dv_t], 1u);
    }
    grp += waves;
    if (grp >= groups) {
      do {
        grp -= groups;
        ++chan;
      } while (grp >= groups);
      if (ALL) cg = chan_geo(P, min(chan, P.n_chan - 1));
    }
  }
  __syncthreads();
  uint32_t *dst = P.chunk_hist + w * ntiles, *dstd = P.chunk_dup + w * ntiles;
  for (int i = threadIdx.x; i < ntiles; i += blockDim.x) {
    dst[i] = h[i];
    dstd[i] = hd[i];
  }
}

// The runs of tile t that image channel ic gathers, those of one segment
// `seg` of `nseg`: segments split the row-chunks.  When image channels gather
// several channels (continuum), a segment takes its runs row-chunk by
// row-chunk, channel by channel within one: the channels of a row, which
// share cache lines, then lie a run apart in the bin instead of a whole
// channel's records apart.
// With `ident` every channel is its own image channel.
// f(i, n) takes n <= kRunBatch runs, the first at i and the others ntiles
// apart: their loads go out together.
constexpr int kRunBatch = 8;
template <typename F>
__device__ inline void chunk_runs(const PlanDev &P, bool ident, int ic, int t, int seg, int nseg,
                                  F f) {
  const int ntiles = P.ntu * P.ntv, K = P.chunks_per_chan;
  const int k0 = (int)((int64_t)K * seg / nseg), k1 = (int)((int64_t)K * (seg + 1) / nseg);
  if (P.chunk_all) {
    for (int k = k0; k < k1; k += kRunBatch)
      f((int64_t)k * ntiles + t, min(kRunBatch, k1 - k));
  } else if (P.n_img_chan < P.n_chan) {
    for (int k = k0; k < k1; ++k)
      for (int c = 0; c < P.n_chan; ++c)
        if (P.chan_map[c] == ic) f(((int64_t)c * K + k) * ntiles + t, 1);
  } else {
    for (int c = ident ? ic : 0; c < (ident ? ic + 1 : P.n_chan); ++c) {
      if (!ident && P.chan_map[c] != ic) continue;
      for (int k = k0; k < k1; k += kRunBatch)
        f(((int64_t)c * K + k) * ntiles + t, min(kRunBatch, k1 - k));
    }
  }
}

// Whether every channel is its own image channel, found by a whole wavefront.
__device__ inline bool chan_identity(const PlanDev &P) {
  bool same = P.n_img_chan == P.n_chan;
  for (int c = (int)__lane_id(); same && c < P.n_chan; c += 64) same = P.chan_map[c] == c;
  return __all(same);
}

// Counts of a batch of runs added to (sp, sd).
__device__ inline void add_runs(const PlanDev &P, int64_t i, int n, uint32_t &sp, uint32_t &sd) {
  const int ntiles = P.ntu * P.ntv;
  uint32_t np[kRunBatch], nd[kRunBatch];
#pragma unroll
  for (int u = 0; u < kRunBatch; ++u) {  // unconditional loads: all in flight
    np[u] = P.chunk_hist[i + (int64_t)min(u, n - 1) * ntiles];
    nd[u] = P.chunk_dup[i + (int64_t)min(u, n - 1) * ntiles];
  }
#pragma unroll
  for (int u = 0; u < kRunBatch; ++u) {
    sp += u < n ? np[u] : 0u;
    sd += u < n ? nd[u] : 0u;
  }
}

// The first slots of a batch of runs written over their counts; (sp, sd) are
// the first free slots before and after.
__device__ inline void place_runs(const PlanDev &P, int64_t i, int n, uint32_t &sp,
                                  uint32_t &sd) {
  const int ntiles = P.ntu * P.ntv;
  uint32_t np[kRunBatch], nd[kRunBatch];
#pragma unroll
  for (int u = 0; u < kRunBatch; ++u) {
    np[u] = P.chunk_hist[i + (int64_t)min(u, n - 1) * ntiles];
    nd[u] = P.chunk_dup[i + (int64_t)min(u, n - 1) * ntiles];
  }
#pragma unroll
  for (int u = 0; u < kRunBatch; ++u)
    if (u < n) {
      P.chunk_hist[i + (int64_t)u * ntiles] = sp;
      P.chunk_dup[i + (int64_t)u * ntiles] = sd;
      sp += np[u];
      sd += nd[u];
    }
}

// Chunked pass 2: the counts of every bin, summed over the chunks of the
// channels that map to its image channel.  A workgroup takes 64 tiles of one
// image channel, a wavefront one segment of their runs: a
// continuum bin has hundreds of runs, and one thread per bin leaves most of
// the chip idle while it walks them.
constexpr int kSegTiles = 64, kMaxSegs = 16;
__global__ void k_chunk_totals(PlanDev P) {
  __shared__ uint32_t part[2][kMaxSegs][kSegTiles];
  const int nbt = (P.ntu * P.ntv + kSegTiles - 1) / kSegTiles;
  const int ic = blockIdx.x / nbt, t = (blockIdx.x - ic * nbt) * kSegTiles + threadIdx.x;
  const int seg = threadIdx.y, nseg = blockDim.y;
  const bool ident = chan_identity(P);
  uint32_t sp = 0, sd = 0;
  if (t < P.ntu * P.ntv)
    chunk_runs(P, ident, ic, t, seg, nseg, [&](int64_t i, int n) { add_runs(P, i, n, sp, sd); });
  part[0][seg][threadIdx.x] = sp;
  part[1][seg][threadIdx.x] = sd;
  __syncthreads();
  if (seg != 0 || t >= P.ntu * P.ntv) return;
  for (int k = 1; k < nseg; ++k) {
    sp += part[0][k][threadIdx.x];
    sd += part[1][k][threadIdx.x];
  }
  const int64_t b = bin_number(P, t, ic);
  P.cnt_prim[b] = sp;
  P.cnt_all[b] = sp + sd;
}

// Chunked pass 3 (after the bin offsets): the first slot of every chunk's
// run in every bin.  The first primary slot overwrites the primary counts
// (chunk_hist), the first duplicate slot the duplicate counts (chunk_dup).
__global__ void k_chunk_bases(PlanDev P) {
  __shared__ uint32_t part[2][kMaxSegs][kSegTiles];
  const int nbt = (P.ntu * P.ntv + kSegTiles - 1) / kSegTiles;
  const int ic = blockIdx.x / nbt, t = (blockIdx.x - ic * nbt) * kSegTiles + threadIdx.x;
  const int seg = threadIdx.y, nseg = blockDim.y;
  const bool ident = chan_identity(P);
  const bool on = t < P.ntu * P.ntv;
  uint32_t sp = 0, sd = 0;
  if (on && nseg > 1)
    chunk_runs(P, ident, ic, t, seg, nseg, [&](int64_t i, int n) { add_runs(P, i, n, sp, sd); });
  part[0][seg][threadIdx.x] = sp;
  part[1][seg][threadIdx.x] = sd;
  __syncthreads();
  if (!on) return;
  const int64_t b = bin_number(P, t, ic);
  sp = P.bin_start[b];
  sd = sp + P.cnt_prim[b];
  for (int k = 0; k < seg; ++k) {
    sp += part[0][k][threadIdx.x];
    sd += part[1][k][threadIdx.x];
  }
  chunk_runs(P, ident, ic, t, seg, nseg, [&](int64_t i, int n) { place_runs(P, i, n, sp, sd); });
}

// Slots for one record per lane from the LDS cursors `cur` (key: the tile,
// or -1 for no record).  A lane whose key equals its left neighbour's joins
// that lane's run; the first lane of a run takes the whole run's slots with
// one LDS atomic, and the run's lanes get consecutive slots in lane order,
// so their record stores are contiguous.  Called by all 64 lanes together.
__device__ inline uint32_t run_slots(uint32_t *cur, int key) {
  if (__ballot(key >= 0) == 0ull) return 0u;
  const int lane = (int)__lane_id();
  const int left = __shfl_up(key, 1u);
  const bool start = lane == 0 || key != left;
  const unsigned long long starts = __ballot(start);
  const unsigned long long upto = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
  const int first = 63 - __clzll((long long)(starts & upto));
  const unsigned long long after = starts & ~upto;
  const int end = after ? __ffsll((long long)after) - 1 : 64;
  uint32_t base = 0u;
  if (start && key >= 0) base = atomicAdd(&cur[key], (uint32_t)(end - lane));
  return (uint32_t)__shfl((int)base, first) + (uint32_t)(lane - first);
}

// p / d for p, d < 2^32 by multiplication, with mul = ceil(2^32 / d):
// the product's high word is p / d or one more.
__device__ inline uint32_t div_by(uint32_t p, uint32_t d, uint64_t mul) {
  uint32_t q = (uint32_t)(((uint64_t)p * mul) >> 32);
  return (uint64_t)q * d > p ? q - 1 : q;
}

// Chunked pass 4: a workgroup per chunk writes the chunk's records.  Its
// runs' first slots are loaded into LDS cursors, and the records take their
// slots from LDS atomics, one per run of equal tiles in a wavefront: no
// global atomics.  When the rows are time-major with order_nb baselines per
// time step, the chunk's rows are visited baseline by baseline: a
// wavefront then holds consecutive times of one baseline, which mostly fall
// in the same tile, so its stores to a bin are contiguous.  A chunk of every
// channel (ALL) visits a row's channels before the next row: they mostly fall
// in one tile, so a bin's records run through contiguous samples, and the
// gridder's gathers and the degridder's stores are whole cache lines: on
// 725,760 rows x 48 channels x 2 polarisations, one 1800 x 1500 plane per
// polarisation, binning 1398 -> 969 us, the FP32 gridder 3788 -> 1421 us and
// the degridder 1403 -> 1160 us, against chunks of one channel.  Where a
// row's channels span many tiles its runs are shorter than a baseline's: 2.0 M
// rows x 64 channels x 4 polarisations on 2048 x 2048, the longest baseline at
// 1.8 half widths, bin in 4.29 ms instead of 3.24, grid in 6.99 instead of
// 9.87 (chunks of 8 channels: 3.93 and 7.04, but the first case 994 and 1275
// us, and 1338 us instead of 989 to grid one polarisation).
// (Numbering the chunks so that 16, 32 or 64 consecutive chunks of a channel
// share an XCD's L2 measured the same as plain numbering.)
template <bool ALL>
__global__ __launch_bounds__(kChunkThreads) void k_scatter_chunks(PlanDev P) {
  extern __shared__ uint32_t lds[];
  const int ntiles = P.ntu * P.ntv;
  uint32_t *cp = lds, *cd = lds + ntiles;  // [n_tiles] each
  const int64_t w = blockIdx.x;
  const int chan0 = ALL ? 0 : (int)(w / P.chunks_per_chan);
  const int64_t r0 = (w - (int64_t)chan0 * P.chunks_per_chan) * P.rows_per_chunk;
  const int64_t r1 = min(r0 + (int64_t)P.rows_per_chunk, P.n_rows);
  const uint32_t *bp = P.chunk_hist + w * ntiles, *bd = P.chunk_dup + w * ntiles;
  for (int i = threadIdx.x; i < ntiles; i += blockDim.x) {
    cp[i] = bp[i];
    cd[i] = bd[i];
  }
  __syncthreads();
  // positions p = b * nt + t over the nt time steps the chunk touches, row
  // (t_lo + t) * nb + b; rows outside [r0, r1) are skipped (nb = 1: p = row -
  // r0).  With ALL, position q = p * n_chan + channel.
  const int64_t nb = P.order_nb;
  const int64_t t_lo = r0 / nb;
  const uint32_t nt = (uint32_t)((r1 - 1) / nb - t_lo + 1);
  const uint32_t nch = ALL ? (uint32_t)P.n_chan : 1u;
  const uint32_t n_pos = nt * (uint32_t)nb * nch;
  const uint64_t nt_mul = ((1ull << 32) + nt - 1) / nt;
  const uint64_t nch_mul = ((1ull << 32) + nch - 1) / nch;
  ChanGeo cg = chan_geo(P, chan0);
  const uint32_t lane = __lane_id();
  for (uint32_t p0 = threadIdx.x - lane; p0 < n_pos; p0 += blockDim.x) {
    uint32_t p = p0 + lane;
    int64_t row = -1;
    int chan = chan0;
    if (p < n_pos) {
      if (ALL) {
        const uint32_t q = div_by(p, nch, nch_mul);
        chan = (int)(p - q * nch);
        p = q;
      }
      const uint32_t b = div_by(p, nt, nt_mul);
      const int64_t r = (t_lo + (int64_t)(p - b * nt)) * nb + b;
      if (r >= r0 && r < r1) row = r;
    }
    if (ALL) cg = chan_geo(P, chan);
    ItemGeo g;
    g.gvalid = g.dvalid = false;
    if (row >= 0) sample_geometry_at(P, row, cg, P.uvw[row * 3 + 0], P.uvw[row * 3 + 1], g);
    const RecPlan rp = record_plan(P, g);
    const int64_t item = row * P.n_chan + chan;
    const uint32_t slot = run_slots(cp, rp.gprim ? rp.tu * P.ntv + rp.tv : -1);
    if (rp.gprim) write_records(P, g, rp, item, slot, rp.tu, rp.tv, true);
    // duplicates: the other tiles of the footprint's (at most) 2 x 2 (a
    // tile is at least `support` wide), in a fixed order so that
    // neighbouring lanes' runs line up
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int a = (k & 2) ? rp.tu1 : rp.tu0, b = (k & 1) ? rp.tv1 : rp.tv0;
      const bool dup = rp.gprim && rp.tu0 <= rp.tu1 && rp.tv0 <= rp.tv1 &&
                       (!(k & 2) || rp.tu1 != rp.tu0) && (!(k & 1) || rp.tv1 != rp.tv0) &&
                       (a != rp.tu || b != rp.tv);
      const uint32_t s2 = run_slots(cd, dup ? a * P.ntv + b : -1);
      if (dup) write_records(P, g, rp, item, s2, a, b, false);
    }
    if (rp.dsep) {
      const uint32_t s3 = atomicAdd(&cp[rp.du_t * P.ntv + rp.dv_t], 1u);
      write_degrid_record(P, g, rp, item, s3);
    }
  }
}

// ---- row-block binning (rows carry their own channel) ---------------------
// A workgroup takes row_block_rows consecutive rows.  Rows of one plane are
// normally stored together, so the records of the block's "own" image
// channel (that of its first row) are gathered per tile in LDS and reach the
// global bins with one atomic per tile the block touches; the records of any
// other image channel take the global path.  This keeps the hot central
// tiles of a plane from being hit by every wavefront on the chip at once.

// Image channel of a row, or -1 when the row's channel is out of range.
__device__ inline int row_image_channel(const PlanDev &P, int64_t row) {
  if (row >= P.n_rows) return -1;
  const int c = P.row_chan[row];
  if (c < 0 || c >= P.n_chan) return -1;
  const int ic = P.chan_map[c];
  return (ic >= 0 && ic < P.n_img_chan) ? ic : -1;
}

// Geometry of a row that carries its channel, most often the block's own,
// whose constants are at hand.
__device__ inline void row_geometry(const PlanDev &P, int64_t row, const ChanGeo &own,
                                    ItemGeo &g) {
  const int c = P.row_chan[row];
  const double uu = P.uvw[row * 3 + 0], vv = P.uvw[row * 3 + 1];
  if (c == own.chan)
    sample_geometry_at(P, row, own, uu, vv, g);
  else
    sample_geometry_at(P, row, chan_geo(P, c), uu, vv, g);
}

// Row-block pass 1: per-tile counts, (primaries) | (duplicates << 16); a row
// adds at most two primaries and one duplicate to a tile and a block has
// at most kMaxRowBlockRows < 32768 rows, so neither half overflows.
__global__ __launch_bounds__(kChunkThreads) void k_count_rows(PlanDev P) {
  extern __shared__ uint32_t h[];  // [n_tiles]
  const int64_t r0 = (int64_t)blockIdx.x * P.row_block_rows;
  const int ntiles = P.ntu * P.ntv;
  const int own = row_image_channel(P, r0);
  const ChanGeo own_geo = chan_geo(P, r0 < P.n_rows ? P.row_chan[r0] : -1);
  for (int i = threadIdx.x; i < ntiles; i += blockDim.x) h[i] = 0u;
  __syncthreads();
  for (int64_t row = r0 + threadIdx.x; row < r0 + P.row_block_rows; row += blockDim.x) {
    ItemGeo g;
    g.gvalid = g.dvalid = false;
    if (row < P.n_rows) row_geometry(P, row, own_geo, g);
    write_masks(P, row, 0, g.gvalid, g.dvalid);
    if (!(g.gvalid || g.dvalid)) continue;
    const RecPlan rp = record_plan(P, g);
    if (g.ic != own) {
      count_global(P, g, rp);
      continue;
    }
    if (rp.gprim) {
      atomicAdd(&h[rp.tu * P.ntv + rp.tv], 1u);
      for (int a = rp.tu0; a <= rp.tu1; ++a)
        for (int b = rp.tv0; b <= rp.tv1; ++b)
          if (a != rp.tu || b != rp.tv) atomicAdd(&h[a * P.ntv + b], 1u << 16);
    }
    if (rp.dsep) atomicAdd(&h[rp.du_t * P.ntv + rp.dv_t], 1u);
  }
  __syncthreads();
  if (own < 0) return;
  uint32_t *keep = P.row_hist + (int64_t)blockIdx.x * ntiles;
  for (int i = threadIdx.x; i < ntiles; i += blockDim.x) {
    const uint32_t hv = h[i];
    keep[i] = hv;
    if (!hv) continue;
    const int64_t b = bin_number(P, i, own);
    const uint32_t np = hv & 0xFFFFu;
    if (np) atomicAdd(&P.cnt_prim[b], np);
    atomicAdd(&P.cnt_all[b], np + (hv >> 16));
  }
}

// Row-block pass 2: the block loads its own-channel counts per tile (kept by
// pass 1), reserves one run of slots per tile from each bin cursor
// (primaries and duplicates), and hands out the slots of each run from LDS
// cursors.
__global__ __launch_bounds__(kChunkThreads) void k_scatter_rows(PlanDev P) {
  extern __shared__ uint32_t lds[];
  const int ntiles = P.ntu * P.ntv;
  uint32_t *cp = lds, *cd = lds + ntiles;  // [n_tiles] each
  const int64_t r0 = (int64_t)blockIdx.x * P.row_block_rows;
  const int64_t r1 = min(r0 + (int64_t)P.row_block_rows, P.n_rows);
  const int own = row_image_channel(P, r0);
  const ChanGeo own_geo = chan_geo(P, r0 < P.n_rows ? P.row_chan[r0] : -1);
  if (own >= 0) {
    const uint32_t *kept = P.row_hist + (int64_t)blockIdx.x * ntiles;
    for (int i = threadIdx.x; i < ntiles; i += blockDim.x) {
      const uint32_t hv = kept[i];
      cp[i] = hv & 0xFFFFu;
      cd[i] = hv >> 16;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < ntiles; i += blockDim.x) {
      const int64_t b = bin_number(P, i, own);
      if (cp[i]) cp[i] = atomicAdd(&P.cur_prim[b], cp[i]);
      if (cd[i]) cd[i] = atomicAdd(&P.cur_dup[b], cd[i]);
    }
    __syncthreads();
  }
  for (int64_t row = r0 + threadIdx.x; row < r1; row += blockDim.x) {
    ItemGeo g;
    row_geometry(P, row, own_geo, g);
    if (!(g.gvalid || g.dvalid)) continue;
    const RecPlan rp = record_plan(P, g);
    if (g.ic != own) {
      scatter_global(P, g, rp, row);
      continue;
    }
    if (rp.gprim) {
      const uint32_t slot = atomicAdd(&cp[rp.tu * P.ntv + rp.tv], 1u);
      write_records(P, g, rp, row, slot, rp.tu, rp.tv, true);
      for (int a = rp.tu0; a <= rp.tu1; ++a)
        for (int b = rp.tv0; b <= rp.tv1; ++b)
          if (a != rp.tu || b != rp.tv) {
            const uint32_t s2 = atomicAdd(&cd[a * P.ntv + b], 1u);
            write_records(P, g, rp, row, s2, a, b, false);
          }
    }
    if (rp.dsep) {
      const uint32_t slot = atomicAdd(&cp[rp.du_t * P.ntv + rp.dv_t], 1u);
      write_degrid_record(P, g, rp, row, slot);
    }
  }
}

// Pair units: the bins of tiles 2j and 2j + 1 (along v) of pair p, and the
// primary records of both.
__device__ inline void pair_bins(const PlanDev &P, int64_t p, int64_t &b0, int64_t &b1,
                                 bool &has1, uint32_t &n) {
  const int ntv2 = (P.ntv + 1) / 2;
  const int64_t per = P.chan_major ? (int64_t)P.ntu * ntv2 : P.n_img_chan, q = p / per;
  const int64_t tp = P.chan_major ? p - q * per : q;
  const int ic = (int)(P.chan_major ? q : p - q * per);
  const int tu = (int)(tp / ntv2), tv = 2 * (int)(tp - (int64_t)tu * ntv2);
  b0 = bin_of(P, tu, tv, ic);
  has1 = tv + 1 < P.ntv;
  b1 = has1 ? bin_of(P, tu, tv + 1, ic) : b0;
  n = P.cnt_prim[b0] + (has1 ? P.cnt_prim[b1] : 0u);
}

// ---- bin offsets and work units --------------------------------------------
// From the bins' counts: the offsets of their records, the grid units (every
// bin has one, an empty bin still owns its tile), the degrid units (primary
// records only) and the pair units, each an exclusive scan of a value formed
// from the counts.  The scans run together: index_bins walks a range of bins
// with the three running totals, index_pairs a range of pairs.

// Exclusive scan of N values per thread over the workgroup; `total` gets the
// sums.  sh: [16][N] LDS words.
template <int N>
__device__ inline void block_scan_n(uint32_t (&v)[N], uint32_t (&total)[N], uint32_t *sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwv = blockDim.x >> 6;
  uint32_t in[N];
#pragma unroll
  for (int k = 0; k < N; ++k) {
    in[k] = v[k];
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t o = __shfl_up(v[k], off);
      if (lane >= off) v[k] += o;
    }
    if (lane == 63) sh[wave * N + k] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) {
    uint32_t before = 0, all = 0;
    for (int w = 0; w < nwv; ++w) {
      const uint32_t s = sh[w * N + k];
      before += w < wave ? s : 0u;
      all += s;
    }
    v[k] += before - in[k];
    total[k] = all;
  }
  __syncthreads();
}

__device__ inline void bin_values(const PlanDev &P, int64_t b, uint32_t (&v)[3]) {
  const uint32_t cap = (uint32_t)P.unit_cap, dcap = (uint32_t)P.dunit_cap;
  const uint32_t na = P.cnt_all[b], np = P.cnt_prim[b];
  v[0] = na;
  v[1] = na == 0 ? 1u : (na + cap - 1) / cap;
  v[2] = (np + dcap - 1) / dcap;
}

__device__ inline uint32_t pair_value(const PlanDev &P, int64_t p) {
  int64_t b0, b1;
  bool has1;
  uint32_t n;
  pair_bins(P, p, b0, b1, has1, n);
  const uint32_t cap = (uint32_t)P.dunit_cap;
  return (n + cap - 1) / cap;
}

// Offsets, cursors and units of bins [b0, b1), whose preceding bins hold
// `carry` records, grid units and degrid units (updated).
__device__ inline void index_bins(const PlanDev &P, int64_t b0, int64_t b1, uint32_t (&carry)[3],
                                  uint32_t *sh) {
  const uint32_t cap = (uint32_t)P.unit_cap, dcap = (uint32_t)P.dunit_cap;
  for (int64_t base = b0; base < b1; base += blockDim.x) {
    const int64_t b = base + threadIdx.x;
    const bool on = b < b1;
    uint32_t v[3] = {0u, 0u, 0u}, n[3], total[3];
    if (on) bin_values(P, b, v);
#pragma unroll
    for (int k = 0; k < 3; ++k) n[k] = v[k];
    block_scan_n<3>(v, total, sh);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      v[k] += carry[k];
      carry[k] += total[k];
    }
    if (!on) continue;
    const uint32_t np = P.cnt_prim[b], na = n[0];
    P.bin_start[b] = v[0];
    P.gunit_start[b] = v[1];
    P.dunit_start[b] = v[2];
    P.cur_prim[b] = v[0];
    P.cur_dup[b] = v[0] + np;
    for (uint32_t k = 0; k < n[1]; ++k) {
      const uint32_t cnt = na > k * cap ? min(cap, na - k * cap) : 0u;
      const uint32_t fl = (n[1] > 1 ? kUnitMulti : 0u) | (k == 0 ? kUnitFirst : 0u);
      P.gunits[v[1] + k] = make_uint4((uint32_t)b, v[0] + k * cap, cnt, fl);
    }
    for (uint32_t k = 0; k < n[2]; ++k)
      P.dunits[v[2] + k] = make_uint4((uint32_t)b, v[0] + k * dcap, min(dcap, np - k * dcap), 0u);
  }
}

// Pair units of pairs [p0, p1), preceded by `carry` units (updated).
__device__ inline void index_pairs(const PlanDev &P, int64_t p0, int64_t p1, uint32_t &carry,
                                   uint32_t *sh) {
  const uint32_t cap = (uint32_t)P.dunit_cap;
  for (int64_t base = p0; base < p1; base += blockDim.x) {
    const int64_t p = base + threadIdx.x;
    const bool on = p < p1;
    int64_t b0 = 0, b1 = 0;
    bool has1 = false;
    uint32_t n = 0u;
    if (on) pair_bins(P, p, b0, b1, has1, n);
    const uint32_t nu = (n + cap - 1) / cap;
    uint32_t v[1] = {nu}, total[1];
    block_scan_n<1>(v, total, sh);
    const uint32_t k0 = v[0] + carry;
    carry += total[0];
    if (!on) continue;
    P.punit_start[p] = k0;
    const uint32_t second = has1 ? (uint32_t)b1 : kNoBin;
    for (uint32_t k = 0; k < nu; ++k)
      P.punits[k0 + k] = make_uint4((uint32_t)b0, k * cap, min(cap, n - k * cap), second);
  }
}

__device__ inline void index_ends(const PlanDev &P, const uint32_t (&carry)[3]) {
  if (threadIdx.x != 0) return;
  P.bin_start[P.n_bins] = carry[0];
  P.gunit_start[P.n_bins] = carry[1];
  P.dunit_start[P.n_bins] = carry[2];
}

// Small plans: the totals (of a chunked plan), every offset and unit and the
// chunks' first slots in one workgroup, where the seven launches of the
// general path cost more than the work (a 128 x 128, 4-channel plan of 28,080
// samples, binned in 21 launches: 85 us; in three: 32 us).
__global__ __launch_bounds__(1024) void k_index_small(PlanDev P) {
  __shared__ uint32_t sh[16 * 3];
  const bool ident = chan_identity(P);
  if (P.chunked && !P.row_chan) {
    for (int64_t b = threadIdx.x; b < P.n_bins; b += blockDim.x) {
      uint32_t t;
      int ic;
      bin_parts(P, (uint32_t)b, t, ic);
      uint32_t sp = 0, sd = 0;
      chunk_runs(P, ident, ic, (int)t, 0, 1, [&](int64_t i, int n) { add_runs(P, i, n, sp, sd); });
      P.cnt_prim[b] = sp;
      P.cnt_all[b] = sp + sd;
    }
    __syncthreads();
  }
  uint32_t carry[3] = {0u, 0u, 0u}, pc = 0u;
  index_bins(P, 0, P.n_bins, carry, sh);
  index_ends(P, carry);
  if (P.n_pairs > 0) {
    index_pairs(P, 0, P.n_pairs, pc, sh);
    if (threadIdx.x == 0) P.punit_start[P.n_pairs] = pc;
  }
  if (P.chunk_scatter) {
    __syncthreads();
    for (int64_t b = threadIdx.x; b < P.n_bins; b += blockDim.x) {
      uint32_t t;
      int ic;
      bin_parts(P, (uint32_t)b, t, ic);
      uint32_t sp = P.bin_start[b], sd = sp + P.cnt_prim[b];
      chunk_runs(P, ident, ic, (int)t, 0, 1, [&](int64_t i, int n) { place_runs(P, i, n, sp, sd); });
    }
  }
}

// General path: per-block sums (kIndexSpan bins or pairs a block), one
// workgroup that scans them in place, then the offsets and units block by
// block.  scan_tmp: [3][bin blocks] then [pair blocks].
constexpr int kIndexSpan = 1024;
__global__ __launch_bounds__(1024) void k_index_sums(PlanDev P, int nb_blocks) {
  __shared__ uint32_t sh[16 * 3];
  const bool pairs = (int)blockIdx.x >= nb_blocks;
  const int64_t blk = pairs ? blockIdx.x - nb_blocks : blockIdx.x;
  const int64_t i1 = min((blk + 1) * (int64_t)kIndexSpan, pairs ? P.n_pairs : P.n_bins);
  uint32_t sum[3] = {0u, 0u, 0u}, total[3];
  for (int64_t i = blk * kIndexSpan + threadIdx.x; i < i1; i += blockDim.x) {
    if (pairs) {
      sum[0] += pair_value(P, i);
    } else {
      uint32_t v[3];
      bin_values(P, i, v);
#pragma unroll
      for (int k = 0; k < 3; ++k) sum[k] += v[k];
    }
  }
  block_scan_n<3>(sum, total, sh);
  if (threadIdx.x != 0) return;
  if (pairs) {
    P.scan_tmp[3 * (int64_t)nb_blocks + blk] = total[0];
  } else {
    for (int k = 0; k < 3; ++k) P.scan_tmp[(int64_t)k * nb_blocks + blk] = total[k];
  }
}

__global__ __launch_bounds__(1024) void k_index_scan(PlanDev P, int nb_blocks, int np_blocks) {
  __shared__ uint32_t sh[16];
  uint32_t ends[4];
  for (int q = 0; q < 4; ++q) {
    uint32_t *a = P.scan_tmp + (int64_t)q * nb_blocks;
    const int n = q < 3 ? nb_blocks : np_blocks;
    uint32_t carry = 0u;
    for (int i0 = 0; i0 < n; i0 += blockDim.x) {
      const int i = i0 + threadIdx.x;
      uint32_t v[1] = {i < n ? a[i] : 0u}, total[1];
      block_scan_n<1>(v, total, sh);
      if (i < n) a[i] = v[0] + carry;
      carry += total[0];
    }
    ends[q] = carry;
  }
  const uint32_t e3[3] = {ends[0], ends[1], ends[2]};
  index_ends(P, e3);
  if (P.n_pairs > 0 && threadIdx.x == 0) P.punit_start[P.n_pairs] = ends[3];
}

__global__ __launch_bounds__(1024) void k_index_apply(PlanDev P, int nb_blocks) {
  __shared__ uint32_t sh[16 * 3];
  if ((int)blockIdx.x >= nb_blocks) {
    const int64_t blk = blockIdx.x - nb_blocks;
    uint32_t carry = P.scan_tmp[3 * (int64_t)nb_blocks + blk];
    index_pairs(P, blk * kIndexSpan, min((blk + 1) * (int64_t)kIndexSpan, P.n_pairs), carry, sh);
    return;
  }
  const int64_t blk = blockIdx.x;
  uint32_t carry[3];
  for (int k = 0; k < 3; ++k) carry[k] = P.scan_tmp[(int64_t)k * nb_blocks + blk];
  index_bins(P, blk * kIndexSpan, min((blk + 1) * (int64_t)kIndexSpan, P.n_bins), carry, sh);
}

// Segments of the chunk totals and bases passes: about eight runs each, one
// where the bins alone fill the chip (a second pass over the counts of a
// million bins: 62 -> 227 us).
static int chunk_segments(const PlanDev &d) {
  if (d.n_bins >= 1 << 16) return 1;
  const int64_t runs =
      (int64_t)d.chunks_per_chan * (d.chunk_all ? 1 : d.n_chan) / d.n_img_chan;
  return (int)std::max<int64_t>(
      1, std::min<int64_t>(std::min<int64_t>(kMaxSegs, d.chunks_per_chan), runs / 8));
}

// Whether one workgroup indexes the plan: its bins and, for a chunked plan,
// its runs are few enough that walking them takes less than the general
// path's launches.
static bool index_is_small(const PlanDev &d) {
  const int64_t runs =
      d.chunked && !d.row_chan
          ? d.n_bins * d.chunks_per_chan *
                (d.chunk_all ? 1 : (d.n_chan + d.n_img_chan - 1) / d.n_img_chan)
          : 0;
  return d.n_bins <= 4096 && runs <= 32768;
}

// Bin offsets, cursors and units from the bins' counts (small chunked plans:
// from the chunks' counts).
static int launch_index(const PlanDev &d, hipStream_t s) {
  if (index_is_small(d)) {
    hipLaunchKernelGGL(k_index_small, dim3(1), dim3(1024), 0, s, d);
    AV_LAUNCH_CHECK("k_index_small");
    return AV_OK;
  }
  const int64_t ntiles = (int64_t)d.ntu * d.ntv;
  const dim3 sg((unsigned)((ntiles + kSegTiles - 1) / kSegTiles * d.n_img_chan));
  const dim3 sb(kSegTiles, (unsigned)chunk_segments(d));
  if (d.chunked && !d.row_chan) {
    hipLaunchKernelGGL(k_chunk_totals, sg, sb, 0, s, d);
    AV_LAUNCH_CHECK("k_chunk_totals");
  }
  const int nbb = (int)((d.n_bins + kIndexSpan - 1) / kIndexSpan);
  const int npb = (int)((d.n_pairs + kIndexSpan - 1) / kIndexSpan);
  hipLaunchKernelGGL(k_index_sums, dim3((unsigned)(nbb + npb)), dim3(1024), 0, s, d, nbb);
  AV_LAUNCH_CHECK("k_index_sums");
  hipLaunchKernelGGL(k_index_scan, dim3(1), dim3(1024), 0, s, d, nbb, npb);
  AV_LAUNCH_CHECK("k_index_scan");
  hipLaunchKernelGGL(k_index_apply, dim3((unsigned)(nbb + npb)), dim3(1024), 0, s, d, nbb);
  AV_LAUNCH_CHECK("k_index_apply");
  if (d.chunk_scatter) {
    hipLaunchKernelGGL(k_chunk_bases, sg, sb, 0, s, d);
    AV_LAUNCH_CHECK("k_chunk_bases");
  }
  return AV_OK;
}

__global__ void k_prepare_tables(PlanDev P, const double *cgk) {
  fill_tables(P, cgk, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

int prepare_tables(const PlanDev &d, const double *cgk, hipStream_t s) {
  hipLaunchKernelGGL(k_prepare_tables, dim3(kTableBlocks), dim3(256), 0, s, d, cgk);
  AV_LAUNCH_CHECK("k_prepare_tables");
  return AV_OK;
}

__global__ void k_popcount(const unsigned long long *m, int64_t n, uint32_t *out) {
  uint32_t c = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    c += (uint32_t)__popcll(m[i]);
  for (int off = 32; off >= 1; off >>= 1) c += __shfl_xor(c, off);
  if (__lane_id() == 0 && c) atomicAdd(out, c);
}

}  // namespace av

using namespace av;

static size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }

// Records per work unit when the caller leaves it open.  A unit is one
// wavefront's serial walk over its records, so a plan of few samples needs
// short units to spread its dense central bins over the chip, and a plan of
// many samples long ones, since the tiles of a split bin are added with
// atomics.  Measured (bin + grid + degrid, us) at caps of 8192, 2048, 1024,
// 512, 256 and 128: 28,080 samples FP64 297, 294, 246, 188, 162, 160; 4.8 M
// FP64 2364, 2340, 2227, 2272, 2320, 2725; 35 M FP32 6586, 6113, 6249, 6639,
// 7889, 12779.
static int32_t default_unit_cap(int64_t n_items) {
  int32_t cap = 256;
  while (cap < 8192 && (int64_t)cap * kCapSamples * 3 < n_items * 2) cap *= 2;
  return cap;
}

// A degrid unit loads its tile's cells before its first record, where a grid
// unit starts from zeros, so short ones cost it more: caps of four grid units
// where a plan has four image channels or more, whose dense bins share the chip,
// the grid unit's own where one plane holds them all.  Degridding alone, us at
// caps of 256, 512, 1024, 2048, 4096 and 8192 (grid caps of 256 and 512): 1.9 M
// samples x 4 polarisations on 8 planes of 1024^2 159, 145, 140, 146, 145 and
// 146, on one plane 128, 116, 122, 141, 167 and 250; 6.5 M on 8 planes 469, 419,
// 403, 391, 403 and 432, on two 438, 389, 371, 380, 407 and 503, on one 396, 347,
// 332, 342, 373 and 442.
static int32_t default_dunit_cap(int64_t n_items, int32_t n_img_chan) {
  return default_unit_cap(n_items * std::min(n_img_chan, 4));
}

// Time steps that a chunk spans before its rows are visited baseline by
// baseline.  Two make runs of two records, and a chunk's positions outside its
// rows are at most half of all; in row order a wavefront's records go to as
// many bins as it has lanes.  Cubes of 64 antennas x 16 channels, binning in row
// order and so: 4.7 steps 341 -> 253 us, 3.1 250 -> 198, 2.3 (FP64) 194 -> 166,
// 15.6 on 2048^2 planes 1248 -> 797; continuum of 4 channels x 2.9 steps 1254 ->
// 843.  Where a chunk takes every channel of a row, many channels fill a
// wavefront already (48 channels x 2.5 steps 1130 -> 1200, 64 x 2 565 -> 640; 16
// x 4 783 -> 661).
// A chunk of one sample a thread is done in one step in row order (a 128^2
// snapshot, bin + grid + degrid 71.7 us, 72.4 in baseline order).
constexpr int64_t kOrderSteps = 2, kOrderStepsWide = 16;
constexpr int kOrderChans = 32;
constexpr int64_t kOrderSamples = 2 * kChunkThreads;

// Rows of a chunk.  Every chunk is a workgroup of the two binning passes:
// kChunkTarget of them in all keep the chip busy, but a chunk also reads and
// writes a word per tile in each of four passes, so it has at least half a
// sample per tile.  Chunks as long as kMaxRowsPerChunk left most CUs idle: a
// 302,400-row, 16-channel plan of 1024 x 1024 was 48 workgroups and binned in
// 611 us, 213 us in 1024 chunks (512: 199, 2048: 246, 4096: 270; a 129 M
// sample plan of 2048 x 2048, already 1024 chunks, 2048 chunks: +12%).
static int32_t chunk_rows(int64_t n_rows, int32_t n_chan, int64_t ntiles, bool all,
                          bool compact) {
  const int64_t per_row = all ? n_chan : 1;  // samples of a chunk per row
  const int64_t step = all ? 64 : kChunkThreads;
  int64_t rows = kMaxRowsPerChunk;
  if (!compact)
    rows = std::max((n_rows * n_chan / per_row + kChunkTarget - 1) / kChunkTarget,
                    ntiles / 2 / per_row);
  // a chunk's positions fit 32 bits
  if (all) rows = std::min<int64_t>(rows, std::max<int64_t>(64, (1ll << 30) / n_chan));
  rows = std::min<int64_t>({rows, n_rows, kMaxRowsPerChunk});
  return (int32_t)(std::max<int64_t>(1, (rows + step - 1) / step) * step);
}

// Validate the plan parameters, fill plan->d's sizes and compute the bytes
// of device memory the plan's arrays need; with base non-NULL, also point
// the arrays into [base, base + bytes).  Shared by av_plan_create (one
// hipMalloc) and av_grid_noalloc (the library's static scratch array).  With
// `compact`, chunks and default units are as long as they may be: the fewest
// bytes.
int plan_layout(int64_t n_rows, int32_t n_chan, int32_t n_img_chan, int32_t n_u, int32_t n_v,
                double cell_u, double cell_v, int32_t support, int32_t oversampling,
                int32_t tile_u, int32_t tile_v, int32_t geometry, int32_t unit_cap, av_plan *p,
                char *base, size_t *bytes, bool compact) {
  if (n_rows < 0 || n_chan < 1 || n_img_chan < 1 || n_u < 1 || n_v < 1)
    return fail(AV_ERR_INVALID, "av_plan_create: sizes must be positive");
  // plans bin footprints up to kMaxPlanSupport wide (the mosaic gridder's
  // max_support); av_grid and av_degrid take supports up to
  // kMaxSupport
  if (support < 2 || support > kMaxPlanSupport)
    return fail(AV_ERR_UNSUPPORTED, "av_plan_create: support must be in [2, 63]");
  if (oversampling < 1 || oversampling > 250)
    return fail(AV_ERR_UNSUPPORTED, "av_plan_create: oversampling must be in [1, 250]");
  if (tile_u == 0) tile_u = 32;
  if (tile_v == 0) tile_v = 32;
  if (tile_u < support || tile_v < support || tile_u > 128 || tile_v > 128)
    return fail(AV_ERR_INVALID, "av_plan_create: tiles must be in [support, 128]");
  if (n_u >= (1 << 24) || n_v >= (1 << 24))
    return fail(AV_ERR_UNSUPPORTED, "av_plan_create: grid sides must be below 2^24");
  const bool row_channels = (geometry & AV_PLAN_ROW_CHANNELS) != 0;
  const bool conjugate = (geometry & AV_GEOM_CONJUGATE) != 0;
  geometry &= ~(AV_PLAN_ROW_CHANNELS | AV_GEOM_CONJUGATE);
  if (geometry != AV_GEOM_REFERENCE && geometry != AV_GEOM_DEGRID)
    return fail(AV_ERR_INVALID, "av_plan_create: unknown geometry");
  if (conjugate && geometry != AV_GEOM_REFERENCE)
    return fail(AV_ERR_INVALID, "av_plan_create: AV_GEOM_CONJUGATE needs AV_GEOM_REFERENCE");
  int64_t n_items = row_channels ? n_rows : n_rows * (int64_t)n_chan;
  if (n_items > ((int64_t)1 << 32) / 5 - 1)
    return fail(AV_ERR_UNSUPPORTED, "av_plan_create: more than 858993458 samples per plan");
  int32_t dunit_cap = unit_cap;
  if (unit_cap == 0) {
    unit_cap = compact ? 8192 : default_unit_cap(n_items);
    dunit_cap = compact ? 8192 : default_dunit_cap(n_items, n_img_chan);
  }
  if (unit_cap < 64) return fail(AV_ERR_INVALID, "av_plan_create: unit_cap < 64");

  PlanDev &d = p->d;
  d.n_rows = n_rows;
  d.n_chan = n_chan;
  d.n_img_chan = n_img_chan;
  d.n_u = n_u;
  d.n_v = n_v;
  d.cell_u = cell_u;
  d.cell_v = cell_v;
  // degrid_spheroid_ms4: scale = -pixelincr * n, offset = n / 2 (float)
  d.dscale_u = (-cell_u) * (double)n_u;
  d.dscale_v = (-cell_v) * (double)n_v;
  d.doff_u = (double)n_u / 2.0;
  d.doff_v = (double)n_v / 2.0;
  d.support = support;
  d.ov = oversampling;
  d.tile_u = tile_u;
  d.tile_v = tile_v;
  d.tile_u_mul = 0xFFFFFFFFu / (uint32_t)tile_u + 1u;
  d.tile_v_mul = 0xFFFFFFFFu / (uint32_t)tile_v + 1u;
  d.geometry = geometry;
  d.conjugate = conjugate ? 1 : 0;
  d.row_channels = row_channels;
  d.unit_cap = unit_cap;
  d.dunit_cap = dunit_cap;
  d.ntu = (n_u + tile_u - 1) / tile_u;
  d.ntv = (n_v + tile_v - 1) / tile_v;
  d.n_bins = (int64_t)d.ntu * d.ntv * n_img_chan;
  d.chan_major = row_channels && d.n_bins < ((int64_t)1 << 32);
  d.bin_minor = d.chan_major ? (uint32_t)(d.ntu * d.ntv) : (uint32_t)n_img_chan;
  d.n_items = n_items;
  // a footprint overlaps at most 2x2 tiles, plus one separate degrid record
  d.max_records = 5 * n_items;
  d.max_gunits = d.n_bins + d.max_records / unit_cap + 1;
  // a sample has at most two primary records (grid + separate degrid)
  d.max_dunits = d.n_bins + 2 * n_items / dunit_cap + 1;
  const bool pairs = tile_u == 16 && tile_v == 16 && support <= 7;
  d.n_pairs = pairs ? (int64_t)d.ntu * ((d.ntv + 1) / 2) * n_img_chan : 0;
  d.max_punits = pairs ? d.n_pairs + 2 * n_items / dunit_cap + 1 : 0;
  d.row_chan = nullptr;
  d.order_nb = 1;
  d.uvw = nullptr;

  const int64_t nb = d.n_bins;
  d.mask_words_per_chan = (n_rows + 63) / 64;
  const int64_t mask_words = d.mask_words_per_chan * (row_channels ? 1 : n_chan) + 1;
  // chunked binning when a channel's tiles fit in LDS
  const int64_t ntiles = (int64_t)d.ntu * d.ntv;
  d.chunked = !row_channels && ntiles <= kMaxChunkTiles && n_rows > 0;
  d.chunk_all = d.chunked && n_img_chan == 1 && n_chan >= kChunkAllChans && !compact;
  d.rows_per_chunk = chunk_rows(n_rows, n_chan, ntiles, d.chunk_all, compact);
  d.chunks_per_chan = (int32_t)((n_rows + d.rows_per_chunk - 1) / d.rows_per_chunk);
  const int64_t chunk_cells =
      d.chunked ? (int64_t)(d.chunk_all ? 1 : n_chan) * d.chunks_per_chan * ntiles : 0;
  // row-block counts, kept for plans whose rows carry their channel when a
  // block's counters and cursors fit in 160 KB of LDS.  Blocks as the chunks:
  // about kChunkTarget of them, at least half a row per tile, and few enough
  // rows for 16-bit counts
  d.row_block_rows = (int32_t)(
      std::min<int64_t>(kMaxRowBlockRows / kChunkThreads,
                        std::max<int64_t>(1, (std::max(n_rows / kChunkTarget, ntiles / 2) +
                                              kChunkThreads - 1) / kChunkThreads)) *
      kChunkThreads);
  const int64_t row_cells = (row_channels && n_rows > 0 && 8 * ntiles <= 160 * 1024)
                                ? (n_rows + d.row_block_rows - 1) / d.row_block_rows * ntiles
                                : 0;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    size_t o = off;
    off += align_up(bytes);
    return o;
  };
  size_t o_gsu = take(sizeof(double) * n_chan), o_gsv = take(sizeof(double) * n_chan),
         o_freq = take(sizeof(double) * n_chan), o_cmap = take(sizeof(int32_t) * n_chan),
         o_call = take(4 * nb), o_cprim = take(4 * nb), o_bstart = take(4 * (nb + 1)),
         o_curp = take(4 * nb), o_curd = take(4 * nb), o_gus = take(4 * (nb + 1)),
         o_dus = take(4 * (nb + 1)),
         o_rec = take(12 * std::max<int64_t>(d.max_records, 1)), o_gun = take(sizeof(uint4) * d.max_gunits),
         o_dun = take(sizeof(uint4) * d.max_dunits), o_pus = take(4 * (d.n_pairs + 1)),
         o_pun = take(sizeof(uint4) * d.max_punits),
         o_gm = take(8 * mask_words), o_dm = take(8 * mask_words),
         o_chh = take(4 * chunk_cells), o_chd = take(4 * chunk_cells), o_rh = take(4 * row_cells),
         o_tab = take(sizeof(float) * oversampling * (support / 2 + 1)),
         o_nrm = take(sizeof(double) * (2 * (oversampling / 2 + 2) + 1)),
         o_wt32 = take(sizeof(float) * (support + 2) * (2 * (oversampling / 2 + 2) + 1)),
         o_wt64 = take(sizeof(double) * (support + 2) * (2 * (oversampling / 2 + 2) + 1)),
         o_upart = take(sizeof(double) * 4 * d.max_gunits), o_ctr = take(4 * 16);
  *bytes = off;
  if (!base) return AV_OK;
  char *c = base;
  d.gscale_u = (double *)(c + o_gsu);
  d.gscale_v = (double *)(c + o_gsv);
  d.freq = (double *)(c + o_freq);
  d.chan_map = (int32_t *)(c + o_cmap);
  d.cnt_all = (uint32_t *)(c + o_call);
  d.cnt_prim = (uint32_t *)(c + o_cprim);
  d.bin_start = (uint32_t *)(c + o_bstart);
  d.cur_prim = (uint32_t *)(c + o_curp);
  d.cur_dup = (uint32_t *)(c + o_curd);
  d.gunit_start = (uint32_t *)(c + o_gus);
  d.dunit_start = (uint32_t *)(c + o_dus);
  d.rec = (uint32_t *)(c + o_rec);
  d.gunits = (uint4 *)(c + o_gun);
  d.dunits = (uint4 *)(c + o_dun);
  d.punit_start = d.n_pairs ? (uint32_t *)(c + o_pus) : nullptr;
  d.punits = d.n_pairs ? (uint4 *)(c + o_pun) : nullptr;
  d.gmask = (unsigned long long *)(c + o_gm);
  d.dmask = (unsigned long long *)(c + o_dm);
  d.n_words = mask_words - 1;
  d.chunk_hist = chunk_cells ? (uint32_t *)(c + o_chh) : nullptr;
  d.chunk_dup = chunk_cells ? (uint32_t *)(c + o_chd) : nullptr;
  d.row_hist = row_cells ? (uint32_t *)(c + o_rh) : nullptr;
  d.tab32 = (float *)(c + o_tab);
  d.nrm = (double *)(c + o_nrm);
  d.wtab32 = (float *)(c + o_wt32);
  d.wtab64 = (double *)(c + o_wt64);
  d.upart = (double *)(c + o_upart);
  // the index passes' block sums (four words per kIndexSpan bins at most):
  // the units' partial sums are written after them, by the gridder
  d.scan_tmp = (uint32_t *)d.upart;
  d.counters = (uint32_t *)(c + o_ctr);
  p->alloc_base = base;
  p->alloc_bytes = off;
  return AV_OK;
}

extern "C" {

int av_plan_create(int64_t n_rows, int32_t n_chan, int32_t n_img_chan, int32_t n_u, int32_t n_v,
                   double cell_u, double cell_v, int32_t support, int32_t oversampling,
                   int32_t tile_u, int32_t tile_v, int32_t geometry, int32_t unit_cap,
                   av_plan **out) {
  if (!out) return fail(AV_ERR_INVALID, "av_plan_create: out is NULL");
  *out = nullptr;
  av_plan probe{};
  size_t bytes = 0;
  int rc = plan_layout(n_rows, n_chan, n_img_chan, n_u, n_v, cell_u, cell_v, support,
                       oversampling, tile_u, tile_v, geometry, unit_cap, &probe, nullptr, &bytes);
  if (rc) return rc;
  void *base = nullptr;
  hipError_t e = hipMalloc(&base, bytes);
  if (e != hipSuccess) return hip_fail(e, "av_plan_create: hipMalloc");
  av_plan *p = new av_plan();
  rc = plan_layout(n_rows, n_chan, n_img_chan, n_u, n_v, cell_u, cell_v, support, oversampling,
                   tile_u, tile_v, geometry, unit_cap, p, (char *)base, &bytes);
  if (rc == AV_OK) {
    e = hipGetDevice(&p->device);
    if (e != hipSuccess) rc = hip_fail(e, "av_plan_create: hipGetDevice");
  }
  if (rc) {
    (void)hipFree(base);
    delete p;
    return rc;
  }
  *out = p;
  return AV_OK;
}

int av_plan_destroy(av_plan *plan) {
  if (!plan) return AV_OK;
  const hipError_t e = plan->alloc_base ? hipFree(plan->alloc_base) : hipSuccess;
  delete plan;
  return e == hipSuccess ? AV_OK : hip_fail(e, "av_plan_destroy: hipFree");
}

int av_plan_set_uvw(av_plan *plan, const double *uvw, const double *freq,
                    const int32_t *chan_map, const int32_t *row_chan, void *stream) {
  if (!plan || !freq || (plan->d.n_rows > 0 && !uvw))
    return fail(AV_ERR_INVALID, "av_plan_set_uvw: NULL argument");
  if (row_chan && plan->d.n_chan < 1)
    return fail(AV_ERR_INVALID, "av_plan_set_uvw: row_chan needs n_chan >= 1");
  if (plan->d.row_channels && !row_chan)
    return fail(AV_ERR_INVALID,
                "av_plan_set_uvw: the plan was created for per-row channels; row_chan is NULL");
  hipStream_t s = (hipStream_t)stream;
  PlanDev &d = plan->d;
  d.uvw = uvw;
  d.row_chan = (int32_t *)row_chan;
  if (row_chan) d.n_items = d.n_rows;  // one sample per row
  else d.n_items = d.n_rows * (int64_t)d.n_chan;
  d.n_words = d.mask_words_per_chan * (row_chan ? 1 : d.n_chan);
  int rc;
  // row-block binning needs a counter and a cursor per tile in LDS
  const int64_t ntiles = (int64_t)d.ntu * d.ntv;
  d.row_blocks = 0;
  d.chunk_scatter = 0;
  if (d.n_rows > 0 && (row_chan || d.chunked)) {
    const DeviceProps &prop = device_props();
    if (prop.error) return hip_fail(prop.error, "av_plan_set_uvw: device properties");
    const bool fits = (size_t)(2 * sizeof(uint32_t) * ntiles) <= prop.lds_per_block;
    if (row_chan) d.row_blocks = fits && d.row_hist != nullptr;
    else d.chunk_scatter = fits;
  }
  const int64_t nchunks = (int64_t)(d.chunk_all ? 1 : d.n_chan) * d.chunks_per_chan;
  const unsigned row_grid = (unsigned)((d.n_rows + d.row_block_rows - 1) / d.row_block_rows);
  const bool by_chunks = d.chunked && !row_chan;
  if (!by_chunks) {  // the counting pass of chunks sets its channels up itself
    hipLaunchKernelGGL(k_chan_setup, dim3((d.n_chan + 255) / 256), dim3(256), 0, s, d, freq,
                       chan_map);
    AV_LAUNCH_CHECK("k_chan_setup");
    // both counts in one fill: they lie one after the other in the plan
    if ((rc = launch_fill_u32(d.cnt_all, 0u, d.cnt_prim - d.cnt_all + d.n_bins, s))) return rc;
  }
  // pass 1: counts per bin, or per chunk and tile
  if (d.row_blocks) {
    const int lds = (int)(sizeof(uint32_t) * ntiles);
    if ((rc = ensure_lds_limit<k_count_rows>(lds, "av_plan_set_uvw: hipFuncSetAttribute")))
      return rc;
    hipLaunchKernelGGL(k_count_rows, dim3(row_grid), dim3(kChunkThreads), lds, s, d);
    AV_LAUNCH_CHECK("k_count_rows");
  } else if (by_chunks) {
    const int lds = (int)(2 * sizeof(uint32_t) * ntiles);
    if ((rc = d.chunk_all ? ensure_lds_limit<k_count_chunks<true>>(
                                lds, "av_plan_set_uvw: hipFuncSetAttribute")
                          : ensure_lds_limit<k_count_chunks<false>>(
                                lds, "av_plan_set_uvw: hipFuncSetAttribute")))
      return rc;
    hipLaunchKernelGGL(d.chunk_all ? k_count_chunks<true> : k_count_chunks<false>,
                       dim3((unsigned)nchunks), dim3(kChunkThreads), lds, s, d, freq, chan_map);
    AV_LAUNCH_CHECK("k_count_chunks");
  } else {
    const int64_t span = d.mask_words_per_chan * 64 * (row_chan ? 1 : d.n_chan);
    int64_t blocks = (span + 255) / 256;
    blocks = std::max<int64_t>(1, std::min<int64_t>(blocks, 16384));
    hipLaunchKernelGGL(k_count, dim3((unsigned)blocks), dim3(256), 0, s, d);
    AV_LAUNCH_CHECK("k_count");
  }
  // pass 2: bin offsets, cursors and units
  if ((rc = launch_index(d, s))) return rc;
  // pass 3: the records
  if (d.chunk_scatter) {
    const int lds = (int)(2 * sizeof(uint32_t) * ntiles);
    if ((rc = d.chunk_all ? ensure_lds_limit<k_scatter_chunks<true>>(
                                lds, "av_plan_set_uvw: hipFuncSetAttribute")
                          : ensure_lds_limit<k_scatter_chunks<false>>(
                                lds, "av_plan_set_uvw: hipFuncSetAttribute")))
      return rc;
    hipLaunchKernelGGL(d.chunk_all ? k_scatter_chunks<true> : k_scatter_chunks<false>,
                       dim3((unsigned)nchunks), dim3(kChunkThreads), lds, s, d);
    AV_LAUNCH_CHECK("k_scatter_chunks");
  } else if (d.row_blocks) {
    const int lds = (int)(2 * sizeof(uint32_t) * ntiles);
    if ((rc = ensure_lds_limit<k_scatter_rows>(lds, "av_plan_set_uvw: hipFuncSetAttribute")))
      return rc;
    hipLaunchKernelGGL(k_scatter_rows, dim3(row_grid), dim3(kChunkThreads), lds, s, d);
    AV_LAUNCH_CHECK("k_scatter_rows");
  } else {
    int64_t blocks = (d.n_items + 255) / 256;
    blocks = std::max<int64_t>(1, std::min<int64_t>(blocks, 16384));
    hipLaunchKernelGGL(k_scatter, dim3((unsigned)blocks), dim3(256), 0, s, d);
    AV_LAUNCH_CHECK("k_scatter");
  }
  return AV_OK;
}

int av_plan_set_degrid_transform(av_plan *plan, double scale_u, double scale_v,
                                 double offset_u, double offset_v) {
  if (!plan) return fail(AV_ERR_INVALID, "av_plan_set_degrid_transform: NULL plan");
  plan->d.dscale_u = scale_u;
  plan->d.dscale_v = scale_v;
  plan->d.doff_u = offset_u;
  plan->d.doff_v = offset_v;
  return AV_OK;
}

int av_plan_set_row_order(av_plan *plan, int32_t n_baseline) {
  if (!plan) return fail(AV_ERR_INVALID, "av_plan_set_row_order: NULL plan");
  PlanDev &d = plan->d;
  if (n_baseline < 1 || (d.n_rows > 0 && d.n_rows % n_baseline != 0))
    return fail(AV_ERR_INVALID, "av_plan_set_row_order: n_baseline must be >= 1 and divide n_rows");
  // a chunk is visited baseline by baseline where it spans a few time steps (see
  // kOrderSteps)
  const int64_t steps = d.chunk_all && d.n_chan >= kOrderChans ? kOrderStepsWide : kOrderSteps;
  const int64_t samples = (int64_t)d.rows_per_chunk * (d.chunk_all ? d.n_chan : 1);
  d.order_nb = (n_baseline > 1 && n_baseline * steps <= d.rows_per_chunk &&
                samples >= kOrderSamples)
                   ? n_baseline
                   : 1;
  return AV_OK;
}

int av_plan_stats(av_plan *plan, int64_t out[8], void *stream) {
  if (!plan || !out) return fail(AV_ERR_INVALID, "av_plan_stats: NULL argument");
  hipStream_t s = (hipStream_t)stream;
  const PlanDev &d = plan->d;
  int rc = launch_fill_u32(d.counters, 0u, 2, s);
  if (rc) return rc;
  if (d.n_words > 0) {
    hipLaunchKernelGGL(k_popcount, dim3(256), dim3(256), 0, s, d.gmask, d.n_words, d.counters);
    AV_LAUNCH_CHECK("k_popcount");
    hipLaunchKernelGGL(k_popcount, dim3(256), dim3(256), 0, s, d.dmask, d.n_words,
                       d.counters + 1);
    AV_LAUNCH_CHECK("k_popcount");
  }
  uint32_t ctr[2], tot[3];
  AV_HIP(hipMemcpyAsync(ctr, d.counters, sizeof(ctr), hipMemcpyDeviceToHost, s));
  AV_HIP(hipMemcpyAsync(&tot[0], d.bin_start + d.n_bins, 4, hipMemcpyDeviceToHost, s));
  AV_HIP(hipMemcpyAsync(&tot[1], d.gunit_start + d.n_bins, 4, hipMemcpyDeviceToHost, s));
  AV_HIP(hipMemcpyAsync(&tot[2], d.dunit_start + d.n_bins, 4, hipMemcpyDeviceToHost, s));
  AV_HIP(hipStreamSynchronize(s));
  out[0] = d.n_items;
  out[1] = ctr[0];
  out[2] = ctr[1];
  out[3] = tot[0];
  out[4] = d.n_bins;
  out[5] = tot[1];
  out[6] = tot[2];
  out[7] = d.n_items - ctr[1];  // samples no degrid unit visits
  return AV_OK;
}

}  // extern "C"

// hogbom.hip -- Hogbom CLEAN on the GPU (replaces the _hogbom_ext extension
// of core/imaging/deconvolvers/hogbom: src/hclean.cpp maximg :51-81 and
// clean :106-210).
//
// CLEAN is a sequence of dependent iterations -- find the residual's peak,
// subtract gain * peak * PSF shifted to it -- so it runs as ONE cooperative
// launch that keeps every workgroup resident and separates iterations with
// a grid-wide exchange, instead of two launches per iteration.  Two kernels
// do so: k_hogbom_reg (below), and, for planes larger than the chip's
// registers and for speed-up thresholds, k_hogbom: workgroup g owns a band of
// image rows.  In every iteration it
//   1. reduces the peak candidate of its band (largest |residual| inside the
//      clean box and the mask; ties go to the lowest row-major index, as the
//      reference's strict > scan does) and publishes it;
//   2. passes the grid barrier, then reduces all bands' candidates itself,
//      so every workgroup reaches the same peak and the same stop decision;
//   3. subtracts gain * peak * PSF over its band and, in the same pass,
//      finds its band's candidate for the next iteration.
// Candidates are double-buffered by iteration parity, so one barrier per
// iteration is enough.  All arithmetic is in the image's type, with separate
// roundings (no contraction), as the reference's C++ does.
#include <algorithm>
#include <cstddef>
#include <type_traits>

#include "tile_common.h"

namespace av {

constexpr int kHogThreads = 1024;
constexpr int kHogMaxGroups = 1024;
constexpr uint32_t kHogSpinLimit = 1u << 25;  // s_sleep rounds before a barrier gives up

// work buffer layout (bytes): header, then two candidate arrays
struct HogHeader {
  uint32_t barrier;  // arrivals, monotonically increasing within a launch
  uint32_t error;    // set when a barrier wait exceeded its spin limit
  int32_t iter, px, py, reason;  // final state; reason 0 = stopped / done, 1 = report
  double maxval;                 // signed peak of the last iteration examined
};
constexpr size_t kHogHeaderBytes = 64;
// What a plane's CLEAN ended with; reason -1: a workgroup did not arrive.
struct HogResult {
  int32_t iter, px, py, reason;
  double maxval;
};
constexpr size_t kHogResultOffset = 8;  // the result of a single plane, in the header
static_assert(offsetof(HogHeader, iter) == kHogResultOffset &&
              offsetof(HogHeader, maxval) == kHogResultOffset + 16, "result in the header");
template <typename T>
struct HogCand {
  T absval, value;
  int32_t idx, pad;
};
constexpr size_t kHogWorkBytes = kHogHeaderBytes + 2 * kHogMaxGroups * sizeof(HogCand<double>);

template <typename T>
__device__ inline bool hog_better(T a, int ia, T b, int ib) {
  return a > b || (a == b && a > (T)0 && ia < ib);
}

// Workgroup reduction of (absval, value, idx); the result is valid in every
// thread.  sv/sx/si are LDS slots for one entry per wave.
template <typename T>
__device__ inline void hog_reduce_wg(T &a, T &v, int &i, T *sa, T *sv, int *si) {
  for (int off = 32; off >= 1; off >>= 1) {
    const T oa = __shfl_xor(a, off, 64);
    const T ov = __shfl_xor(v, off, 64);
    const int oi = __shfl_xor(i, off, 64);
    if (hog_better(oa, oi, a, i)) {
      a = oa;
      v = ov;
      i = oi;
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    sa[wave] = a;
    sv[wave] = v;
    si[wave] = i;
  }
  __syncthreads();
  a = sa[0];
  v = sv[0];
  i = si[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
    if (hog_better(sa[w], si[w], a, i)) {
      a = sa[w];
      v = sv[w];
      i = si[w];
    }
  __syncthreads();
}

template <typename T>
__device__ inline T hog_pow2(T e) {
  if constexpr (sizeof(T) == 4)
    return powf(2.0f, e);
  else
    return pow(2.0, e);
}

// Grid-wide barrier number k of this launch (every workgroup arrives once
// per barrier).  Returns false when the wait exceeded its spin limit (some
// workgroup never arrived); the caller then stops and the host reports it.
__device__ inline bool hog_grid_barrier(HogHeader *h, uint32_t k, uint32_t groups, bool *lds_ok) {
  __syncthreads();
  if (threadIdx.x == 0) {
    __hip_atomic_fetch_add(&h->barrier, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t target = (k + 1) * groups;
    uint32_t spins = 0;
    bool ok = true;
    while (__hip_atomic_load(&h->barrier, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) < target) {
      __builtin_amdgcn_s_sleep(2);
      if (++spins > kHogSpinLimit ||
          __hip_atomic_load(&h->error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        ok = false;
        __hip_atomic_store(&h->error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
    *lds_ok = ok;
  }
  __syncthreads();
  return *lds_ok;
}

template <typename T>
__global__ __launch_bounds__(kHogThreads) void k_hogbom(
    T *__restrict__ model, T *__restrict__ resid, const T *__restrict__ psf,
    const T *__restrict__ mask, int nx, int ny, int xbeg, int xend, int ybeg, int yend,
    int niter, int siter, int start, int report_cycle, int skip_report, T gain, T thres,
    T cspeedup, int px0, int py0, char *work, HogResult *result) {
  HogHeader *h = (HogHeader *)work;
  HogCand<T> *cand = (HogCand<T> *)(work + kHogHeaderBytes);
  __shared__ T s_a[kHogThreads / 64], s_v[kHogThreads / 64];
  __shared__ int s_i[kHogThreads / 64];
  __shared__ bool s_ok;
  const uint32_t G = gridDim.x, g = blockIdx.x;
  const int rpw = (ny + (int)G - 1) / (int)G;
  const int r0 = min(ny, (int)g * rpw), r1 = min(ny, r0 + rpw);
  const int npix = (r1 - r0) * nx;
  const int tid = threadIdx.x;
  const bool domask = mask != nullptr;

  // The band's pixels q = tid + j * B, j = 0, 1, ... (row r0 + q / nx,
  // column q % nx) are walked U at a time (a 2048-row image on 256 bands of
  // 1024 threads gives each thread 16 pixels), the row and column
  // advanced incrementally (one division per thread, not per pixel), and the
  // loads of each group of U pixels issued before their use.
  constexpr int U = sizeof(T) == 4 ? 16 : 8;
  const int B = (int)blockDim.x;
  const int drow = B / nx, dcol = B - drow * nx;
  const int iy_t = r0 + tid / nx, ix_t = tid - (tid / nx) * nx;
  auto in_box = [&](int ix, int iy) {
    return ix >= xbeg && ix < xend && iy >= ybeg && iy < yend &&
           (!domask || mask[iy * nx + ix] > (T)0.5);
  };
  // one pass over the band: subtract pv * PSF shifted to (px, py) inside the
  // window [x1, x2] x [y1, y2] (when SUB), then this thread's candidate for
  // the peak of the clean box
  auto band_pass = [&](auto sub_tag, T pv, int px, int py, int x1, int x2, int y1, int y2,
                       T &ba, T &bv, int &bi) {
    constexpr bool SUB = decltype(sub_tag)::value;
    ba = (T)0;
    bv = (T)0;
    bi = 0x7FFFFFFF;
    int ix = ix_t, iy = iy_t;
    for (int q0 = tid; q0 < npix; q0 += U * B) {
      int cx[U], cy[U];
      bool ok[U], win[U];
      T r[U], pp[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        cx[u] = ix;
        cy[u] = iy;
        ok[u] = q0 + u * B < npix;
        win[u] = false;
        pp[u] = (T)0;
        r[u] = ok[u] ? resid[iy * nx + ix] : (T)0;
        if constexpr (SUB) {
          const int qx = nx / 2 + ix - px, qy = ny / 2 + iy - py;
          win[u] = ok[u] && iy >= y1 && iy <= y2 && ix >= x1 && ix <= x2 && qx >= 0 &&
                   qx < nx && qy >= 0 && qy < ny;
          pp[u] = win[u] ? psf[qy * nx + qx] : (T)0;
        }
        ix += dcol;
        iy += drow;
        if (ix >= nx) {
          ix -= nx;
          ++iy;
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int idx = cy[u] * nx + cx[u];
        if constexpr (SUB) {
          if (win[u]) {
            const T prod = pv * pp[u];
            r[u] = r[u] - prod;
            resid[idx] = r[u];
          }
        }
        if (ok[u] && in_box(cx[u], cy[u])) {
          const T a = fabs(r[u]);
          if (hog_better(a, idx, ba, bi)) {
            ba = a;
            bv = r[u];
            bi = idx;
          }
        }
      }
    }
  };
  T ba, bv;
  int bi;
  band_pass(std::false_type{}, (T)0, 0, 0, 0, -1, 0, -1, ba, bv, bi);

  int px = px0, py = py0;
  T maxval = (T)0;
  int iter = start, reason = 0;
  bool ok = true;
  for (uint32_t k = 0;; ++k, ++iter) {
    if (iter >= niter) break;
    // ---- publish this band's candidate, then reduce all bands
    hog_reduce_wg(ba, bv, bi, s_a, s_v, s_i);
    HogCand<T> *cur = cand + (size_t)(iter & 1) * kHogMaxGroups;
    if (tid == 0) cur[g] = HogCand<T>{ba, bv, bi, 0};
    if (!(ok = hog_grid_barrier(h, k, G, &s_ok))) break;
    T ga = (T)0, gv = (T)0;
    int gi = 0x7FFFFFFF;
    for (uint32_t j = tid; j < G; j += blockDim.x) {
      const T a = __hip_atomic_load(&cur[j].absval, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const T v = __hip_atomic_load(&cur[j].value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int i = __hip_atomic_load(&cur[j].idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (hog_better(a, i, ga, gi)) {
        ga = a;
        gv = v;
        gi = i;
      }
    }
    hog_reduce_wg(ga, gv, gi, s_a, s_v, s_i);
    // ---- the peak (hclean.cpp:127-145): a box with no |r| > 0 keeps the
    // previous position, and the value there is read back
    if (ga > (T)0) {
      py = gi / nx;
      px = gi - py * nx;
      maxval = gv;
    } else {
      maxval = __hip_atomic_load(&resid[py * nx + px], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const T cthres = cspeedup > (T)0 ? thres * hog_pow2((T)(iter - siter) / cspeedup) : thres;
    if (ga < cthres) break;
    if (report_cycle > 0 && iter != skip_report &&
        (iter == siter || (iter % report_cycle) == 1)) {
      reason = 1;
      break;
    }
    // ---- add the component and subtract the shifted PSF (hclean.cpp:166-196)
    const T pv = gain * maxval;
    if (tid == 0 && py >= r0 && py < r1) model[py * nx + px] += pv;
    const int x1 = max(0, px - nx / 2), y1 = max(0, py - ny / 2);
    const int x2 = min(nx - 1, px + nx / 2 - 1), y2 = min(ny - 1, py + ny / 2 - 1);
    band_pass(std::true_type{}, pv, px, py, x1, x2, y1, y2, ba, bv, bi);
  }
  if (g == 0 && tid == 0) {
    result->iter = iter > niter ? niter : iter;
    result->px = px;
    result->py = py;
    result->reason = ok ? reason : -1;
    result->maxval = (double)maxval;
  }
}

// ---- register-resident CLEAN ----------------------------------------------
// The kernel that runs whenever a plane fits the chip's registers and the
// threshold is fixed (a speed-up's 2^x takes the registers of many rows).  What
// bounds an iteration is its chain of dependent latencies (peak, exchange,
// subtraction), not bandwidth, so a plane's residual stays in registers for
// the whole call, the exchange between workgroups needs no memory fence, and
// the planes of a cube run side by side:
//   * a wavefront owns a tile of 64 columns x H rows, a lane one column of
//     it, H residuals in registers; an iteration reads the PSF only, through
//     a uniform row address and one lane offset;
//   * a plane belongs to a group of workgroups, which meet once per iteration
//     through tagged slots: each publishes its candidate (value, index) with
//     one 64-bit store (two for FP64) carrying a phase bit, and reads the
//     others' slots until they carry it.  Slots alternate by parity, so a
//     phase bit per pair of rounds tells a round's slots from those two
//     rounds before.  Only the slots cross workgroups; nothing else needs to
//     be made visible, so no cache is written back or invalidated.
//   * the groups of one launch take the planes in strides.
// 8 planes of 1024 x 1024 FP32, an iteration of all of them: 6.5 us, against
// 165 us plane by plane with the band kernel.
constexpr int kHogWaves = kHogThreads / 64;
// us of an iteration: constant, per row of a lane, per workgroup of a plane,
// and the factor on the rows when two workgroups share a CU (see HogLayout)
constexpr double kHogT0 = 3.1, kHogT1 = 0.085, kHogT2 = 0.0095, kHogCrowd = 3.0;

struct HogRegArgs {
  void *model, *resid;
  const void *psf, *mask;
  int nx, ny, xbeg, xend, ybeg, yend, niter, siter, start, report_cycle, skip_report;
  double gain, thres, cspeedup;
  int px0, py0, n_planes, planes_per_psf;
  int wgs_per_plane, groups, col_tiles;
  unsigned long long *slots;  // [2 parities][workgroup][2 words]
  uint32_t *error;
  HogResult *result;  // [n_planes]
};

// One word of a published candidate: 32 bits of the value, the index (31
// bits) and the phase bit.
__device__ inline unsigned long long hog_word(uint32_t bits, int idx, uint32_t tag) {
  return ((unsigned long long)bits << 32) | ((uint32_t)idx << 1) | tag;
}

template <typename T>
__device__ inline void hog_publish(unsigned long long *slot, T v, int idx, uint32_t tag) {
  if constexpr (sizeof(T) == 4) {
    __hip_atomic_store(slot, hog_word(__float_as_uint(v), idx, tag), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  } else {
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    __hip_atomic_store(slot, hog_word((uint32_t)(b >> 32), idx, tag), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(slot + 1, hog_word((uint32_t)b, idx, tag), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
  }
}

// A slot's candidate, once every word of it carries `tag`.
template <typename T>
__device__ inline bool hog_read(const unsigned long long *slot, uint32_t tag, T &v, int &idx) {
  const unsigned long long a =
      __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  idx = (int)((uint32_t)a >> 1);
  if constexpr (sizeof(T) == 4) {
    v = __uint_as_float((uint32_t)(a >> 32));
    return ((uint32_t)a & 1u) == tag;
  } else {
    const unsigned long long b =
        __hip_atomic_load(slot + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v = __longlong_as_double((long long)((a >> 32 << 32) | (b >> 32)));
    return ((uint32_t)a & 1u) == tag && ((uint32_t)b & 1u) == tag;
  }
}

// The better of two candidates (value, index); `want` >= 0 asks for that
// index instead.
template <typename T>
__device__ inline bool hog_wins(T ov, int oi, T v, int i, int want) {
  if (want >= 0) return oi == want && i != want;
  return hog_better((T)fabs(ov), oi, (T)fabs(v), i);
}

template <typename T>
__device__ inline void hog_wave_reduce(T &v, int &i, int want, int width) {
  for (int off = width / 2; off >= 1; off >>= 1) {
    const T ov = __shfl_xor(v, off, 64);
    const int oi = __shfl_xor(i, off, 64);
    if (hog_wins(ov, oi, v, i, want)) {
      v = ov;
      i = oi;
    }
  }
}

template <typename T>
struct HogShared {
  T v[kHogWaves], gv;
  int i[kHogWaves], gi;
  bool ok;
};

// The best candidate of the plane's workgroups, in every thread; round k of
// this launch.  False when some workgroup never published (spin limit).
template <typename T>
__device__ inline bool hog_exchange(const HogRegArgs &A, HogShared<T> &sh, uint32_t k, int wg0,
                                    int member, T &v, int &i, int want) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  hog_wave_reduce(v, i, want, 64);
  if (lane == 0) {
    sh.v[wave] = v;
    sh.i[wave] = i;
  }
  __syncthreads();
  if (wave == 0) {
    v = sh.v[lane & (kHogWaves - 1)];
    i = sh.i[lane & (kHogWaves - 1)];
    hog_wave_reduce(v, i, want, kHogWaves);
    const uint32_t tag = ((k >> 1) & 1u) ^ 1u;
    unsigned long long *slots =
        A.slots + 2 * ((size_t)(k & 1u) * (A.groups * A.wgs_per_plane) + wg0);
    bool ok = true;
    if (A.wgs_per_plane > 1) {
      if (lane == 0) hog_publish(slots + 2 * member, v, i, tag);
      uint32_t spins = 0;
      T bv = (T)0;
      int bi = 0x7FFFFFFF;
      for (int j = lane; j < A.wgs_per_plane; j += 64) {
        T ov;
        int oi;
        while (!hog_read(slots + 2 * j, tag, ov, oi)) {
          __builtin_amdgcn_s_sleep(1);
          if (++spins > kHogSpinLimit ||
              __hip_atomic_load(A.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            ok = false;
            break;
          }
        }
        if (!ok) {
          __hip_atomic_store(A.error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        if (hog_wins(ov, oi, bv, bi, want)) {
          bv = ov;
          bi = oi;
        }
      }
      v = bv;
      i = bi;
      hog_wave_reduce(v, i, want, 64);
      ok = __all(ok);
    }
    if (lane == 0) {
      sh.gv = v;
      sh.gi = i;
      sh.ok = ok;
    }
  }
  __syncthreads();
  v = sh.gv;
  i = sh.gi;
  return sh.ok;
}

template <typename T, int H>
__global__ __launch_bounds__(kHogThreads, (H * sizeof(T) <= 64 ? 8 : 4)) void k_hogbom_reg(HogRegArgs A) {
  __shared__ HogShared<T> sh;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // consecutive workgroups of a group on one XCD, whose L2 then holds its PSF
  const int total = A.groups * A.wgs_per_plane;
  const int v_blk = (int)gridDim.x % kXcds == 0
                        ? (int)(blockIdx.x % kXcds) * ((int)gridDim.x / kXcds) + blockIdx.x / kXcds
                        : (int)blockIdx.x;
  if (v_blk >= total) return;
  const int group = v_blk / A.wgs_per_plane, member = v_blk - group * A.wgs_per_plane;
  const int wg0 = group * A.wgs_per_plane;
  const int nx = A.nx, ny = A.ny;
  // this wavefront's tile: rows iy0 .., this lane's column ix
  const int t = __builtin_amdgcn_readfirstlane(member * kHogWaves + wave);
  const int iy0 = t / A.col_tiles * H, ix = (t % A.col_tiles) * 64 + lane;
  const bool have = iy0 < ny && ix < nx;
  const int rows = min(H, ny - iy0);  // <= 0 for a wavefront past the plane
  const T *mask = (const T *)A.mask;
  // rows of this column that may hold the peak
  unsigned long long allow = 0ull;
  if (have && ix >= A.xbeg && ix < A.xend)
    for (int h = 0; h < rows; ++h)
      if (iy0 + h >= A.ybeg && iy0 + h < A.yend &&
          (!mask || mask[(size_t)(iy0 + h) * nx + ix] > (T)0.5))
        allow |= 1ull << h;
  const unsigned long long all_rows = rows >= 64 ? ~0ull : rows > 0 ? (1ull << rows) - 1ull : 0ull;
  // every pixel of the tile may (those outside the image stay zero)
  const bool open = __all(!have || allow == all_rows);
  const T gain = (T)A.gain, thres = (T)A.thres;
  uint32_t k = 0;
  bool ok = true;
  for (int plane = group; plane < A.n_planes && ok; plane += A.groups) {
    T *model = (T *)A.model + (size_t)plane * nx * ny;
    T *resid = (T *)A.resid + (size_t)plane * nx * ny;
    const T *psf = (const T *)A.psf + (size_t)(plane / A.planes_per_psf) * nx * ny;
    T r[H];
    T *rp = resid + (size_t)max(iy0, 0) * nx;  // uniform row, lane offset ix
#pragma unroll
    for (int h = 0; h < H; ++h, rp += nx) {
      int n_rows = have ? rows : 0;
      asm volatile("" : "+s"(rp), "+v"(n_rows));
      r[h] = h < n_rows ? rp[ix] : (T)0;
    }
    // the lane's candidate: its first row of the largest |r|
    T bv = (T)0;
    int bh = -1;
    auto candidate = [&](int h) {
      if (fabs(r[h]) > fabs(bv)) {
        bv = r[h];
        bh = h;
      }
    };
#pragma unroll
    for (int hb = 0; hb < H; hb += 8) {
      uint32_t abits = (uint32_t)(allow >> hb);
      asm volatile("" : "+v"(abits));
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if ((abits >> u) & 1u) candidate(hb + u);
    }
    int px = A.px0, py = A.py0, iter = A.start, reason = 0;
    T maxval = (T)0;
    for (;; ++iter) {
      if (iter >= A.niter) break;
      T gv = bv;
      int gi = bh >= 0 ? (iy0 + bh) * nx + ix : 0x7FFFFFFF;
      if (!(ok = hog_exchange(A, sh, k++, wg0, member, gv, gi, -1))) break;
      gi = __builtin_amdgcn_readfirstlane(gi);  // the same in every lane
      const T ga = fabs(gv);
      // the peak (hclean.cpp:127-145): a box with no |r| > 0 keeps the
      // previous position, and the value there is read back
      if (ga > (T)0) {
        py = gi / nx;
        px = gi - py * nx;
        maxval = gv;
      } else {
        const int want = py * nx + px;
        T wv = (T)0;
        int wi = 0x7FFFFFFF;
        if (have && ix == px && py >= iy0 && py < iy0 + rows) {
          wi = want;
#pragma unroll
          for (int h = 0; h < H; ++h) {
            int at = py - iy0;
            asm volatile("" : "+s"(at));
            if (h == at) wv = r[h];
          }
        }
        if (!(ok = hog_exchange(A, sh, k++, wg0, member, wv, wi, want))) break;
        maxval = wv;
      }
      if (ga < thres) break;
      if (A.report_cycle > 0 && iter != A.skip_report &&
          (iter == A.siter || (iter % A.report_cycle) == 1)) {
        reason = 1;
        break;
      }
      // add the component and subtract the shifted PSF (hclean.cpp:166-196)
      const T pv = gain * maxval;
      if (have && ix == px && py >= iy0 && py < iy0 + H) model[(size_t)py * nx + px] += pv;
      const int x1 = max(0, px - nx / 2), y1 = max(0, py - ny / 2);
      const int x2 = min(nx - 1, px + nx / 2 - 1), y2 = min(ny - 1, py + ny / 2 - 1);
      const int qx = nx / 2 + ix - px, qy0 = ny / 2 + iy0 - py;
      const bool colwin = have && ix >= x1 && ix <= x2 && qx >= 0 && qx < nx;
      const int qxc = min(max(qx, 0), nx - 1);
      // rows of the tile inside the window and the PSF: uniform
      const int h0 = max(max(y1 - iy0, -qy0), 0), h1 = min(min(y2 - iy0 + 1, ny - qy0), rows);
      bv = (T)0;
      bh = -1;
      constexpr int U = std::min(H, (H < 64 ? 64 : 32) / (int)sizeof(T));  // loads in flight
      if (open && h0 == 0 && h1 == H && __all(colwin)) {
        // the whole tile is subtracted from and searched
        const T *row = psf + (size_t)qy0 * nx;
#pragma unroll
        for (int hb = 0; hb < H; hb += U) {
          T pp[U];
#pragma unroll
          for (int u = 0; u < U; ++u, row += nx) {
            asm volatile("" : "+s"(row));
            pp[u] = row[(uint32_t)qxc];
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const T prod = pv * pp[u];
            r[hb + u] = r[hb + u] - prod;
            candidate(hb + u);
          }
        }
      } else {
        // one bit per row: subtract there, search there
        const unsigned long long upto = h1 >= 64 ? ~0ull : h1 > 0 ? (1ull << h1) - 1ull : 0ull;
        const unsigned long long win =
            colwin && h0 < 64 ? upto & ~((1ull << h0) - 1ull) : 0ull;
        // (32 rows at a time, opaque to the compiler, which would keep a lane
        // mask per row in scalar registers for the whole loop)
#pragma unroll
        for (int hb = 0; hb < H; hb += U) {
          uint32_t wbits = (uint32_t)(win >> (hb & 32)), abits = (uint32_t)(allow >> (hb & 32));
          asm volatile("" : "+v"(wbits), "+v"(abits));
          T pp[U];
#pragma unroll
          for (int u = 0; u < U; ++u) {
            int qy = qy0 + hb + u;
            asm volatile("" : "+s"(qy));
            pp[u] = (psf + (size_t)min(max(qy, 0), ny - 1) * nx)[(uint32_t)qxc];
          }
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const T prod = pv * pp[u];
            if ((wbits >> ((hb + u) & 31)) & 1u) r[hb + u] = r[hb + u] - prod;
            if ((abits >> ((hb + u) & 31)) & 1u) candidate(hb + u);
          }
        }
      }
    }
    rp = resid + (size_t)max(iy0, 0) * nx;
#pragma unroll
    for (int h = 0; h < H; ++h, rp += nx) {
      int n_rows = have ? rows : 0;
      asm volatile("" : "+s"(rp), "+v"(n_rows));
      if (h < n_rows) rp[ix] = r[h];
    }
    if (member == 0 && threadIdx.x == 0) {
      HogResult *o = A.result + plane;
      o->iter = iter > A.niter ? A.niter : iter;
      o->px = px;
      o->py = py;
      o->reason = ok ? reason : -1;
      o->maxval = (double)maxval;
    }
  }
}

// maxval per workgroup slice, then one reduction: min and max of the
// (masked) image starting from +-1e20 (hclean.cpp:51-81).
template <typename T>
__global__ __launch_bounds__(256) void k_maximg(const T *__restrict__ img,
                                                const T *__restrict__ mask, int64_t n, T *out) {
  __shared__ T smin[4], smax[4];
  T lo = (T)1e20, hi = (T)-1e20;
  for (int64_t k = threadIdx.x; k < n; k += blockDim.x) {
    if (!mask || mask[k] > (T)0.5) {
      const T w = img[k];
      if (w > hi) hi = w;
      if (w < lo) lo = w;
    }
  }
  for (int off = 32; off >= 1; off >>= 1) {
    const T ol = __shfl_xor(lo, off, 64), oh = __shfl_xor(hi, off, 64);
    lo = ol < lo ? ol : lo;
    hi = oh > hi ? oh : hi;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    smin[wave] = lo;
    smax[wave] = hi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      lo = smin[w] < lo ? smin[w] : lo;
      hi = smax[w] > hi ? smax[w] : hi;
    }
    out[0] = lo;
    out[1] = hi;
  }
}

// Before a launch: zero the arrivals, the error mark (unless another plane of
// the call set it: `first` false) and the slots, `n` words in all, and mark the
// planes' results as not reached: a group that misses an exchange leaves its
// remaining planes so.  The header's words between are a single plane's result.
__global__ void k_hog_clear(uint32_t *w, int n, bool first, HogResult *result, int n_planes) {
  constexpr int kHead = (int)(kHogHeaderBytes / 4);
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0 || (i == 1 && first) || (i >= kHead && i < n)) w[i] = 0u;
  if (i < n_planes) result[i].reason = -1;
}

static int launch_hog_clear(void *work, int words, bool first, HogResult *result, int n_planes,
                            hipStream_t s) {
  const int n = std::max(words, n_planes);
  hipLaunchKernelGGL(k_hog_clear, dim3((n + 255) / 256), dim3(256), 0, s, (uint32_t *)work, words,
                     first, result, n_planes);
  AV_LAUNCH_CHECK("k_hog_clear");
  return AV_OK;
}

// One plane by row bands (any size).
template <typename T>
static int launch_hogbom_bands(const HogRegArgs &A, void *model, void *resid, const void *psf,
                               void *work, HogResult *result, const DeviceProps &prop,
                               hipStream_t s) {
  int per_cu = 0;
  AV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_hogbom<T>, kHogThreads, 0));
  int groups = std::min(std::min(prop.num_cus * std::max(per_cu, 0), kHogMaxGroups), A.ny);
  if (groups < 1) return fail(AV_ERR_HIP, "av_hogbom_clean: no resident workgroup possible");
  groups = std::min(groups, prop.num_cus);  // one band per CU
  const int rc = launch_hog_clear(work, (int)(kHogHeaderBytes / 4), result == A.result, result, 1, s);
  if (rc) return rc;
  T *m = (T *)model, *r = (T *)resid;
  const T *p = (const T *)psf, *k = (const T *)A.mask;
  T tg = (T)A.gain, tt = (T)A.thres, tc = (T)A.cspeedup;
  char *w = (char *)work;
  HogRegArgs a = A;
  void *args[] = {&m,     &r,           &p,          &k,  &a.nx, &a.ny, &a.xbeg, &a.xend,
                  &a.ybeg,  &a.yend,        &a.niter,      &a.siter, &a.start, &a.report_cycle,
                  &a.skip_report, &tg, &tt, &tc, &a.px0, &a.py0, &w, &result};
  AV_HIP(hipLaunchCooperativeKernel((const void *)k_hogbom<T>, dim3((unsigned)groups),
                                    dim3(kHogThreads), args, 0, s));
  return AV_OK;
}

// How the register-resident kernel would lay the planes out with H rows per
// lane: workgroups per plane, planes side by side, and the time that takes.
// The model's figures are measured ones (us an iteration of all planes, FP32):
//   planes x side     H = 8    16     32    band kernel, plane by plane
//    1 x  256         3.82   4.52   5.67
//    1 x 1024         4.96   5.03   5.79    20.6
//    1 x 2048        10.34   7.61   7.06    21.5
//    8 x 1024        13.91   7.91   6.47   164.9
//   64 x  256         5.32   4.51   5.66
//    4 x 2048        40.75  19.27  14.98
// 64 rows (FP64: 32) spill registers (10 to 14 us) and serve only planes that
// fit no other way.
struct HogLayout {
  int h = 0, wgs = 0, groups = 0;
  double cost = 0.0;
};

template <typename T, int H>
static int hog_try(const HogRegArgs &A, const DeviceProps &prop, HogLayout &best) {
  int per_cu = 0;
  AV_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (k_hogbom_reg<T, H>), kHogThreads,
                                                      0));
  per_cu = std::min(per_cu, 2);
  const int64_t tiles = (int64_t)A.col_tiles * ((A.ny + H - 1) / H);
  const int64_t wgs = (tiles + kHogWaves - 1) / kHogWaves;
  for (int o = 1; o <= per_cu; ++o) {
    const int64_t room = std::min<int64_t>((int64_t)prop.num_cus * o, kHogMaxGroups);
    if (wgs > room) continue;
    const int64_t groups = std::min<int64_t>(room / wgs, A.n_planes);
    const double rounds = (double)((A.n_planes + groups - 1) / groups);
    // two on a CU only when more planes need them
    const double crowd = groups * wgs > prop.num_cus ? kHogCrowd : 1.0;
    const double cost =
        rounds * (kHogT0 + kHogT1 * H * crowd * (sizeof(T) == 8 ? 1.3 : 1.0) + kHogT2 * wgs);
    if (best.h == 0 || cost < best.cost) best = HogLayout{H, (int)wgs, (int)groups, cost};
  }
  return AV_OK;
}

template <typename T, int H>
static int launch_hogbom_reg(HogRegArgs &A, hipStream_t s) {
  void *args[] = {&A};
  AV_HIP(hipLaunchCooperativeKernel((const void *)k_hogbom_reg<T, H>,
                                    dim3((unsigned)(A.groups * A.wgs_per_plane)),
                                    dim3(kHogThreads), args, 0, s));
  return AV_OK;
}

template <typename T>
static int launch_hogbom(HogRegArgs &A, void *work, hipStream_t s) {
  const DeviceProps &prop = device_props();
  if (prop.error) return hip_fail(prop.error, "av_hogbom_clean: device properties");
  A.col_tiles = (A.nx + 63) / 64;
  HogLayout L;
  int rc = AV_OK;
  constexpr int kMost = sizeof(T) == 4 ? 64 : 32;  // rows: the layout that spills
  if (!(A.cspeedup > 0.0)) {
    if ((rc = hog_try<T, 8>(A, prop, L)) || (rc = hog_try<T, 16>(A, prop, L)) ||
        (rc = hog_try<T, kMost / 2>(A, prop, L)) ||
        (L.h == 0 && (rc = hog_try<T, kMost>(A, prop, L))))
      return rc;
  }
  if (L.h == 0) {
    const size_t plane = (size_t)A.nx * A.ny;
    for (int p = 0; p < A.n_planes; ++p)
      if ((rc = launch_hogbom_bands<T>(A, (T *)A.model + p * plane, (T *)A.resid + p * plane,
                                       (const T *)A.psf + p / A.planes_per_psf * plane, work,
                                       A.result + p, prop, s)))
        return rc;
    return AV_OK;
  }
  A.wgs_per_plane = L.wgs;
  A.groups = L.groups;
  A.error = (uint32_t *)((char *)work + offsetof(HogHeader, error));
  A.slots = (unsigned long long *)((char *)work + kHogHeaderBytes);
  // phase bits 0 in every slot: what no round of the first two expects
  const int words = (int)(kHogHeaderBytes / 4) + L.wgs * L.groups * 8;
  if ((rc = launch_hog_clear(work, words, true, A.result, A.n_planes, s))) return rc;
  if (L.h == 8) return launch_hogbom_reg<T, 8>(A, s);
  if (L.h == 16) return launch_hogbom_reg<T, 16>(A, s);
  if (L.h == kMost / 2) return launch_hogbom_reg<T, kMost / 2>(A, s);
  return launch_hogbom_reg<T, kMost>(A, s);
}

static_assert(kHogHeaderBytes + (size_t)kHogMaxGroups * 32 <= kHogWorkBytes, "slots fit the work");

// Argument checks shared by the two entry points.
static int hog_check(const HogRegArgs &A, const void *work) {
  if (!A.model || !A.resid || !A.psf || !work || !A.result)
    return fail(AV_ERR_INVALID, "av_hogbom_clean: NULL argument");
  if (A.nx < 1 || A.ny < 1 || (int64_t)A.nx * A.ny >= ((int64_t)1 << 31))
    return fail(AV_ERR_INVALID, "av_hogbom_clean: image size out of range");
  if (!(0 <= A.xbeg && A.xbeg < A.xend && A.xend <= A.nx && 0 <= A.ybeg && A.ybeg < A.yend &&
        A.yend <= A.ny))
    return fail(AV_ERR_INVALID, "av_hogbom_clean: clean box outside the image");
  if (A.px0 < 0 || A.px0 >= A.nx || A.py0 < 0 || A.py0 >= A.ny)
    return fail(AV_ERR_INVALID, "av_hogbom_clean: previous peak outside the image");
  return AV_OK;
}

static int hog_launch(HogRegArgs &A, int32_t dtype, void *work, void *stream) {
  if (dtype == AV_F32) return launch_hogbom<float>(A, work, (hipStream_t)stream);
  if (dtype == AV_F64) return launch_hogbom<double>(A, work, (hipStream_t)stream);
  return fail(AV_ERR_INVALID, "av_hogbom_clean: dtype must be AV_F32 or AV_F64");
}

}  // namespace av

using namespace av;

extern "C" {

int av_hogbom_work_bytes(int64_t *bytes) {
  if (!bytes) return fail(AV_ERR_INVALID, "av_hogbom_work_bytes: NULL argument");
  *bytes = (int64_t)kHogWorkBytes;
  return AV_OK;
}

int av_hogbom_maximg(const void *image, const void *mask, int32_t nx, int32_t ny, int32_t dtype,
                     void *out, void *stream) {
  if (!image || !out || nx < 1 || ny < 1)
    return fail(AV_ERR_INVALID, "av_hogbom_maximg: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  const int64_t n = (int64_t)nx * ny;
  if (dtype == AV_F32)
    hipLaunchKernelGGL(k_maximg<float>, dim3(1), dim3(256), 0, s, (const float *)image,
                       (const float *)mask, n, (float *)out);
  else if (dtype == AV_F64)
    hipLaunchKernelGGL(k_maximg<double>, dim3(1), dim3(256), 0, s, (const double *)image,
                       (const double *)mask, n, (double *)out);
  else
    return fail(AV_ERR_INVALID, "av_hogbom_maximg: dtype must be AV_F32 or AV_F64");
  AV_LAUNCH_CHECK("k_maximg");
  return AV_OK;
}

int av_hogbom_clean(void *model, void *residual, const void *psf, const void *mask, int32_t nx,
                    int32_t ny, int32_t xbeg, int32_t xend, int32_t ybeg, int32_t yend,
                    int32_t niter, int32_t siter, int32_t start, int32_t report_cycle,
                    int32_t skip_report, double gain, double thres, double cspeedup,
                    int32_t px0, int32_t py0, int32_t dtype, void *work, void *stream) {
  HogRegArgs A{};
  A.model = model;
  A.resid = residual;
  A.psf = psf;
  A.mask = mask;
  A.nx = nx;
  A.ny = ny;
  A.xbeg = xbeg;
  A.xend = xend;
  A.ybeg = ybeg;
  A.yend = yend;
  A.niter = niter;
  A.siter = siter;
  A.start = start;
  A.report_cycle = report_cycle;
  A.skip_report = skip_report;
  A.gain = gain;
  A.thres = thres;
  A.cspeedup = cspeedup;
  A.px0 = px0;
  A.py0 = py0;
  A.n_planes = A.planes_per_psf = 1;
  A.result = work ? (HogResult *)((char *)work + kHogResultOffset) : nullptr;
  const int rc = hog_check(A, work);
  return rc ? rc : hog_launch(A, dtype, work, stream);
}

int av_hogbom_clean_planes(void *model, void *residual, const void *psf, int32_t n_planes,
                           int32_t planes_per_psf, int32_t nx, int32_t ny, int32_t niter,
                           double gain, double thres, int32_t dtype, void *result, void *work,
                           void *stream) {
  if (n_planes < 0 || planes_per_psf < 1)
    return fail(AV_ERR_INVALID, "av_hogbom_clean_planes: bad plane counts");
  if (n_planes == 0) return AV_OK;
  HogRegArgs A{};
  A.model = model;
  A.resid = residual;
  A.psf = psf;
  A.nx = nx;
  A.ny = ny;
  A.xend = nx;
  A.yend = ny;
  A.niter = niter;
  A.skip_report = -1;
  A.gain = gain;
  A.thres = thres;
  A.n_planes = n_planes;
  A.planes_per_psf = planes_per_psf;
  A.result = (HogResult *)result;
  const int rc = hog_check(A, work);
  return rc ? rc : hog_launch(A, dtype, work, stream);
}

}  // extern "C"

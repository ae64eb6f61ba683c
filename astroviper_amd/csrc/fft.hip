// fft.hip -- the two-dimensional FFTs between the uv grid and real images,
// each in two passes over memory with every step around it fused:
//   uv to image (grid2image_spheroid_ms4, core/imaging/imaging_utils/
//   standard_grid.py:693-708): fold the shifted grid to its Hermitian half,
//   inverse FFT along u | complex-to-real inverse FFT along v, taper
//   correction, 1 / sumwt;
//   image to uv (fft_lm_to_uv, core/imaging/fft.py:5-18, as
//   predict_model_visibilities applies it, imager.py:96-99): taper,
//   real-to-complex FFT along v | FFT along u, the other half from
//   F[-k] = conj(F[k]), fftshift.
// What bounds them is memory, at two thirds to nine tenths of a large copy's 4.67
// TB/s: the grid and the image once, the half spectrum in between written and
// read once.  32 planes of 2048 x 2048, complex64 to FP64 images: 1.41 ms for 4.5
// GB counted (columns 2.35, rows 2.15), 3.2 TB/s, as a block of long columns fills
// a CU's LDS and no other workgroup loads while it computes (fold, rocFFT's
// complex-to-real transform and normalisation: 3.87 ms); 16 planes of 1024 x 1024
// FP64: 0.20 ms to the image for 0.71 GB, 3.5 TB/s, 0.17 to the grid for 0.74, 4.3
// TB/s (transform alone: 0.36).  Groups of planes whose half spectra fit the 256 MB
// Infinity Cache were slower (1.58 ms in groups of two planes): their last
// workgroups leave more idle than the cache saves.  The groups only bound the work
// memory.
//
// A workgroup transforms several columns (or rows) of one plane in LDS, in
// FP64 whatever the types in memory.  The transform is Stockham's
// self-sorting one with radices 8, 4, 2, 3 and 5: pass by pass a thread takes
// butterfly j, reads its R points N / R apart into registers, multiplies by
// the twiddle factors and writes them where the next pass expects them.  The
// first pass reads its points straight from memory and the last writes them
// there.  Twiddle factors come from a table of exp(2 pi i q / n), formed in
// each call with the tapers by one small launch.  Even axes whose sizes have
// no other prime factors are served; torch.fft does the rest.
#include <algorithm>

#include "ps_eval.h"
#include "tile_common.h"

namespace av {

constexpr int kFftMaxPasses = 8;
constexpr int kFftThreads = 1024;                // most threads of a workgroup
constexpr int kFftPoints = 8;                    // most points of a thread
constexpr int kFftWgPoints = kFftThreads * kFftPoints;
constexpr int kFftRowPoints = 1024;              // points of a workgroup of several rows
constexpr int64_t kFftGroupBytes = (int64_t)2 << 30;  // half spectra of a group of planes

// One axis: its length, radices, and per pass 2^32 / Ns (rounded up, the
// quotient j / Ns of j < 2^16 is then exact), Ns the product of the radices
// before it.
struct FftAxis {
  int n, passes;
  int radix[kFftMaxPasses];
  uint32_t ns_inv[kFftMaxPasses];
};

static bool fft_axis(int n, FftAxis &a) {
  a.n = n;
  a.passes = 0;
  int rest = n, ns = 1;
  for (int r : {8, 5, 3, 4, 2}) {
    while (rest % r == 0 && a.passes < kFftMaxPasses) {
      a.radix[a.passes] = r;
      a.ns_inv[a.passes++] = ns == 1 ? 0u : (uint32_t)(((1ull << 32) + ns - 1) / ns);
      rest /= r;
      ns *= r;
    }
  }
  return rest == 1 && a.passes >= 2;
}

__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}
__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
// i a (inverse transforms) or -i a
template <bool INV>
__device__ inline double2 cturn(double2 a) {
  return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

// DFT of R points in place, X[m] = sum_q v[q] exp(+-2 pi i q m / R)
template <int R, bool INV>
__device__ inline void dft(double2 (&v)[R]) {
  if constexpr (R == 2) {
    const double2 a = v[0];
    v[0] = cadd(a, v[1]);
    v[1] = csub(a, v[1]);
  } else if constexpr (R == 3) {
    constexpr double s3 = 0.86602540378443864676;  // sin(pi / 3)
    const double2 t = cadd(v[1], v[2]);
    const double2 d = cturn<INV>(csub(v[1], v[2]));
    const double2 m = make_double2(fma(-0.5, t.x, v[0].x), fma(-0.5, t.y, v[0].y));
    v[0] = cadd(v[0], t);
    v[1] = make_double2(fma(s3, d.x, m.x), fma(s3, d.y, m.y));
    v[2] = make_double2(fma(-s3, d.x, m.x), fma(-s3, d.y, m.y));
  } else if constexpr (R == 4) {
    const double2 a = cadd(v[0], v[2]), b = csub(v[0], v[2]);
    const double2 c = cadd(v[1], v[3]), d = cturn<INV>(csub(v[1], v[3]));
    v[0] = cadd(a, c);
    v[1] = cadd(b, d);
    v[2] = csub(a, c);
    v[3] = csub(b, d);
  } else if constexpr (R == 5) {
    constexpr double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
    constexpr double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
    const double2 a1 = cadd(v[1], v[4]), a2 = cadd(v[2], v[3]);
    const double2 b1 = cturn<INV>(csub(v[1], v[4])), b2 = cturn<INV>(csub(v[2], v[3]));
    const double2 m1 = make_double2(fma(c2, a2.x, fma(c1, a1.x, v[0].x)),
                                    fma(c2, a2.y, fma(c1, a1.y, v[0].y)));
    const double2 m2 = make_double2(fma(c1, a2.x, fma(c2, a1.x, v[0].x)),
                                    fma(c1, a2.y, fma(c2, a1.y, v[0].y)));
    const double2 n1 = make_double2(fma(s2, b2.x, s1 * b1.x), fma(s2, b2.y, s1 * b1.y));
    const double2 n2 = make_double2(fma(-s1, b2.x, s2 * b1.x), fma(-s1, b2.y, s2 * b1.y));
    v[0] = cadd(v[0], cadd(a1, a2));
    v[1] = cadd(m1, n1);
    v[4] = csub(m1, n1);
    v[2] = cadd(m2, n2);
    v[3] = csub(m2, n2);
  } else {
    static_assert(R == 8, "radix");
    constexpr double h = 0.70710678118654752440;
    double2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft<4, INV>(e);
    dft<4, INV>(o);
    // o[m] times exp(+-2 pi i m / 8)
    const double2 t1 = cturn<INV>(o[1]), t3 = cturn<INV>(o[3]);
    o[1] = make_double2(h * (o[1].x + t1.x), h * (o[1].y + t1.y));
    o[2] = cturn<INV>(o[2]);
    o[3] = make_double2(h * (t3.x - o[3].x), h * (t3.y - o[3].y));
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      v[m] = cadd(e[m], o[m]);
      v[m + 4] = csub(e[m], o[m]);
    }
  }
}

// The points of a workgroup in LDS: point i of series c.  A pad point per
// eight keeps the strided writes of the first passes off each other's banks.
// BYC: the series of a point lie together (columns of a plane), else the
// points of a series (rows).
template <bool BYC>
struct FftLds {
  double2 *p;
  int nc, pitch;  // series (a power of two when BYC), points of a series with pads
  __device__ double2 &at(int i, int c) const {
    const int q = i + (i >> 3);
    return BYC ? p[q * nc + c] : p[c * pitch + q];
  }
  __device__ double2 operator()(int i, int c) const { return at(i, c); }
  __device__ void operator()(int i, int c, double2 v) const { at(i, c) = v; }
};

__host__ __device__ inline int fft_pitch(int n) { return n + n / 8 + 1; }

// Butterfly b of the workgroup: its index j in the series and the series c.
template <bool BYC>
__device__ inline void split_butterfly(int b, int nbf, int nc_log2, int &j, int &c) {
  if (BYC) {
    c = b & ((1 << nc_log2) - 1);
    j = b >> nc_log2;
  } else {
    c = b / nbf;
    j = b - c * nbf;
  }
}

// One radix-R pass: reads in(i, c), writes out(i, c, v).  tw[q * tstep] =
// exp(2 pi i q / n).  `wait`: the reads and writes share the LDS.
template <int R, bool INV, bool BYC, typename In, typename Out>
__device__ inline void fft_pass(const FftAxis &a, int nc, int nc_log2, int ns, uint32_t ns_inv,
                                const double2 *tw, int tstep, In in, Out out, bool wait) {
  constexpr int NB = (kFftPoints + R - 1) / R;  // butterflies of a thread
  const int nbf = a.n / R, total = nbf * nc;
  const int T = blockDim.x;
  double2 v[NB][R];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int b = threadIdx.x + i * T;
    if (b < total) {
      int j, c;
      split_butterfly<BYC>(b, nbf, nc_log2, j, c);
#pragma unroll
      for (int m = 0; m < R; ++m) v[i][m] = in(j + m * nbf, c);
    }
  }
  if (wait) __syncthreads();
  const int wstep = nbf / ns * tstep;  // table step of exp(2 pi i / (ns R))
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int b = threadIdx.x + i * T;
    if (b < total) {
      int j, c;
      split_butterfly<BYC>(b, nbf, nc_log2, j, c);
      const int q = ns == 1 ? j : (int)(((uint64_t)(uint32_t)j * ns_inv) >> 32);  // j / ns
      const int k = j - q * ns;
      if (ns > 1) {
#pragma unroll
        for (int m = 1; m < R; ++m) {
          double2 w = tw[(size_t)(k * m) * wstep];
          if (!INV) w.y = -w.y;
          v[i][m] = cmul(v[i][m], w);
        }
      }
      dft<R, INV>(v[i]);
#pragma unroll
      for (int m = 0; m < R; ++m) out(q * ns * R + k + m * ns, c, v[i][m]);
    }
  }
}

template <bool INV, bool BYC, typename In, typename Out>
__device__ inline void fft_pass_any(const FftAxis &a, int pass, int nc, int nc_log2, int ns,
                                    const double2 *tw, int tstep, In in, Out out, bool wait) {
  const uint32_t inv = a.ns_inv[pass];
  switch (a.radix[pass]) {
    case 8: fft_pass<8, INV, BYC>(a, nc, nc_log2, ns, inv, tw, tstep, in, out, wait); break;
    case 5: fft_pass<5, INV, BYC>(a, nc, nc_log2, ns, inv, tw, tstep, in, out, wait); break;
    case 4: fft_pass<4, INV, BYC>(a, nc, nc_log2, ns, inv, tw, tstep, in, out, wait); break;
    case 3: fft_pass<3, INV, BYC>(a, nc, nc_log2, ns, inv, tw, tstep, in, out, wait); break;
    default: fft_pass<2, INV, BYC>(a, nc, nc_log2, ns, inv, tw, tstep, in, out, wait); break;
  }
}

// The passes between the first and the last, all in LDS; returns Ns of the
// next one.  Ends with a barrier.
template <bool INV, bool BYC>
__device__ inline int fft_mid(const FftAxis &a, int from, int to, int nc, int nc_log2, int ns,
                              const double2 *tw, int tstep, const FftLds<BYC> &L) {
  for (int p = from; p < to; ++p) {
    fft_pass_any<INV, BYC>(a, p, nc, nc_log2, ns, tw, tstep, L, L, true);
    __syncthreads();
    ns *= a.radix[p];
  }
  return ns;
}

// ---- tables ----------------------------------------------------------------
// exp(2 pi i q / n), the angle reduced to an eighth of a turn by integer
// arithmetic first, so that its rounding does not grow with q.
__device__ inline double2 unit_root(int q, int n) {
  const int quad = (int)(4 * (int64_t)q / n);
  const int rem = (int)(4 * (int64_t)q - (int64_t)quad * n);  // angle = (quad + rem / n) pi / 2
  double s, c;
  if (2 * rem > n) {
    sincospi(0.5 * (double)(n - rem) / (double)n, &c, &s);
  } else {
    sincospi(0.5 * (double)rem / (double)n, &s, &c);
  }
  if (quad & 1) {
    const double t = c;
    c = -s;
    s = t;
  }
  return (quad & 2) ? make_double2(-c, -s) : make_double2(c, s);
}

struct FftTables {
  double2 *wu, *wv;  // [n_u], [n_v]
  double *tu, *tv;   // tapers
};

__global__ void k_fft_tables(FftTables t, int n_u, int n_v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_u) t.wu[i] = unit_root(i, n_u);
  if (i < n_v) t.wv[i] = unit_root(i, n_v);
  double g, k;
  // grdsf(|2 * coordinates(n)|) (gcf_prolate_spheroidal.py:73-77, :161-163)
  if (i < n_u) {
    ps_eval(fabs(2.0 * ((double)(i - n_u / 2) / (double)n_u)), g, k);
    t.tu[i] = g;
  }
  if (i < n_v) {
    ps_eval(fabs(2.0 * ((double)(i - n_v / 2) / (double)n_v)), g, k);
    t.tv[i] = g;
  }
}

template <typename H>
__device__ inline double2 load_pair(const H *p) {
  typedef H V __attribute__((ext_vector_type(2)));
  const V v = *(const V *)p;
  return make_double2((double)v.x, (double)v.y);
}
template <typename H>
__device__ inline void store_pair(H *p, double x, double y) {
  typedef H V __attribute__((ext_vector_type(2)));
  V v;
  v.x = (H)x;
  v.y = (H)y;
  *(V *)p = v;
}

struct FftShape {
  FftAxis u, v2;  // along u, and along half of v
  int n_u, n_v, nh;
  int nc, nc_log2;  // columns of a workgroup
  int nr;           // rows of a workgroup
  int col_blocks, row_blocks;
  int64_t plane0;
};

// Block b of the grid: a plane and a block of its columns (rows), neighbouring
// blocks of a plane on one XCD, whose L2 then sees whole lines of the columns:
// 32 together (2048 x 2048: 3% faster than 8), 8 where there are few.
__host__ __device__ inline int fft_xcd_group(int64_t grid) { return grid >= 2048 ? 32 : 8; }
static unsigned fft_grid(int64_t blocks) {
  const int64_t g = xcd_grouped_grid(blocks, 32);
  return (unsigned)(fft_xcd_group(g) == 32 ? g : xcd_grouped_grid(blocks, 8));
}
__device__ inline void fft_block(int blocks, int64_t &plane, int &blk) {
  const uint32_t b = xcd_grouped_block(blockIdx.x, fft_xcd_group(gridDim.x));
  plane = b / (uint32_t)blocks;
  blk = (int)(b - (uint32_t)plane * (uint32_t)blocks);
}

// ---- uv to image -----------------------------------------------------------
// Pass 1: columns.  Y[ku][kv] = (-1)^(ku + kv) (X[ku][kv] + conj(X[-ku][-kv])) / 2
// with X = ifftshift(grid): the Hermitian part, whose inverse transform is the
// real part of X's, moved by half a period per axis, which is fftshift for
// even sizes.  half [n_u][nh] gets its inverse FFT along u (unscaled).
template <typename R>
__global__ __launch_bounds__(kFftThreads) void k_uv_columns(FftShape S, int64_t n_planes,
                                                            const R *grid, double *half,
                                                            FftTables t) {
  extern __shared__ __align__(16) char smem[];
  int64_t plane;
  int blk;
  fft_block(S.col_blocks, plane, blk);
  if (plane >= n_planes) return;
  const int kv0 = blk * S.nc, n_u = S.n_u, n_v = S.n_v;
  const FftLds<true> L{(double2 *)smem, S.nc, 0};
  const R *g = grid + (S.plane0 + plane) * (int64_t)n_u * n_v * 2;
  double *h = half + plane * (int64_t)n_u * S.nh * 2;
  auto in = [&](int ku, int c) {
    const int kv = kv0 + c;
    if (kv >= S.nh) return make_double2(0.0, 0.0);
    int su = ku + n_u / 2;
    su -= su >= n_u ? n_u : 0;
    int sv = kv + n_v / 2;
    sv -= sv >= n_v ? n_v : 0;
    int mu = n_u / 2 - ku;
    mu += mu < 0 ? n_u : 0;
    const int mv = n_v / 2 - kv;
    const double2 a = load_pair(g + ((int64_t)su * n_v + sv) * 2);
    const double2 b = load_pair(g + ((int64_t)mu * n_v + mv) * 2);
    const double s = ((ku + kv) & 1) ? -0.5 : 0.5;
    return make_double2(s * (a.x + b.x), s * (a.y - b.y));
  };
  auto out = [&](int i, int c, double2 v) {
    if (kv0 + c < S.nh) *(double2 *)(h + ((int64_t)i * S.nh + kv0 + c) * 2) = v;
  };
  fft_pass_any<true, true>(S.u, 0, S.nc, S.nc_log2, 1, t.wu, 1, in, L, false);
  __syncthreads();
  const int ns = fft_mid<true, true>(S.u, 1, S.u.passes - 1, S.nc, S.nc_log2, S.u.radix[0], t.wu,
                                     1, L);
  fft_pass_any<true, true>(S.u, S.u.passes - 1, S.nc, S.nc_log2, ns, t.wu, 1, L, out, false);
}

// Pass 2: rows.  A real row of n_v = 2 m points from its m + 1 spectral ones
// by an inverse FFT of m complex points: with E = X[k] + conj(X[m - k]) and
// O = (X[k] - conj(X[m - k])) exp(2 pi i k / n_v), Z = E + i O transforms to
// x[2 j] + i x[2 j + 1].  Then out = x / taper / sumwt (each when given).
template <typename O>
__global__ __launch_bounds__(kFftThreads) void k_image_rows(FftShape S, int64_t n_planes,
                                                            const double *half,
                                                            const double *sumwt, int taper,
                                                            O *image, FftTables t) {
  extern __shared__ __align__(16) char smem[];
  int64_t plane;
  int blk;
  fft_block(S.row_blocks, plane, blk);
  if (plane >= n_planes) return;
  const int u0 = blk * S.nr, m = S.v2.n, nr = min(S.nr, S.n_u - u0);
  const FftLds<false> L{(double2 *)smem, S.nr, fft_pitch(m)};
  const double *h = half + (plane * S.n_u + u0) * (int64_t)S.nh * 2;
  const int pairs = m / 2 + 1;
  for (int i = threadIdx.x; i < pairs * nr; i += blockDim.x) {
    const int c = i / pairs, k = i - c * pairs;
    const double *row = h + (int64_t)c * S.nh * 2;
    const double2 x = load_pair(row + 2 * k), y = load_pair(row + 2 * (m - k));
    const double2 e = make_double2(x.x + y.x, x.y - y.y);
    const double2 d = make_double2(x.x - y.x, x.y + y.y);
    const double2 o = cmul(d, t.wv[k]);
    L(k, c, make_double2(e.x - o.y, e.y + o.x));
    // Z[m - k] = conj(E) + i conj(O)
    if (k > 0 && k < m - k) L(m - k, c, make_double2(e.x + o.y, o.x - e.y));
  }
  __syncthreads();
  const int ns = fft_mid<true, false>(S.v2, 0, S.v2.passes - 1, nr, 0, 1, t.wv, 2, L);
  O *dst = image + ((S.plane0 + plane) * S.n_u + u0) * (int64_t)S.n_v;
  const double sw = sumwt ? sumwt[S.plane0 + plane] : 1.0;
  auto out = [&](int i, int c, double2 v) {
    if (taper) {
      const double f = t.tu[u0 + c] * sw;
      v.x = v.x / (f * t.tv[2 * i]);
      v.y = v.y / (f * t.tv[2 * i + 1]);
    } else if (sumwt) {
      v.x = v.x / sw;
      v.y = v.y / sw;
    }
    store_pair(dst + (int64_t)c * S.n_v + 2 * i, v.x, v.y);
  };
  fft_pass_any<true, false>(S.v2, S.v2.passes - 1, nr, 0, ns, t.wv, 2, L, out, false);
}

// ---- image to uv -----------------------------------------------------------
// Pass 1: rows.  z[j] = x[2 j] + i x[2 j + 1] (x over the taper when asked)
// transforms to Z; with E = (Z[k] + conj(Z[m - k])) / 2 and O = (Z[k] -
// conj(Z[m - k])) / 2i exp(-2 pi i k / n_v), X[k] = E + O, X[m - k] =
// conj(E - O).
template <typename I>
__global__ __launch_bounds__(kFftThreads) void k_image_rows_fwd(FftShape S, int64_t n_planes,
                                                                const I *image, int taper,
                                                                double *half, FftTables t) {
  extern __shared__ __align__(16) char smem[];
  int64_t plane;
  int blk;
  fft_block(S.row_blocks, plane, blk);
  if (plane >= n_planes) return;
  const int u0 = blk * S.nr, m = S.v2.n, nr = min(S.nr, S.n_u - u0);
  const FftLds<false> L{(double2 *)smem, S.nr, fft_pitch(m)};
  const I *src = image + ((S.plane0 + plane) * S.n_u + u0) * (int64_t)S.n_v;
  auto in = [&](int j, int c) {
    double2 x = load_pair(src + (int64_t)c * S.n_v + 2 * j);
    if (taper) {
      const double f = t.tu[u0 + c];
      x.x = x.x / (f * t.tv[2 * j]);
      x.y = x.y / (f * t.tv[2 * j + 1]);
    }
    return x;
  };
  fft_pass_any<false, false>(S.v2, 0, nr, 0, 1, t.wv, 2, in, L, false);
  __syncthreads();
  fft_mid<false, false>(S.v2, 1, S.v2.passes, nr, 0, S.v2.radix[0], t.wv, 2, L);
  double *h = half + (plane * S.n_u + u0) * (int64_t)S.nh * 2;
  const int pairs = m / 2 + 1;
  for (int i = threadIdx.x; i < pairs * nr; i += blockDim.x) {
    const int c = i / pairs, k = i - c * pairs;
    const double2 x = L(k, c), y = L(k == 0 ? 0 : m - k, c);
    const double2 e = make_double2(0.5 * (x.x + y.x), 0.5 * (x.y - y.y));
    // (x - conj(y)) / 2i
    const double2 d = make_double2(0.5 * (x.y + y.y), -0.5 * (x.x - y.x));
    double2 w = t.wv[k];
    w.y = -w.y;
    const double2 o = cmul(d, w);
    double *row = h + (int64_t)c * S.nh * 2;
    store_pair(row + 2 * k, e.x + o.x, e.y + o.y);
    if (k < m - k) store_pair(row + 2 * (m - k), e.x - o.x, -(e.y - o.y));
  }
}

// Pass 2: columns.  The FFT along u, then grid[su][sv] = (-1)^(ku + kv)
// F[ku][kv] at the shifted index (the sign is the input's ifftshift), and the
// conjugate at -k for the other half.
template <typename R>
__global__ __launch_bounds__(kFftThreads) void k_uv_columns_fwd(FftShape S, int64_t n_planes,
                                                                const double *half, R *grid,
                                                                FftTables t) {
  extern __shared__ __align__(16) char smem[];
  int64_t plane;
  int blk;
  fft_block(S.col_blocks, plane, blk);
  if (plane >= n_planes) return;
  const int kv0 = blk * S.nc, n_u = S.n_u, n_v = S.n_v;
  const FftLds<true> L{(double2 *)smem, S.nc, 0};
  const double *h = half + plane * (int64_t)n_u * S.nh * 2;
  R *g = grid + (S.plane0 + plane) * (int64_t)n_u * n_v * 2;
  auto in = [&](int i, int c) {
    return kv0 + c < S.nh ? load_pair(h + ((int64_t)i * S.nh + kv0 + c) * 2)
                          : make_double2(0.0, 0.0);
  };
  auto out = [&](int ku, int c, double2 v) {
    const int kv = kv0 + c;
    if (kv >= S.nh) return;
    if ((ku + kv) & 1) v = make_double2(-v.x, -v.y);
    int su = ku + n_u / 2;
    su -= su >= n_u ? n_u : 0;
    int sv = kv + n_v / 2;
    sv -= sv >= n_v ? n_v : 0;
    store_pair(g + ((int64_t)su * n_v + sv) * 2, v.x, v.y);
    if (kv > 0 && kv < n_v / 2) {
      int mu = n_u / 2 - ku;
      mu += mu < 0 ? n_u : 0;
      store_pair(g + ((int64_t)mu * n_v + n_v / 2 - kv) * 2, v.x, -v.y);
    }
  };
  fft_pass_any<false, true>(S.u, 0, S.nc, S.nc_log2, 1, t.wu, 1, in, L, false);
  __syncthreads();
  const int ns = fft_mid<false, true>(S.u, 1, S.u.passes - 1, S.nc, S.nc_log2, S.u.radix[0],
                                      t.wu, 1, L);
  fft_pass_any<false, true>(S.u, S.u.passes - 1, S.nc, S.nc_log2, ns, t.wu, 1, L, out, false);
}

// ---- host ------------------------------------------------------------------
struct FftCall {
  FftShape S;
  FftTables t;
  void *half;
  int64_t group;  // planes of a group
  int col_threads, row_threads, col_lds, row_lds;
  size_t bytes;
};

// Shapes and the work layout; false for sizes torch.fft serves.
static bool fft_layout(int64_t n_planes, int n_u, int n_v, char *work, FftCall &c) {
  FftShape &S = c.S;
  if (n_u < 2 || n_v < 4 || (n_u & 1) || (n_v & 1) || n_u > kFftWgPoints / 2 ||
      n_v / 2 > kFftWgPoints || !fft_axis(n_u, S.u) || !fft_axis(n_v / 2, S.v2))
    return false;
  S.n_u = n_u;
  S.n_v = n_v;
  S.nh = n_v / 2 + 1;
  S.nc_log2 = 3;
  // columns of a workgroup: as many as 8192 points hold for long axes, whose
  // grid lines are then read in pieces of 16 bytes times the columns, and
  // half of that where two workgroups fit a CU (1024 x 1024: 36 -> 33 us)
  while (S.nc_log2 > 0 && (n_u << S.nc_log2) > (n_u > 1024 ? kFftWgPoints : kFftWgPoints / 2))
    --S.nc_log2;
  S.nc = 1 << S.nc_log2;
  S.nr = std::max(1, std::min(n_u, kFftRowPoints / (n_v / 2)));
  S.col_blocks = (S.nh + S.nc - 1) / S.nc;
  S.row_blocks = (n_u + S.nr - 1) / S.nr;
  auto threads = [](int points) {
    return std::min(kFftThreads, std::max(64, (points + kFftPoints * 64 - 1) / (kFftPoints * 64) * 64));
  };
  c.col_threads = threads(n_u * S.nc);
  c.row_threads = threads(n_v / 2 * S.nr);
  c.col_lds = fft_pitch(n_u) * S.nc * (int)sizeof(double2);
  c.row_lds = fft_pitch(n_v / 2) * S.nr * (int)sizeof(double2);
  const int64_t plane_bytes = (int64_t)n_u * S.nh * sizeof(double2);
  c.group = std::max<int64_t>(1, std::min<int64_t>(n_planes, kFftGroupBytes / plane_bytes));
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = off;
    off += (bytes + 255) & ~(size_t)255;
    return work ? work + o : nullptr;
  };
  c.t.wu = (double2 *)take(sizeof(double2) * n_u);
  c.t.wv = (double2 *)take(sizeof(double2) * n_v);
  c.t.tu = (double *)take(sizeof(double) * n_u);
  c.t.tv = (double *)take(sizeof(double) * n_v);
  c.half = take((size_t)(plane_bytes * c.group));
  c.bytes = off;
  return true;
}

static int fft_tables(const FftCall &c, hipStream_t s) {
  const int n = std::max(c.S.n_u, c.S.n_v);
  hipLaunchKernelGGL(k_fft_tables, dim3((n + 255) / 256), dim3(256), 0, s, c.t, c.S.n_u, c.S.n_v);
  AV_LAUNCH_CHECK("k_fft_tables");
  return AV_OK;
}

template <typename R, typename O>
static int uv_to_image(FftCall &c, const R *grid, int64_t n_planes, const double *sumwt,
                       int taper, O *image, hipStream_t s) {
  int rc;
  if ((rc = ensure_lds_limit<k_uv_columns<R>>(c.col_lds, "av_uv_to_image: hipFuncSetAttribute")) ||
      (rc = ensure_lds_limit<k_image_rows<O>>(c.row_lds, "av_uv_to_image: hipFuncSetAttribute")) ||
      (rc = fft_tables(c, s)))
    return rc;
  for (int64_t p = 0; p < n_planes; p += c.group) {
    const int64_t n = std::min(c.group, n_planes - p);
    c.S.plane0 = p;
    hipLaunchKernelGGL(k_uv_columns<R>, dim3(fft_grid(n * c.S.col_blocks)),
                       dim3(c.col_threads), c.col_lds, s, c.S, n, grid, (double *)c.half, c.t);
    AV_LAUNCH_CHECK("k_uv_columns");
    hipLaunchKernelGGL(k_image_rows<O>, dim3(fft_grid(n * c.S.row_blocks)),
                       dim3(c.row_threads), c.row_lds, s, c.S, n, (const double *)c.half, sumwt,
                       taper, image, c.t);
    AV_LAUNCH_CHECK("k_image_rows");
  }
  return AV_OK;
}

template <typename I, typename R>
static int image_to_uv(FftCall &c, const I *image, int64_t n_planes, int taper, R *grid,
                       hipStream_t s) {
  int rc;
  if ((rc = ensure_lds_limit<k_image_rows_fwd<I>>(c.row_lds,
                                                     "av_image_to_uv: hipFuncSetAttribute")) ||
      (rc = ensure_lds_limit<k_uv_columns_fwd<R>>(c.col_lds,
                                                     "av_image_to_uv: hipFuncSetAttribute")) ||
      (rc = fft_tables(c, s)))
    return rc;
  for (int64_t p = 0; p < n_planes; p += c.group) {
    const int64_t n = std::min(c.group, n_planes - p);
    c.S.plane0 = p;
    hipLaunchKernelGGL((k_image_rows_fwd<I>),
                       dim3(fft_grid(n * c.S.row_blocks)),
                       dim3(c.row_threads), c.row_lds, s, c.S, n, image, taper, (double *)c.half, c.t);
    AV_LAUNCH_CHECK("k_image_rows_fwd");
    hipLaunchKernelGGL((k_uv_columns_fwd<R>),
                       dim3(fft_grid(n * c.S.col_blocks)),
                       dim3(c.col_threads), c.col_lds, s, c.S, n, (const double *)c.half, grid, c.t);
    AV_LAUNCH_CHECK("k_uv_columns_fwd");
  }
  return AV_OK;
}

}  // namespace av

using namespace av;

extern "C" {

int av_fft_work_bytes(int64_t n_planes, int32_t n_u, int32_t n_v, int64_t *bytes) {
  if (!bytes || n_planes < 0)
    return fail(AV_ERR_INVALID, "av_fft_work_bytes: bad arguments");
  FftCall c{};
  *bytes = fft_layout(std::max<int64_t>(n_planes, 1), n_u, n_v, nullptr, c) ? (int64_t)c.bytes : 0;
  return AV_OK;
}

int av_uv_to_image(const void *grid, int32_t dtype, int64_t n_planes, int32_t n_u, int32_t n_v,
                   const double *sumwt, int32_t taper, void *image, int32_t image_dtype,
                   void *work, void *stream) {
  if (!grid || !image || !work || n_planes < 0)
    return fail(AV_ERR_INVALID, "av_uv_to_image: bad arguments");
  if (((uintptr_t)grid | (uintptr_t)image | (uintptr_t)work) & 15)
    return fail(AV_ERR_INVALID, "av_uv_to_image: arrays must be 16-byte aligned");
  FftCall c{};
  if (!fft_layout(std::max<int64_t>(n_planes, 1), n_u, n_v, (char *)work, c))
    return fail(AV_ERR_UNSUPPORTED, "av_uv_to_image: sizes must be even, at most 4096 x 16384, "
                                    "with no prime factor beyond 5");
  hipStream_t s = (hipStream_t)stream;
  const bool f = dtype == AV_F32, of = image_dtype == AV_F32;
  if ((!f && dtype != AV_F64) || (!of && image_dtype != AV_F64))
    return fail(AV_ERR_INVALID, "av_uv_to_image: dtype must be AV_F32 or AV_F64");
  if (f && of)
    return uv_to_image(c, (const float *)grid, n_planes, sumwt, taper, (float *)image, s);
  if (f) return uv_to_image(c, (const float *)grid, n_planes, sumwt, taper, (double *)image, s);
  if (of) return uv_to_image(c, (const double *)grid, n_planes, sumwt, taper, (float *)image, s);
  return uv_to_image(c, (const double *)grid, n_planes, sumwt, taper, (double *)image, s);
}

int av_image_to_uv(const void *image, int32_t image_dtype, int64_t n_planes, int32_t n_u,
                   int32_t n_v, int32_t taper, void *grid, int32_t dtype, void *work,
                   void *stream) {
  if (!grid || !image || !work || n_planes < 0)
    return fail(AV_ERR_INVALID, "av_image_to_uv: bad arguments");
  if (((uintptr_t)grid | (uintptr_t)image | (uintptr_t)work) & 15)
    return fail(AV_ERR_INVALID, "av_image_to_uv: arrays must be 16-byte aligned");
  const bool f = dtype == AV_F32, inf = image_dtype == AV_F32;
  if ((!f && dtype != AV_F64) || (!inf && image_dtype != AV_F64))
    return fail(AV_ERR_INVALID, "av_image_to_uv: dtype must be AV_F32 or AV_F64");
  FftCall c{};
  if (!fft_layout(std::max<int64_t>(n_planes, 1), n_u, n_v, (char *)work, c))
    return fail(AV_ERR_UNSUPPORTED, "av_image_to_uv: sizes must be even, at most 4096 x 16384, "
                                    "with no prime factor beyond 5");
  hipStream_t s = (hipStream_t)stream;
  if (inf && f) return image_to_uv(c, (const float *)image, n_planes, taper, (float *)grid, s);
  if (inf) return image_to_uv(c, (const float *)image, n_planes, taper, (double *)grid, s);
  if (f) return image_to_uv(c, (const double *)image, n_planes, taper, (float *)grid, s);
  return image_to_uv(c, (const double *)image, n_planes, taper, (double *)grid, s);
}

}  // extern "C"

// common.hip -- error reporting, device info, fills and the
// prolate-spheroidal table kernels of libavgrid.so.
#include <cstdio>
#include <mutex>

#include "ps_eval.h"

namespace av {

static thread_local std::string g_last_error;

void set_error(const std::string &msg) { g_last_error = msg; }

int fail(int code, const std::string &msg) {
  set_error(msg);
  return code;
}

int hip_fail(hipError_t e, const char *what) {
  set_error(std::string(what) + ": " + hipGetErrorString(e));
  return e == hipErrorOutOfMemory ? AV_ERR_NOMEM : AV_ERR_HIP;
}

const DeviceProps &device_props() {
  static std::mutex mu;
  static DeviceProps cache[64];
  static bool have[64] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  static DeviceProps bad;
  if (e != hipSuccess || dev < 0 || dev >= 64) {
    bad.error = e != hipSuccess ? e : hipErrorInvalidDevice;
    return bad;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (!have[dev]) {
    hipDeviceProp_t prop;
    DeviceProps p;
    p.error = hipGetDeviceProperties(&prop, dev);
    p.num_cus = prop.multiProcessorCount;
    p.lds_per_block = prop.sharedMemPerBlock;
    p.lds_per_cu = prop.maxSharedMemoryPerMultiProcessor;
    cache[dev] = p;
    have[dev] = p.error == hipSuccess;
    if (!have[dev]) return cache[dev];
  }
  return cache[dev];
}

// ------------------------------------------------------------- fill ----
__global__ void k_fill_u32(uint32_t *p, uint32_t v, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = v;
}

int launch_fill_u32(uint32_t *p, uint32_t v, int64_t n, hipStream_t s) {
  if (n <= 0) return AV_OK;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, p, v, n);
  AV_LAUNCH_CHECK("k_fill_u32");
  return AV_OK;
}

// -------------------------------------------------- prolate spheroid ----
__global__ void k_ps_function(const double *u, int64_t n, double *grdsf, double *kern) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double g, k;
  ps_eval(u[i], g, k);
  if (grdsf) grdsf[i] = g;
  if (kern) kern[i] = k;
}

// create_prolate_spheroidal_kernel_1D (gcf_prolate_spheroidal.py:87-99)
__global__ void k_ps_kernel_1d(int ov, int support, double *out) {
  int sc = support / 2;
  int n = ov * sc, ntot = ov * (sc + 1);
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ntot) return;
  double v = 0.0;
  if (i < n) {
    double g;
    ps_eval((double)i / (double)(sc * ov), g, v);
  }
  out[i] = v;
}

// grdsf(|2 * coordinates(n)|) (gcf_prolate_spheroidal.py:73-77, :161-163)
__global__ void k_ps_correction_1d(int n, double *out) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double c = (double)(i - n / 2) / (double)n;
  double g, k;
  ps_eval(fabs(2.0 * c), g, k);
  out[i] = g;
}

// kernel_image of create_prolate_spheroidal_kernel (gcf_prolate_spheroidal.py:72-79)
__global__ void k_ps_taper(int nu, int nv, double *out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)nu * nv) return;
  int a = (int)(i / nv), b = (int)(i - (int64_t)a * nv);
  double gu, gv, k;
  ps_eval(fabs(2.0 * ((double)(a - nu / 2) / (double)nu)), gu, k);
  ps_eval(fabs(2.0 * ((double)(b - nv / 2) / (double)nv)), gv, k);
  out[i] = gu * gv;
}

// gcf_prolate_spheroidal.py:65-67: np.outer of two kernel rows
__global__ void k_ps_outer(const double *k1, int nrow, int nfill, int support, double *k4) {
  int64_t total = (int64_t)nrow * nrow * support * support;
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  int j = (int)(i % support);
  int64_t r = i / support;
  int ii = (int)(r % support);
  r /= support;
  int y = (int)(r % nrow);
  int x = (int)(r / nrow);
  double v = 0.0;
  if (x < nfill && y < nfill) v = k1[(int64_t)x * support + ii] * k1[(int64_t)y * support + j];
  k4[i] = v;
}

}  // namespace av

using namespace av;

extern "C" {

const char *av_last_error(void) { return g_last_error.c_str(); }

int av_version(void) { return AV_ABI_VERSION; }

int av_device_info(int32_t *num_cus, int32_t *lds_bytes_per_cu, int32_t *xcds) {
  int dev = 0;
  AV_HIP(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  AV_HIP(hipGetDeviceProperties(&prop, dev));
  if (num_cus) *num_cus = prop.multiProcessorCount;
  if (lds_bytes_per_cu) *lds_bytes_per_cu = (int32_t)prop.maxSharedMemoryPerMultiProcessor;
  if (xcds) *xcds = 8;
  return AV_OK;
}

int av_ps_function(const double *u, int64_t n, double *grdsf, double *kern, void *stream) {
  if (n < 0 || (n > 0 && !u)) return fail(AV_ERR_INVALID, "av_ps_function: bad arguments");
  if (n == 0) return AV_OK;
  hipLaunchKernelGGL(k_ps_function, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, u, n, grdsf, kern);
  AV_LAUNCH_CHECK("k_ps_function");
  return AV_OK;
}

int av_ps_kernel_1d(int32_t oversampling, int32_t support, double *out, void *stream) {
  if (oversampling < 1 || support < 2 || !out)
    return fail(AV_ERR_INVALID, "av_ps_kernel_1d: need oversampling >= 1, support >= 2");
  int ntot = oversampling * (support / 2 + 1);
  hipLaunchKernelGGL(k_ps_kernel_1d, dim3((ntot + 255) / 256), dim3(256), 0,
                     (hipStream_t)stream, oversampling, support, out);
  AV_LAUNCH_CHECK("k_ps_kernel_1d");
  return AV_OK;
}

int av_ps_correction_1d(int32_t n, double *out, void *stream) {
  if (n < 1 || !out) return fail(AV_ERR_INVALID, "av_ps_correction_1d: bad arguments");
  hipLaunchKernelGGL(k_ps_correction_1d, dim3((n + 255) / 256), dim3(256), 0,
                     (hipStream_t)stream, n, out);
  AV_LAUNCH_CHECK("k_ps_correction_1d");
  return AV_OK;
}

int av_ps_taper(int32_t n_u, int32_t n_v, double *out, void *stream) {
  if (n_u < 1 || n_v < 1 || !out) return fail(AV_ERR_INVALID, "av_ps_taper: bad arguments");
  int64_t n = (int64_t)n_u * n_v;
  hipLaunchKernelGGL(k_ps_taper, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, n_u, n_v, out);
  AV_LAUNCH_CHECK("k_ps_taper");
  return AV_OK;
}

int av_ps_outer(const double *k1, int32_t nrow, int32_t nfill, int32_t support, double *k4,
                void *stream) {
  if (nrow < 1 || support < 1 || nfill < 0 || nfill > nrow || !k1 || !k4)
    return fail(AV_ERR_INVALID, "av_ps_outer: bad arguments");
  int64_t total = (int64_t)nrow * nrow * support * support;
  hipLaunchKernelGGL(k_ps_outer, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, k1, nrow, nfill, support, k4);
  AV_LAUNCH_CHECK("k_ps_outer");
  return AV_OK;
}

}  // extern "C"

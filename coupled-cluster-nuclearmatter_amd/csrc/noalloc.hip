// Correlation energy on caller-owned device buffers without any allocation:
// the variant of ccgpu_energy (ccd_energy_save, ccm_energy.f90:4-71) for
// callers that cannot allocate device memory (code under hipGraph capture,
// serving loops).  Its block partials live in a file-scope device array,
// `scratch`, whose address is taken once per device with
// hipGetSymbolAddress; kernels receive that address as an argument.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <string>

#include "../../include/ccgpu.h"

namespace {

// Block partials of one call: at most kMaxParts complex partial sums, each
// over a span of span_of(n) amplitudes, 2048 to 65536 (so at most kMaxParts *
// kSpan amplitudes per call).  Every call on a GPU shares that GPU's array:
// calls that overlap on one GPU race.  Every partial a call reads was written
// by the same call, so nothing has to be cleared.
constexpr int kMaxParts = 4096;
constexpr int64_t kSpan = 65536;       // largest span
constexpr int64_t kMinSpan = 2048;     // eight amplitudes per thread
__device__ __align__(256) double2 scratch[kMaxParts];

// The sum is HBM-bound (32 bytes per amplitude) and needs every CU: on the
// 1 991 568 amplitudes of PNM A=66 |n_i|<=4, spans of 2048 give 973 blocks and
// 13.3 us per call (4.8 TB/s), spans of 65536 31 blocks and 73 us (0.87 TB/s).
// Below one block per CU the two launches decide.  Above kMaxParts * 2048
// amplitudes the spans grow in whole steps of 2048 to keep to the scratch array.
int64_t span_of(int64_t n) {
  const int64_t s = (n + kMaxParts - 1) / kMaxParts;
  return s <= kMinSpan ? kMinSpan : (s + kMinSpan - 1) / kMinSpan * kMinSpan;
}

constexpr int kMaxDevices = 64;
std::mutex g_mu;
double2 *g_scratch[kMaxDevices] = {};   // device address of `scratch` per device

// Sum of one complex value per thread over a block of NW waves: a butterfly in
// each wave, then the waves in order (fixed, so repeated calls give the same
// bits).  The result is valid in thread 0.
template <int NW>
__device__ __forceinline__ double2 sum_block(double re, double im) {
  __shared__ double sr[NW], si[NW];
  for (int off = 32; off > 0; off >>= 1) {
    re += __shfl_xor(re, off);
    im += __shfl_xor(im, off);
  }
  if ((threadIdx.x & 63) == 0) {
    sr[threadIdx.x >> 6] = re;
    si[threadIdx.x >> 6] = im;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    for (int w = 1; w < NW; ++w) {
      re += sr[w];
      im += si[w];
    }
  return make_double2(re, im);
}

// Partial sum of t * conj(r0) over one span per block; the loads of eight
// amplitudes per thread are in flight together.
__global__ __launch_bounds__(256) void k_energy_spans(const double2 *__restrict__ t, const double2 *__restrict__ r0,
                                                      int64_t n, int64_t span, double2 *__restrict__ part) {
  const int64_t b = (int64_t)blockIdx.x * span;
  const int64_t e = b + span < n ? b + span : n;
  double re = 0.0, im = 0.0;
  int64_t u = b + threadIdx.x;
  for (; u + 7 * 256 < e; u += 8 * 256) {
    double2 x[8], y[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      x[q] = t[u + q * 256];
      y[q] = r0[u + q * 256];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      re += x[q].x * y[q].x + x[q].y * y[q].y;
      im += x[q].y * y[q].x - x[q].x * y[q].y;
    }
  }
  for (; u < e; u += 256) {
    const double2 x = t[u], y = r0[u];
    re += x.x * y.x + x.y * y.y;
    im += x.y * y.x - x.x * y.y;
  }
  const double2 s = sum_block<4>(re, im);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// Fixed-order sum of the partials into the caller's output: four loads per
// thread cover the largest count.
__global__ __launch_bounds__(1024) void k_energy_final(const double2 *__restrict__ part, int nparts,
                                                       double2 *__restrict__ out) {
  double2 v[kMaxParts / 1024];
#pragma unroll
  for (int q = 0; q < kMaxParts / 1024; ++q) {
    const int p = q * 1024 + threadIdx.x;
    v[q] = p < nparts ? part[p] : make_double2(0.0, 0.0);
  }
  double re = 0.0, im = 0.0;
#pragma unroll
  for (int q = 0; q < kMaxParts / 1024; ++q) {
    re += v[q].x;
    im += v[q].y;
  }
  const double2 s = sum_block<16>(re, im);
  if (threadIdx.x == 0) *out = s;
}

// Device address of this GPU's `scratch`, taken once per device with that
// device current (the array's name is only a host-side stand-in).
double2 *scratch_of_current_device() {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) throw std::string("hipGetDevice failed: ") + hipGetErrorString(e);
  if (dev < 0 || dev >= kMaxDevices) throw std::string("device index out of range");
  std::lock_guard<std::mutex> lk(g_mu);
  if (!g_scratch[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) throw std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e);
    g_scratch[dev] = (double2 *)p;
  }
  return g_scratch[dev];
}

}  // namespace

namespace ccgpu {
void set_last_error(const std::string &msg);   // ccgpu_last_error's message (api.cpp)
}

extern "C" {

int ccgpu_energy_noalloc(long long n, const double *t, const double *r0, double *ecorr, void *stream) {
  try {
    if (n < 0) throw std::string("negative amplitude count");
    if (n > (long long)kMaxParts * kSpan)
      throw std::string("amplitude count ") + std::to_string(n) + " above the maximum " +
          std::to_string((long long)kMaxParts * kSpan) + " of ccgpu_energy_noalloc";
    if (!ecorr || (n > 0 && (!t || !r0))) throw std::string("null device pointer");
    double2 *part = scratch_of_current_device();
    const hipStream_t st = (hipStream_t)stream;
    const int64_t span = span_of(n);
    const int nparts = (int)((n + span - 1) / span);
    if (nparts > 0)
      hipLaunchKernelGGL(k_energy_spans, dim3(nparts), dim3(256), 0, st, (const double2 *)t, (const double2 *)r0,
                         (int64_t)n, span, part);
    hipLaunchKernelGGL(k_energy_final, dim3(1), dim3(1024), 0, st, part, nparts, (double2 *)ecorr);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw std::string("kernel launch failed: ") + hipGetErrorString(e);
    return 0;
  } catch (const std::string &m) {
    ccgpu::set_last_error(m);
    return 1;
  }
}

}  // extern "C"

// axh_post.hip -- seismogram post-processing on the GPU.
//
// The reference's post-processing program (SOLVER/UTILS/post_processing.F90)
// sums the moment-tensor runs with their radiation factors, convolves each
// trace with a source time function and rotates the components.  The
// convolution is the costly part: for every trace, every one of nt samples
// sums nj = 2 shift_fact1 t0 / dt terms (convolve_with_stf,
// SOLVER/UTILS/post_processing.F90:1014-1084), tens of millions of terms per
// trace at 5 s and 1800 s.  Here one GPU thread owns four output samples of one
// trace and runs their terms in the reference's order and precision, so the
// result is the reference's bit for bit; a workgroup's consecutive samples read
// a sliding window of the trace in LDS.
#include <hip/hip_runtime.h>

#include <string>

#include "axh_internal.h"

#pragma clang fp contract(off)

namespace axh {

#define HIPCHECK_POST(x)                                                     \
  do {                                                                       \
    hipError_t e_ = (x);                                                     \
    if (e_ != hipSuccess)                                                    \
      fail(AXH_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_));     \
  } while (0)

// Sample i of a trace:
// seis_fil(i) = seis_fil(i) + seis(i-j) * stf(j) * dt over j = 1..nj with
// j < i, the product of two REAL(4) values scaled by a REAL(8) dt and added
// in REAL(8) to the REAL(4) partial sum, then seis_fil * scale in REAL(8).
// The terms of one sample run in ascending j, as in the reference loop.
//
// Bound by the REAL(8) instructions of a term (three conversions, a product and
// a sum, each dependent on the last).  A lane owns kSamples consecutive samples:
// that many chains run side by side, and kSamples terms of each read one 16-byte
// piece of the trace and one of the source time function from LDS instead of two
// words a term.  543 traces of 5001 samples, 401 terms: 296 -> 194 us (43 -> 28
// cycles per wavefront and term).
constexpr int kSamples = 4;
constexpr int kConvTile = 256 * kSamples;   // samples of a workgroup
constexpr int kConvTerms = 512;             // terms staged at a time

__global__ __launch_bounds__(256) void k_convolve(int nt, int nj, const float *__restrict__ seis,
                                                  const float *__restrict__ stf, double dt,
                                                  double scale, float *__restrict__ out) {
  static_assert(kSamples == 4, "the pieces are float4");
  // terms j1 + 1 .. j1 + kConvTerms, and the samples (from 0) they meet:
  // n0 - j1 - kConvTerms .. n0 - j1 + kConvTile - 1, zeros outside the trace
  __shared__ __align__(16) float s_stf[kConvTerms];
  __shared__ __align__(16) float s_tr[kConvTerms + kConvTile];
  const int t = threadIdx.x, n0 = blockIdx.x * kConvTile;
  const float *tr = seis + (size_t)blockIdx.y * nt;
  const int n = n0 + kSamples * t;            // the lane's first sample
  float acc[kSamples] = {0.0f, 0.0f, 0.0f, 0.0f};
  auto term = [&](float &a, float x, float f) {
    const float p = x * f;
    a = (float)((double)a + (double)p * dt);
  };
  for (int j1 = 0; j1 < nj; j1 += kConvTerms) {
    const int nk = min(nj - j1, kConvTerms);
    if (j1 > 0) __syncthreads();
    for (int j = t; j < kConvTerms; j += 256) s_stf[j] = j < nk ? stf[j1 + j] : 0.0f;
    for (int x = t; x < kConvTerms + kConvTile; x += 256) {
      const int m = n0 - j1 - kConvTerms + x;
      s_tr[x] = m >= 0 && m < nt ? tr[m] : 0.0f;
    }
    __syncthreads();
    if (n >= nt) continue;
    const float *w = s_tr + kConvTerms + kSamples * t;   // sample n - j1
    // whole pieces of terms that every sample of the lane has (sample n + r
    // has the terms j <= n + r), the others one by one
    const int full = max(min(nk, n - j1), 0) / kSamples * kSamples;
    int j0 = 0;
    float4 hi = *reinterpret_cast<const float4 *>(w);
    for (; j0 < full; j0 += kSamples) {
      const float4 lo = *reinterpret_cast<const float4 *>(w - j0 - kSamples);
      const float4 f = *reinterpret_cast<const float4 *>(s_stf + j0);
      const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      const float g[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
      for (int q = 0; q < kSamples; q++)
#pragma unroll
        for (int r = 0; r < kSamples; r++) term(acc[r], v[3 + r - q], g[q]);
      hi = lo;
    }
    const int last = min(nk, n - j1 + kSamples - 1);
    for (; j0 < last; j0++)
#pragma unroll
      for (int r = 0; r < kSamples; r++)
        if (n + r > j1 + j0) term(acc[r], w[r - j0 - 1], s_stf[j0]);
  }
  float *o = out + (size_t)blockIdx.y * nt;
#pragma unroll
  for (int r = 0; r < kSamples; r++)
    if (n + r < nt) o[n + r] = (float)((double)acc[r] * scale);
}

void convolve_traces(int nt, int ntraces, const float *seis, int nj, const float *stf,
                     double dt, double scale, float *out) {
  if (nt <= 0 || ntraces <= 0) return;
  const size_t n = (size_t)nt * ntraces;
  float *d_seis = nullptr, *d_out = nullptr, *d_stf = nullptr;
  hipStream_t s = nullptr;
  auto release = [&] {
    if (s) (void)hipStreamSynchronize(s);
    if (d_seis) (void)hipFree(d_seis);
    if (d_out) (void)hipFree(d_out);
    if (d_stf) (void)hipFree(d_stf);
    if (s) (void)hipStreamDestroy(s);
  };
  try {
    HIPCHECK_POST(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    HIPCHECK_POST(hipMalloc(&d_seis, n * sizeof(float)));
    HIPCHECK_POST(hipMalloc(&d_out, n * sizeof(float)));
    HIPCHECK_POST(hipMalloc(&d_stf, (size_t)std::max(nj, 1) * sizeof(float)));
    HIPCHECK_POST(hipMemcpyAsync(d_seis, seis, n * sizeof(float), hipMemcpyHostToDevice, s));
    if (nj > 0)
      HIPCHECK_POST(hipMemcpyAsync(d_stf, stf, (size_t)nj * sizeof(float),
                                   hipMemcpyHostToDevice, s));
    const dim3 grid((nt + kConvTile - 1) / kConvTile, ntraces);
    hipLaunchKernelGGL(k_convolve, grid, dim3(256), 0, s, nt, nj, d_seis, d_stf, dt, scale, d_out);
    HIPCHECK_POST(hipGetLastError());
    HIPCHECK_POST(hipMemcpyAsync(out, d_out, n * sizeof(float), hipMemcpyDeviceToHost, s));
    HIPCHECK_POST(hipStreamSynchronize(s));
  } catch (...) {
    release();
    throw;
  }
  release();
}

}  // namespace axh

// gpu_quotient.hip -- the FP64 step's quotients and square roots
// (Stepper<double, ...>::DIV, DIVR, sqrt of cable_amd/csrc/cbm_step.h) on
// the device, on host operands, for tests/test_gpu_quotient.py to compare with
// IEEE's.  Built with the flags of the FP64 kernels into tests/libgpu_quotient.so.
#include "../cable_amd/csrc/cbm_kernel.h"

using namespace cbm;
using Step = Stepper<double, false, true>;

namespace {
// divisors known to the compiler, as the step has them
constexpr double LITERALS[] = {3.0, 10.0, 0.4, 1.57, 0.85, 237.3, 365.0, 921.0, 1004.64, 1440.0, 2.5014e6, 31536000.0};
constexpr int NLIT = sizeof LITERALS / sizeof *LITERALS;

template <int Q>
__device__ void literal(double n, double *out, long count) {
  *out = Step::DIV(n, LITERALS[Q]);
  if constexpr (Q + 1 < NLIT) literal<Q + 1>(n, out + count, count);
}

// out: [3 + NLIT][count] -- n / d, the same with a shared reciprocal, the root
// of n, and n over each literal
__global__ void __launch_bounds__(256) quotients(const double *n, const double *d, double *out, long count) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  out[i] = Step::DIV(n[i], d[i]);
  out[count + i] = Step::DIVR(n[i], d[i], Step::recip(d[i]));
  out[2 * count + i] = Step::sqrt(n[i]);
  literal<0>(n[i], out + 3 * count + i, count);
}
}  // namespace

extern "C" {
int gpu_quotient_literals(double *lit) {
  for (int q = 0; q < NLIT; q++) lit[q] = LITERALS[q];
  return NLIT;
}

// 0, or the HIP error
int gpu_quotients(const double *n, const double *d, double *out, long count) {
  if (count < 1) return 0;
  const size_t b = sizeof(double) * (size_t)count;
  double *buf = nullptr;
  hipError_t e = hipMalloc((void **)&buf, (5 + NLIT) * b);
  if (e != hipSuccess) return (int)e;
  double *dn = buf, *dd = buf + count, *dout = buf + 2 * count;
  e = hipMemcpy(dn, n, b, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dd, d, b, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(quotients, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, 0, dn, dd, dout, count);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpy(out, dout, (3 + NLIT) * b, hipMemcpyDeviceToHost);
  (void)hipFree(buf);
  return (int)e;
}
}

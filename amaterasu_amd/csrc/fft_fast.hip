// Dispatch of the compile-time-length kernels over the parts of the length list.
#include "fft_fast.hpp"

namespace amt {

bool fast_length_supported(int n) {
  switch (n) {
#define AMT_CASE(N) case N:
    AMT_LENGTHS_A(AMT_CASE) AMT_LENGTHS_B(AMT_CASE) AMT_LENGTHS_C(AMT_CASE) AMT_LENGTHS_D(AMT_CASE)
#undef AMT_CASE
    return true;
    default:
      return false;
  }
}

bool lane_plane_supported(int n, int prec) { return fast_length_supported(n) && lane_count(n, prec == kFP64) > 0; }
int lane_plane_half_width(int n) { return lane_half_width(n); }

// The first part that knows the length answers (-1: not its length).
#define AMT_FIRST_PART(fn, ...)                    \
  int rc = fn##_a(__VA_ARGS__);                    \
  if (rc < 0) rc = fn##_b(__VA_ARGS__);            \
  if (rc < 0) rc = fn##_c(__VA_ARGS__);            \
  if (rc < 0) rc = fn##_d(__VA_ARGS__);            \
  return rc

static int stick(const Plan& p, int prec, int pass, const void* psi, void* hpsi, void* sticks, int nb, int k0,
                 int nkb, hipStream_t s) {
  AMT_FIRST_PART(fast_stick, p, prec, pass, psi, hpsi, sticks, nb, k0, nkb, s);
}
static int plane(const Plan& p, int prec, void* sticks, const void* veff, int nb, int k0, int nkb, hipStream_t s) {
  AMT_FIRST_PART(fast_plane, p, prec, sticks, veff, nb, k0, nkb, s);
}
static int density(const Plan& p, int prec, const void* sticks, int nb, int k0, const int* list, const double* weight,
                   int nlist, int chunk, double* part, hipStream_t s) {
  AMT_FIRST_PART(fast_density, p, prec, sticks, nb, k0, list, weight, nlist, chunk, part, s);
}

// dst[(i m2 + r) m3 + c] = src at plan axes (i, r, c): V_eff in the plan's permuted axes, once per
// call (the kernels then read it along its rows).
template <typename R>
__global__ void k_permute_field(const R* __restrict__ src, R* __restrict__ dst, int m2, int m3, long long n,
                                long long s1, long long s2, long long s3) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const long long i = e / ((long long)m2 * m3), r = e / m3 % m2, c = e % m3;
  dst[e] = src[i * s1 + r * s2 + c * s3];
}

int launch_hpsi_fast(const Plan& p, int prec, const void* psi, void* hpsi, int nb, int k0, int nkk,
                     const void* veff, void* ws, hipStream_t s, int stage, bool pad) {
  const int nkb = nb * nkk;
  void* sticks = static_cast<unsigned char*>(ws) + p.field_bytes(prec);
  if (stage == 0 || stage == 1)
    if (stick(p, prec, kStickInverse, psi, nullptr, sticks, nb, k0, nkb, s)) return 1;
  if (stage == 0 || stage == 2) {
    const void* v = veff;
    if (p.permuted) {
      const long long n = (long long)p.n1 * p.n2 * p.n3;
      const dim3 grid((unsigned)((n + 255) / 256));
      if (prec == kFP64)
        hipLaunchKernelGGL(k_permute_field<double>, grid, dim3(256), 0, s, (const double*)veff, (double*)ws, p.dim(1),
                           p.dim(2), n, p.stride(0), p.stride(1), p.stride(2));
      else
        hipLaunchKernelGGL(k_permute_field<float>, grid, dim3(256), 0, s, (const float*)veff, (float*)ws, p.dim(1),
                           p.dim(2), n, p.stride(0), p.stride(1), p.stride(2));
      if (hipGetLastError() != hipSuccess) return 1;
      v = ws;
    }
    if (plane(p, prec, sticks, v, nb, k0, nkb, s)) return 1;
  }
  if (stage == 0 || stage == 3)
    if (stick(p, prec, pad ? kStickForwardPad : kStickForward, psi, hpsi, sticks, nb, k0, nkb, s)) return 1;
  return 0;
}

int launch_density_fast(const Plan& p, int prec, const void* psi, int nb, int k0, int nkk, const int* list,
                        const double* weight, int nlist, int chunk, void* sticks, double* part, hipStream_t s) {
  if (stick(p, prec, kStickInverse, psi, nullptr, sticks, nb, k0, nb * nkk, s)) return 1;
  return density(p, prec, sticks, nb, k0, list, weight, nlist, chunk, part, s) ? 1 : 0;
}

}  // namespace amt

// Pointwise PBE-form exchange-correlation in FP64: energy per particle, potentials and gradient
// derivatives of one grid in one pass (xc/gga.py, on the PW92 form of xc/lda.py:120-200).
//
// What bounds it: about 40 roots, powers and logarithms a point (FP64 vector work), against 11
// numbers read and written. As some 190 elementwise operations the same formulas were bound by the
// host issuing them (2 ms an evaluation) and by two passes over memory each: with this kernel
// six SCF steps of 8 atoms (12 evaluations) take 119 ms for 136, two of 64 atoms 426 for 434.
#include "kernels.hpp"

namespace amt {
namespace {

constexpr double kXFactor = 0.9305257363491000250020102180716672510262;
constexpr double kRsFactor = 0.6203504908994000166680068120477781673508;
constexpr double kThreshold = 1e-24;
constexpr double kX2s = 0.1282782438530421943003109254455883701296;
constexpr double kFzDen = 0.51984209978974632953442121455650;  // 2^(4/3) - 2
constexpr double kThird = 1.0 / 3.0;

// max(x, lo) that keeps NaN
__device__ __forceinline__ double at_least(double x, double lo) { return x < lo ? lo : x; }

struct Pw92 {
  double g, dg;
};
__device__ __forceinline__ Pw92 pw92_g(double rs, double srs, double a, double al, double b1, double b2, double b3,
                                       double b4) {
  const double q = b1 * srs + b2 * rs + b3 * rs * srs + b4 * rs * rs;
  const double dq = 0.5 * b1 / srs + b2 + 1.5 * b3 * srs + 2.0 * b4 * rs;
  const double lg = log1p(1.0 / (2.0 * a * q));
  return {-2.0 * a * (1.0 + al * rs) * lg, -2.0 * a * al * lg + 2.0 * a * (1.0 + al * rs) * dq / (2.0 * a * q * q + q)};
}

__global__ __launch_bounds__(256) void k_gga(long long n, const double* __restrict__ up, const double* __restrict__ dn,
                                             const double* __restrict__ suu, const double* __restrict__ sud,
                                             const double* __restrict__ sdd, double kappa, double mu, double beta,
                                             double gamma, double* __restrict__ eps, double* __restrict__ vu,
                                             double* __restrict__ vd, double* __restrict__ vsuu,
                                             double* __restrict__ vsud, double* __restrict__ vsdd) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const double rho[2] = {up[i], dn[i]}, sig[2] = {suu[i], sdd[i]}, mixed = sud[i];
  const double tot = rho[0] + rho[1], safe = at_least(tot, kThreshold);
  const bool act = tot > kThreshold;
  const double rs = kRsFactor / cbrt(safe);
  double z = (rho[0] - rho[1]) / safe;
  z = z < -1.0 ? -1.0 : z > 1.0 ? 1.0 : z;
  // exchange, per spin channel
  double ex = 0.0, vx[2], vsx[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const double sp = at_least(rho[s], 0.0), sf = at_least(sp, kThreshold), n13 = cbrt(sf), n43 = sf * n13;
    const double q = kX2s * sqrt(at_least(sig[s], 0.0)) / n43, s2 = q * q;
    const double den = kappa + mu * s2;
    const double fx = 1.0 + kappa * mu * s2 / den, fxs = 2.0 * kappa * kappa * mu * s2 / (den * den);
    const bool live = sp > kThreshold, keep = live && act;
    ex += live ? -kXFactor * n43 * fx : 0.0;
    vx[s] = keep ? -(4.0 / 3.0) * kXFactor * n13 * (fx - fxs) : 0.0;
    vsx[s] = keep ? -kXFactor * kappa * kappa * mu * kX2s * kX2s / (n43 * den * den) : 0.0;
  }
  if (!act) {
    eps[i] = 0.0;
    vu[i] = 0.0;
    vd[i] = 0.0;
    vsuu[i] = 0.0;
    vsud[i] = 0.0;
    vsdd[i] = 0.0;
    return;
  }
  ex /= tot;
  // PW92 (modified parametrisation)
  const double srs = sqrt(rs);
  const Pw92 g0 = pw92_g(rs, srs, 0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294);
  const Pw92 g1 = pw92_g(rs, srs, 0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517);
  const Pw92 g2 = pw92_g(rs, srs, 0.0168869, 0.11125, 10.357, 3.6231, 0.88026, 0.49671);
  constexpr double f20 = 1.709920934161365617563962776245;
  const double pz = at_least(1.0 + z, 0.0), mz = at_least(1.0 - z, 0.0), cp = cbrt(pz), cm = cbrt(mz);
  const double fz = (pz * cp + mz * cm - 2.0) / kFzDen, dfz = (4.0 / 3.0) * (cp - cm) / kFzDen;
  const double z3 = z * z * z, z4 = z3 * z;
  const double br = g1.g - g0.g + g2.g / f20;
  const double elda = g0.g + z4 * fz * br - fz * g2.g / f20;
  const double dl_drs = g0.dg + z4 * fz * (g1.dg - g0.dg + g2.dg / f20) - fz * g2.dg / f20;
  const double dl_dz = (4.0 * z3 * fz + z4 * dfz) * br - dfz * g2.g / f20;
  // gradient correction
  const double op = cbrt(at_least(1.0 + z, kThreshold)), om = cbrt(at_least(1.0 - z, kThreshold));
  const double phi = 0.5 * (op * op + om * om), dphi = kThird * (1.0 / op - 1.0 / om), phi3 = phi * phi * phi;
  const double n13 = cbrt(safe), n43 = safe * n13;
  const double stot = at_least(sig[0] + 2.0 * mixed + sig[1], 0.0);
  const double tpx = 1.0 / (4.0 * 1.2599210498948731647672106072782 * phi * srs);  // 2^(1/3)
  const double xt = sqrt(stot) / n43, t = tpx * xt, t2 = t * t;
  const double et = expm1(-elda / (gamma * phi3)), es = fabs(et) < 1e-300 ? 1e-300 : et;
  const double A = beta / (gamma * es), u = t2 + A * t2 * t2, d = 1.0 + A * u, w = beta * u / (gamma * d);
  const double lg = log1p(w), H = gamma * phi3 * lg, pre = gamma * phi3 / (1.0 + w), gd2 = gamma * d * d;
  const double dh_dt = pre * beta / gd2 * (2.0 * t + 4.0 * A * t2 * t);
  const double dh_da = pre * beta * (t2 * t2 - u * u) / gd2;
  const double da_de = beta * (et + 1.0) / (gamma * gamma * phi3 * es * es);
  const double da_dphi = -3.0 * beta * elda * (et + 1.0) / (gamma * gamma * phi3 * phi * es * es);
  const double de_drs = dl_drs + dh_da * da_de * dl_drs + dh_dt * (-t / (2.0 * rs));
  const double de_dz = dl_dz + 3.0 * gamma * phi * phi * lg * dphi + dh_da * (da_dphi * dphi + da_de * dl_dz) +
                       dh_dt * (-t / phi) * dphi;
  const double ec = elda + H;
  const double common = ec - (rs / 3.0) * de_drs - (4.0 / 3.0) * xt * dh_dt * tpx;
  const double vst = safe * phi3 * beta * (tpx * tpx / (n43 * n43)) * (2.0 + 4.0 * A * t2) / (2.0 * (1.0 + w) * d * d);
  eps[i] = ex + ec;
  vu[i] = vx[0] + common + (1.0 - z) * de_dz;
  vd[i] = vx[1] + common - (1.0 + z) * de_dz;
  vsuu[i] = vsx[0] + vst;
  vsud[i] = 2.0 * vst;
  vsdd[i] = vsx[1] + vst;
}

}  // namespace

int launch_gga(long long n, const double* up, const double* dn, const double* suu, const double* sud, const double* sdd,
               const double par[4], double* const out[6], hipStream_t s) {
  hipLaunchKernelGGL(k_gga, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, up, dn, suu, sud, sdd, par[0], par[1],
                     par[2], par[3], out[0], out[1], out[2], out[3], out[4], out[5]);
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return 0;
  set_error(std::string("gga launch: ") + hipGetErrorString(e));
  return 1;
}

}  // namespace amt

// Entry points of the compile-time-length kernels (fft_fast_impl.hpp, compiled in four parts).
#pragma once

#include "fft_reg.hpp"
#include "kernels.hpp"

namespace amt {

// Every 2,3,5,7,11-smooth length from 20 to 128 with two factors of at most 16, in four parts of
// about equal compile time.
#define AMT_LENGTHS_A(X) X(20) X(28) X(35) X(44) X(50) X(60) X(70) X(80) X(88) X(98) X(105) X(120)
#define AMT_LENGTHS_B(X) X(21) X(25) X(30) X(36) X(45) X(54) X(63) X(72) X(81) X(90) X(99) X(108)
#define AMT_LENGTHS_C(X) X(22) X(27) X(32) X(40) X(48) X(55) X(64) X(75) X(84) X(96) X(110) X(121)
#define AMT_LENGTHS_D(X) X(24) X(33) X(42) X(49) X(56) X(66) X(77) X(100) X(112) X(126) X(128)

// Largest |Miller index| of a plane axis that the one-lane plane kernel takes.
constexpr int lane_half_width(int n) { return n / 4 + 1; }
// Lanes per row or column of that kernel, 0 where the four-step kernel (n = a b, fft_reg.hpp) is used
// at every size. Measured over the lengths with some 13 000 (84 / N)^2 planes, the plane kernel alone
// or the three passes of a local H.psi (us, four-step / one-lane):
//   FP32, one lane (planes): 24 350/248, 32 250/204, 40 253/191, 45 276/216, 54 272/211, 60 287/206;
//     from 63 on its registers leave too few wavefronts (64: 240/322).
//   FP32, four lanes (planes): 84 327/298, 100 432/351, 108 449/349, 112 437/319, 120 465/314, 128
//     382/388; up to 96 the lengths of an 8-point second factor are faster in four steps (72 270/318,
//     96 308/355).
//   FP64, one lane (passes): 20 837/767, 24 810/628, 27 976/898, 28 807/682, 32 719/630, 40 713/587, 44
//     857/732, 45 694/651, 48 679/598. Factors of 5 to 7 points keep both four-step phases short and
//     their tasks even: 25 643/861, 30 703/705, 35 688/699, 36 644/660, 42 656/664, and with a tenth of
//     the planes 70/93, 75/79, 74/79, 70/74, 71/77.
//   FP64, four lanes (planes): 72 768/526, 80 724/662 (64 471/496, 84 690/736, 96 624/877), and above
//     100, where a whole plane does not fit LDS.
constexpr int lane_count(int n, bool fp64) {
  const int a = split_n1(n), b = n / a;
  if (n <= (fp64 ? 48 : 60)) return fp64 && b >= 5 && a <= 7 ? 0 : 1;
  if (n % 4) return 0;
  if (fp64) return (n > 64 && n <= 80) || n * n * 16LL + 24LL * n > 160 * 1024 ? 4 : 0;
  return n >= 84 && !(n % 8 == 0 && n <= 96) ? 4 : 0;
}
// Planes of a call from which it is used: the four-step kernel puts four wavefronts or more on a
// plane, this one a single wavefront (one lane) or a workgroup of longer chains (four), and with fewer
// planes than fill the chip the chain of one plane is the time. Local H.psi, one-lane over four-step
// speed by planes (FP32 unless said):
//   one lane: 28 0.94 at 500, 0.97 at 1030, 1.00 at 1540, 1.04 at 3080; 40 0.81 at 240, 0.94 at 1040, 1.00
//     at 1520, 1.05 at 3080; 24 in FP64 0.95 at 264, 0.97 at 1030, 1.06 at 1536, 1.12 at 3072: six
//     wavefronts a CU. A second factor of 3 or 2 gives the four-step kernel few, long tasks: 33 0.97 at
//     760, 1.21 at 1550; 22 1.04 at 500, 1.34 at 1030. From 48 on, where a lane's row is 96 registers and
//     more, factors of up to 8 points stay ahead until the chip is full many times over: 48 0.74 at 240, 0.96
//     at 6144, 0.97 at 16 368; 56 0.80 at 280, 0.97 at 6160, 1.04 at 16 408.
//   four lanes: one workgroup a CU. 108 0.94 at 216, 1.12 at 324; 120 0.97 at 240, 1.20 at 360; 72 in FP64
//     0.92 at 216, 1.16 at 288 (84: 0.92 at 252, 0.98 at 336, 1.06 at 672).
constexpr long long lane_planes(int n, bool fp64) {
  const int a = split_n1(n), b = n / a;
  if (lane_count(n, fp64) == 0) return 0;
  if (lane_count(n, fp64) == 4) return n * n * (fp64 ? 16LL : 8LL) + 24LL * n > 160 * 1024 ? 1 : 257;
  if (!fp64 && n >= 48 && a <= 8) return 16384;
  return b == 2 ? 512 : b == 3 ? 1024 : 1536;
}

#define AMT_DECLARE_PART(S)                                                                                            \
  int fast_stick_##S(const Plan& p, int prec, int pass, const void* psi, void* hpsi, void* sticks, int nb, int k0, \
                     int nkb, hipStream_t s);                                                                          \
  int fast_plane_##S(const Plan& p, int prec, bool lane, void* sticks, const void* veff, int nb, int k0, int nkb,    \
                     hipStream_t s);                                                                                   \
  int fast_density_##S(const Plan& p, int prec, const void* sticks, int nb, int k0, const int* list,                 \
                       const double* weight, int nlist, int chunk, double* part, hipStream_t s);
AMT_DECLARE_PART(a)
AMT_DECLARE_PART(b)
AMT_DECLARE_PART(c)
AMT_DECLARE_PART(d)
#undef AMT_DECLARE_PART

}  // namespace amt

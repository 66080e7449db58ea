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
// Lanes per row or column of that kernel, 0 where the four-step kernel is used. Measured over
// the lengths at 13 440 (84 / N)^2 planes (us, four-step / one-lane):
//   FP32, one lane: 24 358/263, 32 266/222, 40 240/195, 45 256/219, 54 271/218, 60 273/210; from 63
//     on its registers leave too few wavefronts (64: 240/322).
//   FP32, four lanes: 84 347/310, 108 458/348, 112 444/318, 120 477/309, 128 378/373; up to 96 the
//     lengths of an 8-point second factor are faster in four steps (72 270/318, 96 308/355).
//   FP64, one lane: 24 642/429, 32 496/404, 40 483/339, 45 455/399, 48 441/351. Factors of 6 and 7
//     points keep both four-step phases short and their tasks even: 36 = 6 x 6 and 42 = 7 x 6 gain nothing
//     (440/432, 440/441; the three passes of a local H.psi 644/660 and 656/664, with a tenth of the planes
//     70/74 and 71/77; a factor of 5 leaves them even: 30 703/705, 35 688/699).
//   FP64, four lanes: 72 767/519, 80 723/670 (64 471/496, 84 690/736, 96 624/877), and above 100,
//     where a whole plane does not fit LDS.
// With fewer planes than about six wavefronts a CU the four-step kernel is faster (one band at 48^3 in
// FP32 16 us against 24) and is not used all the same: one-lane results are nearer to 64 bits (24^3 in
// FP64 3.4e-16 against 4.2e-16, 84^3 in FP32 2.24e-7 against 2.35e-7), and an iteration whose calls
// change kernels with their size converges later.
constexpr int lane_count(int n, bool fp64) {
  const int a = split_n1(n), b = n / a;  // the four-step factors
  if (n <= (fp64 ? 48 : 60)) return fp64 && b >= 6 && a <= 7 ? 0 : 1;
  if (n % 4) return 0;
  if (fp64) return (n > 64 && n <= 80) || n * n * 16LL + 24LL * n > 160 * 1024 ? 4 : 0;
  return n >= 84 && !(n % 8 == 0 && n <= 96) ? 4 : 0;
}

#define AMT_DECLARE_PART(S)                                                                                            \
  int fast_stick_##S(const Plan& p, int prec, int pass, const void* psi, void* hpsi, void* sticks, int nb, int k0, \
                     int nkb, hipStream_t s);                                                                          \
  int fast_plane_##S(const Plan& p, int prec, void* sticks, const void* veff, int nb, int k0, int nkb,               \
                     hipStream_t s);                                                                                   \
  int fast_density_##S(const Plan& p, int prec, const void* sticks, int nb, int k0, const int* list,                 \
                       const double* weight, int nlist, int chunk, double* part, hipStream_t s);
AMT_DECLARE_PART(a)
AMT_DECLARE_PART(b)
AMT_DECLARE_PART(c)
AMT_DECLARE_PART(d)
#undef AMT_DECLARE_PART

}  // namespace amt

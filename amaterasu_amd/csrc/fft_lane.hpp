// Length-L complex transforms held in one lane's registers.
//
// Everything is unrolled over compile-time indices, so every twiddle is a literal and every
// permutation is free. L = A * B with coprime factors is split by the prime-factor algorithm
// (Good, Thomas), which needs no twiddles at all: input n = (B a + A b) mod L, output
// k = (B B' ka + A A' kb) mod L with B B' = 1 mod A, A A' = 1 mod B. Only powers of one prime
// (9, 16, 25, 27, 32, ...) take the Cooley-Tukey step with its twiddle multiplications. A
// 42-point transform is 680 arithmetic instructions per lane this way.
#pragma once

#include <utility>

#include "fft_reg.hpp"

namespace amt {

template <typename F, int... I>
__host__ __device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
// f(0), f(1), ..., f(K - 1) with the index as a compile-time constant
template <int K, typename F>
__host__ __device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(std::forward<F>(f), std::make_integer_sequence<int, K>{});
}

constexpr int gcd_of(int a, int b) { return b == 0 ? a : gcd_of(b, a % b); }
// x with a x = 1 mod b
constexpr int inverse_mod(int a, int b) {
  for (int x = 1; x < b; ++x)
    if (a * x % b == 1) return x;
  return 1;
}
constexpr bool one_pass_dft(int l) { return l == 2 || l == 4 || l == 8 || l == 3 || l == 5 || l == 7 || l == 11; }

// Factor of L taken first: the largest power of one prime that leaves a coprime cofactor; for a
// power of one prime (not one of the direct lengths) the radix of its first step.
constexpr int first_factor(int l) {
  const int primes[5] = {2, 3, 5, 7, 11};
  for (int p : primes) {
    if (l % p) continue;
    int q = 1, r = l;
    while (r % p == 0) {
      q *= p;
      r /= p;
    }
    if (r > 1) return q;                                  // coprime split
    if (p == 2) return l % 8 == 0 && l != 16 ? 8 : 4;     // 16 = 4 * 4, 32 = 8 * 4, 64 = 8 * 8
    return p;
  }
  return l;
}

template <int L, int SIGN, typename C>
__host__ __device__ __forceinline__ void lane_dft(C* v) {
  using Rt = decltype(C::x);
  if constexpr (L == 1) {
    return;
  } else if constexpr (one_pass_dft(L)) {
    dft_any<L, SIGN>(v);
  } else {
    constexpr int A = first_factor(L), B = L / A;
    static_assert(A > 1 && B > 1 && A * B == L, "length is not 2,3,5,7,11-smooth");
    constexpr bool coprime = gcd_of(A, B) == 1;
    C t[L];
    static_for<B>([&](auto b_) {
      constexpr int b = b_;
      C u[A];
      static_for<A>([&](auto a_) {
        constexpr int a = a_;
        u[a] = v[coprime ? (B * a + A * b) % L : b + B * a];
      });
      lane_dft<A, SIGN>(u);
      static_for<A>([&](auto a_) {
        constexpr int ka = a_;
        if constexpr (coprime || b * ka == 0) {
          t[ka * B + b] = u[ka];
        } else {
          constexpr double c = cos2pi((long)b * ka, L), s = SIGN * sin2pi((long)b * ka, L);
          t[ka * B + b] = cmake<C>(u[ka].x * (Rt)c - u[ka].y * (Rt)s, u[ka].x * (Rt)s + u[ka].y * (Rt)c);
        }
      });
    });
    static_for<A>([&](auto a_) {
      constexpr int ka = a_;
      lane_dft<B, SIGN>(t + ka * B);
      static_for<B>([&](auto b_) {
        constexpr int kb = b_;
        constexpr int k = coprime ? (B * inverse_mod(B % A, A) * ka + A * inverse_mod(A % B, B) * kb) % L : ka + A * kb;
        v[k] = t[ka * B + kb];
      });
    });
  }
}

}  // namespace amt

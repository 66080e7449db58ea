// Compile-time-length H.psi and density kernels: part a of the lengths.
#define AMT_PART(X) AMT_LENGTHS_A(X)
#define AMT_PART_FN(name) name##_a
#include "fft_fast_impl.hpp"

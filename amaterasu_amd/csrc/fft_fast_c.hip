// Compile-time-length H.psi and density kernels: part c of the lengths.
#define AMT_PART(X) AMT_LENGTHS_C(X)
#define AMT_PART_FN(name) name##_c
#include "fft_fast_impl.hpp"

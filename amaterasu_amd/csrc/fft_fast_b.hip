// Compile-time-length H.psi and density kernels: part b of the lengths.
#define AMT_PART(X) AMT_LENGTHS_B(X)
#define AMT_PART_FN(name) name##_b
#include "fft_fast_impl.hpp"

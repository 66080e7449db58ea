// Compile-time-length H.psi and density kernels: part d of the lengths.
#define AMT_PART(X) AMT_LENGTHS_D(X)
#define AMT_PART_FN(name) name##_d
#include "fft_fast_impl.hpp"

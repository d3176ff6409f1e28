// Instantiations of the in-register Bluestein kernels, compute and storage type float.
#define HPXFFT_INSTANTIATE
#include "blue.hpp"

HPXFFT_DEFINE_BLUE(f32, float)

// Instantiations of the in-register Bluestein kernels, compute and storage type double.
#define HPXFFT_INSTANTIATE
#include "blue.hpp"

HPXFFT_DEFINE_BLUE(f64, double)

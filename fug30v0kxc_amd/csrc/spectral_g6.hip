// spectral_g6.hip -- transform kernels instantiated for one group of
// lengths (split so the kernels compile in parallel).
#include "spectral_expand.hpp"
#include "spectral_mag.hpp"

#define SIZES_G6(X) X(36) X(72) X(100) X(108)
MHD_SPECTRAL_GROUP(launch_spectral_g6, SIZES_G6)

// spectral_g7.hip -- transform kernels instantiated for one group of
// lengths (split so the kernels compile in parallel).
#include "spectral_expand.hpp"
#include "spectral_mag.hpp"

#define SIZES_G7(X) X(144) X(180) X(200) X(216)
MHD_SPECTRAL_GROUP(launch_spectral_g7, SIZES_G7)

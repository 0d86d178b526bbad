// The paired plane pass in FP32: the band density.
#define BD_PLANE_TYPE float
#define BD_PLANE_MODE 1
#include "plane_kernels.hpp"

// The paired plane pass in FP32: dV psi of kept fields.
#define BD_PLANE_TYPE float
#define BD_PLANE_MODE 2
#include "plane_kernels.hpp"

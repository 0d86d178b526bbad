// The paired plane pass in FP32: V psi of the sticks.
#define BD_PLANE_TYPE float
#define BD_PLANE_MODE 0
#include "plane_kernels.hpp"

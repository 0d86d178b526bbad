// The paired plane pass in FP64: dV psi of kept fields.
#define BD_PLANE_TYPE double
#define BD_PLANE_MODE 2
#include "plane_kernels.hpp"

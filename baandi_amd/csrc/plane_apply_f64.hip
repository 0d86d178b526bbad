// The paired plane pass in FP64: V psi of the sticks.
#define BD_PLANE_TYPE double
#define BD_PLANE_MODE 0
#define BD_PLANE_LAYOUTS
#include "plane_kernels.hpp"

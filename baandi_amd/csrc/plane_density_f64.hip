// The paired plane pass in FP64: the band density.
#define BD_PLANE_TYPE double
#define BD_PLANE_MODE 1
#include "plane_kernels.hpp"

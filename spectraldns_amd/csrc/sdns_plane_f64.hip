// Double-precision instantiation of the plane kernels.
#include "sdns_plane.hpp"
SDNS_PLANE_INSTANTIATE(double)

// Plane kernels (passes 1 + 2 and 4 + 5 of small planes), R = float.
#include "gla_planes_impl.hpp"
template hipError_t gla::run_fwd_planes<float>(const gla::Geom&, const gla::DevTab&, const void*, void*, int, hipStream_t);
template hipError_t gla::run_inv_planes<float>(const gla::Geom&, const gla::DevTab&, const void*, void*, int, double,
                                            double, double, double, int, const gla::Epi&, hipStream_t);

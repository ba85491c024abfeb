// procell_filter.hpp -- the error bound of the filtered kernel's
// single-precision times (derived beside normal_pair_f32 in
// procell_kernels.hip), shared by the kernel and the host's choice of a
// kernel.  No HIP.
#pragma once

#include <math.h>
#include <stdint.h>

#ifdef __HIP__
#define PROCELL_FILTER_HD __host__ __device__
#else
#define PROCELL_FILTER_HD
#endif

namespace procell {

// What normal_pair_f32 may be off by.
constexpr float kPairErr = 7.0e-6f;

// Bound of a type's times per level, and of all times of a cell whose row has
// generation cap kcap.
PROCELL_FILTER_HD inline double filter_type_err(double mean, double sd, double t_max)
{
    return fabs(sd) * ((double)kPairErr + 0x1p-20) + 0x1p-22 * fabs(mean) + 0x1p-23 * t_max;
}
PROCELL_FILTER_HD inline float filter_cell_err(uint32_t kcap, float terr) { return (float)(kcap + 4u) * terr; }

}  // namespace procell

// What mcut_amd/csrc/geom.hpp needs of the HIP header, for a host compiler.
#pragma once
#include <math.h>
#include <stdint.h>
#define __device__
#define __host__
#define __forceinline__ inline
static inline double __fma_rn(double a, double b, double c) { return fma(a, b, c); }

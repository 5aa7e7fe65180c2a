// The walk kernels of one family (walk_launch.hpp): Philox4x32-10 draws, one walk per launch.
#include "walk_family.hpp"

SW_SINGLE_FAMILY(philox_f32_half, PhiloxRng, PhaseF32, launch_half)

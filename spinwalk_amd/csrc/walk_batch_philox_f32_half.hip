// The walk kernels of one family (walk_launch.hpp): Philox4x32-10 draws, batched.
#include "walk_family.hpp"

SW_BATCH_FAMILY(philox_f32_half, PhiloxRng, PhaseF32, launch_batch_half)

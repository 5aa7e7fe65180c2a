// The walk kernels of one family (walk_launch.hpp): replayed draws, single and batched.
#include "walk_family.hpp"

SW_SINGLE_FAMILY(replay_f32_wide, ReplayRng, PhaseF32, launch_wide)
SW_BATCH_FAMILY(replay_f32_wide, ReplayRng, PhaseF32, launch_batch_wide)

// The walk kernels of one family (walk_launch.hpp): replayed draws, single and batched.
#include "walk_family.hpp"

SW_SINGLE_FAMILY(replay_f64_wide, ReplayRng, PhaseF64, launch_wide)
SW_BATCH_FAMILY(replay_f64_wide, ReplayRng, PhaseF64, launch_batch_wide)

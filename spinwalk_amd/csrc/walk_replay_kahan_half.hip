// The walk kernels of one family (walk_launch.hpp): replayed draws, single and batched.
#include "walk_family.hpp"

SW_SINGLE_FAMILY(replay_kahan_half, ReplayRng, PhaseKahan, launch_half)
SW_BATCH_FAMILY(replay_kahan_half, ReplayRng, PhaseKahan, launch_batch_half)

// walk_family.hpp -- defines the launchers of one family of walk kernels
// (walk_launch.hpp); each walk_*.hip instantiates one, so that the families
// compile in parallel.
#pragma once
#include "walk_impl.hpp"

#define SW_SINGLE_FAMILY(name, Rng, Phase, launch)                                        \
    namespace sw {                                                                        \
    hipError_t launch_walk_##name(const WalkArgs &a, int field, hipStream_t s) {          \
        return launch<Rng, Phase>(a, field, s);                                           \
    }                                                                                     \
    }

#define SW_BATCH_FAMILY(name, Rng, Phase, launch)                                                                \
    namespace sw {                                                                                               \
    hipError_t launch_walk_batch_##name(const void *items, const BatchChunk *chunks, uint32_t n_slots,           \
                                        uint32_t threads, uint32_t spl, int views, int field, int variant,       \
                                        int addr, size_t lds, hipStream_t s) {                                   \
        return launch<Rng, Phase>(items, chunks, n_slots, threads, spl, views, field, variant, addr, lds, s);    \
    }                                                                                                            \
    }

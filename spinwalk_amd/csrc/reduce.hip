// reduce.hip -- FP64 echo reduction.
//
// The reference reduces on the host in Python: for each scale and echo,
// signal = | mean over spins with T == tissue of (Mx, My) |
// (demo/spinwalk_bold.ipynb:733-736).  Here the sums of Mx, My and the counts
// are formed per (echo, label) in float64 on the device.  Pass 1: block j of a pair
// sums the pair's j-th chunk of spins into partial[pair][j]; pass 2 adds the
// partials of each pair in a fixed order, one block per pair.  The order of
// additions is fixed by the launch shape alone, so results are bit-reproducible.
//
// Small reductions are bound by latency: a chunk's loads, a block's tree, the launches.
// Hence short chunks (a thread adds 4 spins, their loads independent), a block for
// kLabels labels of an echo (one pass over its lines instead of one per label: 8 echoes
// of 2e5 spins in float64, 66 us in pass 1 with a block per label), and for a batch one
// launch per pass for all its tiles.  The batch of 30 tiles of 12 phantoms: 7.17 ms
// with two launches a tile of 4096-spin chunks, 6.69 ms now.  (One pass whose last
// block adds the partials needs a fence per block, which writes an XCD's L2 back:
// 2.24 ms against 1.96 ms for the 8 echoes with their walk.)
// Large ones are bound by the trees (36 lane exchanges per label and wave, 1024 spins
// apart) and the partials, so chunks grow until kBlocks blocks are left, which also
// bounds the grid and the partials (0.8 MB an item) whatever the sizes.  Where an echo
// has more labels than a block takes, a spin's M1 is read by the block of its label
// alone.  Of 1e6 spins, 4 echoes, 64 labels 486 -> 151 us, 1e6, 1, 256 420 -> 129, 2e6, 8, 16
// 985 -> 359, 1e7, 1, 2 65 -> 51 (4096-spin chunks of a label each: 358, 248, 559 and 62).
#include <hip/hip_runtime.h>

#include "walk_launch.hpp"

namespace sw {
namespace {

constexpr uint32_t kThreads = 256;
constexpr uint32_t kPerThread = 4;
constexpr uint32_t kPiece = kThreads * kPerThread;   // spins a block adds at a time
constexpr uint32_t kLabels = 4;                      // labels per block
constexpr uint64_t kBlocks = 4096;                   // 2 workgroups a SIMD: chunks grow above that
constexpr uint64_t kMaxBlocks = (1u << 24) - 1;      // of a launch: a grid holds below 2^32 threads

__host__ __device__ inline uint32_t groups_of(uint32_t n_sub) { return n_sub / kLabels + (n_sub % kLabels != 0); }

// The sums of a block's threads, in thread 0's v.
__device__ __forceinline__ void block_sum(double (&v)[3], double (&sh)[3][kThreads / 64]) {
    #pragma unroll
    for (int i = 0; i < 3; i++) {
        #pragma unroll
        for (int o = 32; o > 0; o >>= 1) v[i] += __shfl_xor(v[i], o);
        if ((threadIdx.x & 63) == 0) sh[i][threadIdx.x >> 6] = v[i];
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int i = 0; i < 3; i++) v[i] = (sh[i][0] + sh[i][1]) + (sh[i][2] + sh[i][3]);
}

// Block b of an item: a chunk (r.pieces pieces) of spins of one echo, for kLabels labels.
// ALL: they are all the labels there are, so M1 is read beside T; else only the spins of
// these labels are read, once their T has come.
template <class R, bool ALL>
__device__ __forceinline__ void reduce_block(const ReduceItem &r, uint32_t b) {
    __shared__ double sh[kLabels][3][kThreads / 64];
    const uint32_t unit = b / r.n_chunks, chunk = b % r.n_chunks;
    const uint32_t groups = groups_of(r.n_sub), te = unit / groups, lab0 = unit % groups * kLabels;
    const R *M1 = (const R *)r.M1;
    double v[kLabels][3] = {};
    const uint64_t first = (uint64_t)chunk * r.pieces * kPiece;
    for (uint32_t j = 0; j < r.pieces; j++) {
        const uint64_t s0 = first + (uint64_t)j * kPiece;
        if (s0 >= r.n) break;
        const uint32_t left = (uint32_t)(r.n - s0);
        const uint64_t base = s0 * r.n_te + te;
        R mx[kPerThread], my[kPerThread];
        uint32_t lab[kPerThread];
        #pragma unroll
        for (uint32_t k = 0; k < kPerThread; k++) {
            const uint32_t i = k * kThreads + threadIdx.x;
            const uint64_t o = base + (uint64_t)i * r.n_te;
            lab[k] = ~0u;
            if (i < left) {
                lab[k] = r.T[o];
                if (ALL) { mx[k] = M1[3 * o]; my[k] = M1[3 * o + 1]; }
            }
        }
        if (!ALL) {
            #pragma unroll
            for (uint32_t k = 0; k < kPerThread; k++) {
                const uint64_t o = base + (uint64_t)(k * kThreads + threadIdx.x) * r.n_te;
                if (lab[k] - lab0 < kLabels) { mx[k] = M1[3 * o]; my[k] = M1[3 * o + 1]; }
            }
        }
        #pragma unroll
        for (uint32_t l = 0; l < kLabels; l++) {
            if (lab0 + l >= r.n_sub) break;
            #pragma unroll
            for (uint32_t k = 0; k < kPerThread; k++)
                if (lab[k] == lab0 + l) { v[l][0] += (double)mx[k]; v[l][1] += (double)my[k]; v[l][2] += 1.0; }
        }
    }
    #pragma unroll
    for (uint32_t l = 0; l < kLabels; l++) {
        if (lab0 + l >= r.n_sub) break;
        block_sum(v[l], sh[l]);
        if (threadIdx.x == 0) {
            const uint64_t pair = (uint64_t)te * r.n_sub + lab0 + l;
            double *p = r.n_chunks == 1 ? r.out + 3 * pair : r.partial + 3 * (pair * r.n_chunks + chunk);
            p[0] = v[l][0]; p[1] = v[l][1]; p[2] = v[l][2];
        }
    }
}
__device__ __forceinline__ void reduce_block(const ReduceItem &r, uint32_t b) {
    const bool all = r.n_sub <= kLabels;
    if (r.f64) all ? reduce_block<double, true>(r, b) : reduce_block<double, false>(r, b);
    else       all ? reduce_block<float, true>(r, b) : reduce_block<float, false>(r, b);
}

// Thread t adds the partials t, t + 256, ... in order, then the block's tree.
__device__ __forceinline__ void finish_pair(const ReduceItem &r, uint32_t pair) {
    __shared__ double sh[3][kThreads / 64];
    const double *part = r.partial + 3 * (uint64_t)pair * r.n_chunks;
    double v[3] = {0., 0., 0.};
    for (uint32_t c = threadIdx.x; c < r.n_chunks; c += kThreads)
        for (int i = 0; i < 3; i++) v[i] += part[3 * (uint64_t)c + i];
    block_sum(v, sh);
    double *out = r.out + 3 * (uint64_t)pair;
    if (threadIdx.x == 0) { out[0] = v[0]; out[1] = v[1]; out[2] = v[2]; }
}

template <class R, bool ALL>
__global__ __launch_bounds__(kThreads) void reduce_pass1(const ReduceItem r) { reduce_block<R, ALL>(r, blockIdx.x); }
__global__ __launch_bounds__(kThreads) void reduce_pass2(const ReduceItem r) { finish_pair(r, blockIdx.x); }

// items[] in device memory: the last item whose first block (pair) is at or before
// x (an item without a second pass has no pairs and shares the next one's first).
__device__ __forceinline__ ReduceItem item_of(const ReduceItem *items, uint32_t n_items, uint32_t ReduceItem::*first,
                                              uint32_t x) {
    uint32_t lo = 0, hi = n_items;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) / 2;
        if (items[mid].*first <= x) lo = mid; else hi = mid;
    }
    return items[lo];
}

__global__ __launch_bounds__(kThreads) void reduce_batch_pass1(const ReduceItem *items, uint32_t n_items) {
    const ReduceItem r = item_of(items, n_items, &ReduceItem::first_block, blockIdx.x);
    reduce_block(r, blockIdx.x - r.first_block);
}
__global__ __launch_bounds__(kThreads) void reduce_batch_pass2(const ReduceItem *items, uint32_t n_items) {
    const ReduceItem r = item_of(items, n_items, &ReduceItem::first_pair, blockIdx.x);
    finish_pair(r, blockIdx.x - r.first_pair);
}

}  // namespace

bool reduce_plan(ReduceItem &r) {
    const uint64_t units = (uint64_t)r.n_te * groups_of(r.n_sub), pieces = (r.n + (uint64_t)kPiece - 1) / kPiece;
    if (units > kMaxBlocks) return false;
    uint64_t per = pieces * units / kBlocks;                 // the factors are at most 2^22 and 2^24
    if (per > pieces) per = pieces;
    if (per == 0) per = 1;
    r.pieces = (uint32_t)per;
    r.n_chunks = (uint32_t)((pieces + per - 1) / per);
    if (r.n_chunks == 0) r.n_chunks = 1;                     // no spins: zeros
    r.blocks = (uint32_t)(units * r.n_chunks);
    r.pairs = r.n_chunks > 1 ? r.n_te * r.n_sub : 0;         // that need the second pass
    return true;
}

uint64_t reduce_partial_len(const ReduceItem &r) { return 3ull * r.n_chunks * r.pairs; }

hipError_t launch_echo_reduce(const ReduceItem &r, hipStream_t s) {
    const bool all = r.n_sub <= kLabels;
    const auto pass1 = r.f64 ? (all ? reduce_pass1<double, true> : reduce_pass1<double, false>)
                             : (all ? reduce_pass1<float, true> : reduce_pass1<float, false>);
    if (r.blocks) hipLaunchKernelGGL(pass1, dim3(r.blocks), dim3(kThreads), 0, s, r);
    if (r.pairs) hipLaunchKernelGGL(reduce_pass2, dim3(r.pairs), dim3(kThreads), 0, s, r);
    return hipGetLastError();
}

std::vector<ReduceLaunch> reduce_launches(std::vector<ReduceItem> &items) {
    std::vector<ReduceLaunch> out;
    for (uint32_t i = 0; i < (uint32_t)items.size(); i++) {
        ReduceItem &r = items[i];
        if (out.empty() || (uint64_t)out.back().n_blocks + r.blocks > kMaxBlocks ||
            (uint64_t)out.back().n_pairs + r.pairs > kMaxBlocks)
            out.push_back({i, 0, 0, 0});
        ReduceLaunch &l = out.back();
        r.first_block = l.n_blocks;
        r.first_pair = l.n_pairs;
        l.n_items++;
        l.n_blocks += r.blocks;
        l.n_pairs += r.pairs;
    }
    return out;
}

hipError_t launch_echo_reduce_batch(const ReduceItem *items, const ReduceLaunch &l, hipStream_t s) {
    if (l.n_blocks)
        hipLaunchKernelGGL(reduce_batch_pass1, dim3(l.n_blocks), dim3(kThreads), 0, s, items + l.first, l.n_items);
    if (l.n_pairs)
        hipLaunchKernelGGL(reduce_batch_pass2, dim3(l.n_pairs), dim3(kThreads), 0, s, items + l.first, l.n_items);
    return hipGetLastError();
}

}  // namespace sw

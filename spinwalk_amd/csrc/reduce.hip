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
// What bounds it is latency: a chunk's loads, a block's tree, the launches.  Hence
// short chunks (a thread adds 4 spins, their loads independent), a block for all
// labels of an echo (one pass over its lines instead of one per label: 8 echoes of
// 2e5 spins in float64, 66 us in pass 1 with a block per label), and for a batch one
// launch per pass for all its tiles.  The batch of 30 tiles of 12 phantoms: 7.17 ms
// with two launches a tile of 4096-spin chunks, 6.69 ms now.  (One pass whose last
// block adds the partials needs a fence per block, which writes an XCD's L2 back:
// 2.24 ms against 1.96 ms for the 8 echoes with their walk.)
#include <hip/hip_runtime.h>

#include "walk_launch.hpp"

namespace sw {
namespace {

constexpr uint32_t kThreads = 256;
constexpr uint32_t kPerThread = 4;
constexpr uint32_t kChunk = kThreads * kPerThread;   // spins per block
constexpr uint32_t kLabels = 4;                      // labels per block

__host__ __device__ inline uint32_t chunks_of(uint32_t n) { return n ? (n + kChunk - 1) / kChunk : 1; }   // no spins: zeros
__host__ __device__ inline uint32_t groups_of(uint32_t n_sub) { return (n_sub + kLabels - 1) / kLabels; }

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

// Block b of an item: a chunk of spins of one echo, for kLabels labels.
template <class R>
__device__ __forceinline__ void reduce_block(const ReduceItem &r, uint32_t b) {
    __shared__ double sh[kLabels][3][kThreads / 64];
    const uint32_t n_chunks = chunks_of(r.n), unit = b / n_chunks, chunk = b % n_chunks;
    const uint32_t groups = groups_of(r.n_sub), te = unit / groups, lab0 = unit % groups * kLabels;
    const R *M1 = (const R *)r.M1;
    R mx[kPerThread], my[kPerThread];
    uint32_t lab[kPerThread];
    #pragma unroll
    for (uint32_t k = 0; k < kPerThread; k++) {
        const uint32_t s = chunk * kChunk + k * kThreads + threadIdx.x;
        const uint64_t o = (uint64_t)s * r.n_te + te;
        lab[k] = ~0u;
        if (s < r.n) { lab[k] = r.T[o]; mx[k] = M1[3 * o]; my[k] = M1[3 * o + 1]; }
    }
    #pragma unroll
    for (uint32_t l = 0; l < kLabels; l++) {
        if (lab0 + l >= r.n_sub) break;
        double v[3] = {0., 0., 0.};
        #pragma unroll
        for (uint32_t k = 0; k < kPerThread; k++)
            if (lab[k] == lab0 + l) { v[0] += (double)mx[k]; v[1] += (double)my[k]; v[2] += 1.0; }
        block_sum(v, sh[l]);
        if (threadIdx.x == 0) {
            const uint64_t pair = (uint64_t)te * r.n_sub + lab0 + l;
            double *p = n_chunks == 1 ? r.out + 3 * pair : r.partial + 3 * (pair * n_chunks + chunk);
            p[0] = v[0]; p[1] = v[1]; p[2] = v[2];
        }
    }
}
__device__ __forceinline__ void reduce_block(const ReduceItem &r, uint32_t b) {
    if (r.f64) reduce_block<double>(r, b);
    else       reduce_block<float>(r, b);
}

// Thread t adds the partials t, t + 256, ... in order, then the block's tree.
__device__ __forceinline__ void finish_pair(const ReduceItem &r, uint32_t pair) {
    __shared__ double sh[3][kThreads / 64];
    const uint32_t n_chunks = chunks_of(r.n);
    const double *part = r.partial + 3 * (uint64_t)pair * n_chunks;
    double v[3] = {0., 0., 0.};
    for (uint32_t c = threadIdx.x; c < n_chunks; c += kThreads)
        for (int i = 0; i < 3; i++) v[i] += part[3 * (uint64_t)c + i];
    block_sum(v, sh);
    double *out = r.out + 3 * pair;
    if (threadIdx.x == 0) { out[0] = v[0]; out[1] = v[1]; out[2] = v[2]; }
}

__global__ __launch_bounds__(kThreads) void reduce_pass1(const ReduceItem r) { reduce_block(r, blockIdx.x); }
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

uint32_t reduce_blocks(uint32_t n_spins, uint32_t n_te, uint32_t n_sub) {
    return chunks_of(n_spins) * n_te * groups_of(n_sub);
}

uint32_t reduce_pairs(uint32_t n_spins, uint32_t n_te, uint32_t n_sub) {
    return chunks_of(n_spins) > 1 ? n_te * n_sub : 0;
}

uint64_t reduce_partial_len(uint32_t n_spins, uint32_t n_te, uint32_t n_sub) {
    return 3ull * chunks_of(n_spins) * n_te * n_sub;
}

hipError_t launch_echo_reduce(const ReduceItem &r, hipStream_t s) {
    const uint32_t blocks = reduce_blocks(r.n, r.n_te, r.n_sub), pairs = reduce_pairs(r.n, r.n_te, r.n_sub);
    if (blocks) hipLaunchKernelGGL(reduce_pass1, dim3(blocks), dim3(kThreads), 0, s, r);
    if (pairs) hipLaunchKernelGGL(reduce_pass2, dim3(pairs), dim3(kThreads), 0, s, r);
    return hipGetLastError();
}

hipError_t launch_echo_reduce_batch(const ReduceItem *items, uint32_t n_items, uint32_t n_blocks, uint32_t n_pairs,
                                    hipStream_t s) {
    if (n_blocks) hipLaunchKernelGGL(reduce_batch_pass1, dim3(n_blocks), dim3(kThreads), 0, s, items, n_items);
    if (n_pairs) hipLaunchKernelGGL(reduce_batch_pass2, dim3(n_pairs), dim3(kThreads), 0, s, items, n_items);
    return hipGetLastError();
}

}  // namespace sw

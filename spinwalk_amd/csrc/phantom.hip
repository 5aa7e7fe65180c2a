// phantom.hip -- phantom preparation kernels: label count, field range and the
// bricked voxel records, 16-bit copies of the fieldmap among them.
//
// The reference keeps the fieldmap in float32 (src/sim/monte_carlo.cu:98-123,
// 254).  The mixed-precision walk gathers a 16-bit copy:
// - float16 or bfloat16 of field_T / half_scale, where half_scale is a power of
//   two chosen so that the largest |field| lands near 2^14: scaling by a power of
//   two is exact, and it keeps the 1/r^2 and 1/r^3 tails of vessel fields out of
//   the float16 subnormal range for as long as possible.  The error is relative:
//   up to 2^-11 of the value for float16;
// - int16 fixed point rint(field_T / q_scale), q_scale = max|field| / 32767.
//   The error is absolute, at most max|field| / 65534, so every value above 3 %
//   of the largest is held more closely than in float16; a field that is one
//   constant inside every inclusion (cylinders along B0) is held exactly at its
//   largest value.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include "walk_launch.hpp"

namespace sw {
namespace {

// Largest label and largest |field| of the phantom.  Streams 16 voxels a thread
// and trip (one 16-byte load of labels, four of field), reduces in the workgroup
// and sends one atomic per value and workgroup, and only where it would raise the
// value: atomics of all workgroups meet in one line, about 11 ns each.  (One
// atomic per wave and value from 16384 waves took 380 us at 256^3, whatever the
// phantom's size; this takes 23 us, 3.7 TB/s.)
constexpr uint32_t kStatsThreads = 256, kStatsBlocks = 1024;
__global__ __launch_bounds__(kStatsThreads) void stats_kernel(const uint8_t *mask, const float *field, uint64_t n,
                                                              uint32_t *stats) {
    uint32_t mlab = 0, mabs = 0;
    const uint64_t first = (uint64_t)blockIdx.x * kStatsThreads + threadIdx.x, stride = (uint64_t)gridDim.x * kStatsThreads;
    auto bits = [](float f) { return __float_as_uint(fabsf(f)); };                // |f| bits order like values
    const uint64_t n16 = n / 16;                                                  // mask and field are 16-byte aligned
    for (uint64_t i = first; i < n16; i += stride) {
        const uint4 m = ((const uint4 *)mask)[i];
        for (uint32_t w : {m.x, m.y, m.z, m.w})
            mlab = max(mlab, max(max(w & 0xFFu, (w >> 8) & 0xFFu), max((w >> 16) & 0xFFu, w >> 24)));
        if (field) {
            #pragma unroll
            for (int k = 0; k < 4; k++) {
                const float4 f = ((const float4 *)field)[4 * i + k];
                mabs = max(mabs, max(max(bits(f.x), bits(f.y)), max(bits(f.z), bits(f.w))));
            }
        }
    }
    for (uint64_t i = 16 * n16 + first; i < n; i += stride) {                     // the last n mod 16
        mlab = max(mlab, (uint32_t)mask[i]);
        if (field) mabs = max(mabs, bits(field[i]));
    }
    for (int o = 32; o > 0; o >>= 1) {
        mlab = max(mlab, (uint32_t)__shfl_xor((int)mlab, o));
        mabs = max(mabs, (uint32_t)__shfl_xor((int)mabs, o));
    }
    __shared__ uint32_t sh[2][kStatsThreads / 64];
    if ((threadIdx.x & 63) == 0) { sh[0][threadIdx.x >> 6] = mlab; sh[1][threadIdx.x >> 6] = mabs; }
    __syncthreads();
    if (threadIdx.x < 2) {
        uint32_t v = 0;
        for (uint32_t w = 0; w < kStatsThreads / 64; w++) v = max(v, sh[threadIdx.x][w]);
        if (v > __atomic_load_n(&stats[threadIdx.x], __ATOMIC_RELAXED)) atomicMax(&stats[threadIdx.x], v);
    }
}

// The 16-bit field of a voxel: KIND 1 fp16, 2 bf16 of field_T / half_scale;
// 4 int16 fixed point rint(field_T / q_scale).
template <int KIND>
__device__ __forceinline__ uint32_t field16(float field, float inv_scale) {
    uint32_t h = 0;
    if (KIND == 1) h = __half_as_ushort(__float2half_rn(field * inv_scale));
    if (KIND == 2) {
        const uint32_t bits = __float_as_uint(field * inv_scale);
        h = (bits + 0x7FFFu + ((bits >> 16) & 1u)) >> 16;          // round to nearest even
    }
    if (KIND == 4) {
        // nearest step, ties to even; |q| <= 32767 up to the rounding of inv_scale
        const double q = rint((double)field * (double)inv_scale);
        h = (uint32_t)(int32_t)fmin(32767.0, fmax(-32767.0, q)) & 0xFFFFu;
    }
    return h & 0xFFFFu;
}

// Row-major mask/field -> bricked records (walk_args.hpp).  One thread builds one
// 128-byte line, a brick, in registers and writes it whole, padding included, so
// the array needs no clearing; neighbouring lanes take bricks neighbouring in z,
// so their reads of a row of voxels are contiguous.  The two float32 copies of the
// production walks have the same bricks and are built together.  (One thread per voxel, its
// record written byte by byte into a cleared array, took 104 us a copy at 256^3
// for the float32 formats; this takes 55 us for the 8-byte records, 5 B read and 8 B
// written a voxel, 4 TB/s, and 87 us for the two copies, 110 us one by one.)
enum : int { REC_F32 = 0, REC_F16 = 1, REC_BF16 = 2, REC_NONE = 3, REC_Q16 = 4, REC_F32_PAIR = 5 };
template <int KIND> struct BrickOf {         // voxels of a line per axis
    static constexpr bool k16 = KIND == REC_F16 || KIND == REC_BF16 || KIND == REC_Q16;
    static constexpr int bx = KIND == REC_F32 ? 1 << kBrick8.lbx : KIND == REC_NONE ? 1 << kBrick4.lbx : k16 ? kPack16.bx : kPackF32.bx;
    static constexpr int by = KIND == REC_F32 ? 1 << kBrick8.lby : KIND == REC_NONE ? 1 << kBrick4.lby : k16 ? kPack16.by : kPackF32.by;
    static constexpr int bz = KIND == REC_F32 ? 1 << kBrick8.lbz : KIND == REC_NONE ? 1 << kBrick4.lbz : k16 ? kPack16.bz : kPackF32.bz;
};

// ors the low `bytes` bytes of v into a line at byte `at` (a constant after unrolling)
__device__ __forceinline__ void put_bytes(uint32_t w[32], int at, uint32_t v, int bytes) {
    const int k = at / 4, sh = 8 * (at % 4);
    w[k] |= v << sh;
    if (sh + 8 * bytes > 32) w[k + 1] |= v >> (32 - sh);
}

// n_x, n_y, n_z: bricks per axis, padding included; nb_y, nb_z: the array's pitch.
template <int KIND>
__global__ __launch_bounds__(256) void bricks_kernel(const uint8_t *mask, const float *field, uint32_t nx, uint32_t ny,
                                                     uint32_t nz, uint32_t n_x, uint32_t n_y, uint32_t n_z, uint64_t nb_y,
                                                     uint64_t nb_z, bool sup, float inv_scale, uint4 *out, uint4 *out2) {
    using B = BrickOf<KIND>;
    const uint64_t id = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (id >= (uint64_t)n_x * n_y * n_z) return;
    const uint32_t id32 = (uint32_t)id;                                // below 2^32: 512 GiB of lines
    const uint32_t gz = id32 % n_z, gy = (id32 / n_z) % n_y, gx = id32 / n_z / n_y;
    uint32_t w[32] = {}, w2[KIND == REC_F32_PAIR ? 32 : 1] = {};
    #pragma unroll
    for (int x = 0; x < B::bx; x++)
        #pragma unroll
        for (int y = 0; y < B::by; y++) {
            const uint32_t ix = gx * B::bx + x, iy = gy * B::by + y;
            if (ix >= nx || iy >= ny) continue;
            const uint64_t row = ((uint64_t)ix * ny + iy) * nz;
            #pragma unroll
            for (int z = 0; z < B::bz; z++) {
                const uint32_t iz = gz * B::bz + z;
                if (iz >= nz) continue;
                const uint32_t lab = mask[row + iz];
                const float f = KIND != REC_NONE && field ? field[row + iz] : 0.f;
                const int j = (x * B::by + y) * B::bz + z;
                if (KIND == REC_F32) { w[2 * j] = __float_as_uint(f); w[2 * j + 1] = lab; }
                else if (KIND == REC_NONE) w[j] = lab << 16;
                else if (KIND == REC_F32_PAIR) {
                    put_bytes(w, 5 * j, lab, 1); put_bytes(w, 5 * j + 1, __float_as_uint(f), 4);
                    put_bytes(w2, j, lab, 1); w2[kSoaF32.nvox / 4 + j] = __float_as_uint(f);
                }
                else { put_bytes(w, 3 * j, lab, 1); put_bytes(w, 3 * j + 1, field16<KIND>(f, inv_scale), 2); }
            }
        }
    constexpr bool kPacked = KIND != REC_F32 && KIND != REC_NONE;
    const uint64_t line = kPacked ? pack_line(gx, gy, gz, nb_y, nb_z, sup) : ((uint64_t)gx * nb_y + gy) * nb_z + gz;
    #pragma unroll
    for (int k = 0; k < 8; k++) out[line * 8 + k] = make_uint4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
    if constexpr (KIND == REC_F32_PAIR) {
        #pragma unroll
        for (int k = 0; k < 8; k++) out2[line * 8 + k] = make_uint4(w2[4 * k], w2[4 * k + 1], w2[4 * k + 2], w2[4 * k + 3]);
    }
}

template <int KIND>
hipError_t launch_bricks(const uint8_t *mask, const float *field, uint64_t nx, uint64_t ny, uint64_t nz, float inv_scale,
                         void *out, hipStream_t s, void *out2 = nullptr) {
    using B = BrickOf<KIND>;
    uint64_t n_x, n_y, n_z, nb_y, nb_z;
    bool sup = false;
    if (KIND == REC_F32 || KIND == REC_NONE) {
        n_x = (nx + B::bx - 1) / B::bx;
        nb_y = n_y = (ny + B::by - 1) / B::by;
        nb_z = n_z = (nz + B::bz - 1) / B::bz;
    } else {
        const PackShape &S = BrickOf<KIND>::k16 ? kPack16 : kPackF32;
        sup = pack_super(nx, ny, nz, S);
        nb_y = pack_pitch_y(ny, S, sup); nb_z = pack_pitch_z(nz, S, sup);
        n_x = pack_super_count(nx, S.bx, sup ? kSuper.sx : 1) * (sup ? kSuper.sx : 1);
        n_y = nb_y * (sup ? kSuper.sy : 1);
        n_z = nb_z * (sup ? kSuper.sz : 1);
    }
    const uint64_t lines = n_x * n_y * n_z;
    if (lines == 0) return hipSuccess;
    if (lines >= (1ull << 32)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(bricks_kernel<KIND>, dim3((unsigned)((lines + 255) / 256)), dim3(256), 0, s, mask, field,
                       (uint32_t)nx, (uint32_t)ny, (uint32_t)nz, (uint32_t)n_x, (uint32_t)n_y, (uint32_t)n_z, nb_y, nb_z,
                       sup, inv_scale, (uint4 *)out, (uint4 *)out2);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_f32_records(const uint8_t *mask, const float *field, uint64_t nx, uint64_t ny, uint64_t nz,
                              void *packed, void *soa, hipStream_t s) {
    return launch_bricks<REC_F32_PAIR>(mask, field, nx, ny, nz, 1.f, packed, s, soa);
}

hipError_t launch_phantom_stats(const uint8_t *mask, const float *field, uint64_t n, uint32_t *stats,
                                hipStream_t s) {
    if (n == 0) return hipSuccess;
    const uint64_t blocks = (n / 16 + kStatsThreads) / kStatsThreads;
    hipLaunchKernelGGL(stats_kernel, dim3((unsigned)(blocks < kStatsBlocks ? blocks : kStatsBlocks)), dim3(kStatsThreads), 0,
                       s, mask, field, n, stats);
    return hipGetLastError();
}

hipError_t launch_records(const uint8_t *mask, const float *field, uint64_t nx, uint64_t ny, uint64_t nz, int kind,
                          float inv_scale, void *out, hipStream_t s) {
    switch (kind) {
    case REC_F32:  return launch_bricks<REC_F32>(mask, field, nx, ny, nz, inv_scale, out, s);
    case REC_F16:  return launch_bricks<REC_F16>(mask, field, nx, ny, nz, inv_scale, out, s);
    case REC_BF16: return launch_bricks<REC_BF16>(mask, field, nx, ny, nz, inv_scale, out, s);
    case REC_NONE: return launch_bricks<REC_NONE>(mask, field, nx, ny, nz, inv_scale, out, s);
    case REC_Q16:  return launch_bricks<REC_Q16>(mask, field, nx, ny, nz, inv_scale, out, s);
    default:       return hipErrorInvalidValue;
    }
}

}  // namespace sw

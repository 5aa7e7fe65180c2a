// walk_prod.hpp -- the production walk's step loop for scans of one TR and for
// recorded trajectories (Philox draws, float voxel-unit positions).  Included by
// walk_impl.hpp, which holds the records, lookups, phases and rotations it is
// made of.
//
// What bounds it: few waves per SIMD (small launches) leave a wave alone with its
// instruction stream, about 4 cycles an instruction and 20 to 40 more wherever the
// scalar unit waits for a vector comparison or a branch is taken; many waves
// (batches) share the SIMD's issue slots.  Both gain from a shorter stream, so
// against the general loop (walk_spin) this one
// - counts attempts on the scalar unit where they are uniform, with the two draw
//   products that then are uniform too, and keeps the round keys in scalar
//   registers (with the rest, 87.5 instead of 94.4 VALU instructions a wave-step on the
//   FoV sweep's FP32 batch);
// - holds the gathered record in place: a lane that stays in its voxel keeps the
//   one it has, so neither record index nor field is selected per step;
// - reads T1 and T2 at events instead of at every change of tissue;
// - decides a crossing between closed tissues without the probability table;
// - reads the arguments that rare blocks need when they run, so that the step
//   loop's scalar registers hold no more than it uses.
// Measured, start of this change against now: 200 k spins, 1201 time points,
// permeable, FP64: 2.39 -> 1.91 ms; 12 phantoms, GRE/SE/PGSE, Kahan + int16 batch:
// 7.53 -> 7.21 ms; 64 tiles of the FoV sweep, FP32 batch: 120.4 -> 118.5 ms.  Where walls
// are met at nearly every step and a wave has a SIMD to itself, its longer rare blocks
// cost more than that (general_loop).
#pragma once

namespace sw {
namespace {

// Launch arguments through the constant address space: reads are scalar loads
// wherever they stand, also after the walk's own stores.
using ArgsPtr = const __attribute__((address_space(4))) WalkArgs *;
using ViewPtr = const __attribute__((address_space(4))) WalkView *;

// The arguments for a block that runs rarely: the empty statement keeps the
// compiler from reading its fields ahead of the step loop, where they would
// hold scalar registers (and spill) for the whole walk.
template <class P> __device__ __forceinline__ P cold(P p) {
    asm volatile("" : "+s"(p));
    return p;
}

// Field of view v of a fused walk: view 0 is the WalkArgs fields, views 1.. are xv[v - 1].
#define SW_VIEW(a, xv, v, name) ((v) == 0 ? (a)->name : (xv)[(v) - 1].name)

// What the step loop and its rarer blocks (walls, changes of tissue) read of the
// arguments, as scalar registers.
struct Hot {
    uint32_t n[3], n_sub, max_iter;
    uint32_t tis;                    // where the tissue tables stand in LDS, in words
    uint32_t flags;
};
enum : uint32_t { HOT_TISSUE_LDS = 1, HOT_CLOSED = 2, HOT_CROSS = 4 };

// Per-tissue values of the production walk: the workgroup's LDS copies after the
// per-axis tables (tissue_lds, 32-bit mode), else the global tables.
// LDS layout: crossing probabilities [n_sub^2], T1 [n_sub], T2 [n_sub], step sizes
// [3 n_sub] in voxels (PosVox::Step).
template <bool IDX32> struct ProdTissue {
    __device__ static float *tab(ArgsPtr a) {
        return reinterpret_cast<float *>(axis_tab) + (uint32_t)(a->nx + a->ny + a->nz);
    }
    // Copies the tables; every thread of the workgroup calls it, and the caller
    // synchronises the workgroup before the first walk.
    __device__ static void fill(ArgsPtr a) {
        if (!IDX32 || !a->tissue_lds) return;
        float *t = tab(a);
        const uint32_t n = a->n_sub, nn = n * n;
        for (uint32_t i = threadIdx.x; i < nn; i += blockDim.x) t[i] = a->pXY[i];
        for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
            t[nn + i] = a->T1s[i];
            t[nn + n + i] = a->T2s[i];
            step_of(a, i, t + nn + 2 * n + 3 * i);
        }
    }
    __device__ static void step_of(ArgsPtr a, uint32_t ts, float *d) {
        const double D = gload<double>(a->diffusivity, (uint64_t)ts * 8) * kDrawScale;
        d[0] = D != 0. ? (float)(D * a->s2g[0]) : __builtin_nanf("");
        d[1] = (float)(D * a->s2g[1]);
        d[2] = (float)(D * a->s2g[2]);
    }
    __device__ static float pxy(ArgsPtr a, const Hot &h, uint32_t from, uint32_t to) {   // kernels.cu:155
        const uint32_t i = from * h.n_sub + to;
        if (IDX32 && (h.flags & HOT_TISSUE_LDS)) return reinterpret_cast<const float *>(axis_tab)[h.tis + i];
        const float v = gload<float>(a->pXY, (uint64_t)i * 4);
        asm volatile("" ::);
        return v;
    }
    template <class R> __device__ static void relax(ArgsPtr a, uint32_t ts, R &T1, R &T2) {   // kernels.cu:167-168
        // Before the first accepted step T1 = T2 = 0 (kernels.cu:91), which only
        // a TR without time points can show.
        T1 = T2 = 0;
        if (a->n_timepoints == 0) return;
        if constexpr (sizeof(R) == 8) {
            T1 = gload<double>(a->T1d, (uint64_t)ts * 8);
            T2 = gload<double>(a->T2d, (uint64_t)ts * 8);
        } else {
            T1 = gload<float>(a->T1s, (uint64_t)ts * 4);
            T2 = gload<float>(a->T2s, (uint64_t)ts * 4);
        }
    }
    __device__ static void step(ArgsPtr a, const Hot &h, uint32_t ts, float d[3]) {      // kernels.cu:169
        if (IDX32 && (h.flags & HOT_TISSUE_LDS)) {
            const float *t = reinterpret_cast<const float *>(axis_tab) + h.tis + h.n_sub * (h.n_sub + 2) + 3 * ts;
            d[0] = t[0]; d[1] = t[1]; d[2] = t[2];
            return;
        }
        step_of(a, ts, d);
    }
};

// The events of one TR: next times of each kind and where their tables stand.
struct Events {
    uint32_t rf_i, te_i, dp_i, gr_i, next_rf, next_te, next_dp, next_gr, next, old_tp;
    __device__ void start(ArgsPtr a, bool last) {                                   // kernels.cu:123-126
        rf_i = 1; te_i = dp_i = gr_i = 0; old_tp = 0;
        next_rf = (a->n_rf > 1) ? (uint32_t)a->rf[1].t : kNever;
        next_te = (last && a->n_te > 0) ? (uint32_t)a->TE_t[0] : kNever;
        next_dp = (a->n_deph > 0) ? (uint32_t)a->deph_t[0] : kNever;
        next_gr = (a->n_grad > 0) ? (uint32_t)a->grad_t[0] : kNever;
        next = next_event(next_rf, next_te, next_dp, next_gr);
    }
};

// The events of time point tp of a spin in tissue ts at x (kernels.cu:175-215).
// T1 and T2 are read here, not when the spin changes tissue: events are rarer.
template <class Phase, int NV>
__device__ __forceinline__ void prod_events(ArgsPtr a, ViewPtr xv, Events &ev, uint32_t tp, uint32_t ts, uint32_t li,
                                            const float x[3], typename Phase::R m[][3], Phase *ph) {
    using R = typename Phase::R;
    if (tp == ev.next_dp) {                                            // :175-178
        const uint32_t spin = a->spin_offset + li;
        #pragma unroll
        for (int v = 0; v < NV; v++) {
            const float dd = SW_VIEW(a, xv, v, deph_deg)[ev.dp_i];
            if (sizeof(R) == 8) ph[v].add((R)((double)spin * dd / (double)a->n_spins_total));
            else                ph[v].add((R)((float)spin * dd / (float)a->n_spins_total));
        }
        ++ev.dp_i;
        ev.next_dp = (ev.dp_i < a->n_deph) ? (uint32_t)a->deph_t[ev.dp_i] : kNever;
    }
    if (tp == ev.next_gr) {                                            // :181-187
        #pragma unroll
        for (int v = 0; v < NV; v++) {
            const float gs = SW_VIEW(a, xv, v, gradient_scale);
            const float Gx = SW_VIEW(a, xv, v, gx)[ev.gr_i] * gs;
            const float Gy = SW_VIEW(a, xv, v, gy)[ev.gr_i] * gs;
            const float Gz = SW_VIEW(a, xv, v, gz)[ev.gr_i] * gs;
            PosVox::add_grad(ph[v], *a, Gx, Gy, Gz, x);
        }
        ++ev.gr_i;
        ev.next_gr = (ev.gr_i < a->n_grad) ? (uint32_t)a->grad_t[ev.gr_i] : kNever;
    }
    if (tp == ev.next_rf) {                                            // :190-199
        R T1, T2;
        ProdTissue<false>::relax(a, ts, T1, T2);
        const R te = (R)((tp - ev.old_tp) * (uint32_t)a->timestep_us * 1e-6);
        #pragma unroll
        for (int v = 0; v < NV; v++) {
            dephase_relax(m[v], ph[v].angle(), T1, T2, te);
            const RfPulse *p = SW_VIEW(a, xv, v, rf) + ev.rf_i;
            if (sizeof(R) == 8) rot_apply<R>(p->kind_d, (R)p->sd, (R)p->cd, (R)p->spd, (R)p->cpd, m[v]);
            else                rot_apply<R>(p->kind, (R)p->s, (R)p->c, (R)p->sp, (R)p->cp, m[v]);
            ph[v].reset();
        }
        ev.old_tp = tp;
        ++ev.rf_i;
        ev.next_rf = (ev.rf_i < a->n_rf) ? (uint32_t)a->rf[ev.rf_i].t : kNever;
    }
    if (tp == ev.next_te) {                                            // :202-215
        R T1, T2;
        ProdTissue<false>::relax(a, ts, T1, T2);
        const R te = (R)((tp - ev.old_tp) * (uint32_t)a->timestep_us * 1e-6);
        const uint64_t o = (uint64_t)li * a->n_te + ev.te_i;
        #pragma unroll
        for (int v = 0; v < NV; v++) {
            dephase_relax(m[v], ph[v].angle(), T1, T2, te);
            R *M1 = (R *)SW_VIEW(a, xv, v, M1);
            M1[3 * o + 0] = m[v][0]; M1[3 * o + 1] = m[v][1]; M1[3 * o + 2] = m[v][2];
            SW_VIEW(a, xv, v, T)[o] = (uint8_t)ts;
            ph[v].reset();
        }
        ev.old_tp = tp;
        ++ev.te_i;
        ev.next_te = (ev.te_i < a->n_te) ? (uint32_t)a->TE_t[ev.te_i] : kNever;
    }
    ev.next = next_event(ev.next_rf, ev.next_te, ev.next_dp, ev.next_gr);
}

// The factors of the field a record holds (Rec::field), kept in scalar registers.
struct FieldFactor { float t2d, h2d; double t2d_f64; };

// d = s in the lanes that run this, in d's own register.  A plain assignment in
// a rare block would be a merge of two values that the compiler places in a
// third register, with a copy on the common path of every step.
template <class T> __device__ __forceinline__ void put(T &d, T s) {
    static_assert(sizeof(T) == 4, "one register");
    asm volatile("v_mov_b32 %0, %1" : "+v"(d) : "v"(s));
}

// The draws of attempt `att` of the spin whose first-round product is (m_hi, m_lo).
// UNI: att is the same in every lane of the wave, so the products of the first
// round and one of the second are scalar (philox4x32_10_pre's rounds 1 to 3 with
// the uniform words folded; the same words as there).
struct ProdDraw { float x, y, z; uint32_t u; };
template <bool UNI>
__device__ __forceinline__ ProdDraw prod_draw(uint64_t att, uint32_t m_hi, uint32_t m_lo, uint32_t k0, uint32_t k1) {
    U32x4 r;
    if constexpr (UNI) r = philox4x32_10_uniform(att, m_hi, m_lo, k0, k1);
    else r = philox4x32_10_pre((uint32_t)att, (uint32_t)(att >> 32), m_hi, m_lo, 0u, k0, k1);
    ProdDraw q;
    draw_bundle(r, q.x, q.y, q.z, q.u);
    return q;
}

// An attempt with some lane of the wave outside the FoV or in still tissue
// (PosVox::advance's checked path): corrects y and the subscripts i of its voxel.
// Returns false for a lane whose voxel the reference finds outside the volume.
template <class Rec, bool IDX32>
__device__ __forceinline__ bool prod_outside(ArgsPtr a, const Hot &h, const float nf[3], const float q[3], const float step[3], const float x[3],
                                             float y[3], uint32_t i[3]) {
    float z[3];
    if (step[0] == step[0]) {
        if (h.flags & HOT_CROSS) {
            for (int k = 0; k < 3; k++) z[k] = fix_axis_vox<true>(nf[k], q[k] * step[k], y[k]);
        } else {
            for (int k = 0; k < 3; k++) z[k] = fix_axis_vox<false>(nf[k], q[k] * step[k], y[k]);
        }
    } else {
        for (int k = 0; k < 3; k++) z[k] = x[k];                       // a spin that does not move stays put
    }
    uint32_t s[3] = {cvt_i32_sat_f(z[0]), cvt_i32_sat_f(z[1]), cvt_i32_sat_f(z[2])};
    bool ok = s[0] < h.n[0] && s[1] < h.n[1] && s[2] < h.n[2];
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!ok) != 0, 0)) {
        if (!ok) ok = wrapped_subscripts(*cold(a), (double)z[0], (double)z[1], (double)z[2], s);
    }
    for (int k = 0; k < 3; k++) {
        put(y[k], ok ? z[k] : x[k]);
        put(i[k], ok ? s[k] : 0u);                                     // a lost lane reads record 0
    }
    return ok;
}

enum : int { TRAJ_NONE = 0, TRAJ_DIRECT = 1, TRAJ_STAGED = 2 };

// Recorded positions on their way to XYZ1.  Each spin has a row of its own, so a
// store per step is 64 pieces of 12 bytes in 64 lines, and the L2 sends nearly each of
// them on by itself: 63 M write requests, 3.3 GB, for the 0.96 GB of 1e5 spins and 800
// steps, which is what such walks wait for.  So a lane keeps its words in a ring of two
// 64-byte sectors in LDS, and when some lane's ring is full the wave writes the whole
// sectors: four lanes exchange pieces, so that each store of the four is one lane's
// sector, aligned.  The ends of a row go word by word.  200^3: 1e5 spins of 800 steps 1.41
// -> 0.85 ms, 2e5 of 400 1.99 -> 0.85 ms, 5e5 of 200 1.96 -> 0.96 ms.  Only from
// kStageSpins on: with fewer rows open the L2 gathers the pieces itself, and the ring
// costs more than it saves (5e4 spins 0.65 ms without, 0.74 with; 6.5e4 0.75 and 0.75;
// 8e4 1.21 and 0.82).  Compiled for 4 waves a SIMD, which is what the rings leave room for
// and where nothing of the step loop spills.
// A lane's words: absolute word w (row words from the row's 64-byte boundary) in
// piece w / 4 mod 8, the pieces 64 lanes apart.
typedef uint32_t Piece __attribute__((ext_vector_type(4)));
typedef uint32_t PieceOut __attribute__((ext_vector_type(4), aligned(4)));
template <bool IDX32> struct Recorder {
    uint32_t ring;               // this lane's place in the wave's ring, axis_tab[ring ..]
    uint32_t first, w, done;     // words: the row's first, the next, the first not yet written
    float vs[3];
    __device__ Recorder(ArgsPtr a, ViewPtr, uint64_t xoff)
        : ring(stage_ring<IDX32>(*a) + 4 * (threadIdx.x & 63)), vs{a->vsf[0], a->vsf[1], a->vsf[2]} {
        first = w = done = (uint32_t)((uintptr_t)(a->XYZ1 + xoff) / 4) & 15u;
    }
    __device__ bool any() const { return w != first; }
    // word i's place
    __device__ uint32_t place(uint32_t i) const { return ring + (i & 28u) * 64 + (i & 3u); }
    template <int NV> __device__ void add(ArgsPtr a, ViewPtr xv, uint64_t xoff, const float y[3]) {
        for (uint32_t i = 0; i < 3; i++) axis_tab[place(w + i)] = __float_as_uint(y[i] * vs[i]);
        w += 3;
    }
    // Called by every lane of the wave that still walks.
    template <int NV> __device__ void spill(ArgsPtr a, ViewPtr xv, uint64_t xoff) {
        if (__builtin_amdgcn_ballot_w64(w - (done & ~15u) > 29) != 0) write<NV>(a, xv, xoff);
    }
    template <int NV> __device__ void write(ArgsPtr a, ViewPtr xv, uint64_t xoff) {
        // a row's first words, up to its first 64-byte boundary
        if (done & 15u && w >= 16) words<NV>(a, xv, xoff, 16);
        const bool full = w - done >= 16 && !(done & 15u);
        __builtin_amdgcn_wave_barrier();                              // other lanes read what this one wrote
        const uint64_t m = __builtin_amdgcn_ballot_w64(true);
        const uint64_t q = m & m >> 1 & m >> 2 & m >> 3 & 0x1111111111111111ull;
        const uint64_t off = xoff + done - first;                     // of the sector in XYZ1
        if (q * 15 == m) {                                            // whole quads of lanes
            const uint32_t st = full ? (done & 16u) | 1u : 0u;
            exchange<0, NV>(a, xv, off, st);
            exchange<1, NV>(a, xv, off, st);
            exchange<2, NV>(a, xv, off, st);
            exchange<3, NV>(a, xv, off, st);
        } else if (full) {
            #pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                const Piece p = *(const Piece *)(axis_tab + ring + ((done & 16u) + 4 * j) * 64);
                #pragma unroll
                for (int v = 0; v < NV; v++) *(PieceOut *)(SW_VIEW(a, xv, v, XYZ1) + off + 4 * j) = p;
            }
        }
        if (full) done += 16;
    }
    // The sector of the quad's lane K: its lanes store a piece each.
    template <int K, int NV> __device__ void exchange(ArgsPtr a, ViewPtr xv, uint64_t off, uint32_t st) {
        const auto of_k = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)x, K * 0x55, 0xF, 0xF, true); };
        const uint64_t o = (uint64_t)of_k((uint32_t)(off >> 32)) << 32 | of_k((uint32_t)off);
        const uint32_t j4 = 4 * (threadIdx.x & 3);
        st = of_k(st);
        if (st) {
            const Piece p = *(const Piece *)(axis_tab + ring + ((st & 16u) + j4) * 64 + 4 * K - j4);
            #pragma unroll
            for (int v = 0; v < NV; v++) *(PieceOut *)(SW_VIEW(a, xv, v, XYZ1) + o + j4) = p;
        }
    }
    template <int NV> __device__ void finish(ArgsPtr a, ViewPtr xv, uint64_t xoff) { words<NV>(a, xv, xoff, w); }
    // this lane's words up to `end`, one by one
    template <int NV> __device__ void words(ArgsPtr a, ViewPtr xv, uint64_t xoff, uint32_t end) {
        for (; done < end; done++) {
            const float f = __uint_as_float(axis_tab[place(done)]);
            #pragma unroll
            for (int v = 0; v < NV; v++) (SW_VIEW(a, xv, v, XYZ1) + xoff)[done - first] = f;
        }
    }
};

// Recorded positions written as they come: few rows, or no room in LDS (WalkArgs::stage).
// A walk of its own instead of a branch per step: 2e4 spins 217 -> 210 us.
struct DirectRecorder {
    uint64_t at;                 // the next word of XYZ1
    float vs[3];
    bool some = false;
    __device__ DirectRecorder(ArgsPtr a, ViewPtr, uint64_t xoff) : at(xoff), vs{a->vsf[0], a->vsf[1], a->vsf[2]} {}
    __device__ bool any() const { return some; }
    template <int NV> __device__ void add(ArgsPtr a, ViewPtr xv, uint64_t, const float y[3]) {
        #pragma unroll
        for (int v = 0; v < NV; v++) {
            float *dst = SW_VIEW(a, xv, v, XYZ1) + at;
            for (int i = 0; i < 3; i++) dst[i] = y[i] * vs[i];
        }
        at += 3;
        some = true;
    }
    template <int NV> __device__ void spill(ArgsPtr, ViewPtr, uint64_t) {}
    template <int NV> __device__ void finish(ArgsPtr, ViewPtr, uint64_t) {}
};

// One spin.  ONE_TR: the scan has no dummy TRs, so every lane of the wave that
// still walks is at the same attempt, and the attempt counter and the draw's
// first products run on the scalar unit.
template <class Rec, class Phase, bool IDX32, int NV, bool ONE_TR, int TRAJ>
__device__ __forceinline__ int walk_spin_prod(ArgsPtr a, ViewPtr xv, uint32_t li, uint64_t &n_acc, uint32_t &n_rej) {
    using R = typename Phase::R;
    using RI = RecIdx<IDX32>;
    using Tis = ProdTissue<IDX32>;
    const uint32_t k0 = (uint32_t)a->seed, k1 = (uint32_t)(a->seed >> 32);
    const uint64_t first = (uint64_t)kPhiloxM1 * (a->spin_offset + li);
    const uint32_t m_hi = (uint32_t)(first >> 32), m_lo = (uint32_t)first;
    const uint64_t xoff = 3 * (uint64_t)li * a->traj_len;              // this spin's XYZ1 slots
    float x[3];
    R m[NV][3];
    for (int i = 0; i < 3; i++) {                                      // kernels.cu:95-99
        const float x0 = a->XYZ0[3 * (uint64_t)li + i] * a->xyz_scale;
        x[i] = PosVox::start(*a, x0, i);
        #pragma unroll
        for (int v = 0; v < NV; v++) m[v][i] = (R)a->M0[3 * (uint64_t)li + i];
    }
    Hot h;
    h.n[0] = (uint32_t)a->nx; h.n[1] = (uint32_t)a->ny; h.n[2] = (uint32_t)a->nz;
    h.n_sub = a->n_sub;
    h.tis = h.n[0] + h.n[1] + h.n[2];
    h.max_iter = (uint32_t)(a->max_iterations >> 32) ? 0xFFFFFFFFu : (uint32_t)a->max_iterations;
    // HOT_TISSUE_LDS, HOT_CLOSED, HOT_CROSS of arguments that are 0 or 1
    h.flags = (IDX32 ? a->tissue_lds : 0u) | a->closed << 1 | (uint32_t)a->cross_fov << 2;
    int st = ST_OK;
    bool recorded = false;
    uint32_t d = 0, tp = 0;
    const Vox<IDX32> vx = PosVox::find<Rec, IDX32>(*a, x);             // kernels.cu:102
    if (!vx.ok) {                                                      // the reference reads out of bounds here
        st = ST_LOST;
    } else {
        typename Rec::T raw = rec_load<Rec, IDX32>(a->rec, vx.rec);
        uint32_t ts = Rec::label(raw);                                 // :103
        float step[3];
        [[maybe_unused]] typename std::conditional<TRAJ == TRAJ_STAGED, Recorder<IDX32>, DirectRecorder>::type rec1(a, xv, xoff);
        uint64_t att = 0;
        uint32_t itr = 0, last_rej = 0;
        ProdDraw q = prod_draw<ONE_TR>(0, m_hi, m_lo, k0, k1);
        Phase ph[NV];
        const uint32_t n_tp = a->n_timepoints;
        const void *const recs = a->rec;
        const float nf[3] = {a->nf[0], a->nf[1], a->nf[2]};
        FieldFactor ff = {a->t2d, a->h2d, a->t2d_f64};
        asm volatile("" : "+s"(ff.t2d), "+s"(ff.h2d), "+s"(ff.t2d_f64));
        Tis::step(a, h, ts, step);                                     // :104
        for (d = 0;; ++d) {                                            // :107
            const bool last = ONE_TR || d == a->n_dummy;
            Events ev;
            {                                                          // :110-120 excitation
                const ArgsPtr c = cold(a);
                #pragma unroll
                for (int v = 0; v < NV; v++) {
                    const Excitation *e = SW_VIEW(c, xv, v, exc) + d;
                    if (sizeof(R) == 8)
                        rot_apply<R>(e->kind_d, (R)SW_VIEW(c, xv, v, exc_sd), (R)SW_VIEW(c, xv, v, exc_cd), (R)e->spd,
                                     (R)e->cpd, m[v]);
                    else
                        rot_apply<R>(e->kind, (R)SW_VIEW(c, xv, v, exc_s), (R)SW_VIEW(c, xv, v, exc_c), (R)e->sp,
                                     (R)e->cp, m[v]);
                    ph[v].reset();
                }
                ev.start(c, last);
            }
            RI rec_old = ~(RI)0;                                       // no voxel: the first gather is made
            tp = 0;
            while (tp < n_tp) {                                        // :128
                float y[3] = {__builtin_fmaf(q.x, step[0], x[0]), __builtin_fmaf(q.y, step[1], x[1]),
                              __builtin_fmaf(q.z, step[2], x[2])};
                uint32_t i[3] = {cvt_i32_sat_f(y[0]), cvt_i32_sat_f(y[1]), cvt_i32_sat_f(y[2])};
                const uint32_t out = maybe_outside_f(y[0], nf[0]) | maybe_outside_f(y[1], nf[1]) |
                                     maybe_outside_f(y[2], nf[2]);     // a NaN step is outside
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(out != 0) != 0, 0)) {
                    const float qq[3] = {q.x, q.y, q.z};
                    if (!prod_outside<Rec, IDX32>(a, h, nf, qq, step, x, y, i)) {   // :141-147: lost
                        put(tp, tp | kParked);
                        put(ts, ~0u);                                  // no label: seen by the test below
                    }
                }
                const RI rec = (RI)record_of<Rec, IDX32>(*a, i[0], i[1], i[2]);
                // One gather brings label and field.  Lanes still in their voxel keep
                // the record they hold, whose label is their tissue's.
                if (rec != rec_old) raw = rec_load<Rec, IDX32>(recs, rec);
                const uint32_t u = q.u;
                ++att;                                                 // the next attempt's draws while it flies
                q = prod_draw<ONE_TR>(att, m_hi, m_lo, k0, k1);
                after_draws(raw, q.x, q.y, q.z);
                rec_old = rec;
                bool acc = true;                                       // the attempt becomes a step
                const uint32_t to = Rec::label(raw);                   // :152
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(to != ts) != 0, 0)) {
                    if (to != ts) {                                    // :153-163
                        bool in = false;
                        if ((int32_t)tp >= 0) {                        // not lost
                            if (!(h.flags & HOT_CLOSED)) in = !(u24_to_unit(u) >= Tis::pxy(a, h, ts, to));
                            if (!in) {
                                ++n_rej;
                                // rejections in a row: consecutive attempts
                                if (last_rej + 1 != (uint32_t)att) itr = 0;
                                last_rej = (uint32_t)att;
                                if (itr++ > h.max_iter) put(tp, tp | kParked);
                            }
                        }
                        if (in) {
                            put(ts, to);
                            Tis::step(a, h, ts, step);
                        } else {
                            put(y[0], x[0]); put(y[1], x[1]); put(y[2], x[2]);
                            rec_old = ~(RI)0;                          // the gathered record is not the spin's
                            acc = false;
                        }
                    }
                }
                if (acc) {
                    const R f = Rec::template field<R>(ff, raw);       // :166
                    #pragma unroll
                    for (int v = 0; v < NV; v++) ph[v].add(f);         // :171
                    if (__builtin_expect(tp == ev.next, 0))
                        prod_events<Phase, NV>(cold(a), xv, ev, tp, ts, li, y, m, ph);
                    if constexpr (TRAJ) rec1.template add<NV>(a, xv, xoff, y);   // :218-221
                    ++tp;
                }
                x[0] = y[0]; x[1] = y[1]; x[2] = y[2];
                if constexpr (TRAJ) rec1.template spill<NV>(a, xv, xoff);
            }
            if (tp & kParked) { st = ST_LOST; tp &= ~kParked; break; }
            {
                const ArgsPtr c = cold(a);
                R T1, T2;
                Tis::relax(c, ts, T1, T2);
                const R te = (R)((tp - ev.old_tp) * (uint32_t)c->timestep_us * 1e-6);   // :226-231
                #pragma unroll
                for (int v = 0; v < NV; v++) dephase_relax(m[v], ph[v].angle(), T1, T2, te);
            }
            if (last) { ++d; tp = 0; break; }                          // every TR done
        }
        if constexpr (TRAJ) {
            rec1.template finish<NV>(a, xv, xoff);                     // the row's last words, also of a lost spin
            recorded = rec1.any();
        }
    }
    // Without trajectories XYZ1 holds the last accepted position: the reference
    // stores every accepted position in place (kernels.cu:222-223), and a spin
    // that is lost keeps the one before.  Then the count of accepted steps.
    // With trajectories a spin without a step shows its start (kernels.cu:95-99).
    const ArgsPtr c = cold(a);
    if (!TRAJ || (!recorded && c->traj_len)) {
        #pragma unroll
        for (int v = 0; v < NV; v++)
            for (int i = 0; i < 3; i++)
                (SW_VIEW(c, xv, v, XYZ1) + xoff)[i] =
                    TRAJ ? c->XYZ0[3 * (uint64_t)li + i] * c->xyz_scale : PosVox::metres(*c, x[i], i);
    }
    n_acc += (uint64_t)d * c->n_timepoints + tp;
    return st;
}

// This lane walks the spins at positions t0 + k * blockDim.x, k = 0 .. spl-1, of
// the launch's visiting order, those below n_local, one after the other.
template <class Rec, class Phase, bool IDX32, int NV, bool ONE_TR, bool TRAJ>
__device__ __forceinline__ void prod_block(ArgsPtr a, ViewPtr xv, uint32_t n_views, uint32_t t0, uint32_t spl) {
    if (IDX32) {
        const uint32_t n_tab = (uint32_t)(a->nx + a->ny + a->nz);
        for (uint32_t i = threadIdx.x; i < n_tab; i += blockDim.x) axis_tab[i] = axis_entry<Rec>(*a, i);
        ProdTissue<IDX32>::fill(a);
        __syncthreads();
    }
    uint64_t n_acc = 0;
    uint32_t n_rej = 0, lost = 0;
    for (uint32_t k = 0; k < spl; k++) {
        const uint32_t t = t0 + k * blockDim.x;
        if (t >= a->n_local) continue;
        const uint32_t li = a->order ? a->order[t] : t;
        int st;
        if constexpr (!TRAJ) st = walk_spin_prod<Rec, Phase, IDX32, NV, ONE_TR, TRAJ_NONE>(a, xv, li, n_acc, n_rej);
        else if (a->stage) st = walk_spin_prod<Rec, Phase, IDX32, NV, ONE_TR, TRAJ_STAGED>(a, xv, li, n_acc, n_rej);
        else st = walk_spin_prod<Rec, Phase, IDX32, NV, ONE_TR, TRAJ_DIRECT>(a, xv, li, n_acc, n_rej);
        lost += st == ST_LOST;
    }
    const uint64_t s_acc = wave_sum_u64(n_acc), s_rej = wave_sum_u64(n_rej), s_lost = wave_sum_u64(lost);
    if ((threadIdx.x & 63) == 0) {
        #pragma unroll
        for (int v = 0; v < NV; v++) {                 // every view walked these steps
            unsigned long long *c = SW_VIEW(a, xv, v, counters);
            if (c && (v == 0 || (uint32_t)v < n_views)) {
                if (s_lost) atomicAdd(&c[0], (unsigned long long)s_lost);
                atomicAdd(&c[2], (unsigned long long)s_acc);
                atomicAdd(&c[3], (unsigned long long)(s_acc + s_rej));
            }
        }
    }
}

}  // namespace
}  // namespace sw

/* persist.h - persistent multi-frame tracer (device code, included by bhrt.hip).

   Workgroups stay resident and pull rays from per-frame work queues (one atomic counter per frame;
   queue entries are the rays of 8 x 8 pixel tiles, so the rays a wave takes at once are image
   neighbours). The tiles of a frame are queued in row order or in a given order (the launcher sorts
   them by their centre ray's impact parameter, or by its predicted length, longest first, so the
   rays that orbit the hole longest start first). Every `interval` integration steps a wave retires finished lanes (one ballot),
   writes their pixels, and refills the free lanes with new rays when at least `refill_min` lanes are
   free: lane 0 claims a contiguous range with one atomic add and each free lane takes the entry at
   its rank among the free lanes. A wave refills only from its current frame and moves to the next
   frame once its lanes are drained, so the frame parameters stay wave-uniform (scalar loads).
   Every wave exits when all frames are exhausted and its lanes are idle; each ray runs at most
   max_steps steps, so the grid always drains. With prio_age > 0 a wave that holds a ray older than
   prio_age steps raises its issue priority, so the longest rays run at their own latency instead
   of sharing the SIMD evenly with younger waves. What an entry means (which pixel and sample, where
   the finished ray is written) is a Work policy: frame batches, the tile interface's ray records,
   and the two passes of adaptive sampling. Launches of few radio rays take pair_body (below) instead. */
#pragma once
#include "../../include/bhrt.h"
#include "trace_fp64.h"
#include "trace_mixed.h"

namespace bhp {

constexpr int MAX_BLOCK = 256;   // largest workgroup of the persistent kernel
constexpr int NSTAT = 5;         // per-ray statistics summed per lane (steps, accepted, flow, escaped, FP64)

using bhd::RayResult;
using bhd::TraceParams;

struct BatchFrame {
    TraceParams P;         // scene + frame; P.w/P.h = frame size, P.spp = 1
    bhm32::MixedParams M;  // the frame's mixed-precision policy and emission constants
    unsigned int nentries; // queue entries of the frame
    int tiles_x;
    float4* out;           // W*H pixels (frame batches)
    unsigned int* order;   // queue position -> tile (null: row order)
};

__device__ __forceinline__ unsigned int queued_tile(const BatchFrame& F, unsigned int pos) {
    return F.order ? F.order[pos] : pos;
}

__device__ __forceinline__ void tile_pixel(int tiles_x, unsigned int tile, unsigned int within, int* px, int* py) {
    *px = (int)(tile % (unsigned)tiles_x) * 8 + (int)(within & 7u);
    *py = (int)(tile / (unsigned)tiles_x) * 8 + (int)(within >> 3);
}

/* Work mappings: entry e of frame f -> (pixel, sample index) and where a finished ray goes. RECORDS: the
   finished ray's coordinate time is part of the output.
   Entries of 64 consecutive indices are 8 x 8 pixel tiles, so a wave's rays are image neighbours. */

// Frame batches: one pixel-centre (or jittered sample 0) ray per pixel, written as a float4 pixel.
struct BatchWork {
    static constexpr bool RECORDS = false;
    const BatchFrame* frames;
    int n;
    __device__ __forceinline__ bool begin(int f, unsigned int e, int* px, int* py, int* s) const {
        tile_pixel(frames[f].tiles_x, queued_tile(frames[f], e >> 6), e & 63u, px, py);
        *s = 0;
        return *px < frames[f].P.w && *py < frames[f].P.h;
    }
    __device__ __forceinline__ void finish(int f, unsigned int e, const RayResult& r) const {
        int px, py;
        tile_pixel(frames[f].tiles_x, queued_tile(frames[f], e >> 6), e & 63u, &px, &py);
        frames[f].out[(size_t)py * frames[f].P.w + px] =
            make_float4((float)r.I[0], (float)r.I[1], (float)r.I[2], (float)r.I[3]);
    }
};

// Every per-ray output of a finished ray as the tile interface's record.
__device__ __forceinline__ void write_record(bh_ray_out* __restrict__ q, const RayResult& r) {
    for (int i = 0; i < 6; ++i) q->y[i] = r.y[i];
    q->th_inf = r.th_inf;
    q->ph_inf = r.ph_inf;
    q->I[0] = r.I[0]; q->I[1] = r.I[1]; q->I[2] = r.I[2]; q->I[3] = r.I[3];
    q->trans = r.trans;
    q->psi = r.psi;
    q->fate = r.fate;
    q->ncross = r.ncross;
    q->order = r.order;
    q->steps = r.steps;
    q->accepted = r.accepted;
    q->flow_steps = r.flow_steps;
    q->sky_u = r.sky_u;
    q->sky_v = r.sky_v;
}

// Ray records of a w x h region at (x0, y0) of a frame (the tile interface): P.w / P.h are the
// region's size and P.x0 / P.y0 its origin; one ray per pixel (centre, or jittered sample 0), its
// record at out[(py - y0) * w + (px - x0)].
struct RecordWork {
    static constexpr bool RECORDS = true;
    const BatchFrame* frames;   // one frame
    int n;
    bh_ray_out* out;
    __device__ __forceinline__ bool begin(int f, unsigned int e, int* px, int* py, int* s) const {
        const TraceParams& P = frames[f].P;
        int lx, ly;
        tile_pixel(frames[f].tiles_x, queued_tile(frames[f], e >> 6), e & 63u, &lx, &ly);
        *px = P.x0 + lx;
        *py = P.y0 + ly;
        *s = 0;
        return lx < P.w && ly < P.h;
    }
    __device__ __forceinline__ void finish(int f, unsigned int e, const RayResult& r) const {
        int lx, ly;
        tile_pixel(frames[f].tiles_x, queued_tile(frames[f], e >> 6), e & 63u, &lx, &ly);
        write_record(out + (size_t)ly * frames[f].P.w + lx, r);
    }
};

// First pass of adaptive sampling: samples 0..spp-1 of every pixel (entry = tile, sample, pixel in
// tile), each kept in FP64 at out[pixel * spp + sample].
struct SampleWork {
    static constexpr bool RECORDS = false;
    const BatchFrame* frames;   // one frame
    int n;
    int spp;
    double4* out;
    __device__ __forceinline__ bool begin(int f, unsigned int e, int* px, int* py, int* s) const {
        const unsigned int per_tile = 64u * (unsigned)spp, rem = e % per_tile;
        tile_pixel(frames[f].tiles_x, queued_tile(frames[f], e / per_tile), rem & 63u, px, py);
        *s = (int)(rem >> 6);
        return *px < frames[f].P.w && *py < frames[f].P.h;
    }
    __device__ __forceinline__ void finish(int f, unsigned int e, const RayResult& r) const {
        const unsigned int per_tile = 64u * (unsigned)spp, rem = e % per_tile;
        int px, py;
        tile_pixel(frames[f].tiles_x, queued_tile(frames[f], e / per_tile), rem & 63u, &px, &py);
        out[((size_t)py * frames[f].P.w + px) * spp + (rem >> 6)] = make_double4(r.I[0], r.I[1], r.I[2], r.I[3]);
    }
};

// Second pass: chunk g of the exclusive prefix sum `offsets` of per-pixel chunk counts belongs to
// the last pixel p with offsets[p] <= g; its 8 samples continue p's sequence at
// spp + 8 * (g - offsets[p]). Each sample is kept in FP64 at out[entry].
struct ChunkWork {
    static constexpr bool RECORDS = false;
    const BatchFrame* frames;   // one frame
    int n;
    int spp;
    int npix;
    const unsigned int* offsets;
    double4* out;
    __device__ __forceinline__ bool begin(int f, unsigned int e, int* px, int* py, int* s) const {
        const unsigned int g = e >> 3;
        int lo = 0, hi = npix;   // upper bound of g in offsets
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (offsets[mid] <= g) lo = mid + 1;
            else hi = mid;
        }
        const int p = lo - 1;
        const int W = frames[f].P.w;
        *px = p % W;
        *py = p / W;
        *s = spp + 8 * (int)(g - offsets[p]) + (int)(e & 7u);
        return true;
    }
    __device__ __forceinline__ void finish(int, unsigned int e, const RayResult& r) const {
        out[e] = make_double4(r.I[0], r.I[1], r.I[2], r.I[3]);
    }
};

template <int PREC, int RADIO, bool TIME>
struct Tracer;

template <int RADIO, bool TIME>
struct Tracer<BH_PREC_FP64, RADIO, TIME> {
    using State = bhd::RayState;
    static __device__ __forceinline__ void init(const TraceParams& P, const bhm32::MixedParams&, double x, double y,
                                                State& R) {
        bhd::ray_init<RADIO>(P, x, y, R);
    }
    static __device__ __forceinline__ void step(const TraceParams& P, const bhm32::MixedParams&, const TraceParams& F,
                                                const bhm32::MixedParams&, State& R) {
        bhd::ray_step<RADIO, TIME>(P, F, R);
    }
    template <bool SETTLE>
    static __device__ __forceinline__ bool move(const TraceParams& P, const bhm32::MixedParams&, State& R,
                                                bhd::StepSample& q) {
        return bhd::ray_move<RADIO, TIME, SETTLE>(P, R, q);
    }
    // whether the ray's last attempt counted as an FP64 one, and taking some back (here every attempt does, and
    // they are not counted apart)
    static __device__ __forceinline__ bool last_fp64(const State&) { return false; }
    static __device__ __forceinline__ void undo_fp64(State&, int) {}
    // what a ray's samples add up to, in the wave that evaluates them
    struct Sums {
        double acc0, acc1, acc2, acc3, trans, psi;
        bhd::Direction d;
        bool first;
    };
    static __device__ __forceinline__ void begin(Sums& S) {
        S = Sums{0.0, 0.0, 0.0, 0.0, 1.0, 0.0, bhd::Direction{0.0, 0.0, 0.0}, true};
    }
    static __device__ __forceinline__ bool add(const TraceParams& F, const bhm32::MixedParams&, double lam, double E,
                                               const bhd::StepSample& q, Sums& S) {
        if (S.first) S.d = bhd::direction_of(q.u0, q.phi0);
        S.first = false;
        double ang, dI, e;
        bhd::sample_eval<RADIO>(F, lam, E, q, S.d, &ang, &dI, &e);
        S.psi += ang;
        return q.flow && bhd::ray_absorb(S, (int)(S.psi * (1.0 / bhd::PI)), dI, e);
    }
    static __device__ __forceinline__ int result(const TraceParams& P, const State& R, RayResult& out) {
        bhd::ray_result(P, R, out);
        return out.steps;
    }
};

template <int RADIO, bool TIME>
struct Tracer<BH_PREC_MIXED, RADIO, TIME> {
    using State = bhm32::RayStateM;
    static __device__ __forceinline__ void init(const TraceParams& P, const bhm32::MixedParams& M, double x, double y,
                                                State& R) {
        bhm32::ray_init_m<RADIO>(P, M, x, y, R);
    }
    static __device__ __forceinline__ void step(const TraceParams& P, const bhm32::MixedParams& M, const TraceParams& F,
                                                const bhm32::MixedParams& FM, State& R) {
        bhm32::ray_step_m<RADIO, TIME>(P, M, F, FM, R);
    }
    template <bool SETTLE>
    static __device__ __forceinline__ bool move(const TraceParams& P, const bhm32::MixedParams& M, State& R,
                                                bhd::StepSample& q) {
        return bhm32::ray_move_m<RADIO, TIME, SETTLE>(P, M, R, q);
    }
    static __device__ __forceinline__ bool last_fp64(const State& R) { return !R.k1_f32; }
    static __device__ __forceinline__ void undo_fp64(State& R, int n) { R.fp64_attempts -= n; }
    struct Sums {
        double acc0, acc1, acc2, acc3, trans;
        float psi;
        bhm32::TurbCache tc;
    };
    static __device__ __forceinline__ void begin(Sums& S) {
        S.acc0 = S.acc1 = S.acc2 = S.acc3 = 0.0;
        S.trans = 1.0;
        S.psi = 0.f;
        S.tc.v = bhm32::Corners{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        S.tc.key = ~0u;
    }
    static __device__ __forceinline__ bool add(const TraceParams& F, const bhm32::MixedParams& FM, double lam, double E,
                                               const bhd::StepSample& q, Sums& S) {
        float ang;
        bool emits;
        double dI, e;
        bhm32::sample_eval_m<RADIO>(F, FM, lam, E, q, S.tc, &ang, &emits, &dI, &e);
        S.psi += ang;
        return emits && bhd::ray_absorb(S, (int)(S.psi * 0.31830988618379067f), dI, e);
    }
    static __device__ __forceinline__ int result(const TraceParams& P, const State& R, RayResult& out) {
        return bhm32::ray_result_m(P, R, out);
    }
};

// The refill of persist_body (below, where it stands in the loop: as a function it costs that kernel registers)
// for pair_body.
template <class T, class Work>
__device__ __forceinline__ void refill(const Work& Wk, unsigned int* __restrict__ queue, int refill_min, int* cur,
                                       bool* active, unsigned int* ent, typename T::State& R) {
    const int lane = threadIdx.x & 63;
    const unsigned long long freem = __ballot(!*active);
    const int nfree = __popcll(freem);
    if (nfree >= refill_min || nfree == 64) {
        while (*cur < Wk.n) {
            const unsigned int n = Wk.frames[*cur].nentries;
            unsigned int base = 0;
            if (lane == 0) {
                // read before adding, so an exhausted counter grows by at most one claim per wave
                base = __hip_atomic_load(&queue[*cur], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (base < n) base = atomicAdd(&queue[*cur], (unsigned int)nfree);
            }
            base = __builtin_amdgcn_readfirstlane(__shfl(base, 0, 64));
            if (base < n) {
                if (!*active) {
                    const unsigned int rank = (unsigned int)__popcll(freem & ((1ull << lane) - 1ull));
                    const unsigned int e = base + rank;
                    int px, py, s = 0;
                    if (e < n && Wk.begin(*cur, e, &px, &py, &s)) {
                        const TraceParams& P = Wk.frames[*cur].P;
                        double ox, oy;
                        bhd::sample_offsets(P, px, py, s, &ox, &oy);
                        T::init(P, Wk.frames[*cur].M, ox, oy, R);
                        *ent = e;
                        *active = true;
                    }
                }
                break;
            }
            if (nfree == 64) {
                ++*cur;   // this frame's queue is empty and the wave is idle: next frame
                continue;
            }
            break;   // tail of the frame: keep stepping the live lanes
        }
    }
}

template <int PREC, int RADIO, bool TIME, class Work>
__device__ __forceinline__ void persist_body(const Work& Wk, unsigned int* __restrict__ queue, int interval,
                                             int refill_min, int prio_age, double* flux_out,
                                             unsigned long long* cnt_out) {
    using T = Tracer<PREC, RADIO, TIME>;
    const BatchFrame* __restrict__ frames = Wk.frames;
    const int nframes = Wk.n;
    const int lane = threadIdx.x & 63;
    int cur = 0;   // the wave's frame (wave-uniform)
    bool active = false;
    unsigned int ent = 0;   // the lane's queue entry (the work mapping recovers pixel and sample)
    typename T::State R;
    // per-lane sums over the lane's finished rays, in the lane's own LDS slots (updated once per ray,
    // so they need no registers during the integration)
    __shared__ double s_flux[MAX_BLOCK];
    __shared__ unsigned long long s_stat[NSTAT][MAX_BLOCK];
    const int tid = threadIdx.x;
    s_flux[tid] = 0.0;
    for (int i = 0; i < NSTAT; ++i) s_stat[i][tid] = 0ull;
    for (;;) {
        // retire-and-refill
        const unsigned long long freem = __ballot(!active);
        const int nfree = __popcll(freem);
        if (nfree >= refill_min || nfree == 64) {
            while (cur < nframes) {
                const unsigned int n = frames[cur].nentries;
                unsigned int base = 0;
                if (lane == 0) {
                    // read before adding, so an exhausted counter grows by at most one claim per wave
                    base = __hip_atomic_load(&queue[cur], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (base < n) base = atomicAdd(&queue[cur], (unsigned int)nfree);
                }
                base = __builtin_amdgcn_readfirstlane(__shfl(base, 0, 64));
                if (base < n) {
                    if (!active) {
                        const unsigned int rank = (unsigned int)__popcll(freem & ((1ull << lane) - 1ull));
                        const unsigned int e = base + rank;
                        int px, py, s = 0;
                        if (e < n && Wk.begin(cur, e, &px, &py, &s)) {
                            const TraceParams& P = frames[cur].P;
                            double ox, oy;
                            bhd::sample_offsets(P, px, py, s, &ox, &oy);
                            T::init(P, frames[cur].M, ox, oy, R);
                            ent = e;
                            active = true;
                        }
                    }
                    break;
                }
                if (nfree == 64) {
                    ++cur;   // this frame's queue is empty and the wave is idle: next frame
                    continue;
                }
                break;   // tail of the frame: keep stepping the live lanes
            }
        }
        if (__ballot(active) == 0ull && cur >= nframes) break;
        if (prio_age > 0) {   // wave-uniform: any lane with an old ray lifts the wave
            if (__ballot(active && R.it >= prio_age)) __builtin_amdgcn_s_setprio(2);
            else __builtin_amdgcn_s_setprio(0);
        }
        const int cf = __builtin_amdgcn_readfirstlane(cur < nframes ? cur : nframes - 1);
        // frame parameters through the constant address space: wave-uniform scalar loads
        using CFrame = const __attribute__((address_space(4))) BatchFrame;
        CFrame* cfr = (CFrame*)frames;
        const TraceParams& P0 = *(const TraceParams*)&cfr[cf].P;
        const bhm32::MixedParams& M0 = *(const bhm32::MixedParams*)&cfr[cf].M;
        // What every attempt reads of them is loaded once per interval, into scalar registers: read
        // through P0, each field is loaded again at its use and the wave waits for the scalar cache, 5
        // times an attempt in the vacuum and some 25 times in the flow. The flow's tables stay behind P0
        // and M0 (with them the registers spill). FP64 vacuum records of 256^2 3.2 -> 2.8 ms; mixed
        // radio, 8 frames of 4.0 M rays, 11.0 -> 9.8; 1024^2 with the surrogate 2.9 -> 2.6 (kernel).
        const TraceParams P = P0;
        const bhm32::MixedParams M = M0;
        for (int k = 0; k < interval; ++k)
            if (active && !R.done) T::step(P, M, P0, M0, R);
        // Finished rays are written here, all of the interval's together: inside the loop nearly every
        // step of a 64-ray wave would end some ray and hold the others up for its output (LDS sums, a
        // store, the escape direction). Mixed radio, 8 frames of 4.0 M rays: 11.6 -> 11.0 ms; 1024^2 with
        // the surrogate: 3.02 -> 2.94.
        if (active && R.done) {
            RayResult r;
            const int f64 = T::result(P0, R, r);
            Wk.finish(cf, ent, r);
            s_flux[tid] += r.I[0];
            s_stat[0][tid] += (unsigned long long)r.steps;
            s_stat[1][tid] += (unsigned long long)r.accepted;
            s_stat[2][tid] += (unsigned long long)r.flow_steps;
            s_stat[3][tid] += r.fate == 0 ? 1ull : 0ull;
            s_stat[4][tid] += (unsigned long long)f64;
            active = false;
        }
    }
    if (prio_age > 0) __builtin_amdgcn_s_setprio(0);
    *flux_out = s_flux[tid];
    for (int i = 0; i < NSTAT; ++i) cnt_out[i] = s_stat[i][tid];
}

/* Two waves per 64 rays, for radio launches that leave most of the chip's issue slots idle. A SIMD issues one
   wave's instructions at half its rate, so where every SIMD holds at most one wave of rays a launch lasts as
   long as its longest ray's chain of instructions. Of an attempt's chain only the integration is a chain: the
   flow sample and the ring angle (nearly half) feed nothing back but the end of an opaque ray. So the
   workgroup's first wave integrates and leaves each accepted step in LDS, and the second evaluates it during
   the next attempt: one barrier per attempt, two slots by turns. Every value is formed by the same operations
   in the same order as in ray_step: same outputs. One wave -> two, ms of the launch (frames 30 M wide at 17
   degrees, the 0.6 Jy flow): mixed 64^2 1.32 -> 0.98, 256^2 2.04 -> 1.69; FP64 64^2 3.9 -> 2.9, 256^2 5.6 -> 4.4.
   A ray that turned out opaque in attempt k is known to be so after the barrier of attempt k + 1. Its flag is
   read then, and used after attempt k + 2 so that nothing waits for the read; the ray takes no further attempts,
   and at the interval's end its counters are taken back by the tags of the attempts since. So it costs two
   attempts more than it has. Ray records hold its state before attempt k too: they save the rays' state at the
   interval's start, from which its attempts up to k are repeated (keeping every attempt's state for that cost all
   records 2 %). Learning of the flag at the interval's end only, with every opaque ray's attempts repeated, cost a
   thick flow (3000 times the density, 69 degrees) the gain and more: mixed 256^2 0.73 ms, 448^2 1.25, 640^2 1.88;
   now 0.51, 0.84, 1.26; one wave 0.63, 0.81, 1.20.
   Both waves take every branch around a barrier on a value that both read from LDS. */
constexpr int PAIR_BLOCK = 128;

// What an attempt of a lane left (PairLDS::tag)
constexpr int TAG_SAMPLE = 1, TAG_FLOW = 2, TAG_TRIED = 4, TAG_FP64 = 8;   // an accepted step; inside the flow; an attempt

template <class T, bool RECORDS>
struct PairLDS {
    double v[2][7][64];        // StepSample
    int tag[2][64];
    int opaque[2][64];         // the attempt's sample made the ray opaque
    int more[2];               // some ray runs on after this attempt
    int frame;                 // the rays' frame; -1: no rays are left
    int fresh[64];             // the lane has a new ray
    double lam[64], E[64];
    double sums[6][64];        // acc0..3, trans, psi
    double flux[64];
    unsigned long long stat[NSTAT][64];
    typename T::State start[RECORDS ? 64 : 1];   // ray records: at the interval's start
};

// What the ray's statistics hold of an attempt, three bits each (it, fp64_attempts, accepted, flow_steps)
__device__ __forceinline__ int counts_of(int tag) {
    return (tag & TAG_TRIED ? 1 : 0) | (tag & TAG_FP64 ? 1 << 3 : 0) | (tag & TAG_SAMPLE ? 1 << 6 : 0) |
           (tag & TAG_FLOW ? 1 << 9 : 0);
}
constexpr int ENDED = 1 << 12;   // beside the counts to take back: a sample made the ray opaque

template <class T>
__device__ __forceinline__ void take_back(int back, typename T::State& R) {
    R.it -= back & 7;
    T::undo_fp64(R, back >> 3 & 7);
    R.accepted -= back >> 6 & 7;
    R.flow_steps -= back >> 9 & 7;
}

template <int PREC, int RADIO, bool TIME, class Work>
__device__ __forceinline__ void pair_body(const Work& Wk, unsigned int* __restrict__ queue, int interval,
                                          int refill_min, double* flux_out, unsigned long long* cnt_out) {
    using T = Tracer<PREC, RADIO, TIME>;
    using CFrame = const __attribute__((address_space(4))) BatchFrame;
    CFrame* cfr = (CFrame*)Wk.frames;
    constexpr bool RECORDS = Work::RECORDS;
    __shared__ PairLDS<T, RECORDS> L;
    const int lane = threadIdx.x & 63;
    const bool mover = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0;
    *flux_out = 0.0;
    for (int i = 0; i < NSTAT; ++i) cnt_out[i] = 0ull;
    if (mover) {
        int cur = 0;   // the wave's frame (wave-uniform)
        bool active = false;
        unsigned int ent = 0;
        typename T::State R;
        L.flux[lane] = 0.0;
        for (int i = 0; i < NSTAT; ++i) L.stat[i][lane] = 0ull;
        for (;;) {
            const bool was = active;
            refill<T>(Wk, queue, refill_min, &cur, &active, &ent, R);
            const bool any = __ballot(active) != 0ull;
            const int cf = __builtin_amdgcn_readfirstlane(cur < Wk.n ? cur : Wk.n - 1);
            L.fresh[lane] = active && !was;
            if (active) {
                L.lam[lane] = R.c.lam;
                L.E[lane] = R.c.E;
                if constexpr (RECORDS) L.start[lane] = R;
            }
            if (lane == 0) L.frame = !any && cur >= Wk.n ? -1 : cf;
            __syncthreads();   // A: the interval's rays
            if (!any && cur >= Wk.n) break;
            const TraceParams P = *(const TraceParams*)&cfr[cf].P;
            const bhm32::MixedParams M = *(const bhm32::MixedParams*)&cfr[cf].M;
            // of a ray that a sample made opaque: its counts to take back (ray records: that sample's attempt + 1)
            int k = 0, back = 0;
            for (;; ++k) {
                const int b = k & 1;
                const int opaque = L.opaque[b][lane];   // by attempt k - 2; an older interval's before that
                const bool run = active && !R.done;
                bhd::StepSample q;
                bool push = run && T::template move<true>(P, M, R, q);
                int tag = (run ? TAG_TRIED | (T::last_fp64(R) ? TAG_FP64 : 0) : 0) |
                          (push ? TAG_SAMPLE | (q.flow ? TAG_FLOW : 0) : 0);
                if (opaque && k >= 2) {
                    if constexpr (RECORDS) back = k - 1;
                    else
                        back = ENDED + counts_of(tag) + counts_of(L.tag[b ^ 1][lane]);
                    R.done = true;
                    push = false;
                    tag = 0;
                }
                if (push) {
                    L.v[b][0][lane] = q.r;
                    L.v[b][1][lane] = q.u;
                    L.v[b][2][lane] = q.phi;
                    L.v[b][3][lane] = q.t;
                    L.v[b][4][lane] = q.h;
                    L.v[b][5][lane] = q.u0;
                    L.v[b][6][lane] = q.phi0;
                }
                L.tag[b][lane] = tag;
                const bool more = k + 1 < interval && __ballot(active && !R.done) != 0ull;
                if (lane == 0) L.more[b] = more;
                __syncthreads();   // B: attempt k's samples
                if (!more) break;
            }
            __syncthreads();   // C: the interval's sums
            {   // the last two attempts' samples
                const int b = k & 1;
                if (k > 0 && L.opaque[b ^ 1][lane])
                    back = RECORDS ? k : ENDED + counts_of(L.tag[b][lane]);
                else if (L.opaque[b][lane])
                    back = RECORDS ? k + 1 : ENDED;
            }
            if (back) {
                if constexpr (RECORDS) {
                    bhd::StepSample q;
                    R = L.start[lane];
                    for (int i = 1; i < back; ++i) T::template move<true>(P, M, R, q);
                    T::template move<false>(P, M, R, q);
                } else {
                    take_back<T>(back, R);
                }
                R.fate = -1;
                R.done = true;
            }
            if (active && R.done) {
                R.acc0 = L.sums[0][lane];
                R.acc1 = L.sums[1][lane];
                R.acc2 = L.sums[2][lane];
                R.acc3 = L.sums[3][lane];
                R.trans = L.sums[4][lane];
                R.psi = (decltype(R.psi))L.sums[5][lane];
                RayResult r;
                const int f64 = T::result(*(const TraceParams*)&cfr[cf].P, R, r);
                Wk.finish(cf, ent, r);
                L.flux[lane] += r.I[0];
                L.stat[0][lane] += (unsigned long long)r.steps;
                L.stat[1][lane] += (unsigned long long)r.accepted;
                L.stat[2][lane] += (unsigned long long)r.flow_steps;
                L.stat[3][lane] += r.fate == 0 ? 1ull : 0ull;
                L.stat[4][lane] += (unsigned long long)f64;
                active = false;
            }
        }
        *flux_out = L.flux[lane];
        for (int i = 0; i < NSTAT; ++i) cnt_out[i] = L.stat[i][lane];
    } else {
        typename T::Sums S;
        T::begin(S);
        double lam = 0.0, E = 0.0;
        for (;;) {
            __syncthreads();   // A
            const int cf = __builtin_amdgcn_readfirstlane(L.frame);
            if (cf < 0) break;
            const TraceParams& F = *(const TraceParams*)&cfr[cf].P;
            const bhm32::MixedParams& FM = *(const bhm32::MixedParams*)&cfr[cf].M;
            if (L.fresh[lane]) {
                T::begin(S);
                lam = L.lam[lane];
                E = L.E[lane];
            }
            bool opaque = false;
            for (int k = 0;; ++k) {
                __syncthreads();   // B
                const int b = k & 1, tag = L.tag[b][lane];
                const bool more = __builtin_amdgcn_readfirstlane(L.more[b]) != 0;
                bool now = false;
                if ((tag & TAG_SAMPLE) && !opaque) {
                    const bhd::StepSample q{L.v[b][0][lane], L.v[b][1][lane], L.v[b][2][lane], L.v[b][3][lane],
                                            L.v[b][4][lane], L.v[b][5][lane], L.v[b][6][lane], (tag & TAG_FLOW) != 0};
                    now = T::add(F, FM, lam, E, q, S);
                }
                L.opaque[b][lane] = now;
                opaque = opaque || now;
                if (!more) break;
            }
            L.sums[0][lane] = S.acc0;
            L.sums[1][lane] = S.acc1;
            L.sums[2][lane] = S.acc2;
            L.sums[3][lane] = S.acc3;
            L.sums[4][lane] = S.trans;
            L.sums[5][lane] = (double)S.psi;
            __syncthreads();   // C
        }
    }
}

}  // namespace bhp

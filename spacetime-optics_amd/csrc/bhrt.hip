/* bhrt.hip - gfx950 kernels and the C ABI (include/bhrt.h) of the Kerr tracer.

   Launch geometry: a 256-lane workgroup traces a 16x16 pixel tile; each wave64 owns an 8x8
   sub-tile, so the rays of a wave are image neighbours with similar step counts (less divergence)
   and similar paths through the turbulence grid (shared cache lines). Workgroups are renumbered so
   that each of the 8 XCDs (workgroup i runs on XCD i % 8) receives a contiguous band of tiles and
   the grid lines its rays touch stay in that XCD's L2.

   Per-block partial sums (flux and integrator counters) are reduced by a second kernel in a fixed
   order, so frame totals are deterministic (no floating-point atomics). */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/bhrt.h"
#include "trace_fp64.h"
#include "trace_mixed.h"
#include "ctx.h"
#include "launch.h"
#include "persist.h"

using bhd::RayResult;
using bhd::TraceParams;

namespace {

constexpr int TILE = 16;          // pixels per tile side
constexpr int BLOCK = TILE * TILE;
constexpr int NXCD = 8;



// tile index of this workgroup after the XCD-aware renumbering; -1 for padding workgroups
__device__ __forceinline__ int xcd_tile(int bid, int ntiles, int per_xcd) {
    int t = (bid % NXCD) * per_xcd + bid / NXCD;
    return t < ntiles ? t : -1;
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}
__device__ __forceinline__ unsigned long long wave_sum(unsigned long long v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    return v;
}

// Two waves per SIMD at least: with 256-lane workgroups alone the compiler may take VGPRs and AGPRs
// beyond 256 together (one wave per SIMD); the bound makes it spill to scratch instead.
template <int PREC, int RADIO, bool TIME, bool RAYS>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(2))) void k_trace(
    const TraceParams P, const bhm32::MixedParams M, float4* __restrict__ px_out, bh_ray_out* __restrict__ rays_out,
    BlockOut* __restrict__ blk, int per_xcd) {
    const int tiles_x = (P.w + TILE - 1) / TILE, tiles_y = (P.h + TILE - 1) / TILE;
    const int tile = xcd_tile(blockIdx.x, tiles_x * tiles_y, per_xcd);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double flux = 0.0;
    unsigned long long c[NCNT] = {0, 0, 0, 0, 0};
    if (tile >= 0) {
        const int lx = (wave & 1) * 8 + (lane & 7), ly = (wave >> 1) * 8 + (lane >> 3);
        const int tx = (tile % tiles_x) * TILE + lx, ty = (tile / tiles_x) * TILE + ly;
        if (tx < P.w && ty < P.h) {
            const int px = P.x0 + tx, py = P.y0 + ty;
            double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
            RayResult r;
            for (int s = 0; s < P.spp; ++s) {
                double ox, oy;
                bhd::sample_offsets(P, px, py, s, &ox, &oy);
                int fp64_attempts;
                if (PREC == BH_PREC_FP64) {
                    bhd::trace_ray_fp64<RADIO, TIME>(P, ox, oy, r);
                    fp64_attempts = r.steps;
                } else {
                    fp64_attempts = bhm32::trace_ray_mixed<RADIO, TIME>(P, M, ox, oy, r);
                }
                a0 += r.I[0];
                a1 += r.I[1];
                a2 += r.I[2];
                a3 += r.I[3];
                c[0] += (unsigned long long)r.steps;
                c[1] += (unsigned long long)r.accepted;
                c[2] += (unsigned long long)r.flow_steps;
                c[3] += r.fate == 0 ? 1ull : 0ull;
                c[4] += (unsigned long long)fp64_attempts;
            }
            flux = a0;
            const size_t o = (size_t)ty * P.w + tx;
            if (RAYS) {
                bhp::write_record(rays_out + o, r);
            } else {
                const double m = (double)P.spp;   // mean as sum / count, as the adaptive resolve and the oracle
                px_out[o] = make_float4((float)(a0 / m), (float)(a1 / m), (float)(a2 / m), (float)(a3 / m));
            }
        }
    }
    // deterministic block partials: wave64 shuffles, then the 4 waves in order through LDS
    __shared__ double s_flux[BLOCK / 64];
    __shared__ unsigned long long s_cnt[BLOCK / 64][NCNT];
    flux = wave_sum(flux);
    for (int i = 0; i < NCNT; ++i) c[i] = wave_sum(c[i]);
    if (lane == 0) {
        s_flux[wave] = flux;
        for (int i = 0; i < NCNT; ++i) s_cnt[wave][i] = c[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        BlockOut b;
        b.flux = ((s_flux[0] + s_flux[1]) + s_flux[2]) + s_flux[3];
        for (int i = 0; i < NCNT; ++i) b.cnt[i] = s_cnt[0][i] + s_cnt[1][i] + s_cnt[2][i] + s_cnt[3][i];
        blk[blockIdx.x] = b;
    }
}

// The frame kernel's block partials of the flux from samples already traced (samp[pixel * spp + sample]):
// the same workgroups, lanes and order of additions, so the total has the same bits.
__global__ __launch_bounds__(BLOCK) void k_flux_blocks(const double4* __restrict__ samp, int w, int h, int spp,
                                                       BlockOut* __restrict__ blk, int per_xcd) {
    const int tiles_x = (w + TILE - 1) / TILE, tiles_y = (h + TILE - 1) / TILE;
    const int tile = xcd_tile(blockIdx.x, tiles_x * tiles_y, per_xcd);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double flux = 0.0;
    if (tile >= 0) {
        const int tx = (tile % tiles_x) * TILE + (wave & 1) * 8 + (lane & 7);
        const int ty = (tile / tiles_x) * TILE + (wave >> 1) * 8 + (lane >> 3);
        if (tx < w && ty < h)
            for (int s = 0; s < spp; ++s) flux += samp[((size_t)ty * w + tx) * spp + s].x;
    }
    __shared__ double s_flux[BLOCK / 64];
    flux = wave_sum(flux);
    if (lane == 0) s_flux[wave] = flux;
    __syncthreads();
    if (threadIdx.x == 0) {
        BlockOut b{};
        b.flux = ((s_flux[0] + s_flux[1]) + s_flux[2]) + s_flux[3];
        blk[blockIdx.x] = b;
    }
}

// Sums nb block partials in index order (one workgroup; each lane a strided slice, then a fixed tree).
__global__ __launch_bounds__(256) void k_reduce(const BlockOut* __restrict__ blk, int nb, BlockOut* __restrict__ tot) {
    __shared__ double s_f[256];
    __shared__ unsigned long long s_c[256][NCNT];
    double f = 0.0;
    unsigned long long c[NCNT] = {0, 0, 0, 0, 0};
    for (int i = threadIdx.x; i < nb; i += 256) {
        f += blk[i].flux;
        for (int k = 0; k < NCNT; ++k) c[k] += blk[i].cnt[k];
    }
    s_f[threadIdx.x] = f;
    for (int k = 0; k < NCNT; ++k) s_c[threadIdx.x][k] = c[k];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            s_f[threadIdx.x] += s_f[threadIdx.x + w];
            for (int k = 0; k < NCNT; ++k) s_c[threadIdx.x][k] += s_c[threadIdx.x + w][k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        BlockOut b;
        b.flux = s_f[0];
        for (int k = 0; k < NCNT; ++k) b.cnt[k] = s_c[0][k];
        *tot = b;
    }
}

}  // namespace

/* Scratch memory of bh_render_noalloc: the frame kernel's per-workgroup partials followed by the
   reduced total, for frames of up to NOALLOC_MAX_BLOCKS workgroups (16 x 16 tiles, padded to a
   multiple of the 8 XCDs): 65536 x 48 B = 3 MiB per device, held until the process ends. Host code
   never uses this name as an address: bh_create resolves each device's copy with
   hipGetSymbolAddress and keeps the pointer per device (g_noalloc_scratch). */
constexpr int NOALLOC_MAX_BLOCKS = 65536;
constexpr int NOALLOC_MAX_DEVICES = 64;
static __device__ __align__(256) BlockOut scratch[NOALLOC_MAX_BLOCKS + 1];

namespace {

// WAVES > 1 asks the compiler for at least that many resident waves per SIMD (fewer VGPRs, possibly
// spills); 1 leaves the register budget to the compiler.
static_assert(BLOCK == bhp::MAX_BLOCK && NCNT == bhp::NSTAT, "persistent kernel slots");

// The workgroup's flux and counters from its lanes' sums
__device__ __forceinline__ void block_out(double flux, unsigned long long c[NCNT], BlockOut* __restrict__ blk) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    __shared__ double s_flux[BLOCK / 64];
    __shared__ unsigned long long s_cnt[BLOCK / 64][NCNT];
    flux = wave_sum(flux);
    for (int i = 0; i < NCNT; ++i) c[i] = wave_sum(c[i]);
    if (lane == 0) {
        s_flux[wave] = flux;
        for (int i = 0; i < NCNT; ++i) s_cnt[wave][i] = c[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        BlockOut b;
        b.flux = 0.0;
        for (int i = 0; i < NCNT; ++i) b.cnt[i] = 0;
        for (int w = 0; w < nw; ++w) {
            b.flux += s_flux[w];
            for (int i = 0; i < NCNT; ++i) b.cnt[i] += s_cnt[w][i];
        }
        blk[blockIdx.x] = b;
    }
}

template <int PREC, int RADIO, bool TIME, int WAVES, class Work>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WAVES))) void k_persist(
    const Work wk, unsigned int* __restrict__ queue, int interval, int refill_min, int prio_age,
    BlockOut* __restrict__ blk) {
    double flux;
    unsigned long long c[NCNT];
    bhp::persist_body<PREC, RADIO, TIME>(wk, queue, interval, refill_min, prio_age, &flux, c);
    block_out(flux, c, blk);
}

// Two waves per 64 rays (persist.h): an integrating and an evaluating wave per SIMD.
template <int PREC, int RADIO, bool TIME, class Work>
__global__ __launch_bounds__(bhp::PAIR_BLOCK) __attribute__((amdgpu_waves_per_eu(2))) void k_pair(
    const Work wk, unsigned int* __restrict__ queue, int interval, int refill_min, int, BlockOut* __restrict__ blk) {
    double flux;
    unsigned long long c[NCNT];
    bhp::pair_body<PREC, RADIO, TIME>(wk, queue, interval, refill_min, &flux, c);
    block_out(flux, c, blk);
}

/* ---- adaptive sampling (render.cu:89-242, 677-721), deterministic form ----
   Pass-1 samples are kept per (pixel, sample) and summed per pixel in sample order; the frame sum of
   the luminance goes through fixed blocks of 256 pixels; pass-2 samples are kept per entry and added
   in order. The decisions (extra samples per pixel) use the reference's float formulas. */
constexpr int ADAPT_CHUNK = 8;     // samples per pass-2 work item (render.cu:30)
constexpr int FSUM_BLOCK = 256;    // pixels per partial of the frame luminance sum

// Per pixel: FP64 sums of the pass-1 samples (sample order) and the float luminance sums.
__global__ void k_adapt_stats(const double4* __restrict__ samp, int npix, int spp, int lum,
                              double4* __restrict__ acc, float2* __restrict__ ystat) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npix) return;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
    float ys = 0.f, yq = 0.f;
    for (int s = 0; s < spp; ++s) {
        const double4 v = samp[(size_t)p * spp + s];
        a0 += v.x;
        a1 += v.y;
        a2 += v.z;
        a3 += v.w;
        const float Y = (float)(lum == 0 ? v.x : v.y);
        ys += Y;
        yq += Y * Y;
    }
    acc[p] = make_double4(a0, a1, a2, a3);
    ystat[p] = make_float2(ys, yq);
}

// Partial luminance sums over FSUM_BLOCK consecutive pixels, each in pixel order.
__global__ void k_adapt_fsum(const float2* __restrict__ ystat, int npix, double* __restrict__ part) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    const int p0 = b * FSUM_BLOCK;
    if (p0 >= npix) return;
    double s = 0.0;
    for (int p = p0; p < npix && p < p0 + FSUM_BLOCK; ++p) s += (double)ystat[p].x;
    part[b] = s;
}

// render.cu:130-139 with yref = 0.03 * (frame luminance sum) / (npix * spp) + 1e-37 (render.cu:702).
// The partials are summed in order by every thread (a few thousand L2-resident loads).
__global__ void k_adapt_extra(const float2* __restrict__ ystat, int npix, int spp, const double* __restrict__ part,
                              int nparts, float target, int extra_max, unsigned int* __restrict__ extra) {
    __shared__ float s_yref;
    if (threadIdx.x == 0) {
        double fsum = 0.0;
        for (int b = 0; b < nparts; ++b) fsum += part[b];
        s_yref = (float)(0.03 * fsum / ((double)npix * spp) + 1e-37);
    }
    __syncthreads();
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npix) return;
    const float n = (float)spp;
    const float2 st = ystat[p];
    const float mean = st.x / n, var = fmaxf(st.y / n - mean * mean, 0.f);
    const float se = sqrtf(var / n), den = target * (mean + s_yref);
    const float want = n * (se / den) * (se / den);
    extra[p] = (unsigned int)fminf(fmaxf(ceilf(want) - n, 0.f), (float)extra_max);
}

// render.cu:141-150: 3 x 3 maximum, clamped at the edges, in chunks of ADAPT_CHUNK samples.
__global__ void k_adapt_dilate(const unsigned int* __restrict__ extra, int W, int H, int extra_max,
                               unsigned int* __restrict__ chunks) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y * blockDim.y + threadIdx.y;
    if (x >= W || y >= H) return;
    unsigned int m = 0;
    for (int dy = -1; dy <= 1; ++dy)
        for (int dx = -1; dx <= 1; ++dx)
            m = max(m, extra[(size_t)min(max(y + dy, 0), H - 1) * W + min(max(x + dx, 0), W - 1)]);
    chunks[(size_t)y * W + x] = (min(m, (unsigned int)extra_max) + ADAPT_CHUNK - 1) / ADAPT_CHUNK;
}

// Exclusive prefix sum of unsigned ints: per-1024 block scans (wave64 shuffles, then the 16 wave
// totals), the block totals scanned by one workgroup in rounds of 1024, then added back.
__device__ __forceinline__ unsigned int wave_incl_scan(unsigned int v, int lane) {
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned int t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

__device__ __forceinline__ unsigned int block_excl_scan(unsigned int v, unsigned int* total) {
    __shared__ unsigned int ws[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const unsigned int inc = wave_incl_scan(v, lane);
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    if (w == 0) {   // one wave scans the 16 wave totals in place (its reads precede its writes)
        unsigned int t = lane < 16 ? ws[lane] : 0u;
        t = wave_incl_scan(t, lane);
        if (lane < 16) ws[lane] = t;
    }
    __syncthreads();
    const unsigned int pre = w > 0 ? ws[w - 1] : 0u;
    *total = ws[15];
    __syncthreads();   // ws is rewritten by the next call
    return pre + inc - v;
}

__global__ __launch_bounds__(1024) void k_scan_block(const unsigned int* __restrict__ in, unsigned int* __restrict__ out,
                                                     unsigned int* __restrict__ bsum, int n) {
    const int i = blockIdx.x * 1024 + threadIdx.x;
    unsigned int tot;
    const unsigned int ex = block_excl_scan(i < n ? in[i] : 0u, &tot);
    if (i < n) out[i] = ex;
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

__global__ __launch_bounds__(1024) void k_scan_top(unsigned int* __restrict__ bsum, int nb) {
    unsigned int carry = 0;
    for (int base = 0; base < nb; base += 1024) {
        const int i = base + threadIdx.x;
        unsigned int tot;
        const unsigned int ex = block_excl_scan(i < nb ? bsum[i] : 0u, &tot);
        if (i < nb) bsum[i] = carry + ex;
        carry += tot;
    }
}

__global__ void k_scan_add(unsigned int* __restrict__ out, const unsigned int* __restrict__ bsum, int n) {
    const int i = blockIdx.x * 1024 + threadIdx.x;
    if (i < n) out[i] += bsum[blockIdx.x];
}

// Pixel = (pass-1 sum + pass-2 samples in order) / sample count.
__global__ void k_adapt_resolve(const double4* __restrict__ acc, const double4* __restrict__ samp2,
                                const unsigned int* __restrict__ offsets, const unsigned int* __restrict__ chunks,
                                int npix, int spp, float4* __restrict__ out, unsigned int* __restrict__ nsamp) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= npix) return;
    double4 a = acc[p];
    const unsigned int k = chunks ? chunks[p] : 0u;
    if (k) {
        const double4* v = samp2 + (size_t)offsets[p] * ADAPT_CHUNK;
        for (unsigned int i = 0; i < k * ADAPT_CHUNK; ++i) {
            a.x += v[i].x;
            a.y += v[i].y;
            a.z += v[i].z;
            a.w += v[i].w;
        }
    }
    const unsigned int m = (unsigned int)spp + k * ADAPT_CHUNK;
    const double dm = (double)m;
    out[p] = make_float4((float)(a.x / dm), (float)(a.y / dm), (float)(a.z / dm), (float)(a.w / dm));
    if (nsamp) nsamp[p] = m;
}

// graph-safe reset of the work queues (a kernel, not a memset node)
__global__ void k_zero_u32(unsigned int* __restrict__ p, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// Bake of the sheared turbulence slices (render.cu:449-460): one work-item per cell, phi fastest.
__global__ __launch_bounds__(256) void k_bake_sheared(const bhd::ShearedBake B, float* __restrict__ out,
                                                      unsigned long long total) {
    const unsigned long long idx = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    unsigned long long rest = idx;
    const int i = (int)(rest % (unsigned)B.nphi);
    rest /= (unsigned)B.nphi;
    const int j = (int)(rest % (unsigned)B.nlr);
    rest /= (unsigned)B.nlr;
    const int l = (int)(rest % (unsigned)B.nz);
    const int k = (int)(rest / (unsigned)B.nz);
    out[idx] = bhd::sh_cell(B, i, j, l, k);
}

/* Queue orders of a persistent launch, from the tile's centre ray (lam, eta):
   - impact: by the impact parameter b, smallest first. b^2 = eta + lam^2 (+ a^2 cos^2 theta_cam, the
     same for the whole frame) is the distance from the hole's image for a distant camera.
   - critical: by the predicted length of the ray, longest first. Near the critical curve the radial
     potential R(r) = (r^2 + a^2 - a lam)^2 - Delta (eta + (lam - a)^2) has a near-double root at a
     spherical photon orbit radius, and the number of orbits (so the step count) grows as
     -ln |min R| over those radii; key = -ln(|min R(r) / r^4| + 1e-9) over 24 radii spanning the
     prograde to retrograde circular photon orbits (Bardeen 1972). On the 1024^2 230 GHz frame its
     rank correlation with the tile's longest ray is 0.97, and the tiles with rays above 800 steps
     come within the first 44 of 16384.
   Counting sort over ORDER_BUCKETS bins (the order inside a bin is whatever the atomics give, which
   changes no pixel). SCATTER = false counts the bins, true writes each tile at its bin's next
   position. */
constexpr int ORDER_BUCKETS = 1024;
constexpr double ORDER_BINS_PER_M = 16.0;   // impact order: bins of b
constexpr double ORDER_BINS_PER_KEY = 40.0; // critical order: bins of key + 4, reversed

__device__ __forceinline__ unsigned int critical_bin(double a, double lam, double eta) {
    const double aa = fabs(a);
    const double r_lo = 2.0 * (1.0 + cos(2.0 / 3.0 * acos(-aa))) - 0.05;   // prograde photon orbit
    const double r_hi = 2.0 * (1.0 + cos(2.0 / 3.0 * acos(aa))) + 0.05;    // retrograde photon orbit
    const double K = eta + (lam - a) * (lam - a);
    double m = 1e300;
    for (int i = 0; i < 24; ++i) {
        const double r = r_lo + (r_hi - r_lo) * (i * (1.0 / 23.0));
        const double P = r * r + a * a - a * lam, D = r * r - 2.0 * r + a * a;
        const double v = fabs((P * P - D * K) / (r * r * r * r));
        m = fmin(m, v);
    }
    const double key = -log(m + 1e-9);
    const unsigned int k = (unsigned int)fmin(fmax((key + 4.0) * ORDER_BINS_PER_KEY, 0.0), (double)(ORDER_BUCKETS - 1));
    return (unsigned int)(ORDER_BUCKETS - 1) - k;
}

template <bool SCATTER, int ORDER>
__global__ __launch_bounds__(256) void k_order_tiles(const bhp::BatchFrame* __restrict__ frames,
                                                     unsigned int* __restrict__ hist) {
    const int f = blockIdx.y;
    const bhp::BatchFrame& F = frames[f];
    const unsigned int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (F.nentries >> 6)) return;
    int px, py;
    bhp::tile_pixel(F.tiles_x, t, 36u, &px, &py);   // pixel (4, 4) of the 8 x 8 tile
    px = min(px, F.P.w - 1);
    py = min(py, F.P.h - 1);
    double ox, oy;
    bhd::sample_offsets(F.P, F.P.x0 + px, F.P.y0 + py, 0, &ox, &oy);   // x0 = y0 = 0 but for tile records
    bhd::RayConst rc;
    bhd::State st;
    bhd::camera_photon(F.P, ox, oy, rc, st);
    unsigned int k;
    if (ORDER == BH_ORDER_CRITICAL) {
        k = critical_bin(F.P.a, rc.lam, rc.eta);
    } else {
        const double b = sqrt(fmax(rc.eta + rc.lam * rc.lam, 0.0));
        k = (unsigned int)fmin(b * ORDER_BINS_PER_M, (double)(ORDER_BUCKETS - 1));
    }
    unsigned int* h = hist + (size_t)f * ORDER_BUCKETS + k;
    if (!SCATTER) {
        atomicAdd(h, 1u);
    } else {
        F.order[atomicAdd(h, 1u)] = t;
    }
}

// Exclusive prefix sum of each frame's ORDER_BUCKETS bin counts, in place (one workgroup per frame).
__global__ __launch_bounds__(256) void k_order_scan(unsigned int* __restrict__ hist) {
    static_assert(ORDER_BUCKETS == 4 * 256, "4 bins per thread");
    unsigned int* h = hist + (size_t)blockIdx.x * ORDER_BUCKETS;
    __shared__ unsigned int part[256];
    const int t = threadIdx.x;
    unsigned int v[4], sum = 0u;
    for (int i = 0; i < 4; ++i) {
        v[i] = h[4 * t + i];
        sum += v[i];
    }
    part[t] = sum;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const unsigned int x = t >= off ? part[t - off] : 0u;
        __syncthreads();
        part[t] += x;
        __syncthreads();
    }
    unsigned int run = part[t] - sum;
    for (int i = 0; i < 4; ++i) {
        h[4 * t + i] = run;
        run += v[i];
    }
}

__global__ __launch_bounds__(64) void k_vacuum_fates(const TraceParams P, const double* __restrict__ photons, int n,
                                                     double tol, double r_escape, int max_steps,
                                                     int* __restrict__ fates) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double ph[9];
    for (int k = 0; k < 9; ++k) ph[k] = photons[9 * (size_t)i + k];
    fates[i] = bhd::vacuum_fate(P, ph, tol, r_escape, max_steps);
}

__global__ void k_math_eval(int fn, const double* __restrict__ x, const double* __restrict__ y,
                            double* __restrict__ out, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double a = x[i], b = y[i], r = 0.0, s, c;
    switch (fn) {
        case 0: r = bhm::exp(a); break;
        case 1: r = bhm::log(a); break;
        case 2: r = bhm::expm1(a); break;
        case 3: r = bhm::cbrt(a); break;
        case 4: r = bhm::pow_m02(a); break;
        case 5: bhm::sincos(a, &s, &c); r = s; break;
        case 6: bhm::sincos(a, &s, &c); r = c; break;
        case 7: r = bhm::atan2(a, b); break;
        case 8: r = bhm::acos(a); break;
        case 11: r = bhm::asin(a); break;
        case 9: r = sqrt(a); break;
        case 12: r = bhm::quot_ieee_(a, b); break;
        case 13: r = bhm::sqrt_nn_(a); break;
        case 14: r = bhd::step_factor(a); break;
        case 15: r = bhd::angle_pos(a, b); break;
        default: r = a / b; break;
    }
    out[i] = r;
}

double now_ms() {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

std::string g_create_error;

// Device address of `scratch` on each device (resolved once per device by bh_create)
BlockOut* g_noalloc_scratch[NOALLOC_MAX_DEVICES] = {};
std::mutex g_noalloc_mu;

}  // namespace


#define HIPCK(ctx, x)                                                                                      \
    do {                                                                                                   \
        hipError_t e_ = (x);                                                                               \
        if (e_ != hipSuccess) {                                                                            \
            (ctx)->err = std::string(#x) + ": " + hipGetErrorString(e_);                                   \
            return BH_ERR_HIP;                                                                             \
        }                                                                                                  \
    } while (0)

namespace {

int fail(bh_ctx* c, int code, const std::string& msg) {
    c->err = msg;
    return code;
}

template <typename T>
int ensure(bh_ctx* c, T** p, size_t* cap, size_t n) {
    if (*cap >= n && *p) return BH_OK;
    if (*p) {
        HIPCK(c, hipStreamSynchronize(c->st));
        HIPCK(c, hipFree(*p));
        *p = nullptr;
        *cap = 0;
    }
    HIPCK(c, hipMalloc((void**)p, std::max<size_t>(n, 1) * sizeof(T)));
    *cap = n;
    return BH_OK;
}

// Whether a buffer can be had; if not, the caller takes a path without it.
template <typename T>
bool try_ensure(bh_ctx* c, T** p, size_t* cap, size_t n) {
    const std::string err = c->err;
    if (ensure(c, p, cap, n) == BH_OK) return true;
    (void)hipGetLastError();   // it would be taken for a later launch's
    c->err = err;
    return false;
}

TraceParams make_params_scene(const bh_ctx* c, const bh_scene& S, const bh_frame* f) {
    TraceParams P;
    std::memset(&P, 0, sizeof P);
    P.a = S.a;
    P.a2 = S.a * S.a;
    P.rh = S.rh;
    P.r_isco = S.r_isco;
    P.tol = S.tol;
    P.inv_tol = 1.0 / S.tol;
    // numerators of the scaled error above which a step is rejected unscaled: far above any scale, and
    // low enough that the quotients below it stay finite. A tolerance of zero rejects every error, one
    // below zero none.
    P.err_big = S.tol >= 1e-280 ? 1e200 * std::min(1.0, S.tol) : (S.tol >= 0.0 ? 0.0 : HUGE_VAL);
    P.r_escape = S.r_escape;
    P.r_stop = S.r_stop;
    P.step_frac = S.step_frac;
    P.max_steps = S.max_steps;
    P.mode = S.mode;
    P.flow_on = S.flow_on;
    P.turb_on = (S.flow_turb_amp > 0.f && c->d_turb && c->turb_n > 1) ? 1 : 0;
    P.n0 = S.n0;
    P.n_index = S.n_index;
    P.theta_index = S.theta_index;
    P.theta0 = S.theta0;
    P.h_r = S.h_r;
    P.beta_p = S.beta_p;
    P.r_flow_max = S.r_flow_max;
    P.nu_obs = S.nu_obs;
    P.rg_cm = S.rg_cm;
    P.flow_kep = S.flow_kep;
    P.k2 = c->d_k2;
    P.k2_n = c->k2_n;
    P.k2_l0 = c->k2_l0;
    P.k2_dl = c->k2_dl;
    P.k2_inv_dl = 1.f / c->k2_dl;
    P.turb = c->d_turb;
    P.turb_n = c->turb_n;
    P.turb_nt = c->turb_nt;
    P.turb_half = c->turb_half;
    P.turb_inv_dx = c->turb_n > 0 ? c->turb_n / (2.0 * c->turb_half) : 0.0;
    P.turb_t0 = c->turb_t0;
    P.turb_inv_dt = c->turb_dt > 0 ? 1.0 / c->turb_dt : 0.0;
    if (c->turb_model == BH_TURB_SHEARED) {
        // the slices baked for this scene and camera (prepare_turbulence runs before every launch)
        P.turb_on = (S.flow_turb_amp > 0.f && c->ts_valid) ? 1 : 0;
        P.ts = c->d_tsv;
    }
    P.sky_on = S.mode == BH_MODE_VISIBLE && S.sky_on && S.sky_nu > 0 && S.sky_nv > 0 ? 1 : 0;
    P.sky_nu = S.sky_nu;
    P.sky_nv = S.sky_nv;
    P.sky_scale = S.sky_scale;
    for (int i = 0; i < 9; ++i) P.sky_rot[i] = S.sky_rot[i];
    if (f) {
        P.ph0 = f->ph;
        P.t0 = f->t;
        for (int i = 0; i < 11; ++i) P.kp[i] = f->kp[i];
        for (int i = 0; i < 3; ++i) {
            P.F[i] = f->F[i];
            P.R[i] = f->R[i];
            P.U[i] = f->U[i];
            P.beta[i] = f->beta[i];
        }
        P.cx = f->cx;
        P.cy = f->cy;
        P.pix = f->pix;
        P.W = f->W;
        P.H = f->H;
        P.seed = f->seed;
    }
    return P;
}

TraceParams make_params(const bh_ctx* c, const bh_frame* f) { return make_params_scene(c, c->S, f); }

// Sheared turbulence of a radio scene seen from frame f: bakes the slices (render.cu:594-619,
// 679-682) unless the ones in memory belong to the same noise parameters and camera.
// With may_alloc false the slice buffers must already hold this bake (BH_ERR_UNSUPPORTED otherwise).
int prepare_turbulence(bh_ctx* c, const bh_scene& S, const bh_frame* f, bool may_alloc = true) {
    if (c->turb_model != BH_TURB_SHEARED || !f || S.mode != BH_MODE_RADIO || !S.flow_on || !(S.flow_turb_amp > 0.f))
        return BH_OK;
    if (!(S.flow_turb_scale > 0.f) || !(S.flow_tcorr > 0.f))
        return fail(c, BH_ERR_ARG, "sheared turbulence needs flow_turb_scale > 0 and flow_tcorr > 0");
    if (!(f->r > 0.0)) return fail(c, BH_ERR_ARG, "sheared turbulence needs the camera radius (frame r > 0)");
    bhd::ShearedBake B{};
    B.a = S.a;
    B.r_isco = S.r_isco;
    B.cam_t = f->t;
    B.cam_r = f->r;
    B.lr0 = (float)std::log(0.8 * S.rh);
    B.lr1 = (float)std::log(S.r_flow_max * 1.05);
    B.zmax = (float)std::min(2.0, 5.0 * S.h_r);
    B.nphi = c->ts_dims[0];
    B.nlr = c->ts_dims[1];
    B.nz = c->ts_dims[2];
    B.nt = c->ts_dims[3];
    B.d0 = -250.f;
    B.dd = 260.f / (float)(B.nt - 1);
    B.amp = S.flow_turb_amp;
    B.scale = S.flow_turb_scale;
    B.tcorr = S.flow_tcorr;
    B.seed = S.seed ^ 0x51f15eedu;
    const std::array<double, 16> key = {B.a, B.r_isco, B.cam_t, B.cam_r, S.rh, S.r_flow_max, S.h_r, (double)B.amp,
                                        (double)B.scale, (double)B.tcorr, (double)B.seed, (double)B.nphi,
                                        (double)B.nlr, (double)B.nz, (double)B.nt, 1.0};
    if (c->ts_valid && key == c->ts_key) return BH_OK;
    const unsigned long long total = (unsigned long long)B.nphi * B.nlr * B.nz * B.nt;
    if (!may_alloc && (!c->d_ts || c->ts_cap < total || !c->d_tsv))
        return fail(c, BH_ERR_UNSUPPORTED,
                    "sheared turbulence slices are not allocated yet: trace one frame with bh_render first");
    c->ts_valid = false;
    int rc = ensure(c, &c->d_ts, &c->ts_cap, (size_t)total);
    if (rc) return rc;
    rc = ensure(c, &c->d_tsv, &c->tsv_cap, 1);
    if (rc) return rc;
    hipLaunchKernelGGL(k_bake_sheared, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, c->st, B, c->d_ts, total);
    HIPCK(c, hipGetLastError());
    bhd::ShearedView& V = c->tsv_host;   // lives in the context until the copy has run
    V.data = c->d_ts;
    V.nphi = B.nphi;
    V.nlr = B.nlr;
    V.nz = B.nz;
    V.nt = B.nt;
    V.lr0 = B.lr0;
    V.lr1 = B.lr1;
    V.zmax = B.zmax;
    V.d0 = B.d0;
    V.dd = B.dd;
    V.inv_dd = 1.f / B.dd;
    V.inv_lr = 1.0 / (double)(B.lr1 - B.lr0);
    V.inv_zmax = 1.0 / (double)B.zmax;
    V.cam_t = B.cam_t;
    V.cam_r = B.cam_r;
    HIPCK(c, hipMemcpyAsync(c->d_tsv, &V, sizeof V, hipMemcpyHostToDevice, c->st));
    c->ts_key = key;
    c->ts_valid = true;
    return BH_OK;
}

int check_frame(bh_ctx* c, const bh_frame* f) {
    if (!f) return fail(c, BH_ERR_ARG, "frame is NULL");
    if (f->W <= 0 || f->H <= 0 || f->W > 65536 || f->H > 65536) return fail(c, BH_ERR_ARG, "bad frame size");
    if (!(f->pix > 0.0)) return fail(c, BH_ERR_ARG, "frame pixel scale must be > 0");
    if (c->S.mode == BH_MODE_RADIO && c->S.flow_on && !c->d_k2) return fail(c, BH_ERR_ARG, "radio mode needs the K2 table");
    return BH_OK;
}

using KernelFn = void (*)(const TraceParams, const bhm32::MixedParams, float4*, bh_ray_out*, BlockOut*, int);

// The tracers' RADIO and TIME arguments for a scene, the context's turbulence model and the call.
struct Variant {
    int radio;
    bool time;
};

// coordinate-time bound of a mixed-tracer call: the caller's, or the default where the emission
// depends on the time a sample is emitted at
double time_bound(const bh_ctx* c, const bh_scene& S, const bh_trace_opts& o);

// The emission reads the coordinate time: time slices, or the sheared model
bool flow_reads_time(const bh_ctx* c, const bh_scene& S) {
    return S.mode == BH_MODE_RADIO && S.flow_on &&
           ((c->turb_model == BH_TURB_GRID && c->d_turb && c->turb_nt > 1) || c->turb_model == BH_TURB_SHEARED);
}

Variant variant_of(const bh_ctx* c, const bh_scene& S, const bh_trace_opts& o) {
    Variant v{bhd::RADIO_OFF, flow_reads_time(c, S)};
    if (S.mode == BH_MODE_RADIO) v.radio = c->turb_model == BH_TURB_SHEARED ? bhd::RADIO_SHEARED : bhd::RADIO_GRID;
    if (o.precision == BH_PREC_MIXED && time_bound(c, S, o) > 0.0) v.time = true;
    return v;
}

// The kernel `at<RADIO, TIME>()` of a variant. ALWAYS: the kernel reads the coordinate time whatever
// the frame (ray records). The sheared model always reads it, and the FP64 tracer of a vacuum frame
// never does.
template <int PREC, bool ALWAYS, class At>
auto pick_variant(const Variant& v, const At& at) {
    switch (v.radio) {
        case bhd::RADIO_SHEARED: return at.template operator()<bhd::RADIO_SHEARED, true>();
        case bhd::RADIO_GRID:
            return v.time ? at.template operator()<bhd::RADIO_GRID, true>() : at.template operator()<bhd::RADIO_GRID, ALWAYS>();
        default:
            return v.time ? at.template operator()<bhd::RADIO_OFF, ALWAYS || PREC == BH_PREC_MIXED>()
                          : at.template operator()<bhd::RADIO_OFF, ALWAYS>();
    }
}

template <int PREC, bool RAYS>
struct TraceAt {
    template <int RADIO, bool TIME>
    KernelFn operator()() const {
        return k_trace<PREC, RADIO, TIME, RAYS>;
    }
};

template <bool RAYS>
KernelFn pick_kernel_r(int prec, const Variant& v) {
    return prec == BH_PREC_FP64 ? pick_variant<BH_PREC_FP64, RAYS>(v, TraceAt<BH_PREC_FP64, RAYS>{})
                                : pick_variant<BH_PREC_MIXED, RAYS>(v, TraceAt<BH_PREC_MIXED, RAYS>{});
}

KernelFn pick_kernel(int prec, const Variant& v, bool rays) {
    return rays ? pick_kernel_r<true>(prec, v) : pick_kernel_r<false>(prec, v);
}

constexpr double C_C = 2.99792458e10, C_H = 6.62607015e-27, C_ME = 9.1093837e-28, C_MP = 1.67262192e-24,
                 C_QE = 4.80320471e-10, C_PI = 3.14159265358979323846;

// Emission weight j r^2 and absorption coefficient of the mid-plane flow at radius r
void flow_cell(const bh_scene& S, const std::vector<float>& k2, float k2_l0, float k2_dl, double r, double* w,
               double* alpha) {
    const double ne = S.n0 * std::pow(r, -S.n_index) * (1.0 - std::exp(-(r - S.rh) * (r - S.rh) / 0.25));
    const double th = S.theta0 * std::pow(r, -S.theta_index);
    const double B = std::sqrt(8.0 * C_PI * ne * C_MP * C_C * C_C / (6.0 * r * S.beta_p));
    const double nus = 2.0 / 9.0 * (C_QE * B / (2.0 * C_PI * C_ME * C_C)) * th * th;
    const double X = S.nu_obs / nus, x3 = std::cbrt(X);
    float f = ((float)std::log(th) - k2_l0) / k2_dl;
    f = std::min(f > 0.f ? f : 0.f, (float)(k2.size() - 2) + 0.9999f);   // a NaN reads the first entry
    const int k = (int)f;
    const double lk2 = k2[k] + (k2[k + 1] - k2[k]) * (f - k);
    const double brk = std::sqrt(X) + 1.887748625363387 * std::sqrt(x3);
    // j_nu in cgs (emission.cuh:165-166) and alpha_nu = j_nu / B_nu(T_e) (Kirchhoff)
    const double j = ne * std::sqrt(2.0) * C_PI * C_QE * C_QE * nus / (3.0 * C_C) * std::exp(-lk2) * brk * brk *
                     std::exp(-x3);
    const double bnu = 2.0 * C_H * S.nu_obs * S.nu_obs * S.nu_obs / (C_C * C_C) /
                       std::expm1(C_H * S.nu_obs / (C_ME * C_C * C_C * th));
    *w = std::isfinite(j) ? j * r * r : 0.0;
    *alpha = std::isfinite(j) && bnu > 0.0 ? j / bnu : 0.0;
}

// Beyond it a vacuum ray does not circle the hole: the photon orbits and the horizon lie well inside
double near_radius(const bh_scene& S) {
    const double r_ph = 2.0 * (1.0 + std::cos(2.0 / 3.0 * std::acos(std::min(1.0, std::fabs(S.a)))));
    return std::max(3.0 * S.rh, r_ph) + 1.0;
}

// Whether the mid-plane optical depth from the flow's edge down to near_radius exceeds 1, from 16 cells in ln r
bool flow_opaque(const bh_ctx* c, const bh_scene& S) {
    constexpr int N = 16;
    const double r0 = near_radius(S), r1 = S.r_flow_max;
    if (!S.flow_on || !(r1 > r0) || c->k2_host.size() < 2) return false;
    const double dl = std::log(r1 / r0) / N;
    double tau = 0.0, w, alpha;
    for (int i = 0; i < N; ++i) {
        const double r = r0 * std::exp(dl * (i + 0.5));
        flow_cell(S, c->k2_host, c->k2_l0, c->k2_dl, r, &w, &alpha);
        tau += alpha * r * dl * S.rg_cm;
    }
    return tau > 1.0;
}

/* Radius outside which the scene's flow model emits a fraction `frac` of its emission: the thermal
   synchrotron emissivity (emission.cuh:130-170 at nu_obs, in the mid-plane, sin theta_B = 1, no
   Doppler factor, no turbulence) weighted by r^2 (a face-on annulus of height ~ h_r r), integrated
   outward from the horizon on a fine radial grid. Host-side, once per launch. */
double emission_radius(const bh_scene& S, const std::vector<float>& k2, float k2_l0, float k2_dl, double frac,
                       double tau_max) {
    const int n = 2000;
    const double r0 = S.rh * 1.001, r1 = S.r_flow_max;
    if (!(r1 > r0) || k2.size() < 2) return r1;
    const double dr = (r1 - r0) / n;
    // no storage: the bh_render_noalloc path must not allocate, so the two passes below evaluate each cell twice
    auto cell = [&](int i, double* w, double* alpha) { flow_cell(S, k2, k2_l0, k2_dl, r0 + dr * (i + 0.5), w, alpha); };
    double tot = 0.0, w, alpha;
    for (int i = 0; i < n; ++i) {
        cell(i, &w, &alpha);
        tot += w;
    }
    if (!(tot > 0.0)) return r1;
    // outermost radius where the emission outside still exceeds frac of the total, or the mid-plane
    // radial optical depth from there to the flow's edge exceeds tau_max
    double out = 0.0, tau = 0.0;
    for (int i = n - 1; i >= 0; --i) {
        cell(i, &w, &alpha);
        out += w;
        tau += alpha * dr * S.rg_cm;
        if (out > frac * tot || tau > tau_max) return r0 + dr * (i + 1.0);
    }
    return r0;
}

// Default bound on a mixed-tracer step's coordinate-time error (M) for time-dependent turbulence
constexpr double DEFAULT_TOL_T = 1e-3;
double time_bound(const bh_ctx* c, const bh_scene& S, const bh_trace_opts& o) {
    if (o.tol_t > 0) return o.tol_t;
    return o.tol_t == 0 && flow_reads_time(c, S) && S.flow_turb_amp > 0.f ? DEFAULT_TOL_T : 0.0;
}
// Default long-ray relaxation: off until measured
constexpr int DEFAULT_RELAX_AFTER = 0;
constexpr double DEFAULT_TOL_RELAX = 1e-9;
constexpr double DEFAULT_RELAX_CAP = 1.0;

// Log-space emission constants and the region split of the mixed policy
bhm32::MixedParams make_mixed(bh_ctx* c, const bh_scene& S, const bh_frame* f, const bh_trace_opts& o) {
    constexpr double C = C_C, H = C_H, ME = C_ME, MP = C_MP, QE = C_QE, PI = C_PI;
    bhm32::MixedParams M;
    std::memset(&M, 0, sizeof M);
    const bool radio = S.mode == BH_MODE_RADIO && S.flow_on;
    M.tol_mid = std::max(1e-6, S.tol);
    M.tol_far = M.tol_mid;
    if (o.tol_far > 0) {
        M.tol_far = o.tol_far;
    } else if (radio && f && f->pix > 0 && f->r > 0) {
        // far-field error that stays far below a pixel: 1e-4 on 0.04 M pixels (1024^2 over 40 M, where
        // CPU sweeps against the FP64 oracle give 6e-7 flux and 2e-5 median pixel error), scaled
        // with the pixel size at the hole (pix is an angle: pix * r in M), at most 1e-4. A camera
        // within 15 degrees of the spin axis scales it further by sin(theta_cam) / sin(15 deg): the
        // norm bounds the error of u = cos(theta), and near the axis the polar angle's error is that
        // divided by sin(theta) (a 5.7-degree view of turbulent flow lost 8e-4 of its flux at 1e-4,
        // 2e-6 at 5e-5). At least max(1e-6, tol).
        const double axis = std::min(1.0, std::fabs(std::sin(f->th)) / std::sin(15.0 * PI / 180.0));
        M.tol_far = std::max(M.tol_mid, std::min(1e-4, 1e-4 * (f->pix * f->r) / 0.04) * axis);
    }
    const double r_near = o.r_near > 0 ? o.r_near : near_radius(S);
    M.r_far = r_near;
    M.r_tol = r_near;
    if (S.mode == BH_MODE_RADIO && S.flow_on) {
        double r_emit = o.r_emit;
        if (!(r_emit > 0)) {
            // cached per flow model: a batch of frames usually shares a few scenes
            const double key[10] = {S.n0, S.n_index, S.theta0, S.theta_index, S.beta_p, S.nu_obs, S.rh, S.r_flow_max,
                                    (double)c->k2_l0, S.rg_cm};
            for (const auto& e : c->emit_cache)
                if (std::memcmp(e.first.data(), key, sizeof key) == 0) r_emit = e.second;
            if (!(r_emit > 0)) {
                r_emit = emission_radius(S, c->k2_host, c->k2_l0, c->k2_dl, 1e-6, 1e-7);
                if (c->emit_cache.size() >= 64) c->emit_cache.clear();
                std::array<double, 10> k;
                std::memcpy(k.data(), key, sizeof key);
                c->emit_cache.emplace_back(k, r_emit);
            }
        }
        M.r_far = std::max(S.r_flow_max, r_near);
        M.r_tol = std::max(std::min(r_emit, S.r_flow_max), r_near);
        M.r_cut = o.full_flow ? S.r_flow_max : M.r_tol;
        // outside the emission region the steps no longer follow the transfer step cap: a tolerance
        // between the scene's and the far field's keeps the entry point into the region accurate
        if (!o.full_flow) M.tol_mid = std::max(M.tol_mid, M.tol_far * 0.1);
    }
    M.r_f32 = o.far_fp32 ? M.r_far : 1e300;
    const double tol_t = time_bound(c, S, o);
    M.inv_tol_t = tol_t > 0 ? 1.0 / tol_t : 0.0;
    // long-ray relaxation of the emission-region tolerance
    M.relax_after = o.relax_after > 0 ? o.relax_after : (o.relax_after == 0 ? DEFAULT_RELAX_AFTER : 0x7fffffff);
    M.tol_relax = o.tol_relax > 0 ? o.tol_relax : std::max(S.tol, DEFAULT_TOL_RELAX);
    M.relax_cap = o.relax_cap > 0 ? o.relax_cap : DEFAULT_RELAX_CAP;
    if (M.relax_after <= 0) M.relax_after = 0x7fffffff;
    M.inv_tol = 1.0 / S.tol;
    M.inv_tol_mid = 1.0 / M.tol_mid;
    M.inv_tol_far = 1.0 / M.tol_far;
    M.inv_tol_relax = 1.0 / M.tol_relax;
    bhm32::EmisParams& E = M.E;
    E.ln_n0 = (float)std::log(S.n0);
    E.n_index = (float)S.n_index;
    E.ln_theta0 = (float)std::log(S.theta0);
    E.theta_index = (float)S.theta_index;
    E.h_r = (float)S.h_r;
    E.inv_h_r = (float)(1.0 / S.h_r);
    E.r_flow_max = (float)S.r_flow_max;
    E.rh = (float)S.rh;
    E.r_isco = (float)S.r_isco;
    E.flow_kep = (float)S.flow_kep;
    E.a = (float)S.a;
    E.a2 = (float)(S.a * S.a);
    E.ln_bconst = (float)std::log(8.0 * PI * MP * C * C / (6.0 * S.beta_p));
    E.ln_nuc_per_B = (float)std::log(QE / (2.0 * PI * ME * C));
    E.ln_jconst = (float)std::log(1.4142135623730951 * PI * QE * QE / (3.0 * C));
    E.ln_bnu_const = (float)std::log(2.0 * H / (C * C));
    E.ln_h_over_mec2 = (float)std::log(H / (ME * C * C));
    E.ln_nu_obs = (float)std::log(S.nu_obs);
    E.ln_rg = (float)std::log(S.rg_cm);
    E.k2_inv_dl = c->k2_dl > 0.f ? 1.f / c->k2_dl : 0.f;
    M.ln_e2_over_c = (float)std::log(QE * QE / C);
    M.ln_e2_over_mec = (float)std::log(QE * QE / (ME * C));
    return M;
}

int check_opts(bh_ctx* c, const bh_trace_opts& o) {
    if (o.precision != BH_PREC_FP64 && o.precision != BH_PREC_MIXED) return fail(c, BH_ERR_ARG, "bad precision");
    if (o.emissivity != BH_EMIS_EXACT && o.emissivity != BH_EMIS_MLP) return fail(c, BH_ERR_ARG, "bad emissivity");
    if (o.emissivity == BH_EMIS_MLP && o.precision != BH_PREC_MIXED)
        return fail(c, BH_ERR_ARG, "the MLP emissivity runs in the mixed-precision tracer");
    if (o.emissivity == BH_EMIS_MLP && !c->stab_ready)
        return fail(c, BH_ERR_UNSUPPORTED, "no baked surrogate: call bh_mlp_train (or bh_mlp_set) and bh_mlp_bake first");
    if (o.engine != BH_ENGINE_AUTO && o.engine != BH_ENGINE_FRAME) return fail(c, BH_ERR_ARG, "engine must be 0 or 1");
    if (o.precision == BH_PREC_MIXED && !(c->S.tol > 0.0))
        return fail(c, BH_ERR_ARG, "the mixed-precision tracer needs a scene tolerance > 0");
    return BH_OK;
}

// Workgroups of the frame kernel for a w x h tile: 16 x 16 tiles padded to a multiple of the XCDs.
int trace_blocks(int w, int h, int* per_xcd) {
    const int ntiles = ((w + TILE - 1) / TILE) * ((h + TILE - 1) / TILE);
    *per_xcd = (ntiles + NXCD - 1) / NXCD;
    return *per_xcd * NXCD;
}

// Frame-kernel launch of a w x h tile at (x0, y0) into the given device buffers (px or rays, the
// block partials blk[nb] and the total), then the block reduction; fills the stats counters.
// Allocates nothing: the callers provide every buffer, and the sheared turbulence slices must already
// have room for this frame's bake when may_alloc is false.
int launch_trace_into(bh_ctx* c, const bh_frame* f, const bh_trace_opts& o, int x0, int y0, int w, int h, bool rays,
                      float4* px, bh_ray_out* rays_out, BlockOut* blk, BlockOut* tot_dev, bool may_alloc,
                      bh_stats* st) {
    bhm32::MixedParams M = make_mixed(c, c->S, f, o);
    if (o.emissivity == BH_EMIS_MLP) {
        M.use_surrogate = 1;
        M.S = c->stab;
    }
    int rc = prepare_turbulence(c, c->S, f, may_alloc);
    if (rc) return rc;
    TraceParams P = make_params(c, f);
    P.x0 = x0;
    P.y0 = y0;
    P.w = w;
    P.h = h;
    P.spp = o.spp > 0 ? o.spp : (f->spp > 0 ? f->spp : 1);
    if (rays) P.spp = 1;
    P.jitter = o.jitter;
    int per_xcd;
    const int nb = trace_blocks(w, h, &per_xcd);
    KernelFn k = pick_kernel(o.precision, variant_of(c, c->S, o), rays);
    HIPCK(c, hipEventRecord(c->ev0, c->st));
    hipLaunchKernelGGL(k, dim3(nb), dim3(BLOCK), 0, c->st, P, M, px, rays_out, blk, per_xcd);
    HIPCK(c, hipGetLastError());
    HIPCK(c, hipEventRecord(c->ev1, c->st));
    hipLaunchKernelGGL(k_reduce, dim3(1), dim3(256), 0, c->st, blk, nb, tot_dev);
    HIPCK(c, hipGetLastError());
    BlockOut tot;
    HIPCK(c, hipMemcpyAsync(&tot, tot_dev, sizeof tot, hipMemcpyDeviceToHost, c->st));
    HIPCK(c, hipStreamSynchronize(c->st));
    if (st) {
        float ms = 0.f;
        HIPCK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
        st->ms_kernel = ms;
        st->samples = (long long)w * h * P.spp;
        st->step_attempts = (long long)tot.cnt[0];
        st->steps_accepted = (long long)tot.cnt[1];
        st->flow_steps = (long long)tot.cnt[2];
        st->step_limited = (long long)tot.cnt[3];
        st->fp64_steps = (long long)tot.cnt[4];
        st->flux_sum = tot.flux;
    }
    return BH_OK;
}

// Launches the trace of a w x h tile at (x0, y0) and the block reduction into the context's buffers;
// fills stats counters.
int launch_trace(bh_ctx* c, const bh_frame* f, const bh_trace_opts* opts, int x0, int y0, int w, int h, bool rays,
                 bh_stats* st) {
    int rc = check_frame(c, f);
    if (rc) return rc;
    if (w <= 0 || h <= 0) return fail(c, BH_ERR_ARG, "empty tile");
    bh_trace_opts o{};
    if (opts) o = *opts;
    rc = check_opts(c, o);
    if (rc) return rc;
    int per_xcd;
    const int nb = trace_blocks(w, h, &per_xcd);
    rc = ensure(c, &c->d_blk, &c->blk_cap, (size_t)nb);
    if (rc) return rc;
    if (rays) rc = ensure(c, &c->d_rays, &c->rays_cap, (size_t)w * h);
    else rc = ensure(c, &c->d_px, &c->px_cap, (size_t)w * h);
    if (rc) return rc;
    return launch_trace_into(c, f, o, x0, y0, w, h, rays, c->d_px, c->d_rays, c->d_blk, c->d_tot, true, st);
}

using PersistFn = void (*)(const bhp::BatchWork, unsigned int*, int, int, int, BlockOut*);

template <class Work>
using WorkFn = void (*)(const Work, unsigned int*, int, int, int, BlockOut*);

template <int PREC, int W, class Work>
struct PersistAt {
    template <int RADIO, bool TIME>
    WorkFn<Work> operator()() const {
        return k_persist<PREC, RADIO, TIME, W, Work>;
    }
};

template <int W, class Work>
WorkFn<Work> pick_persist_w(int prec, const Variant& v) {
    return prec == BH_PREC_FP64 ? pick_variant<BH_PREC_FP64, Work::RECORDS>(v, PersistAt<BH_PREC_FP64, W, Work>{})
                                : pick_variant<BH_PREC_MIXED, Work::RECORDS>(v, PersistAt<BH_PREC_MIXED, W, Work>{});
}

template <int PREC, class Work>
struct PairAt {
    template <int RADIO, bool TIME>
    WorkFn<Work> operator()() const {
        if constexpr (RADIO == bhd::RADIO_OFF) return nullptr;
        else return k_pair<PREC, RADIO, TIME, Work>;
    }
};

template <class Work>
WorkFn<Work> pick_pair(int prec, const Variant& v) {
    return prec == BH_PREC_FP64 ? pick_variant<BH_PREC_FP64, Work::RECORDS>(v, PairAt<BH_PREC_FP64, Work>{})
                                : pick_variant<BH_PREC_MIXED, Work::RECORDS>(v, PairAt<BH_PREC_MIXED, Work>{});
}

// adaptive passes and ray records: the kernel compiled for at least 3 waves per SIMD (waves 3 or 4) or
// for the compiler's register budget (waves 0)
template <class Work>
WorkFn<Work> pick_adaptive(int prec, const Variant& v, int waves) {
    return waves >= 3 ? pick_persist_w<3, Work>(prec, v) : pick_persist_w<1, Work>(prec, v);
}

PersistFn pick_persist(int prec, const Variant& v, int waves) {
    switch (waves) {
        case 3: return pick_persist_w<3, bhp::BatchWork>(prec, v);
        case 4: return pick_persist_w<4, bhp::BatchWork>(prec, v);
        default: return pick_persist_w<1, bhp::BatchWork>(prec, v);
    }
}

// Grid of a persistent launch: grid_per_cu workgroups per CU, but no more than the CU holds at once
// for this kernel and block size (register file, LDS). A workgroup beyond that waits for a slot and
// only starts once others have drained most of the queue, so its rays become the frame's tail.
int persist_grid(const bh_ctx* c, const void* k, int block, int grid_per_cu) {
    int resident = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&resident, k, block, 0) == hipSuccess && resident > 0)
        grid_per_cu = std::min(grid_per_cu, resident);
    return c->n_cu * grid_per_cu;
}

constexpr size_t PLAIN_SPP_SAMPLE_BUDGET = size_t(1) << 30;   // bytes of per-sample storage of bh_render, spp > 1
constexpr size_t FLUX_SAMPLES_KEPT = size_t(64) << 20;   // bytes of bh_radio_flux's samples that outlive the call (n = 1024)
constexpr long long BATCH_MAX_PIXELS = 1ll << 30;   // per frame: keeps the 32-bit queue counters from wrapping

// Replaces the 0 ("default") fields of a launch configuration and checks the ranges.
int resolve_cfg(bh_ctx* c, const bh_batch_cfg& d, bh_batch_cfg* g) {
    if (g->block == 0) g->block = d.block;
    if (g->grid_per_cu == 0) g->grid_per_cu = d.grid_per_cu;
    if (g->interval == 0) g->interval = d.interval;
    if (g->refill_min == 0) g->refill_min = d.refill_min;
    if (g->order == 0) g->order = d.order;
    if (g->prio_age == 0) g->prio_age = d.prio_age;
    if (g->block != 64 && g->block != 128 && g->block != 256) return fail(c, BH_ERR_ARG, "block must be 64, 128 or 256");
    if (g->grid_per_cu < 1 || g->grid_per_cu > 32) return fail(c, BH_ERR_ARG, "grid_per_cu must be in [1, 32]");
    if (g->interval < 1 || g->interval > 4096) return fail(c, BH_ERR_ARG, "interval must be in [1, 4096]");
    if (g->refill_min < 1 || g->refill_min > 64) return fail(c, BH_ERR_ARG, "refill_min must be in [1, 64]");
    if (g->waves != 0 && g->waves != 3 && g->waves != 4) return fail(c, BH_ERR_ARG, "waves must be 0, 3 or 4");
    if (g->order != BH_ORDER_ROWS && g->order != BH_ORDER_IMPACT && g->order != BH_ORDER_CRITICAL)
        return fail(c, BH_ERR_ARG, "order must be 0, 1, 2 or 3");
    if (g->prio_age > (1 << 24)) return fail(c, BH_ERR_ARG, "prio_age must be at most 2^24");
    return BH_OK;
}

// What a launch over `n` frames' descriptors has to do; entries: its rays. With regions: the frames' P.x0 .. P.h
// are the regions traced, each with nentries rays; else where its rays lie is not known, and all of them count
// as reaching the flow.
launch::Load load_of(bh_ctx* c, int prec, const Variant& v, const bhp::BatchFrame* B, const bh_scene* const* scenes,
                     int n, long long entries, bool regions) {
    launch::Load l;
    l.precision = prec;
    l.radio = v.radio;
    l.w = (double)entries / 64.0 / c->n_cu;
    l.reach = l.w;
    // only where launch::pairs asks
    if (v.radio == bhd::RADIO_OFF || prec != BH_PREC_MIXED || l.w <= launch::PAIR_REACH_OPAQUE || l.w > launch::PAIR_W_MIXED)
        return l;
    double rays = 0.0;
    const bh_scene* last = nullptr;   // frames of a batch usually share their flow
    for (int i = 0; i < n; ++i) {
        const TraceParams& P = B[i].P;
        if (regions)
            rays += (double)B[i].nentries * launch::share_within(B[i].M.r_cut, P.kp[0], P.cx, P.cy, P.pix, P.W, P.H, P.x0,
                                                                 P.y0, P.w, P.h);
        if (l.opaque || (last && std::memcmp(last, scenes[i], sizeof *last) == 0)) continue;
        last = scenes[i];
        l.opaque = flow_opaque(c, *last);
    }
    if (regions) l.reach = rays / 64.0 / c->n_cu;
    return l;
}

// The kernel and grid of a persistent launch: two waves per 64 rays where launch::pairs and the
// configuration's shape say so, else the kernel `plain`.
template <class Work>
struct PersistPlan {
    WorkFn<Work> k;
    int block, grid;
};

template <class Work>
PersistPlan<Work> plan_persist(const bh_ctx* c, const launch::Load& load, const Variant& v, const bh_batch_cfg& g,
                               WorkFn<Work> plain) {
    PersistPlan<Work> p{plain, g.block, 0};
    if (launch::pairs(load) && launch::pair_shape(g)) {
        p.k = pick_pair<Work>(load.precision, v);
        p.block = bhp::PAIR_BLOCK;
    }
    p.grid = persist_grid(c, (const void*)p.k, p.block, g.grid_per_cu);
    return p;
}

// Enqueues the counting sort that fills each frame's tile order (frames already on the device;
// hist holds n * ORDER_BUCKETS counters).
void enqueue_tile_order(hipStream_t st, const bhp::BatchFrame* dframes, int n, unsigned int max_tiles,
                        unsigned int* hist, int order) {
    const int nh = n * ORDER_BUCKETS;
    hipLaunchKernelGGL(k_zero_u32, dim3((nh + 255) / 256), dim3(256), 0, st, hist, nh);
    const dim3 og((max_tiles + 255) / 256, n);
    using OrderFn = void (*)(const bhp::BatchFrame*, unsigned int*);
    const bool crit = order == BH_ORDER_CRITICAL;
    const OrderFn count = crit ? k_order_tiles<false, BH_ORDER_CRITICAL> : k_order_tiles<false, BH_ORDER_IMPACT>;
    const OrderFn scatter = crit ? k_order_tiles<true, BH_ORDER_CRITICAL> : k_order_tiles<true, BH_ORDER_IMPACT>;
    hipLaunchKernelGGL(count, og, dim3(256), 0, st, dframes, hist);
    hipLaunchKernelGGL(k_order_scan, dim3(n), dim3(256), 0, st, hist);
    hipLaunchKernelGGL(scatter, og, dim3(256), 0, st, dframes, hist);
}

// Traces a batch with one persistent launch: [queue reset, k_persist, k_reduce], captured into a
// hipGraph (rebuilt when a buffer, the kernel or the launch shape changes) or launched directly.
// cfg_out (nullable): the configuration with its defaults filled in.
int launch_batch(bh_ctx* c, const bh_batch_frame* frames, int n, const bh_trace_opts* opts, const bh_batch_cfg* cfg_in,
                 long long* npix_out, bh_stats* st, bh_batch_cfg* cfg_out = nullptr) {
    if (!frames || n <= 0) return fail(c, BH_ERR_ARG, "empty batch");
    bh_trace_opts o{};
    if (opts) o = *opts;
    int rc = check_opts(c, o);
    if (rc) return rc;
    // one kernel for all frames: it integrates the coordinate time if any of them reads it
    Variant v = variant_of(c, frames[0].scene, o);
    for (int i = 1; i < n; ++i) v.time = v.time || variant_of(c, frames[i].scene, o).time;
    const int mode = frames[0].scene.mode;
    if (c->turb_model == BH_TURB_SHEARED) {
        // one set of slices per launch: every frame must see the same turbulence bake
        for (int i = 1; i < n; ++i) {
            const bh_scene& A = frames[0].scene;
            const bh_scene& Bs = frames[i].scene;
            if (frames[i].frame.t != frames[0].frame.t || frames[i].frame.r != frames[0].frame.r || Bs.a != A.a ||
                Bs.flow_turb_amp != A.flow_turb_amp || Bs.flow_turb_scale != A.flow_turb_scale ||
                Bs.flow_tcorr != A.flow_tcorr || Bs.seed != A.seed || Bs.h_r != A.h_r || Bs.rh != A.rh ||
                Bs.r_flow_max != A.r_flow_max)
                return fail(c, BH_ERR_UNSUPPORTED,
                            "sheared turbulence: the frames of a batch must share the camera time and radius and "
                            "the scene's noise parameters (one bake per launch)");
        }
        rc = prepare_turbulence(c, frames[0].scene, &frames[0].frame);
        if (rc) return rc;
    }
    long long total = 0, entries = 0;
    std::vector<bhp::BatchFrame> hb((size_t)n);
    std::vector<const bh_scene*> scenes((size_t)n);
    for (int i = 0; i < n; ++i) {
        const bh_frame* f = &frames[i].frame;
        const bh_scene& S = frames[i].scene;
        scenes[(size_t)i] = &S;
        if (f->W <= 0 || f->H <= 0 || (long long)f->W * f->H > BATCH_MAX_PIXELS)
            return fail(c, BH_ERR_ARG, "bad frame size in batch (at most 2^30 pixels per frame)");
        if (!(f->pix > 0.0)) return fail(c, BH_ERR_ARG, "frame pixel scale must be > 0");
        if (S.mode != mode) return fail(c, BH_ERR_ARG, "all frames of a batch must share the render mode");
        if (S.mode == BH_MODE_RADIO && S.flow_on && !c->d_k2) return fail(c, BH_ERR_ARG, "radio mode needs the K2 table");
        bhp::BatchFrame& B = hb[(size_t)i];
        std::memset(&B, 0, sizeof B);
        B.P = make_params_scene(c, S, f);
        B.P.w = f->W;
        B.P.h = f->H;
        B.P.spp = 1;
        B.P.jitter = o.jitter;
        B.M = make_mixed(c, S, f, o);
        if (o.emissivity == BH_EMIS_MLP) {
            B.M.use_surrogate = 1;
            B.M.S = c->stab;
        }
        B.tiles_x = (f->W + 7) / 8;
        B.nentries = (unsigned int)((long long)B.tiles_x * ((f->H + 7) / 8) * 64);
        entries += B.nentries;
        total += (long long)f->W * f->H;
    }
    const launch::Load load = load_of(c, o.precision, v, hb.data(), scenes.data(), n, entries, true);
    const bh_batch_cfg dflt = launch::defaults(load);
    bh_batch_cfg cfg = cfg_in ? *cfg_in : launch::choose(c->tuned[o.precision], load, dflt);
    rc = resolve_cfg(c, dflt, &cfg);
    if (rc) return rc;
    if (cfg_out) *cfg_out = cfg;
    rc = ensure(c, &c->d_bout, &c->bout_cap, (size_t)total);
    if (rc) return rc;
    long long off = 0;
    for (int i = 0; i < n; ++i) {
        hb[(size_t)i].out = c->d_bout + off;
        off += (long long)frames[i].frame.W * frames[i].frame.H;
    }
    // tile order (grid y = frame, so at most 65535 frames are sorted; larger batches keep row order)
    const bool ordered = cfg.order != BH_ORDER_ROWS && n <= 65535;
    unsigned int max_tiles = 0;
    if (ordered) {
        rc = ensure(c, &c->d_order, &c->order_cap, (size_t)(total + 63));   // >= tiles of all frames
        if (rc) return rc;
        rc = ensure(c, &c->d_ohist, &c->ohist_cap, (size_t)n * ORDER_BUCKETS);
        if (rc) return rc;
        long long toff = 0;
        for (int i = 0; i < n; ++i) {
            const unsigned int nt = hb[(size_t)i].nentries >> 6;
            hb[(size_t)i].order = c->d_order + toff;
            toff += nt;
            max_tiles = std::max(max_tiles, nt);
        }
    }
    const int prio = cfg.prio_age > 0 ? cfg.prio_age : 0;
    const auto plan = plan_persist<bhp::BatchWork>(c, load, v, cfg, pick_persist(o.precision, v, cfg.waves));
    const PersistFn k = plan.k;
    const int grid = plan.grid;
    rc = ensure(c, &c->d_bframes, &c->bframes_cap, sizeof(bhp::BatchFrame) * (size_t)n);
    if (rc) return rc;
    rc = ensure(c, &c->d_queue, &c->queue_cap, (size_t)n);
    if (rc) return rc;
    rc = ensure(c, &c->d_blk, &c->blk_cap, (size_t)grid);
    if (rc) return rc;
    HIPCK(c, hipMemcpyAsync(c->d_bframes, hb.data(), sizeof(bhp::BatchFrame) * (size_t)n, hipMemcpyHostToDevice, c->st));
    const bhp::BatchFrame* dframes = (const bhp::BatchFrame*)c->d_bframes;
    auto enqueue = [&]() -> hipError_t {
        hipLaunchKernelGGL(k_zero_u32, dim3((n + 255) / 256), dim3(256), 0, c->st, c->d_queue, n);
        if (ordered) enqueue_tile_order(c->st, dframes, n, max_tiles, c->d_ohist, cfg.order);
        hipLaunchKernelGGL(k, dim3(grid), dim3(plan.block), 0, c->st, bhp::BatchWork{dframes, n}, c->d_queue,
                           cfg.interval, cfg.refill_min, prio, c->d_blk);
        hipLaunchKernelGGL(k_reduce, dim3(1), dim3(256), 0, c->st, c->d_blk, grid, c->d_tot);
        return hipGetLastError();
    };
    HIPCK(c, hipEventRecord(c->ev0, c->st));
    if (cfg.use_graph) {
        // everything the captured launches depend on, except the frame descriptors (copied above)
        unsigned long long key = 1469598103934665603ull;
        const unsigned long long parts[] = {(unsigned long long)(uintptr_t)k, (unsigned long long)(uintptr_t)dframes,
                                            (unsigned long long)(uintptr_t)c->d_queue,
                                            (unsigned long long)(uintptr_t)c->d_blk,
                                            (unsigned long long)(uintptr_t)c->d_tot, (unsigned long long)n,
                                            (unsigned long long)grid, (unsigned long long)plan.block,
                                            (unsigned long long)cfg.interval, (unsigned long long)cfg.refill_min,
                                            (unsigned long long)ordered, (unsigned long long)max_tiles,
                                            (unsigned long long)(uintptr_t)c->d_ohist, (unsigned long long)prio,
                                            (unsigned long long)cfg.order};
        for (unsigned long long v : parts) key = (key ^ v) * 1099511628211ull;
        if (!c->graph || c->graph_key != key) {
            if (c->graph) {
                HIPCK(c, hipGraphExecDestroy(c->graph));
                c->graph = nullptr;
            }
            if (c->graph_def) {
                HIPCK(c, hipGraphDestroy(c->graph_def));
                c->graph_def = nullptr;
            }
            HIPCK(c, hipStreamBeginCapture(c->st, hipStreamCaptureModeThreadLocal));
            hipError_t le = enqueue();
            hipGraph_t g = nullptr;
            hipError_t ce = hipStreamEndCapture(c->st, &g);
            HIPCK(c, le);
            HIPCK(c, ce);
            c->graph_def = g;
            HIPCK(c, hipGraphInstantiate(&c->graph, g, nullptr, nullptr, 0));
            c->graph_key = key;
        }
        HIPCK(c, hipGraphLaunch(c->graph, c->st));
    } else {
        HIPCK(c, enqueue());
    }
    HIPCK(c, hipEventRecord(c->ev1, c->st));
    BlockOut tot;
    HIPCK(c, hipMemcpyAsync(&tot, c->d_tot, sizeof tot, hipMemcpyDeviceToHost, c->st));
    HIPCK(c, hipStreamSynchronize(c->st));
    if (npix_out) *npix_out = total;
    if (st) {
        float ms = 0.f;
        HIPCK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
        st->ms_kernel = ms;
        st->samples = total;
        st->step_attempts = (long long)tot.cnt[0];
        st->steps_accepted = (long long)tot.cnt[1];
        st->flow_steps = (long long)tot.cnt[2];
        st->step_limited = (long long)tot.cnt[3];
        st->fp64_steps = (long long)tot.cnt[4];
        st->flux_sum = tot.flux;
    }
    return BH_OK;
}

// Ray records of a w x h region at (x0, y0) (bh_trace_tile) with one persistent launch: the region's
// 8 x 8 tiles are the queue entries, in the launch configuration's order; the records land in d_rays.
// The rays and their records are those of the frame kernel (same per-ray code).
int launch_records(bh_ctx* c, const bh_frame* f, const bh_trace_opts* opts, int x0, int y0, int w, int h) {
    int rc = check_frame(c, f);
    if (rc) return rc;
    if (w <= 0 || h <= 0) return fail(c, BH_ERR_ARG, "empty tile");
    if ((long long)w * h > BATCH_MAX_PIXELS) return fail(c, BH_ERR_ARG, "tile too large (2^30 rays)");
    bh_trace_opts o{};
    if (opts) o = *opts;
    rc = check_opts(c, o);
    if (rc) return rc;
    const int tiles_x = (w + 7) / 8, tiles = tiles_x * ((h + 7) / 8);
    const Variant v = variant_of(c, c->S, o);
    rc = prepare_turbulence(c, c->S, f);
    if (rc) return rc;
    bhp::BatchFrame B;
    std::memset(&B, 0, sizeof B);
    B.P = make_params(c, f);
    B.P.x0 = x0;
    B.P.y0 = y0;
    B.P.w = w;
    B.P.h = h;
    B.P.spp = 1;
    B.P.jitter = o.jitter;
    B.M = make_mixed(c, c->S, f, o);
    if (o.emissivity == BH_EMIS_MLP) {
        B.M.use_surrogate = 1;
        B.M.S = c->stab;
    }
    B.tiles_x = tiles_x;
    B.nentries = (unsigned int)tiles * 64u;
    const bh_scene* scene = &c->S;
    const launch::Load load = load_of(c, o.precision, v, &B, &scene, 1, (long long)tiles * 64, true);
    const bh_batch_cfg cfg = launch::choose(c->tuned[o.precision], load, launch::defaults(load));
    const auto plan = plan_persist<bhp::RecordWork>(c, load, v, cfg,
                                                    pick_adaptive<bhp::RecordWork>(o.precision, v, cfg.waves));
    const int grid = plan.grid;
    const bool ordered = cfg.order != BH_ORDER_ROWS;
    if (ordered) {
        if ((rc = ensure(c, &c->d_order, &c->order_cap, (size_t)tiles)) ||
            (rc = ensure(c, &c->d_ohist, &c->ohist_cap, (size_t)ORDER_BUCKETS)))
            return rc;
        B.order = c->d_order;
    }
    if ((rc = ensure(c, &c->d_bframes, &c->bframes_cap, sizeof B)) || (rc = ensure(c, &c->d_queue, &c->queue_cap, 1)) ||
        (rc = ensure(c, &c->d_blk, &c->blk_cap, (size_t)grid)) ||
        (rc = ensure(c, &c->d_rays, &c->rays_cap, (size_t)w * h)))
        return rc;
    const bhp::BatchFrame* dB = (const bhp::BatchFrame*)c->d_bframes;
    HIPCK(c, hipMemcpyAsync(c->d_bframes, &B, sizeof B, hipMemcpyHostToDevice, c->st));
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, c->st, c->d_queue, 1);
    if (ordered) enqueue_tile_order(c->st, dB, 1, (unsigned int)tiles, c->d_ohist, cfg.order);
    hipLaunchKernelGGL(plan.k, dim3(grid), dim3(plan.block), 0, c->st, bhp::RecordWork{dB, 1, c->d_rays}, c->d_queue,
                       cfg.interval, cfg.refill_min, cfg.prio_age > 0 ? cfg.prio_age : 0, c->d_blk);
    HIPCK(c, hipGetLastError());
    return BH_OK;
}

// A persistent launch over the samples of a frame: every (tile, sample, pixel) entry's intensities in
// d_samp1[pixel * spp + sample]. Enqueues the launch and fills B[0] (the frame's descriptor) and B[1]
// (the same with one entry per pixel). The caller has checked the frame, the options and the sizes.
int launch_samples(bh_ctx* c, const bh_frame* f, const bh_trace_opts& o, int spp, bhp::BatchFrame B[2],
                   bh_batch_cfg* cfg_out, int* grid_out) {
    const int W = f->W, H = f->H;
    const int tiles_x = (W + 7) / 8, tiles = tiles_x * ((H + 7) / 8);
    const Variant v = variant_of(c, c->S, o);
    int rc = prepare_turbulence(c, c->S, f);
    if (rc) return rc;
    std::memset(B, 0, 2 * sizeof B[0]);
    B[0].P = make_params(c, f);
    B[0].P.w = W;
    B[0].P.h = H;
    B[0].P.spp = spp;
    B[0].P.jitter = o.jitter;
    B[0].M = make_mixed(c, c->S, f, o);
    if (o.emissivity == BH_EMIS_MLP) {
        B[0].M.use_surrogate = 1;
        B[0].M.S = c->stab;
    }
    B[0].tiles_x = tiles_x;
    B[0].nentries = (unsigned int)(tiles * 64 * spp);
    const bh_scene* scene = &c->S;
    const launch::Load load = load_of(c, o.precision, v, B, &scene, 1, (long long)tiles * 64 * spp, true);
    const bh_batch_cfg cfg = launch::choose(c->tuned[o.precision], load, launch::defaults(load));
    const auto plan = plan_persist<bhp::SampleWork>(c, load, v, cfg,
                                                    pick_adaptive<bhp::SampleWork>(o.precision, v, cfg.waves));
    const int grid = plan.grid;
    const bool ordered = cfg.order != BH_ORDER_ROWS;
    if (ordered) {
        if ((rc = ensure(c, &c->d_order, &c->order_cap, (size_t)tiles)) ||
            (rc = ensure(c, &c->d_ohist, &c->ohist_cap, (size_t)ORDER_BUCKETS)))
            return rc;
        B[0].order = c->d_order;
    }
    // the sort reads nentries / 64 tiles from its descriptor and pass 1 has spp entries per pixel, so the
    // sort gets slot 1 (pass 2's, written again before pass 2) with one entry per pixel
    B[1] = B[0];
    B[1].nentries = (unsigned int)(tiles * 64);
    if ((rc = ensure(c, &c->d_bframes, &c->bframes_cap, 2 * sizeof B[0])) ||
        (rc = ensure(c, &c->d_queue, &c->queue_cap, 1)) || (rc = ensure(c, &c->d_blk, &c->blk_cap, (size_t)grid)) ||
        (rc = ensure(c, &c->d_samp1, &c->samp1_cap, (size_t)W * H * spp)))
        return rc;
    const bhp::BatchFrame* dB = (const bhp::BatchFrame*)c->d_bframes;
    HIPCK(c, hipEventRecord(c->ev0, c->st));
    HIPCK(c, hipMemcpyAsync(c->d_bframes, B, 2 * sizeof B[0], hipMemcpyHostToDevice, c->st));
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, c->st, c->d_queue, 1);
    if (ordered) enqueue_tile_order(c->st, dB + 1, 1, (unsigned int)tiles, c->d_ohist, cfg.order);
    hipLaunchKernelGGL(plan.k, dim3(grid), dim3(plan.block), 0, c->st, bhp::SampleWork{dB, 1, spp, c->d_samp1}, c->d_queue,
                       cfg.interval, cfg.refill_min, cfg.prio_age > 0 ? cfg.prio_age : 0, c->d_blk);
    HIPCK(c, hipGetLastError());
    *cfg_out = cfg;
    *grid_out = grid;
    return BH_OK;
}

// Adaptive render (render.cu:677-721): persistent pass 1 over (tile, sample, pixel) entries, the
// statistics and decisions on the device, one host read of the pass-2 size, persistent pass 2 over
// chunks, resolve. px_out / nsamp_out are device pointers (d_px, d_nsamp).
// plain_spp > 0: pass 1 only with that many samples per pixel (the plain mean of bh_render).
int launch_adaptive(bh_ctx* c, const bh_frame* f, const bh_trace_opts* opts, long long* samples, bh_stats* st,
                    int plain_spp = 0) {
    int rc = check_frame(c, f);
    if (rc) return rc;
    bh_trace_opts o{};
    if (opts) o = *opts;
    rc = check_opts(c, o);
    if (rc) return rc;
    const int spp = plain_spp > 0 ? plain_spp : (o.spp > 0 ? o.spp : (c->rs.spp > 0 ? c->rs.spp : 8));
    const int spp_max = plain_spp > 0 ? plain_spp : (c->rs.spp_max > 0 ? c->rs.spp_max : 128);
    const float target = c->rs.target_err > 0.f ? c->rs.target_err : 0.03f;
    const int W = f->W, H = f->H, npix = W * H;
    const int extra_max = std::max(spp_max - spp, 0);
    const long long tiles = (long long)((W + 7) / 8) * ((H + 7) / 8);
    if (tiles * 64 * spp >= (1ll << 31) ||
        (long long)npix * ((extra_max + ADAPT_CHUNK - 1) / ADAPT_CHUNK) * ADAPT_CHUNK >= (1ll << 31))
        return fail(c, BH_ERR_ARG, "frame too large for adaptive sampling (2^31 samples)");
    const size_t n = (size_t)npix;
    if ((rc = ensure(c, &c->d_acc, &c->acc_cap, n)) ||
        (rc = ensure(c, &c->d_ystat, &c->ystat_cap, n)) || (rc = ensure(c, &c->d_extra, &c->extra_cap, n)) ||
        (rc = ensure(c, &c->d_chunks, &c->chunks_cap, n)) || (rc = ensure(c, &c->d_offsets, &c->offsets_cap, n)) ||
        (rc = ensure(c, &c->d_bsum, &c->bsum_cap, (n + 1023) / 1024)) ||
        (rc = ensure(c, &c->d_fpart, &c->fpart_cap, (n + FSUM_BLOCK - 1) / FSUM_BLOCK)) ||
        (rc = ensure(c, &c->d_nsamp, &c->nsamp_cap, n)) || (rc = ensure(c, &c->d_px, &c->px_cap, n)))
        return rc;
    const bool radio = c->S.mode == BH_MODE_RADIO;
    bhp::BatchFrame B[2];
    bh_batch_cfg cfg;
    int grid;
    rc = launch_samples(c, f, o, spp, B, &cfg, &grid);
    if (rc) return rc;
    hipLaunchKernelGGL(k_reduce, dim3(1), dim3(256), 0, c->st, c->d_blk, grid, c->d_tot);
    HIPCK(c, hipGetLastError());
    BlockOut tot1, tot2{};
    HIPCK(c, hipMemcpyAsync(&tot1, c->d_tot, sizeof tot1, hipMemcpyDeviceToHost, c->st));
    const int lum = radio ? 0 : 1;
    hipLaunchKernelGGL(k_adapt_stats, dim3((npix + 255) / 256), dim3(256), 0, c->st, c->d_samp1, npix, spp, lum,
                       c->d_acc, c->d_ystat);
    unsigned int total = 0;
    if (extra_max > 0) {
        const int nparts = (npix + FSUM_BLOCK - 1) / FSUM_BLOCK;
        hipLaunchKernelGGL(k_adapt_fsum, dim3((nparts + 255) / 256), dim3(256), 0, c->st, c->d_ystat, npix, c->d_fpart);
        hipLaunchKernelGGL(k_adapt_extra, dim3((npix + 255) / 256), dim3(256), 0, c->st, c->d_ystat, npix, spp,
                           c->d_fpart, nparts, target, extra_max, c->d_extra);
        hipLaunchKernelGGL(k_adapt_dilate, dim3((W + 15) / 16, (H + 15) / 16), dim3(16, 16), 0, c->st, c->d_extra, W, H,
                           extra_max, c->d_chunks);
        const int nb = (npix + 1023) / 1024;
        hipLaunchKernelGGL(k_scan_block, dim3(nb), dim3(1024), 0, c->st, c->d_chunks, c->d_offsets, c->d_bsum, npix);
        hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, c->st, c->d_bsum, nb);
        hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(1024), 0, c->st, c->d_offsets, c->d_bsum, npix);
        HIPCK(c, hipGetLastError());
        unsigned int last[2];
        HIPCK(c, hipMemcpyAsync(&last[0], c->d_offsets + npix - 1, 4, hipMemcpyDeviceToHost, c->st));
        HIPCK(c, hipMemcpyAsync(&last[1], c->d_chunks + npix - 1, 4, hipMemcpyDeviceToHost, c->st));
        HIPCK(c, hipStreamSynchronize(c->st));
        total = last[0] + last[1];
        if (total > 0) {
            // pass 2's launch by its own number of rays
            const Variant v = variant_of(c, c->S, o);
            const bh_scene* scene = &c->S;
            const launch::Load load = load_of(c, o.precision, v, B, &scene, 1, (long long)total * ADAPT_CHUNK, false);
            cfg = launch::choose(c->tuned[o.precision], load, launch::defaults(load));
            const auto plan = plan_persist<bhp::ChunkWork>(c, load, v, cfg,
                                                           pick_adaptive<bhp::ChunkWork>(o.precision, v, cfg.waves));
            grid = plan.grid;
            if ((rc = ensure(c, &c->d_samp2, &c->samp2_cap, (size_t)total * ADAPT_CHUNK)) ||
                (rc = ensure(c, &c->d_blk, &c->blk_cap, (size_t)grid)))
                return rc;
            const bhp::BatchFrame* dB = (const bhp::BatchFrame*)c->d_bframes;
            B[1].nentries = total * ADAPT_CHUNK;
            B[1].order = nullptr;
            HIPCK(c, hipMemcpyAsync(c->d_bframes + sizeof(bhp::BatchFrame), &B[1], sizeof B[1], hipMemcpyHostToDevice,
                                    c->st));
            hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, c->st, c->d_queue, 1);
            hipLaunchKernelGGL(plan.k, dim3(grid), dim3(plan.block), 0, c->st,
                               bhp::ChunkWork{dB + 1, 1, spp, npix, c->d_offsets, c->d_samp2}, c->d_queue,
                               cfg.interval, cfg.refill_min, cfg.prio_age > 0 ? cfg.prio_age : 0, c->d_blk);
            hipLaunchKernelGGL(k_reduce, dim3(1), dim3(256), 0, c->st, c->d_blk, grid, c->d_tot);
            HIPCK(c, hipGetLastError());
            HIPCK(c, hipMemcpyAsync(&tot2, c->d_tot, sizeof tot2, hipMemcpyDeviceToHost, c->st));
        }
    }
    hipLaunchKernelGGL(k_adapt_resolve, dim3((npix + 255) / 256), dim3(256), 0, c->st, c->d_acc, c->d_samp2,
                       c->d_offsets, total > 0 ? c->d_chunks : nullptr, npix, spp, c->d_px, c->d_nsamp);
    HIPCK(c, hipGetLastError());
    HIPCK(c, hipEventRecord(c->ev1, c->st));
    HIPCK(c, hipStreamSynchronize(c->st));
    const long long ns = (long long)npix * spp + (long long)total * ADAPT_CHUNK;
    if (samples) *samples = ns;
    if (st) {
        float ms = 0.f;
        HIPCK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
        st->ms_kernel = ms;
        st->samples = ns;
        st->step_attempts = (long long)(tot1.cnt[0] + tot2.cnt[0]);
        st->steps_accepted = (long long)(tot1.cnt[1] + tot2.cnt[1]);
        st->flow_steps = (long long)(tot1.cnt[2] + tot2.cnt[2]);
        st->step_limited = (long long)(tot1.cnt[3] + tot2.cnt[3]);
        st->fp64_steps = (long long)(tot1.cnt[4] + tot2.cnt[4]);
        st->flux_sum = tot1.flux + tot2.flux;
    }
    return BH_OK;
}

// A whole frame on the context's scene, on the persistent engine (launched with bh_autotune's
// result for this precision or the defaults): one sample per pixel as a batch of one frame, more as
// the adaptive render's first pass alone (samples summed in index order, then divided by their
// number). The same pixels and counters as the frame kernel, without its per-tile tails. Frames
// beyond the engine's 2^31 work entries, or engine BH_ENGINE_FRAME, run the frame kernel.
// *d_out receives the device image.
int render_frame(bh_ctx* c, const bh_frame* f, const bh_trace_opts* opts, const float4** d_out, bh_stats* st) {
    int rc = check_frame(c, f);
    if (rc) return rc;
    bh_trace_opts o{};
    if (opts) o = *opts;
    const int spp = o.spp > 0 ? o.spp : (f->spp > 0 ? f->spp : 1);
    const long long entries = (long long)((f->W + 7) / 8) * ((f->H + 7) / 8) * 64 * spp;
    // the persistent path keeps every sample (FP64 x 4) until the per-pixel sums; beyond this budget
    // the frame kernel, which sums a pixel's samples in registers, gives the same pixels
    const bool samples_fit = (double)entries * sizeof(double4) <= (double)PLAIN_SPP_SAMPLE_BUDGET;
    if (o.engine == BH_ENGINE_AUTO && spp == 1 && (long long)f->W * f->H <= BATCH_MAX_PIXELS) {
        const bh_batch_frame bf{c->S, *f};
        rc = launch_batch(c, &bf, 1, &o, nullptr, nullptr, st);
        *d_out = c->d_bout;
    } else if (o.engine == BH_ENGINE_AUTO && spp > 1 && entries < (1ll << 31) && samples_fit) {
        rc = launch_adaptive(c, f, &o, nullptr, st, spp);
        *d_out = c->d_px;
    } else {
        rc = launch_trace(c, f, &o, 0, 0, f->W, f->H, false, st);
        *d_out = c->d_px;
    }
    return rc;
}

}  // namespace

extern "C" {

int bh_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int bh_create(int device, const bh_scene* scene, const bh_tables* tables, const bh_settings* settings, bh_ctx** out,
              char* err, size_t errlen) {
    auto set_err = [&](const std::string& m) {
        g_create_error = m;
        if (err && errlen) {
            std::strncpy(err, m.c_str(), errlen - 1);
            err[errlen - 1] = 0;
        }
    };
    if (!out || !scene) {
        set_err("bh_create: NULL argument");
        return BH_ERR_ARG;
    }
    *out = nullptr;
    int ndev = bh_device_count();
    if (ndev <= 0) {
        set_err("bh_create: no HIP device");
        return BH_ERR_NODEVICE;
    }
    if (device < 0 || device >= ndev) {
        set_err("bh_create: device index out of range");
        return BH_ERR_ARG;
    }
    bh_ctx* c = new bh_ctx;
    c->device = device;
    c->S = *scene;
    if (settings) c->rs = *settings;
    auto bail = [&](int code) {
        set_err(c->err);
        bh_destroy(c);
        return code;
    };
    if (hipSetDevice(device) != hipSuccess) {
        c->err = "hipSetDevice failed";
        return bail(BH_ERR_HIP);
    }
    if (hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess ||
        hipMalloc((void**)&c->d_tot, sizeof(BlockOut)) != hipSuccess) {
        c->err = "stream/event/alloc creation failed";
        return bail(BH_ERR_HIP);
    }
    if (hipDeviceGetAttribute(&c->n_cu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || c->n_cu <= 0) {
        c->err = "cannot query the compute-unit count";
        return bail(BH_ERR_HIP);
    }
    try {
        c->transfer = Transfer::of_device(device);
    } catch (...) {
        c->err = "host allocation failed";
        return bail(BH_ERR_HIP);
    }
    c->emit_cache.reserve(64);   // make_mixed then never allocates (bh_render_noalloc)
    if (device < NOALLOC_MAX_DEVICES) {
        // this device's copy of the no-alloc scratch array, resolved once with the device current
        std::lock_guard<std::mutex> lock(g_noalloc_mu);
        if (!g_noalloc_scratch[device]) {
            void* ptr = nullptr;
            if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) {
                c->err = "hipGetSymbolAddress of the no-alloc scratch array failed";
                return bail(BH_ERR_HIP);
            }
            g_noalloc_scratch[device] = static_cast<BlockOut*>(ptr);
        }
    }
    if (tables) {
        if (tables->k2_ln && tables->k2_n >= 2) {
            c->k2_n = tables->k2_n;
            c->k2_l0 = tables->k2_l0;
            c->k2_dl = tables->k2_dl;
            c->k2_host.assign(tables->k2_ln, tables->k2_ln + tables->k2_n);
            if (hipMalloc((void**)&c->d_k2, sizeof(float) * c->k2_n) != hipSuccess ||
                hipMemcpy(c->d_k2, tables->k2_ln, sizeof(float) * c->k2_n, hipMemcpyHostToDevice) != hipSuccess) {
                c->err = "K2 table upload failed";
                return bail(BH_ERR_HIP);
            }
        }
        if (tables->turb_model != BH_TURB_GRID && tables->turb_model != BH_TURB_SHEARED) {
            c->err = "turb_model must be BH_TURB_GRID or BH_TURB_SHEARED";
            return bail(BH_ERR_ARG);
        }
        if (tables->turb_model == BH_TURB_SHEARED) {
            c->turb_model = BH_TURB_SHEARED;
            const int def[4] = {512, 192, 48, 24};   // render.cu:448
            for (int i = 0; i < 4; ++i) c->ts_dims[i] = tables->ts_dims[i] > 0 ? tables->ts_dims[i] : def[i];
            const long long cells = (long long)c->ts_dims[0] * c->ts_dims[1] * c->ts_dims[2] * c->ts_dims[3];
            if (c->ts_dims[0] < 2 || c->ts_dims[1] < 2 || c->ts_dims[2] < 2 || c->ts_dims[3] < 2 ||
                cells > (1ll << 31)) {
                c->err = "sheared turbulence dimensions must be >= 2 with at most 2^31 cells";
                return bail(BH_ERR_ARG);
            }
        } else if (tables->turb && tables->turb_n >= 2) {
            int nt = tables->turb_nt > 0 ? tables->turb_nt : 1;
            if (nt > 1 && !(tables->turb_dt > 0.0)) {
                c->err = "turbulence time slices need turb_dt > 0";
                return bail(BH_ERR_ARG);
            }
            if (!(tables->turb_half > 0.0)) {
                c->err = "turbulence grid needs turb_half > 0";
                return bail(BH_ERR_ARG);
            }
            size_t n = (size_t)tables->turb_n * tables->turb_n * tables->turb_n * nt;
            if (n >= (1ull << 31)) {   // the mixed tracer addresses the slices with 32-bit offsets
                c->err = "turbulence grid must hold fewer than 2^31 cells";
                return bail(BH_ERR_ARG);
            }
            c->turb_n = tables->turb_n;
            c->turb_nt = nt;
            c->turb_half = tables->turb_half;
            c->turb_t0 = tables->turb_t0;
            c->turb_dt = tables->turb_dt;
            if (hipMalloc((void**)&c->d_turb, sizeof(float) * n) != hipSuccess ||
                hipMemcpy(c->d_turb, tables->turb, sizeof(float) * n, hipMemcpyHostToDevice) != hipSuccess) {
                c->err = "turbulence grid upload failed";
                return bail(BH_ERR_HIP);
            }
        }
    }
    *out = c;
    return BH_OK;
}

int bh_update_scene(bh_ctx* c, const bh_scene* s) {
    if (!c || !s) return BH_ERR_ARG;
    c->S = *s;
    return BH_OK;
}

int bh_get_scene(const bh_ctx* c, bh_scene* s) {
    if (!c || !s) return BH_ERR_ARG;
    *s = c->S;
    return BH_OK;
}

int bh_render(bh_ctx* c, const bh_frame* f, const bh_trace_opts* opts, float* px_out, bh_stats* st) {
    if (!c) return BH_ERR_ARG;
    double t0 = now_ms();
    HIPCK(c, hipSetDevice(c->device));
    bh_stats local{};
    const float4* img = nullptr;
    int rc = render_frame(c, f, opts, &img, &local);
    if (rc) return rc;
    if (px_out) {
        HIPCK(c, c->transfer->to_host(px_out, img, sizeof(float4) * (size_t)f->W * f->H, c->st));
    }
    local.ms_trace = now_ms() - t0;
    if (st) *st = local;
    return BH_OK;
}

int bh_render_adaptive(bh_ctx* c, const bh_frame* f, const bh_trace_opts* opts, float* px_out,
                       unsigned int* nsamp_out, bh_stats* st) {
    if (!c) return BH_ERR_ARG;
    double t0 = now_ms();
    HIPCK(c, hipSetDevice(c->device));
    bh_stats local{};
    int rc = launch_adaptive(c, f, opts, nullptr, &local);
    if (rc) return rc;
    const size_t n = (size_t)f->W * f->H;
    if (px_out) HIPCK(c, c->transfer->to_host(px_out, c->d_px, sizeof(float4) * n, c->st));
    if (nsamp_out) HIPCK(c, c->transfer->to_host(nsamp_out, c->d_nsamp, sizeof(unsigned int) * n, c->st));
    local.ms_trace = now_ms() - t0;
    if (st) *st = local;
    return BH_OK;
}

int bh_render_resident(bh_ctx* c, const bh_frame* f, const bh_trace_opts* opts, const void** d_px, bh_stats* st) {
    if (!c) return BH_ERR_ARG;
    double t0 = now_ms();
    HIPCK(c, hipSetDevice(c->device));
    bh_stats local{};
    const float4* img = nullptr;
    int rc = render_frame(c, f, opts, &img, &local);
    if (rc) return rc;
    if (d_px) *d_px = img;
    local.ms_trace = now_ms() - t0;
    if (st) *st = local;
    return BH_OK;
}

int bh_render_noalloc(bh_ctx* c, const bh_frame* f, const bh_trace_opts* opts, void* d_px, bh_stats* st) {
    if (!c) return BH_ERR_ARG;
    double t0 = now_ms();
    HIPCK(c, hipSetDevice(c->device));
    int rc = check_frame(c, f);
    if (rc) return rc;
    if (!d_px) return fail(c, BH_ERR_ARG, "bh_render_noalloc: d_px is NULL");
    bh_trace_opts o{};
    if (opts) o = *opts;
    rc = check_opts(c, o);
    if (rc) return rc;
    int per_xcd;
    const int nb = trace_blocks(f->W, f->H, &per_xcd);   // W, H <= 65536: no overflow
    if (nb > NOALLOC_MAX_BLOCKS)
        return fail(c, BH_ERR_ARG, "bh_render_noalloc: the frame needs " + std::to_string(nb) +
                                       " workgroups of 16x16 pixels; the scratch array holds " +
                                       std::to_string(NOALLOC_MAX_BLOCKS) + " (e.g. 4096 x 4096 pixels)");
    BlockOut* s = c->device < NOALLOC_MAX_DEVICES ? g_noalloc_scratch[c->device] : nullptr;
    if (!s) return fail(c, BH_ERR_UNSUPPORTED, "bh_render_noalloc: no scratch array on this device");
    bh_stats local{};
    rc = launch_trace_into(c, f, o, 0, 0, f->W, f->H, false, static_cast<float4*>(d_px), nullptr, s, s + nb, false,
                           &local);
    if (rc) return rc;
    local.ms_trace = now_ms() - t0;
    if (st) *st = local;
    return BH_OK;
}

int bh_trace_tile(bh_ctx* c, const bh_frame* f, int x0, int y0, int w, int h, const bh_trace_opts* opts,
                  bh_ray_out* out) {
    if (!c) return BH_ERR_ARG;
    if (!out) return fail(c, BH_ERR_ARG, "output is NULL");
    HIPCK(c, hipSetDevice(c->device));
    const bool frame_kernel = opts && opts->engine == BH_ENGINE_FRAME;
    int rc = frame_kernel ? launch_trace(c, f, opts, x0, y0, w, h, true, nullptr)
                          : launch_records(c, f, opts, x0, y0, w, h);
    if (rc) return rc;
    HIPCK(c, c->transfer->to_host(out, c->d_rays, sizeof(bh_ray_out) * (size_t)w * h, c->st));
    return BH_OK;
}

int bh_sheared_slices(bh_ctx* c, const bh_frame* f, float* out, size_t n) {
    if (!c || !f || !out) return BH_ERR_ARG;
    HIPCK(c, hipSetDevice(c->device));
    if (c->turb_model != BH_TURB_SHEARED) return fail(c, BH_ERR_ARG, "the context has no sheared turbulence");
    const size_t total = (size_t)c->ts_dims[0] * c->ts_dims[1] * c->ts_dims[2] * c->ts_dims[3];
    if (n < total) return fail(c, BH_ERR_ARG, "output too small for the turbulence slices");
    bh_scene S = c->S;
    S.mode = BH_MODE_RADIO;
    S.flow_on = 1;
    if (!(S.flow_turb_amp > 0.f)) return fail(c, BH_ERR_ARG, "the scene has no turbulence (flow_turb_amp = 0)");
    int rc = prepare_turbulence(c, S, f);
    if (rc) return rc;
    HIPCK(c, c->transfer->to_host(out, c->d_ts, sizeof(float) * total, c->st));
    return BH_OK;
}

int bh_radio_flux(bh_ctx* c, const bh_frame* f, int n, double pix_sr, double* jy) {
    if (!c || !f || !jy || n <= 0) return BH_ERR_ARG;
    HIPCK(c, hipSetDevice(c->device));
    bh_frame g = *f;
    g.W = n;
    g.H = n;
    g.spp = 2;
    bh_trace_opts o{};
    o.precision = BH_PREC_FP64;
    o.jitter = 1;
    o.spp = 2;
    bh_stats st{};
    int rc = check_frame(c, &g);
    if (rc) return rc;
    const long long entries = (long long)((n + 7) / 8) * ((n + 7) / 8) * 64 * o.spp;
    const size_t samples = (size_t)n * n * o.spp, had = c->samp1_cap;
    if ((double)entries * sizeof(double4) <= (double)PLAIN_SPP_SAMPLE_BUDGET &&
        try_ensure(c, &c->d_samp1, &c->samp1_cap, samples)) {
        // Each sample a ray of its own on the persistent engine. The frame kernel traces a pixel's two
        // samples one after the other and n = 160 is 100 workgroups for 256 CUs: it ends with the longest
        // pair of rays on a lane, this with the longest ray (the 0.6 Jy flow at 17 degrees, n = 160, 512,
        // 1024, 2048: 8.1, 28, 73, 178 ms there, 3.7, 24, 51, 140 here).
        bhp::BatchFrame B[2];
        bh_batch_cfg cfg;
        int grid, per_xcd;
        rc = launch_samples(c, &g, o, o.spp, B, &cfg, &grid);
        if (rc) return rc;
        const int nb = trace_blocks(n, n, &per_xcd);
        rc = ensure(c, &c->d_blk, &c->blk_cap, (size_t)nb);
        if (rc) return rc;
        hipLaunchKernelGGL(k_flux_blocks, dim3(nb), dim3(BLOCK), 0, c->st, c->d_samp1, n, n, o.spp, c->d_blk, per_xcd);
        hipLaunchKernelGGL(k_reduce, dim3(1), dim3(256), 0, c->st, c->d_blk, nb, c->d_tot);
        HIPCK(c, hipGetLastError());
        BlockOut tot;
        HIPCK(c, hipMemcpyAsync(&tot, c->d_tot, sizeof tot, hipMemcpyDeviceToHost, c->st));
        HIPCK(c, hipStreamSynchronize(c->st));
        st.flux_sum = tot.flux;
        if (samples > had && samples * sizeof(double4) > FLUX_SAMPLES_KEPT) {
            HIPCK(c, hipFree(c->d_samp1));
            c->d_samp1 = nullptr;
            c->samp1_cap = 0;
        }
    } else {   // the frame kernel, which needs no memory for them
        rc = launch_trace(c, &g, &o, 0, 0, n, n, false, &st);
        if (rc) return rc;
    }
    // render.cu:803-808: sum of the per-pixel means times the pixel solid angle, in Jy
    *jy = st.flux_sum / 2.0 * pix_sr / 1e-23;
    return BH_OK;
}

int bh_trace_batch(bh_ctx* c, const bh_batch_frame* frames, int n, const bh_trace_opts* opts,
                   const bh_batch_cfg* cfg, float* px_out, bh_stats* st) {
    if (!c) return BH_ERR_ARG;
    double t0 = now_ms();
    HIPCK(c, hipSetDevice(c->device));
    bh_stats local{};
    long long npix = 0;
    int rc = launch_batch(c, frames, n, opts, cfg, &npix, &local);
    if (rc) return rc;
    if (px_out) {
        HIPCK(c, c->transfer->to_host(px_out, c->d_bout, sizeof(float4) * (size_t)npix, c->st));
    }
    local.ms_trace = now_ms() - t0;
    if (st) *st = local;
    return BH_OK;
}

int bh_autotune(bh_ctx* c, const bh_batch_frame* frames, int n, const bh_trace_opts* opts, bh_batch_cfg* best,
                double* best_ms, double* tried, int max_tried, int* n_tried) {
    if (!c || !best) return BH_ERR_ARG;
    HIPCK(c, hipSetDevice(c->device));
    // coordinate descent from the defaults: one parameter at a time over its candidate list, two passes
    const int prec = opts ? opts->precision : BH_PREC_FP64;
    if (!frames || n <= 0) return fail(c, BH_ERR_ARG, "empty batch");
    bh_batch_cfg cur{};   // the defaults, filled in by the first timed launches
    cur.use_graph = 1;
    cur.waves = 3;
    int count = 0;
    double cur_ms = 0.0;
    auto time_cfg = [&](const bh_batch_cfg& asked, double* ms, bh_batch_cfg* filled) -> int {
        bh_stats s{};
        bh_batch_cfg g;
        int rc = launch_batch(c, frames, n, opts, &asked, nullptr, &s, &g);   // first run: warm caches and graph
        if (rc) return rc;
        double t[3];   // the median of three timed runs (launch-to-launch spread is up to 10 %)
        for (int rep = 0; rep < 3; ++rep) {
            rc = launch_batch(c, frames, n, opts, &g, nullptr, &s);
            if (rc) return rc;
            t[rep] = s.ms_kernel;
        }
        const double best_of = std::max(std::min(t[0], t[1]), std::min(std::max(t[0], t[1]), t[2]));
        *ms = best_of;
        if (tried && count < max_tried) {
            double* row = tried + 8 * (size_t)count;
            row[0] = g.block;
            row[1] = g.grid_per_cu;
            row[2] = g.interval;
            row[3] = g.refill_min;
            row[4] = best_of;
            row[5] = g.waves;
            row[6] = g.order;
            row[7] = g.prio_age;
        }
        ++count;
        if (filled) *filled = g;
        return BH_OK;
    };
    int rc = time_cfg(cur, &cur_ms, &cur);
    if (rc) return rc;
    const bh_batch_cfg from = cur;
    const int blocks[] = {64, 128, 256}, grids[] = {1, 2, 3, 4, 8}, intervals[] = {2, 4, 8, 16, 32, 64},
              refills[] = {1, 8, 16, 32, 48}, waves[] = {0, 3, 4},
              orders[] = {BH_ORDER_ROWS, BH_ORDER_IMPACT, BH_ORDER_CRITICAL}, ages[] = {-1, 64, 128, 256, 512};
    for (int pass = 0; pass < 2; ++pass) {
        for (int p = 0; p < 7; ++p) {
            const int* vals = p == 0 ? waves : p == 1 ? blocks : p == 2 ? grids : p == 3 ? intervals
                            : p == 4 ? refills : p == 5 ? orders : ages;
            const int nv = p == 0 ? 3 : p == 1 ? 3 : p == 2 ? 5 : p == 3 ? 6 : p == 4 ? 5 : p == 5 ? 3 : 5;
            for (int i = 0; i < nv; ++i) {
                bh_batch_cfg g = cur;
                int* field = p == 0 ? &g.waves : p == 1 ? &g.block : p == 2 ? &g.grid_per_cu
                           : p == 3 ? &g.interval : p == 4 ? &g.refill_min : p == 5 ? &g.order : &g.prio_age;
                if (*field == vals[i]) continue;
                *field = vals[i];
                double ms;
                rc = time_cfg(g, &ms, nullptr);
                if (rc) return rc;
                if (ms < cur_ms) {
                    cur = g;
                    cur_ms = ms;
                }
            }
        }
    }
    *best = cur;
    if (best_ms) *best_ms = cur_ms;
    if (n_tried) *n_tried = count;
    c->tuned[prec] = launch::Tuned{true, frames[0].scene.mode == BH_MODE_RADIO, from, cur};   // the launches checked prec
    return BH_OK;
}

int bh_vacuum_fates(bh_ctx* c, const double* photons, int n, double tol, double r_escape, int max_steps, int* fates) {
    if (!c || !photons || !fates || n < 0) return BH_ERR_ARG;
    if (n == 0) return BH_OK;
    HIPCK(c, hipSetDevice(c->device));
    if (c->ph_cap < (size_t)n) {
        c->ph_cap = 0;
        if (c->d_ph) {
            HIPCK(c, hipFree(c->d_ph));
            c->d_ph = nullptr;
        }
        if (c->d_fates) {
            HIPCK(c, hipFree(c->d_fates));
            c->d_fates = nullptr;
        }
        HIPCK(c, hipMalloc((void**)&c->d_ph, sizeof(double) * 9 * n));
        HIPCK(c, hipMalloc((void**)&c->d_fates, sizeof(int) * n));
        c->ph_cap = n;
    }
    HIPCK(c, hipMemcpyAsync(c->d_ph, photons, sizeof(double) * 9 * n, hipMemcpyHostToDevice, c->st));
    TraceParams P = make_params(c, nullptr);
    hipLaunchKernelGGL(k_vacuum_fates, dim3((n + 63) / 64), dim3(64), 0, c->st, P, c->d_ph, n, tol, r_escape,
                       max_steps, c->d_fates);
    HIPCK(c, hipGetLastError());
    HIPCK(c, hipMemcpyAsync(fates, c->d_fates, sizeof(int) * n, hipMemcpyDeviceToHost, c->st));
    HIPCK(c, hipStreamSynchronize(c->st));
    return BH_OK;
}

int bh_math_eval(int fn, const double* x, const double* y, double* out, int n) {
    if (!x || !y || !out || n < 0 || fn < 0 || fn > 15) return BH_ERR_ARG;
    if (n == 0) return BH_OK;
    if (bh_device_count() <= 0) return BH_ERR_NODEVICE;
    double *dx = nullptr, *dy = nullptr, *dout = nullptr;
    size_t bytes = sizeof(double) * (size_t)n;
    int rc = BH_OK;
    if (hipSetDevice(0) != hipSuccess || hipMalloc((void**)&dx, bytes) != hipSuccess ||
        hipMalloc((void**)&dy, bytes) != hipSuccess || hipMalloc((void**)&dout, bytes) != hipSuccess ||
        hipMemcpy(dx, x, bytes, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dy, y, bytes, hipMemcpyHostToDevice) != hipSuccess) {
        rc = BH_ERR_HIP;
    } else {
        hipLaunchKernelGGL(k_math_eval, dim3((n + 255) / 256), dim3(256), 0, 0, fn, dx, dy, dout, n);
        if (hipGetLastError() != hipSuccess || hipMemcpy(out, dout, bytes, hipMemcpyDeviceToHost) != hipSuccess)
            rc = BH_ERR_HIP;
    }
    if (dx) (void)hipFree(dx);
    if (dy) (void)hipFree(dy);
    if (dout) (void)hipFree(dout);
    return rc;
}

void bh_destroy(bh_ctx* c) {
    if (!c) return;
    // best-effort teardown: errors here have nowhere to go
    (void)hipSetDevice(c->device);
    if (c->st) (void)hipStreamSynchronize(c->st);
    if (c->graph) (void)hipGraphExecDestroy(c->graph);
    if (c->graph_def) (void)hipGraphDestroy(c->graph_def);
    void* bufs[] = {c->d_k2,     c->d_turb,   c->d_px,     c->d_rays,    c->d_blk,    c->d_tot,    c->d_ph,
                    c->d_fates,  c->d_mlp,    c->d_adam_m, c->d_adam_v,  c->d_stab,   c->d_sbad,   c->d_bframes,
                    c->d_queue,  c->d_bout,   c->d_samp1,  c->d_acc,     c->d_ystat,  c->d_extra,  c->d_chunks,
                    c->d_offsets, c->d_bsum,  c->d_nsamp,  c->d_fpart,   c->d_samp2,  c->d_order,  c->d_ohist,
                    c->d_post_lev, c->d_post_tmp, c->d_post_wt, c->d_post_rgb, c->d_hud, c->d_ts, c->d_tsv};
    for (void* b : bufs)
        if (b) (void)hipFree(b);
    if (c->ev0) (void)hipEventDestroy(c->ev0);
    if (c->ev1) (void)hipEventDestroy(c->ev1);
    if (c->st) (void)hipStreamDestroy(c->st);
    delete c;
}

const char* bh_last_error(const bh_ctx* c) { return c ? c->err.c_str() : g_create_error.c_str(); }

}  // extern "C"

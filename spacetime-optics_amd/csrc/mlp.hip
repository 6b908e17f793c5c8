/* mlp.hip - thermal-synchrotron surrogate on gfx950: exact-routine sampler, BF16-MFMA training
   (forward + backward + Adam) and inference kernels, and the deployment table with its exact-routine
   judge. C ABI in include/bhrt.h (bh_mlp_*).

   Matrix products of the two 64 x 64 hidden layers use v_mfma_f32_16x16x16_bf16 with FP32
   accumulation. Each FP32 operand is split into a BF16 head and a BF16 tail (x = hi + lo, both
   rounded to nearest even) and a product is accumulated as lo*hi + hi*lo + hi*hi: three MFMAs that
   keep about 16 significant bits of every operand, so BF16 rounding does not bound the surrogate's
   accuracy. The 3 -> 64 input layer and the 64 -> 2 output layer run on the FP32 VALU.

   Work layout: tiles of 16 samples, four waves per tile, each wave owning 16 columns of every layer.
   MFMA operand layout (16x16x16, wave64): A[i][k] lane i + 16*(k/4), element k % 4; B[k][j] lane
   j + 16*(k/4), element k % 4; D[i][j] lane j + 16*(i/4), element i % 4. The products are taken
   transposed (weights as A, activations as B): a wave's result then has the layout that the next
   product's B operand needs, so a layer is handed on through LDS as whole 16-byte fragments. The
   weights stay in registers, each wave its own columns' share, loaded and split once. */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

#include "ctx.h"
#include "trace_fp64.h"

using namespace bhmlp;

namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int TM = 16;           // samples per tile
constexpr int LDA = NH + 4;      // padded row of an activation tile (floats)
constexpr int PSTRIDE = (NPARAM + 3) / 4 * 4;   // row of a partial gradient (floats): 16-byte aligned rows

typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float fl2 __attribute__((ext_vector_type(2)));
typedef unsigned int u2 __attribute__((ext_vector_type(2)));

// two floats to packed BF16 (a in the low half), rounded to nearest even: one v_cvt_pk_bf16_f32
__device__ __forceinline__ unsigned int bf16x2(float a, float b) {
    return __builtin_bit_cast(unsigned int, __builtin_convertvector((fl2){a, b}, bf2));
}
// the low / high BF16 of a packed pair as a float
__device__ __forceinline__ float bf16_lo(unsigned int p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi(unsigned int p) { return __uint_as_float(p & 0xffff0000u); }

// x = hi + lo with hi = bf16(x) and lo = bf16(x - hi), four values at once
__device__ __forceinline__ void split4(const float v[4], s4& hi, s4& lo) {
    const unsigned int h01 = bf16x2(v[0], v[1]), h23 = bf16x2(v[2], v[3]);
    const unsigned int l01 = bf16x2(v[0] - bf16_lo(h01), v[1] - bf16_hi(h01));
    const unsigned int l23 = bf16x2(v[2] - bf16_lo(h23), v[3] - bf16_hi(h23));
    hi = __builtin_bit_cast(s4, (u2){h01, h23});
    lo = __builtin_bit_cast(s4, (u2){l01, l23});
}

__device__ __forceinline__ f4 mfma3(s4 ah, s4 al, s4 bh, s4 bl, f4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(al, bh, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, bl, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, bh, c, 0, 0, 0);
}

// logistic sigmoid from the hardware exp2 and reciprocal (about 1 ulp each; the library expf and
// the IEEE division cost ~30 instructions per element, on ~100 elements per lane and tile)
__device__ __forceinline__ float sigm(float z) {
    return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}

constexpr int TILE_WAVES = 4;    // waves per tile: wave w owns columns 16 w .. 16 w + 15 of every layer
typedef unsigned int u4 __attribute__((ext_vector_type(4)));
typedef u4 Frag[TILE_WAVES][64];     // B operands of the transposed products: (head, tail) per wave and lane

// a D-layout fragment of the transposed activations as the next product's B operand
__device__ __forceinline__ u4 pack_frag(const float v[4]) {
    s4 h, l;
    split4(v, h, l);
    const u2 hh = __builtin_bit_cast(u2, h), ll = __builtin_bit_cast(u2, l);
    return u4{hh[0], hh[1], ll[0], ll[1]};
}
__device__ __forceinline__ void unpack_frag(u4 f, s4& h, s4& l) {
    h = __builtin_bit_cast(s4, (u2){f[0], f[1]});
    l = __builtin_bit_cast(s4, (u2){f[2], f[3]});
}

// A wave's 16 columns of a 64 x 64 matrix as A operands, split into head and tail: four steps of the
// contraction. Forward: A[j][k] = W[k][16 w + j]; backward: A[k][j] = W[16 w + k][j].
struct WFrag {
    s4 h[4], l[4];
};
__device__ __forceinline__ void load_fwd(const float* __restrict__ M, int w, int r, int g, WFrag& F) {
    float v[4][4];
    for (int kb = 0; kb < 4; ++kb)
        for (int e = 0; e < 4; ++e) v[kb][e] = M[(16 * kb + 4 * g + e) * NH + 16 * w + r];
    for (int kb = 0; kb < 4; ++kb) split4(v[kb], F.h[kb], F.l[kb]);
}
__device__ __forceinline__ void load_bwd(const float* __restrict__ M, int w, int r, int g, WFrag& F) {
    f4 v[4];
    for (int jb = 0; jb < 4; ++jb) v[jb] = *(const f4*)&M[(16 * w + r) * NH + 16 * jb + 4 * g];
    for (int jb = 0; jb < 4; ++jb) {
        const float q[4] = {v[jb][0], v[jb][1], v[jb][2], v[jb][3]};
        split4(q, F.h[jb], F.l[jb]);
    }
}

// The wave's 16 rows of (W^T or W) X^T, X^T from the fragments that the tile's four waves left. The
// products are taken activation tail first, then the weight's, then the heads.
__device__ __forceinline__ f4 gemm_t(const WFrag& W, const Frag& X, int lane) {
    f4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int kb = 0; kb < 4; ++kb) {
        s4 xh, xl;
        unpack_frag(X[kb][lane], xh, xl);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(W.h[kb], xl, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(W.l[kb], xh, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(W.h[kb], xh, acc, 0, 0, 0);
    }
    return acc;
}

// gW[m][j] = sum_i H[i][m] G[i][j] over a tile's 16 samples, m of the wave's 16 columns; D layout [jb]
__device__ __forceinline__ void gemm_wgrad(const float* H, const float* G, int w, int r, int g, f4 gW[4]) {
    float av[4];
    for (int e = 0; e < 4; ++e) av[e] = H[(4 * g + e) * LDA + 16 * w + r];
    s4 ah, al;
    split4(av, ah, al);
    for (int jb = 0; jb < 4; ++jb) {
        float bv[4];
        for (int e = 0; e < 4; ++e) bv[e] = G[(4 * g + e) * LDA + 16 * jb + r];
        s4 bh, bl;
        split4(bv, bh, bl);
        gW[jb] = mfma3(ah, al, bh, bl, f4{0.f, 0.f, 0.f, 0.f});
    }
}

// silu and its derivative from one sigmoid
__device__ __forceinline__ void act4(const f4 z, float h[4], float d[4]) {
    for (int e = 0; e < 4; ++e) {
        const float s = sigm(z[e]);
        h[e] = z[e] * s;
        d[e] = s * (1.f + z[e] * (1.f - s));
    }
}

// the lane's four columns of row i of an FP32 tile
__device__ __forceinline__ void put_row(float* X, int i, int j, const float v[4]) {
    *(f4*)&X[i * LDA + j] = f4{v[0], v[1], v[2], v[3]};
}

// A wave's share of the network in the forward direction, in registers
struct FwdWeights {
    f4 w1[3], b1, b2, b3;
    WFrag W2, W3;
};
__device__ __forceinline__ void load_forward(const float* __restrict__ P, int w, int r, int g, FwdWeights& F) {
    const int j = 16 * w + 4 * g;
    for (int k = 0; k < 3; ++k) F.w1[k] = *(const f4*)&P[OFF_W1 + k * NH + j];
    F.b1 = *(const f4*)&P[OFF_B1 + j];
    F.b2 = *(const f4*)&P[OFF_B2 + j];
    F.b3 = *(const f4*)&P[OFF_B3 + j];
    load_fwd(P + OFF_W2, w, r, g, F.W2);
    load_fwd(P + OFF_W3, w, r, g, F.W3);
}
__device__ __forceinline__ f4 layer1(const FwdWeights& F, const float x[3]) {
    f4 z;
    for (int e = 0; e < 4; ++e) z[e] = F.b1[e] + x[0] * F.w1[0][e] + x[1] * F.w1[1][e] + x[2] * F.w1[2][e];
    return z;
}

// The output layer's 64 weights of each output, and its 32 sums (one per lane 0..31 of a tile's first wave)
struct alignas(16) OutLayer {
    float w[NOUT][NH];
};
__device__ __forceinline__ void load_out(const float* __restrict__ P, OutLayer& O) {
    for (int q = threadIdx.x; q < NH * NOUT; q += blockDim.x) O.w[q % NOUT][q / NOUT] = P[OFF_W4 + q];
}
__device__ __forceinline__ float out_sum(float b4, const OutLayer& O, const float* X, int i, int o) {
    float y = b4;
    for (int k = 0; k < NH; k += 4) {
        const f4 h = *(const f4*)&X[i * LDA + k], w = *(const f4*)&O.w[o][k];
        for (int e = 0; e < 4; ++e) y += h[e] * w[e];
    }
    return y;
}

__device__ __forceinline__ uint64_t splitmix(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}
__device__ __forceinline__ double uniform01(uint64_t seed, uint64_t i) {   // (0, 1)
    return ((splitmix(seed ^ splitmix(i)) >> 11) + 0.5) * 0x1p-53;
}

}  // namespace

// Exact coefficients in the surrogate coordinates (emission.cuh:159-170 normalised; FP64, bh_math
// elementary functions, the tracer's K2 table): (ln f_j, ln f_a) at ln X = lx, ln Theta = lth,
// ln sin theta_B = ls.
__device__ void exact_lnf_s(const float* __restrict__ k2, int k2_n, float k2_l0, float k2_dl, double lx, double lth,
                            double ls, double* lfj, double* lfa) {
    const double X = bhm::exp(lx), x3 = bhm::exp(lx * (1.0 / 3.0));
    const double brk = sqrt(X) + 1.887748625363387 * sqrt(x3);
    const double lk2 = (double)bhd::table_lerp(k2, k2_n, k2_l0, k2_dl, (float)lth);
    const double fj = LN_FJ_CONST + 2.0 * lth + ls - lk2 + 2.0 * bhm::log(brk) - x3;
    const double u0ln10 = lx + LN_2_9 + 2.0 * lth + ls;
    *lfj = fj;
    *lfa = fj - 0.6931471805599453 - lth - 2.0 * u0ln10;
}

// The same at u0 = log10(nu/nu_c), Theta, theta_B (sin theta_B >= 1e-3, as in the tracer).
__device__ void exact_lnf(const float* __restrict__ k2, int k2_n, float k2_l0, float k2_dl, double u0, double th,
                          double tb, double* lfj, double* lfa) {
    double s, c;
    bhm::sincos(tb, &s, &c);
    const double lth = bhm::log(th), ls = bhm::log(fmax(s, 1e-3));
    exact_lnf_s(k2, k2_n, k2_l0, k2_dl, u0 * LN10 - LN_2_9 - 2.0 * lth - ls, lth, ls, lfj, lfa);
}

namespace {

// training set: normalised inputs, raw (clamped) targets and loss weights
__global__ __launch_bounds__(256) void k_mlp_sample(uint64_t seed, int n, const float* __restrict__ k2, int k2_n,
                                                   float k2_l0, float k2_dl, Norm N, float hot_weight,
                                                   float* __restrict__ xs, float* __restrict__ ts,
                                                   float* __restrict__ ws) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double u0 = U0_LO + (U0_HI - U0_LO) * uniform01(seed, 3ull * i);
    const double lth = LTH_LO + (LTH_HI - LTH_LO) * uniform01(seed, 3ull * i + 1);
    const double tb = TB_LO + (TB_HI - TB_LO) * uniform01(seed, 3ull * i + 2);
    double sb, cb;
    bhm::sincos(tb, &sb, &cb);
    const double ls = bhm::log(fmax(sb, 1e-3));
    const double lx = u0 * LN10 - LN_2_9 - 2.0 * lth - ls;
    double fj, fa;
    exact_lnf_s(k2, k2_n, k2_l0, k2_dl, lx, lth, ls, &fj, &fa);
    const double sc[3] = {fmin(lx, LX_HI), lth, ls};
    for (int k = 0; k < 3; ++k) xs[3 * (size_t)i + k] = (float)((sc[k] - N.x_c[k]) / N.x_h[k]);
    ts[2 * (size_t)i] = (float)fmax(fj, FLOOR_J);
    ts[2 * (size_t)i + 1] = (float)fmax(fa, FLOOR_A);
    ws[i] = 1.f + hot_weight / (1.f + expf(-(float)(fj + 12.0)));
}

// One training step is a chain of small products, so its time is latency: the longest chain of one tile,
// not the matrix rate (1.3 GFLOP). Four waves share a tile, so each runs a quarter of every product, and the
// weight gradients, which nothing waits for, come after the chain. Two tiles per workgroup: the default
// batch of 8192 samples is 256 workgroups, one per CU with two waves per SIMD. Per step of that batch:
// one wave per tile with the split weights in LDS, read 2 bytes at a time: 26.7 us; this one 13.6. Beyond
// the chain that is the first touch of weights and samples, and the 8.9 MB of partial gradients.
constexpr int GRAD_TILES = 2, GRAD_BLOCK = 64 * TILE_WAVES * GRAD_TILES;
static_assert(GRAD_TILES == 2, "the two tiles' halves add the partial gradient of one matrix each");

struct alignas(16) GradTile {
    float h1[TM * LDA], h2[TM * LDA], h3[TM * LDA];    // activations
    float g1[TM * LDA], g2[TM * LDA], g3[TM * LDA];    // gradients by the pre-activations
    Frag f1, f2;                                       // fragments, by turns
    float x[TM][4], dy[TM][2];
};

// Row index of a partial gradient: everything but W2 and W3 lies as in the parameters; each of W2 and W3
// as a lane holds it (wave, jb, lane, e), so that the partials are stored 16 bytes at a time (the reduction
// reads whole rows, 4 bytes a lane).
__device__ __forceinline__ int partial_param(int q) {
    const int off = q >= OFF_W3 && q < OFF_B3 ? OFF_W3 : OFF_W2;
    if (q < OFF_W2 || q >= OFF_B3 || (q >= OFF_B2 && q < OFF_W3)) return q;
    const int v = q - off, e = v & 3, lane = (v >> 2) & 63, jb = (v >> 8) & 3, w = v >> 10;
    return off + (16 * w + 4 * (lane >> 4) + e) * NH + 16 * jb + (lane & 15);
}

/* One training step's gradient over `count` samples starting at `first` (indices mod n): each
   workgroup takes two consecutive 16-sample tiles and writes the sum of their partial gradients
   (8706 floats, rows as partial_param) and of their losses.
   Loss = sum_i w_i |y_i - t_i|^2 / count on normalised outputs. */
__global__ __launch_bounds__(GRAD_BLOCK) void k_mlp_grad(const float* __restrict__ P, Norm N, const float* __restrict__ xs,
                                                 const float* __restrict__ ts, const float* __restrict__ ws, int n,
                                                 int first, int count, float* __restrict__ partial,
                                                 float* __restrict__ loss_partial) {
    __shared__ GradTile TT[GRAD_TILES];
    __shared__ OutLayer O;
    __shared__ f4 swap[GRAD_TILES][4 * 64 * TILE_WAVES];   // a tile's gradient of the other tile's matrix
    __shared__ float small[2 * NH + 2 * NH + NIN * NH + NH * NOUT];
    __shared__ float tile_loss[GRAD_TILES], small4[NOUT];
    const int tile = threadIdx.x / (64 * TILE_WAVES), w = (threadIdx.x >> 6) & (TILE_WAVES - 1);
    GradTile& T = TT[tile];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int col = 16 * w + 4 * g;        // the lane's four columns of sample r
    const float inv_count = 1.f / (float)count;
    const int base = (blockIdx.x * GRAD_TILES + tile) * TM;   // sample offset in the batch
    // the lane's sample, and on the first wave the target and weight of its output sum
    float x[3];
    {
        const bool in = base + r < count;
        const size_t idx = (size_t)((first + base + r) % n);
        for (int k = 0; k < 3; ++k) x[k] = in ? xs[3 * idx + k] : 0.f;
    }
    const int oi = (lane >> 1) & 15, oo = lane & 1;
    float tgt = 0.f, wgt = 0.f, b4 = 0.f;
    if (w == 0) {
        const bool in = base + oi < count;
        const size_t idx = (size_t)((first + base + oi) % n);
        tgt = in ? (ts[2 * idx + oo] - N.y_mu[oo]) / N.y_sd[oo] : 0.f;
        wgt = in ? ws[idx] : 0.f;
        b4 = P[OFF_B4 + oo];
    }
    FwdWeights F;
    load_forward(P, w, r, g, F);
    WFrag B2, B3;
    load_bwd(P + OFF_W3, w, r, g, B3);
    load_bwd(P + OFF_W2, w, r, g, B2);
    float w4[4][2];
    for (int e = 0; e < 4; ++e)
        for (int o = 0; o < 2; ++o) w4[e][o] = P[OFF_W4 + (col + e) * NOUT + o];
    load_out(P, O);
    if (w == 0 && g == 0)
        for (int k = 0; k < 3; ++k) T.x[r][k] = x[k];
    // forward
    float h[4], d1[4], d2[4], d3[4];
    act4(layer1(F, x), h, d1);
    T.f1[w][lane] = pack_frag(h);
    put_row(T.h1, r, col, h);
    __syncthreads();
    act4(gemm_t(F.W2, T.f1, lane) + F.b2, h, d2);
    T.f2[w][lane] = pack_frag(h);
    put_row(T.h2, r, col, h);
    __syncthreads();
    act4(gemm_t(F.W3, T.f2, lane) + F.b3, h, d3);
    put_row(T.h3, r, col, h);
    __syncthreads();
    // outputs, loss and its gradient: lanes 0..31 of the tile's first wave
    if (w == 0) {
        float loss = 0.f;
        if (lane < 2 * TM) {
            const float d = out_sum(b4, O, T.h3, oi, oo) - tgt;
            loss += wgt * d * d * inv_count;
            T.dy[oi][oo] = 2.f * wgt * d * inv_count;
        }
        for (int off = 32; off > 0; off >>= 1) loss += __shfl_down(loss, off, 64);
        if (lane == 0) tile_loss[tile] = loss;
    }
    __syncthreads();
    // backward: the chain first
    float q[4];
    {
        const float dy0 = T.dy[r][0], dy1 = T.dy[r][1];
        for (int e = 0; e < 4; ++e) q[e] = (dy0 * w4[e][0] + dy1 * w4[e][1]) * d3[e];
    }
    T.f1[w][lane] = pack_frag(q);
    put_row(T.g3, r, col, q);
    __syncthreads();
    {
        const f4 a = gemm_t(B3, T.f1, lane);
        for (int e = 0; e < 4; ++e) q[e] = a[e] * d2[e];
    }
    T.f2[w][lane] = pack_frag(q);
    put_row(T.g2, r, col, q);
    __syncthreads();
    {
        const f4 a = gemm_t(B2, T.f2, lane);
        for (int e = 0; e < 4; ++e) q[e] = a[e] * d1[e];
    }
    put_row(T.g1, r, col, q);
    // the weight gradients: this tile's of the other tile's matrix first
    f4 gW2[4], gW3[4];
    gemm_wgrad(T.h2, T.g3, w, r, g, gW3);
    gemm_wgrad(T.h1, T.g2, w, r, g, gW2);
    for (int jb = 0; jb < 4; ++jb) swap[tile][(w * 4 + jb) * 64 + lane] = tile == 0 ? gW3[jb] : gW2[jb];
    __syncthreads();
    // the vectors' gradients, a share per wave: lane = column, sums over the samples in order
    float v0 = 0.f, v1 = 0.f, v2 = 0.f;
    if (w < 2) {
        for (int i = 0; i < TM; ++i) v0 += T.h3[i * LDA + lane] * T.dy[i][w];            // W4[lane][w]
        const float* G = w == 0 ? T.g3 : T.g2;
        for (int i = 0; i < TM; ++i) v1 += G[i * LDA + lane];                            // b3, b2
        if (w == 0 && lane < 2)
            for (int i = 0; i < TM; ++i) v2 += T.dy[i][lane];                            // b4
    } else if (w == 2) {
        for (int i = 0; i < TM; ++i) {
            const float d = T.g1[i * LDA + lane];
            v0 += T.x[i][0] * d;
            v1 += T.x[i][1] * d;
        }
    } else {
        for (int i = 0; i < TM; ++i) {
            const float d = T.g1[i * LDA + lane];
            v0 += T.x[i][2] * d;
            v1 += d;
        }
    }
    // tile 1 hands its vectors over; tile 0 adds and stores them. Each tile adds and stores one matrix.
    constexpr int S_W4 = 0, S_B3 = 2 * NH, S_B2 = 3 * NH, S_W1 = 4 * NH, S_B1 = 7 * NH;
    const int i0 = w < 2 ? S_W4 + w * NH : S_W1 + (w == 2 ? 0 : 2) * NH;
    const int i1 = w == 0 ? S_B3 : w == 1 ? S_B2 : w == 2 ? S_W1 + NH : S_B1;
    if (tile == 1) {
        small[i0 + lane] = v0;
        small[i1 + lane] = v1;
        if (w == 0 && lane < 2) small4[lane] = v2;
    }
    float* out = partial + (size_t)blockIdx.x * PSTRIDE;
    for (int jb = 0; jb < 4; ++jb) {
        const int k = (w * 4 + jb) * 64 + lane;
        const f4 own = tile == 0 ? gW2[jb] : gW3[jb], other = swap[1 - tile][k];
        *(f4*)&out[(tile == 0 ? OFF_W2 : OFF_W3) + 4 * k] = own + other;
    }
    __syncthreads();
    if (tile == 0) {
        const int p0 = w < 2 ? OFF_W4 + lane * NOUT + w : OFF_W1 + (w == 2 ? 0 : 2) * NH + lane;
        const int p1 = (w == 0 ? OFF_B3 : w == 1 ? OFF_B2 : w == 2 ? OFF_W1 + NH : OFF_B1) + lane;
        out[p0] = v0 + small[i0 + lane];
        out[p1] = v1 + small[i1 + lane];
        if (w == 0 && lane < 2) out[OFF_B4 + lane] = v2 + small4[lane];
        if (threadIdx.x == 0) loss_partial[blockIdx.x] = tile_loss[0] + tile_loss[1];
    }
}

// grad[p] = sum over workgroups of partial[w][p]; loss likewise. A workgroup takes 64 parameters; its
// eight waves each sum an eighth of the workgroups' partials (w = q, q + 8, ...) in eight running
// sums, and the eighths are added through LDS. Every sum is taken in a fixed order, so the result
// does not depend on timing. 256 partials: four rounds of eight loads, all in flight at once: 6.6 -> 4.9 us.
// With P set, the same lane then takes the Adam step of its parameter (bias-corrected moments).
struct AdamStep {
    float* P;   // nullptr: gradient only
    float* m;
    float* v;
    float lr, b1, b2, eps, bc1, bc2;
};

constexpr int RED_PARAMS = 64, RED_SPLIT = 8, RED_BLOCK = RED_PARAMS * RED_SPLIT;
__global__ __launch_bounds__(RED_BLOCK) void k_mlp_reduce(const float* __restrict__ partial, int nw,
                                                         const float* __restrict__ loss_partial,
                                                         float* __restrict__ grad, float* __restrict__ loss,
                                                         AdamStep A) {
    __shared__ float part_sum[RED_SPLIT][RED_PARAMS];
    static_assert(RED_SPLIT == 8, "the final sum below adds eight parts");
    const int lp = threadIdx.x % RED_PARAMS, qt = threadIdx.x / RED_PARAMS;
    const int row = blockIdx.x * RED_PARAMS + lp, p = partial_param(row);
    float total = 0.f;
    if (p < NPARAM) {
        constexpr size_t STEP = (size_t)RED_SPLIT * PSTRIDE;   // between this group's rows
        float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f, s4 = 0.f, s5 = 0.f, s6 = 0.f, s7 = 0.f, sr = 0.f;
        const float* q = partial + (size_t)qt * PSTRIDE + row;
        int w = qt;
#pragma unroll 4
        for (; w + 7 * RED_SPLIT < nw; w += 8 * RED_SPLIT, q += 8 * STEP) {
            s0 += q[0];
            s1 += q[STEP];
            s2 += q[2 * STEP];
            s3 += q[3 * STEP];
            s4 += q[4 * STEP];
            s5 += q[5 * STEP];
            s6 += q[6 * STEP];
            s7 += q[7 * STEP];
        }
        for (; w < nw; w += RED_SPLIT, q += STEP) sr += q[0];
        total = (((s0 + s1) + (s2 + s3)) + ((s4 + s5) + (s6 + s7))) + sr;
    }
    part_sum[qt][lp] = total;
    __syncthreads();
    if (qt == 0 && p < NPARAM) {
        const float(&q)[RED_SPLIT][RED_PARAMS] = part_sum;
        const float gr = ((q[0][lp] + q[1][lp]) + (q[2][lp] + q[3][lp])) + ((q[4][lp] + q[5][lp]) + (q[6][lp] + q[7][lp]));
        grad[p] = gr;
        if (A.P) {
            const float mm = A.b1 * A.m[p] + (1.f - A.b1) * gr, vv = A.b2 * A.v[p] + (1.f - A.b2) * gr * gr;
            A.m[p] = mm;
            A.v[p] = vv;
            A.P[p] -= A.lr * (mm / A.bc1) / (sqrtf(vv / A.bc2) + A.eps);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < 64) {   // the loss: one wave, strided sums and a fixed tree
        float sl = 0.f;
        for (int v = threadIdx.x; v < nw; v += 64) sl += loss_partial[v];
        for (int off = 32; off > 0; off >>= 1) sl += __shfl_down(sl, off, 64);
        if (threadIdx.x == 0) *loss = sl;
    }
}


constexpr int INFER_GRID = 2048;   // persistent workgroups of the inference, eight per CU

/* Inference: n samples of raw inputs (u0, Theta, theta_B) or, with lattice != 0, the nodes of the
   (n0 x n1 x n2) lattice over (u0, log10 Theta, theta_B in [lo2, hi2]); writes (ln f_j, ln f_a). */
struct Lattice {
    int n0, n1, n2;
    float lo0, lo1, lo2, d0, d1, d2;
};
// Four waves per tile as in the training step, the weights in registers over all of a workgroup's tiles.
// 200 003 points: one wave per tile with the split weights in LDS 215 us, this one 39 us.
__global__ __launch_bounds__(64 * TILE_WAVES) void k_mlp_infer(const float* __restrict__ P, Norm N,
                                                  const float* __restrict__ in, int n, int lattice, Lattice L,
                                                  float* __restrict__ out) {
    __shared__ Frag f1, f2;
    __shared__ alignas(16) float h3[TM * LDA];
    __shared__ OutLayer O;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    FwdWeights F;
    load_forward(P, w, r, g, F);
    load_out(P, O);
    const int oi = lane >> 1, oo = lane & 1;
    const float b4 = P[OFF_B4 + oo];
    const int ntiles = (n + TM - 1) / TM;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        float x[3];
        {
            const int s = tile * TM + r;
            float sc[3] = {0.f, 0.f, 0.f};   // surrogate coordinates
            if (s < n) {
                if (lattice) {
                    const int i0 = s % L.n0, i1 = (s / L.n0) % L.n1, i2 = s / (L.n0 * L.n1);
                    sc[0] = L.lo0 + i0 * L.d0;
                    sc[1] = L.lo1 + i1 * L.d1;
                    sc[2] = L.lo2 + i2 * L.d2;
                } else {
                    const float u0 = in[3 * (size_t)s], lth = logf(in[3 * (size_t)s + 1]);
                    const float ls = logf(fmaxf(sinf(in[3 * (size_t)s + 2]), 1e-3f));
                    sc[0] = fminf(u0 * (float)LN10 - (float)LN_2_9 - 2.f * lth - ls, (float)LX_HI);
                    sc[1] = lth;
                    sc[2] = ls;
                }
            }
            for (int k = 0; k < 3; ++k) x[k] = (sc[k] - N.x_c[k]) / N.x_h[k];
        }
        // every buffer is written behind a barrier that its readers in the tile before have passed: f1
        // behind that tile's second and third, f2 and h3 behind this tile's first and second
        float h[4], d[4];
        act4(layer1(F, x), h, d);
        f1[w][lane] = pack_frag(h);
        __syncthreads();
        act4(gemm_t(F.W2, f1, lane) + F.b2, h, d);
        f2[w][lane] = pack_frag(h);
        __syncthreads();
        act4(gemm_t(F.W3, f2, lane) + F.b3, h, d);
        put_row(h3, r, 16 * w + 4 * g, h);
        __syncthreads();
        if (w == 0 && lane < 2 * TM) {
            const int s = tile * TM + oi;
            const float y = out_sum(b4, O, h3, oi, oo);
            if (s < n) out[2 * (size_t)s + oo] = y * N.y_sd[oo] + N.y_mu[oo];
        }
    }
}

__global__ __launch_bounds__(256) void k_mlp_exact(const float* __restrict__ in, int n, const float* __restrict__ k2,
                                                   int k2_n, float k2_l0, float k2_dl, double* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double fj, fa;
    exact_lnf(k2, k2_n, k2_l0, k2_dl, in[3 * (size_t)i], in[3 * (size_t)i + 1], in[3 * (size_t)i + 2], &fj, &fa);
    out[2 * (size_t)i] = fj;
    out[2 * (size_t)i + 1] = fa;
}

/* Judge: for every lattice cell, the exact coefficients at 4 interior points against the trilinear
   interpolation of the tabulated network; a cell fails when |d ln f_j| > tol where ln f_j > floor
   (or the same for ln f_a). */
__global__ __launch_bounds__(256) void k_mlp_judge(const float2* __restrict__ tab, Lattice L, const float* __restrict__ k2,
                                                   int k2_n, float k2_l0, float k2_dl, float tol, float floor_j,
                                                   float floor_a, unsigned char* __restrict__ bad,
                                                   unsigned int* __restrict__ counts) {
    const int c0 = L.n0 - 1, c1 = L.n1 - 1, c2 = L.n2 - 1;
    const int cell = blockIdx.x * blockDim.x + threadIdx.x;
    if (cell >= c0 * c1 * c2) return;
    const int i0 = cell % c0, i1 = (cell / c0) % c1, i2 = cell / (c0 * c1);
    const float2* b = tab + ((size_t)i2 * L.n1 + i1) * L.n0 + i0;
    const size_t s1 = L.n0, s2 = (size_t)L.n0 * L.n1;
    const float2 v[8] = {b[0], b[1], b[s1], b[s1 + 1], b[s2], b[s2 + 1], b[s2 + s1], b[s2 + s1 + 1]};
    const float fr[4][3] = {{0.5f, 0.5f, 0.5f}, {0.25f, 0.25f, 0.75f}, {0.75f, 0.75f, 0.25f}, {0.25f, 0.75f, 0.5f}};
    bool fail = false, hot = false;
    for (int p = 0; p < 4; ++p) {
        const float f0 = fr[p][0], f1 = fr[p][1], f2 = fr[p][2];
        float iv[2];
        for (int o = 0; o < 2; ++o) {
            auto at = [&](int q) { return o == 0 ? v[q].x : v[q].y; };
            float c00 = at(0) + (at(1) - at(0)) * f0, c10 = at(2) + (at(3) - at(2)) * f0;
            float c01 = at(4) + (at(5) - at(4)) * f0, c11 = at(6) + (at(7) - at(6)) * f0;
            float c0v = c00 + (c10 - c00) * f1, c1v = c01 + (c11 - c01) * f1;
            iv[o] = c0v + (c1v - c0v) * f2;
        }
        const double lx = L.lo0 + (i0 + f0) * L.d0, lth = L.lo1 + (i1 + f1) * L.d1, ls = L.lo2 + (i2 + f2) * L.d2;
        double fj, fa;
        exact_lnf_s(k2, k2_n, k2_l0, k2_dl, lx, lth, ls, &fj, &fa);
        if (fj > floor_j) {
            hot = true;
            if (fabs(iv[0] - fj) > tol) fail = true;
        }
        if (fa > floor_a && fabs(iv[1] - fa) > tol) fail = true;
    }
    bad[cell] = fail ? 1 : 0;
    if (hot) atomicAdd(&counts[0], 1u);
    if (hot && fail) atomicAdd(&counts[1], 1u);
}

}  // namespace

#define MCK(ctx, x)                                                                                        \
    do {                                                                                                   \
        hipError_t e_ = (x);                                                                               \
        if (e_ != hipSuccess) {                                                                            \
            (ctx)->err = std::string(#x) + ": " + hipGetErrorString(e_);                                   \
            return BH_ERR_HIP;                                                                             \
        }                                                                                                  \
    } while (0)

namespace {

Norm default_norm() {
    Norm N;
    const double lo[3] = {LX_LO, LTH_LO, LS_LO}, hi[3] = {LX_HI, LTH_HI, LS_HI};
    for (int k = 0; k < 3; ++k) {
        N.x_c[k] = (float)(0.5 * (lo[k] + hi[k]));
        N.x_h[k] = (float)(0.5 * (hi[k] - lo[k]));
    }
    N.y_mu[0] = N.y_mu[1] = 0.f;
    N.y_sd[0] = N.y_sd[1] = 1.f;
    return N;
}

void norm_to_floats(const Norm& N, float* v) {
    for (int k = 0; k < 3; ++k) {
        v[k] = N.x_c[k];
        v[3 + k] = N.x_h[k];
    }
    v[6] = N.y_mu[0];
    v[7] = N.y_mu[1];
    v[8] = N.y_sd[0];
    v[9] = N.y_sd[1];
}

Norm norm_from_floats(const float* v) {
    Norm N;
    for (int k = 0; k < 3; ++k) {
        N.x_c[k] = v[k];
        N.x_h[k] = v[3 + k];
    }
    N.y_mu[0] = v[6];
    N.y_mu[1] = v[7];
    N.y_sd[0] = v[8];
    N.y_sd[1] = v[9];
    return N;
}

int ensure_params(bh_ctx* c) {
    if (c->d_mlp) return BH_OK;
    MCK(c, hipMalloc((void**)&c->d_mlp, sizeof(float) * NPARAM));
    MCK(c, hipMalloc((void**)&c->d_adam_m, sizeof(float) * NPARAM));
    MCK(c, hipMalloc((void**)&c->d_adam_v, sizeof(float) * NPARAM));
    return BH_OK;
}

// He-style uniform initialisation (host, seeded)
void init_params(uint64_t seed, std::vector<float>* p) {
    p->assign(NPARAM, 0.f);
    uint64_t s = seed * 0x9E3779B97F4A7C15ull + 1;
    auto next = [&]() {
        s ^= s << 13;
        s ^= s >> 7;
        s ^= s << 17;
        return (double)(s >> 11) * 0x1p-53 * 2.0 - 1.0;
    };
    auto fill = [&](int off, int fan_in, int count) {
        const double a = std::sqrt(6.0 / fan_in);
        for (int i = 0; i < count; ++i) (*p)[off + i] = (float)(a * next());
    };
    fill(OFF_W1, NIN, NIN * NH);
    fill(OFF_W2, NH, NH * NH);
    fill(OFF_W3, NH, NH * NH);
    fill(OFF_W4, NH, NH * NOUT);
}

double now_ms() {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

}  // namespace

extern "C" {

int bh_mlp_train(bh_ctx* c, const bh_mlp_train_cfg* cfg_in, bh_mlp_report* rep) {
    if (!c) return BH_ERR_ARG;
    if (!c->d_k2) {
        c->err = "the surrogate's exact routine needs the K2 table (radio scene)";
        return BH_ERR_ARG;
    }
    bh_mlp_train_cfg cfg{};
    if (cfg_in) cfg = *cfg_in;
    if (cfg.n_samples <= 0) cfg.n_samples = 1 << 22;
    if (cfg.batch <= 0) cfg.batch = 8192;
    if (cfg.epochs <= 0) cfg.epochs = 200;
    if (!(cfg.lr > 0)) cfg.lr = 2e-3f;
    if (!(cfg.lr_min > 0)) cfg.lr_min = 2e-5f;
    if (cfg.seed == 0) cfg.seed = 1;
    if (!(cfg.hot_weight >= 0)) cfg.hot_weight = 20.f;
    if (cfg.batch % TM != 0 || cfg.batch > cfg.n_samples) {
        c->err = "batch must be a multiple of 16 and at most n_samples";
        return BH_ERR_ARG;
    }
    MCK(c, hipSetDevice(c->device));
    int rc = ensure_params(c);
    if (rc) return rc;
    const int n = cfg.n_samples;
    float *xs = nullptr, *ts = nullptr, *ws = nullptr, *partial = nullptr, *lpart = nullptr, *grad = nullptr,
          *loss = nullptr;
    const int nwg = (cfg.batch / TM + GRAD_TILES - 1) / GRAD_TILES;
    auto cleanup = [&]() {
        for (float* p : {xs, ts, ws, partial, lpart, grad, loss})
            if (p) (void)hipFree(p);
    };
    double t0 = now_ms();
    if (hipMalloc((void**)&xs, sizeof(float) * 3 * (size_t)n) != hipSuccess ||
        hipMalloc((void**)&ts, sizeof(float) * 2 * (size_t)n) != hipSuccess ||
        hipMalloc((void**)&ws, sizeof(float) * (size_t)n) != hipSuccess ||
        hipMalloc((void**)&partial, sizeof(float) * PSTRIDE * (size_t)nwg) != hipSuccess ||
        hipMalloc((void**)&lpart, sizeof(float) * nwg) != hipSuccess ||
        hipMalloc((void**)&grad, sizeof(float) * NPARAM) != hipSuccess ||
        hipMalloc((void**)&loss, sizeof(float)) != hipSuccess) {
        cleanup();
        c->err = "surrogate training buffers: hipMalloc failed";
        return BH_ERR_HIP;
    }
    Norm N = default_norm();
    hipLaunchKernelGGL(k_mlp_sample, dim3((n + 255) / 256), dim3(256), 0, c->st, cfg.seed, n, c->d_k2, c->k2_n,
                       c->k2_l0, c->k2_dl, N, cfg.hot_weight, xs, ts, ws);
    // output normalisation from the samples
    std::vector<float> th((size_t)2 * n);
    if (hipMemcpyAsync(th.data(), ts, sizeof(float) * 2 * (size_t)n, hipMemcpyDeviceToHost, c->st) != hipSuccess ||
        hipStreamSynchronize(c->st) != hipSuccess) {
        cleanup();
        c->err = "surrogate sampler failed";
        return BH_ERR_HIP;
    }
    for (int o = 0; o < 2; ++o) {
        double s = 0, s2 = 0;
        for (int i = 0; i < n; ++i) {
            s += th[2 * (size_t)i + o];
            s2 += (double)th[2 * (size_t)i + o] * th[2 * (size_t)i + o];
        }
        const double mu = s / n;
        N.y_mu[o] = (float)mu;
        N.y_sd[o] = (float)std::sqrt(std::max(s2 / n - mu * mu, 1e-12));
    }
    double t1 = now_ms();
    std::vector<float> p0;
    init_params(cfg.seed, &p0);
    std::vector<float> zeros(NPARAM, 0.f);
    if (hipMemcpyAsync(c->d_mlp, p0.data(), sizeof(float) * NPARAM, hipMemcpyHostToDevice, c->st) != hipSuccess ||
        hipMemcpyAsync(c->d_adam_m, zeros.data(), sizeof(float) * NPARAM, hipMemcpyHostToDevice, c->st) != hipSuccess ||
        hipMemcpyAsync(c->d_adam_v, zeros.data(), sizeof(float) * NPARAM, hipMemcpyHostToDevice, c->st) != hipSuccess) {
        cleanup();
        c->err = "surrogate parameter upload failed";
        return BH_ERR_HIP;
    }
    const int steps_per_epoch = n / cfg.batch;
    const int total = steps_per_epoch * cfg.epochs;
    float first_loss = -1.f, last_loss = -1.f;
    for (int step = 0; step < total; ++step) {
        const int first = (int)(((long long)step * cfg.batch) % n);
        hipLaunchKernelGGL(k_mlp_grad, dim3(nwg), dim3(GRAD_BLOCK), 0, c->st, c->d_mlp, N, xs, ts, ws, n, first,
                           cfg.batch, partial, lpart);
        const double prog = (double)step / std::max(total - 1, 1);
        const float lr = (float)(cfg.lr_min + 0.5 * (cfg.lr - cfg.lr_min) * (1.0 + std::cos(3.141592653589793 * prog)));
        const float bc1 = (float)(1.0 - std::pow(0.9, step + 1)), bc2 = (float)(1.0 - std::pow(0.999, step + 1));
        const AdamStep A{c->d_mlp, c->d_adam_m, c->d_adam_v, lr, 0.9f, 0.999f, 1e-8f, bc1, bc2};
        hipLaunchKernelGGL(k_mlp_reduce, dim3((NPARAM + RED_PARAMS - 1) / RED_PARAMS), dim3(RED_BLOCK), 0, c->st,
                           partial, nwg, lpart, grad, loss, A);
        if (step == 0 || step == total - 1) {
            float l = 0;
            if (hipMemcpyAsync(&l, loss, sizeof(float), hipMemcpyDeviceToHost, c->st) != hipSuccess ||
                hipStreamSynchronize(c->st) != hipSuccess) {
                cleanup();
                c->err = "surrogate training step failed";
                return BH_ERR_HIP;
            }
            if (step == 0) first_loss = l;
            else last_loss = l;
        }
    }
    if (hipStreamSynchronize(c->st) != hipSuccess || hipGetLastError() != hipSuccess) {
        cleanup();
        c->err = "surrogate training failed";
        return BH_ERR_HIP;
    }
    double t2 = now_ms();
    cleanup();
    c->mlp_norm = N;
    c->mlp_trained = true;
    c->stab_ready = false;
    if (rep) {
        rep->ms_sample = t1 - t0;
        rep->ms_train = t2 - t1;
        rep->steps = total;
        rep->loss_first = first_loss;
        rep->loss_last = last_loss;
        // 3 MFMA products per hidden GEMM, forward + 2 backward GEMMs per hidden layer
        rep->train_flop = (double)total * cfg.batch * 2.0 * (2.0 * NH * NH) * 3.0 * 3.0;
    }
    return BH_OK;
}

int bh_mlp_get(bh_ctx* c, float* params, float* norm) {
    if (!c || !params) return BH_ERR_ARG;
    if (!c->mlp_trained) {
        c->err = "no surrogate parameters";
        return BH_ERR_ARG;
    }
    MCK(c, hipSetDevice(c->device));
    MCK(c, hipMemcpy(params, c->d_mlp, sizeof(float) * NPARAM, hipMemcpyDeviceToHost));
    if (norm) norm_to_floats(c->mlp_norm, norm);
    return BH_OK;
}

int bh_mlp_set(bh_ctx* c, const float* params, const float* norm) {
    if (!c || !params || !norm) return BH_ERR_ARG;
    MCK(c, hipSetDevice(c->device));
    int rc = ensure_params(c);
    if (rc) return rc;
    MCK(c, hipMemcpy(c->d_mlp, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice));
    c->mlp_norm = norm_from_floats(norm);
    c->mlp_trained = true;
    c->stab_ready = false;
    return BH_OK;
}

int bh_mlp_infer(bh_ctx* c, const float* in, int n, float* out) {
    if (!c || !in || !out || n < 0) return BH_ERR_ARG;
    if (!c->mlp_trained) {
        c->err = "no surrogate parameters";
        return BH_ERR_ARG;
    }
    if (n == 0) return BH_OK;
    MCK(c, hipSetDevice(c->device));
    float* din = nullptr;
    float2* dout = nullptr;
    int rc = BH_OK;
    if (hipMalloc((void**)&din, sizeof(float) * 3 * (size_t)n) != hipSuccess ||
        hipMalloc((void**)&dout, sizeof(float2) * (size_t)n) != hipSuccess ||
        hipMemcpy(din, in, sizeof(float) * 3 * (size_t)n, hipMemcpyHostToDevice) != hipSuccess) {
        rc = BH_ERR_HIP;
    } else {
        const int ntiles = (n + TM - 1) / TM;
        Lattice L{};
        hipLaunchKernelGGL(k_mlp_infer, dim3(std::min(ntiles, INFER_GRID)), dim3(64 * TILE_WAVES), 0, c->st, c->d_mlp,
                           c->mlp_norm, din, n, 0, L, (float*)dout);
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(out, dout, sizeof(float2) * (size_t)n, hipMemcpyDeviceToHost, c->st) != hipSuccess ||
            hipStreamSynchronize(c->st) != hipSuccess)
            rc = BH_ERR_HIP;
    }
    if (din) (void)hipFree(din);
    if (dout) (void)hipFree(dout);
    if (rc) c->err = "surrogate inference failed";
    return rc;
}

int bh_mlp_exact(bh_ctx* c, const float* in, int n, double* out) {
    if (!c || !in || !out || n < 0) return BH_ERR_ARG;
    if (!c->d_k2) {
        c->err = "the exact routine needs the K2 table";
        return BH_ERR_ARG;
    }
    if (n == 0) return BH_OK;
    MCK(c, hipSetDevice(c->device));
    float* din = nullptr;
    double* dout = nullptr;
    int rc = BH_OK;
    if (hipMalloc((void**)&din, sizeof(float) * 3 * (size_t)n) != hipSuccess ||
        hipMalloc((void**)&dout, sizeof(double) * 2 * (size_t)n) != hipSuccess ||
        hipMemcpy(din, in, sizeof(float) * 3 * (size_t)n, hipMemcpyHostToDevice) != hipSuccess) {
        rc = BH_ERR_HIP;
    } else {
        hipLaunchKernelGGL(k_mlp_exact, dim3((n + 255) / 256), dim3(256), 0, c->st, din, n, c->d_k2, c->k2_n, c->k2_l0,
                           c->k2_dl, dout);
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(out, dout, sizeof(double) * 2 * (size_t)n, hipMemcpyDeviceToHost, c->st) != hipSuccess ||
            hipStreamSynchronize(c->st) != hipSuccess)
            rc = BH_ERR_HIP;
    }
    if (din) (void)hipFree(din);
    if (dout) (void)hipFree(dout);
    if (rc) c->err = "exact routine failed";
    return rc;
}

int bh_mlp_grad(bh_ctx* c, const float* params, const float* norm, const float* xn, const float* tn, const float* w,
                int n, float* loss_out, float* grad_out) {
    if (!c || !params || !norm || !xn || !tn || !w || !grad_out || n <= 0 || n % TM != 0) return BH_ERR_ARG;
    MCK(c, hipSetDevice(c->device));
    const Norm N = norm_from_floats(norm);
    const int nwg = (n / TM + GRAD_TILES - 1) / GRAD_TILES;
    float *dp = nullptr, *dx = nullptr, *dt = nullptr, *dw = nullptr, *part = nullptr, *lp = nullptr, *g = nullptr,
          *l = nullptr;
    int rc = BH_OK;
    if (hipMalloc((void**)&dp, sizeof(float) * NPARAM) != hipSuccess ||
        hipMalloc((void**)&dx, sizeof(float) * 3 * (size_t)n) != hipSuccess ||
        hipMalloc((void**)&dt, sizeof(float) * 2 * (size_t)n) != hipSuccess ||
        hipMalloc((void**)&dw, sizeof(float) * (size_t)n) != hipSuccess ||
        hipMalloc((void**)&part, sizeof(float) * PSTRIDE * (size_t)nwg) != hipSuccess ||
        hipMalloc((void**)&lp, sizeof(float) * nwg) != hipSuccess ||
        hipMalloc((void**)&g, sizeof(float) * NPARAM) != hipSuccess || hipMalloc((void**)&l, sizeof(float)) != hipSuccess ||
        hipMemcpy(dp, params, sizeof(float) * NPARAM, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dx, xn, sizeof(float) * 3 * (size_t)n, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dt, tn, sizeof(float) * 2 * (size_t)n, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(dw, w, sizeof(float) * (size_t)n, hipMemcpyHostToDevice) != hipSuccess) {
        rc = BH_ERR_HIP;
    } else {
        hipLaunchKernelGGL(k_mlp_grad, dim3(nwg), dim3(GRAD_BLOCK), 0, c->st, dp, N, dx, dt, dw, n, 0, n, part, lp);
        hipLaunchKernelGGL(k_mlp_reduce, dim3((NPARAM + RED_PARAMS - 1) / RED_PARAMS), dim3(RED_BLOCK), 0, c->st, part,
                           nwg, lp, g, l, AdamStep{});
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(grad_out, g, sizeof(float) * NPARAM, hipMemcpyDeviceToHost, c->st) != hipSuccess ||
            (loss_out && hipMemcpyAsync(loss_out, l, sizeof(float), hipMemcpyDeviceToHost, c->st) != hipSuccess) ||
            hipStreamSynchronize(c->st) != hipSuccess)
            rc = BH_ERR_HIP;
    }
    for (float* p : {dp, dx, dt, dw, part, lp, g, l})
        if (p) (void)hipFree(p);
    if (rc) c->err = "surrogate gradient failed";
    return rc;
}

int bh_mlp_bake(bh_ctx* c, int n0, int n1, int n2, float judge_tol, bh_mlp_bake_report* rep) {
    if (!c) return BH_ERR_ARG;
    if (!c->mlp_trained || !c->d_k2) {
        c->err = "baking needs trained surrogate parameters and the K2 table";
        return BH_ERR_ARG;
    }
    if (n0 <= 0) n0 = 1024;
    if (n1 <= 0) n1 = 128;
    if (n2 <= 0) n2 = 8;
    if (!(judge_tol > 0)) judge_tol = 2e-3f;
    if (n0 < 2 || n1 < 2 || n2 < 2 || (size_t)n0 * n1 * n2 > (size_t)1 << 24) {
        c->err = "bad surrogate lattice size";
        return BH_ERR_ARG;
    }
    MCK(c, hipSetDevice(c->device));
    if (c->d_stab) (void)hipFree(c->d_stab);
    if (c->d_sbad) (void)hipFree(c->d_sbad);
    c->d_stab = nullptr;
    c->d_sbad = nullptr;
    c->stab_ready = false;
    const size_t nodes = (size_t)n0 * n1 * n2, cells = (size_t)(n0 - 1) * (n1 - 1) * (n2 - 1);
    MCK(c, hipMalloc((void**)&c->d_stab, sizeof(float2) * nodes));
    MCK(c, hipMalloc((void**)&c->d_sbad, cells));
    unsigned int* counts = nullptr;
    MCK(c, hipMalloc((void**)&counts, 2 * sizeof(unsigned int)));
    // lattice over the surrogate coordinates (ln X, ln Theta, ln sin theta_B)
    Lattice L;
    L.n0 = n0;
    L.n1 = n1;
    L.n2 = n2;
    L.lo0 = (float)LX_LO;
    L.d0 = (float)((LX_HI - LX_LO) / (n0 - 1));
    L.lo1 = (float)LTH_LO;
    L.d1 = (float)((LTH_HI - LTH_LO) / (n1 - 1));
    L.lo2 = (float)LS_LO;
    L.d2 = (float)((LS_HI - LS_LO) / (n2 - 1));
    double t0 = now_ms();
    const int ntiles = (int)((nodes + TM - 1) / TM);
    hipLaunchKernelGGL(k_mlp_infer, dim3(std::min(ntiles, INFER_GRID)), dim3(64 * TILE_WAVES), 0, c->st, c->d_mlp,
                       c->mlp_norm, nullptr, (int)nodes, 1, L, (float*)c->d_stab);
    hipEvent_t e0, e1;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    (void)hipEventRecord(e0, c->st);
    (void)hipMemsetAsync(counts, 0, 2 * sizeof(unsigned int), c->st);
    hipLaunchKernelGGL(k_mlp_judge, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0, c->st, c->d_stab, L, c->d_k2,
                       c->k2_n, c->k2_l0, c->k2_dl, judge_tol, (float)(FLOOR_J + 10.0), (float)(FLOOR_A + 10.0),
                       c->d_sbad, counts);
    (void)hipEventRecord(e1, c->st);
    unsigned int hc[2] = {0, 0};
    int rc = BH_OK;
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(hc, counts, sizeof hc, hipMemcpyDeviceToHost, c->st) != hipSuccess ||
        hipStreamSynchronize(c->st) != hipSuccess)
        rc = BH_ERR_HIP;
    float ms_judge = 0.f;
    (void)hipEventElapsedTime(&ms_judge, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(counts);
    if (rc) {
        c->err = "surrogate bake failed";
        return rc;
    }
    SurrogateTable& T = c->stab;
    T.tab = (const float*)c->d_stab;
    T.bad = c->d_sbad;
    T.n0 = n0;
    T.n1 = n1;
    T.n2 = n2;
    T.lo0 = L.lo0;
    T.lo1 = L.lo1;
    T.lo2 = L.lo2;
    T.inv_d0 = 1.f / L.d0;
    T.inv_d1 = 1.f / L.d1;
    T.inv_d2 = 1.f / L.d2;
    T.hi0 = (float)LX_HI;
    c->stab_ready = true;
    if (rep) {
        rep->ms_bake = now_ms() - t0;
        rep->ms_judge = ms_judge;
        rep->cells = (long long)cells;
        rep->hot_cells = hc[0];
        rep->failed_hot_cells = hc[1];
    }
    return BH_OK;
}

}  // extern "C"

/* trace_fp64.h - plain FP64 per-ray Kerr tracer for gfx950 (device code, included by bhrt.hip).

   Parity contract: with -ffp-contract=off every value below rounds exactly like the reference
   integrator's host build (blackholes/src/kerr.hpp, trace.cuh, emission.cuh), except that the
   elementary functions come from bh_math.h; the CPU oracle built on bh_math.h reproduces the
   results bit for bit.

   MI355X layout of the work:
   - One ray per lane, wave64; the integrator state lives in VGPRs for the whole trace.
   - Dormand-Prince 5(4) is evaluated incrementally: after each stage derivative k_i the partial
     sums of every later stage, of the 5th-order solution and of the error estimate are updated in
     the reference's left-to-right association order, so the live set is partial sums instead of
     seven stored derivative vectors.
   - The phi and t components never enter the right-hand side (kerr.hpp:103-116), so their stage
     states are never formed; only their 5th-order sums (and phi's error term) are kept.
   - d[0] = y[1] and d[2] = y[3]: the r and u components of each stage derivative are the stage
     state's r' and u' and are not stored separately.
   - The coordinate time enters neither the right-hand side nor the error norm, so a frame that reads
     it nowhere (static turbulence, no ray records) does not integrate it.
   - The kernels are bound by VALU issue, so the correctly rounded quotients and roots take their
     shortest form (bh_math.h quot_, sqrt_pos_): the operators' range scaling and fix-up are half of
     their instructions and the operands here stay far from the ends of the exponent range. Where one
     can leave it (a stage inside the horizon or past the pole, a step that diverged), the code below
     says what catches it. With the time left out where nothing reads it, one power per attempt and the
     sine, cosine and root of the swept angle handed on to the flow, the bound per attempt fell by a
     third at the same bits: 1024^2 230 GHz frame 27.8 -> 20.3 ms, 160^2 normalising flux 15.5 -> 9.7
     ms, 256^2 vacuum records 5.2 -> 4.1 ms (static VALU instructions of the frame's persistent kernel
     3997 -> 2885, 164 -> 140 VGPRs). */
#pragma once
#include "bh_math.h"

namespace bhd {

// blackholes/src/common.hpp:17-28
constexpr double C_C = 2.99792458e10, C_KB = 1.380649e-16, C_H = 6.62607015e-27, C_ME = 9.1093837e-28,
                 C_MP = 1.67262192e-24, C_QE = 4.80320471e-10;
constexpr double PI = 3.14159265358979323846;

// The tracers' RADIO template argument: no flow (thermal disk), or the radio flow with the grid
// turbulence or with the sheared turbulence. The turbulence model is a compile-time choice so a
// kernel carries the lookup code of one model only (registers and instruction cache).
constexpr int RADIO_OFF = 0, RADIO_GRID = 1, RADIO_SHEARED = 2;
// The TIME template argument: whether something reads the coordinate time (time-dependent turbulence,
// ray records, a bound on its error); without it t is not integrated. A compile-time choice too: both
// steps in one kernel cost 26 registers (166 and 140 alone, 168 and spills together).
constexpr int MODE_VISIBLE = 0;   // bh_scene.mode: vacuum geodesics and the celestial sphere

// Dormand-Prince 1980 tableau (kerr.hpp:124-129): the same constant expressions, folded by the compiler.
constexpr double a21 = 1.0 / 5, a31 = 3.0 / 40, a32 = 9.0 / 40, a41 = 44.0 / 45, a42 = -56.0 / 15, a43 = 32.0 / 9;
constexpr double a51 = 19372.0 / 6561, a52 = -25360.0 / 2187, a53 = 64448.0 / 6561, a54 = -212.0 / 729;
constexpr double a61 = 9017.0 / 3168, a62 = -355.0 / 33, a63 = 46732.0 / 5247, a64 = 49.0 / 176, a65 = -5103.0 / 18656;
constexpr double b1 = 35.0 / 384, b3 = 500.0 / 1113, b4 = 125.0 / 192, b5 = -2187.0 / 6784, b6 = 11.0 / 84;
constexpr double e1 = 71.0 / 57600, e3 = -71.0 / 16695, e4 = 71.0 / 1920, e5 = -17253.0 / 339200, e6 = 22.0 / 525,
                 e7 = -1.0 / 40;

// Baked sheared-turbulence slices (turb_sheared.h): nt slices of nz x nlr x nphi floats, phi fastest,
// with the slice coordinates and the camera they were baked for.
struct ShearedView {
    const float* data;
    int nphi, nlr, nz, nt;
    float lr0, lr1, zmax, d0, dd;
    float inv_dd;               // 1 / dd
    double inv_lr, inv_zmax;    // 1 / (lr1 - lr0), 1 / zmax
    double cam_t, cam_r;
};

// Uniform scene and frame parameters: passed by value as the kernel argument, so they sit in SGPRs.
struct TraceParams {
    // scene (bh_scene)
    double a, a2, rh, r_isco, tol, r_escape, r_stop, step_frac;
    double inv_tol;   // 1 / tol
    double err_big;   // scaled errors whose numerators exceed this are rejected unscaled (dp54_step)
    int max_steps, mode, flow_on, turb_on;
    double n0, n_index, theta_index, theta0, h_r, beta_p, r_flow_max, nu_obs, rg_cm, flow_kep;
    const float* __restrict__ k2;
    int k2_n;
    float k2_l0, k2_dl, k2_inv_dl;
    const float* __restrict__ turb;
    int turb_n, turb_nt;
    double turb_half, turb_inv_dx, turb_t0, turb_inv_dt;
    // sheared turbulence (RADIO_SHEARED kernels): the slices and their coordinates, in device memory
    // so the kernel arguments stay small
    const struct ShearedView* __restrict__ ts;
    // frame (bh_frame)
    double ph0, t0;
    double kp[11];
    double F[3], R[3], U[3], beta[3];
    double cx, cy, pix;
    int W, H;
    uint32_t seed;
    // visible mode: checkerboard celestial sphere (sky_nu x sky_nv squares of galactic u, v)
    int sky_on, sky_nu, sky_nv;
    float sky_scale;
    double sky_rot[9];
    // launch
    int x0, y0, w, h, spp, jitter;
};

struct RayResult {
    double y[6];
    double th_inf, ph_inf;
    double I[4];
    double trans, psi;
    int fate, ncross, order, steps, accepted, flow_steps;
    float sky_u, sky_v;
};

struct RayConst {
    double lam, eta, E, K, lam2, alam;
};

// blackholes/src/device_util.cuh:15-29, render.cu:70-80
__device__ __forceinline__ uint32_t pcg(uint32_t v) {
    uint32_t s = v * 747796405u + 2891336453u;
    uint32_t w = ((s >> ((s >> 28u) + 4u)) ^ s) * 277803737u;
    return (w >> 22u) ^ w;
}
// the reference's sheared turbulence (bake and lookup), in this namespace
#include "turb_sheared.h"

__device__ __forceinline__ void sample_offsets(const TraceParams& P, int px, int py, int s, double* tx, double* ty) {
    float jx = 0.5f, jy = 0.5f;
    if (P.jitter) {
        uint32_t hs = pcg((uint32_t)(py * P.W + px) * 0x9E3779B9u ^ P.seed);
        hs = pcg(hs);
        float r0 = (hs >> 8) * (1.0f / 16777216.0f);
        hs = pcg(hs);
        float r1 = (hs >> 8) * (1.0f / 16777216.0f);
        // fmod(n a, 1) for n a >= 0 is n a - floor(n a), exactly
        double q1 = (double)(uint32_t)s * 0.7548776662466927, q2 = (double)(uint32_t)s * 0.5698402909980532;
        float fx = r0 + (float)(q1 - floor(q1)), fy = r1 + (float)(q2 - floor(q2));
        jx = fx - floorf(fx);
        jy = fy - floorf(fy);
    }
    *tx = (px + jx - 0.5 * P.W) * P.pix;
    *ty = (0.5 * P.H - (py + jy)) * P.pix;
}

// blackholes/src/kerr.hpp:103-116 (components 1, 3, 4, 5; d0 = y1 and d2 = y3)
struct Rhs {
    double d1, d3, d4, d5;
};
// The quotients by Delta share its reciprocal; Delta may vanish or overflow at a wild stage, which
// the fix-up instruction turns into the IEEE result. s2 is at least 1e-300, so lam / s2 needs none
// (past the pole it is finite for |lam| < 1e8). Without TIME d5 is not formed.
template <bool TIME>
__device__ __forceinline__ Rhs rhs(const TraceParams& P, const RayConst& c, double r, double u) {
    double r2 = r * r;
    double Delta = r2 - 2.0 * r + P.a2;
    double Pp = r2 + P.a2 - c.alam;
    double s2 = fmax(1.0 - u * u, 1e-300);
    Rhs o;
    o.d1 = 2.0 * r * Pp - (r - 1.0) * c.K;
    o.d3 = u * (P.a2 * (1.0 - 2.0 * u * u) - c.eta - c.lam2);
    const bhm::Recip iD = bhm::recip_(Delta);
    const double n4 = P.a * Pp;
    o.d4 = -(__builtin_amdgcn_div_fixup(bhm::quot_(n4, iD), Delta, n4) + bhm::quot_(c.lam, s2) - P.a);
    if (TIME) {
        const double n5 = (r2 + P.a2) * Pp;
        o.d5 = -(__builtin_amdgcn_div_fixup(bhm::quot_(n5, iD), Delta, n5) + P.a * (c.lam - P.a * s2));
    } else {
        o.d5 = 0.0;
    }
    return o;
}

// Integrator state: y and the FSAL derivative k1 (k1[0] == y[1] and k1[2] == y[3] always hold).
struct State {
    double y0, y1, y2, y3, y4, y5;
    double k1, k3, k4, k5;   // k1[1], k1[3], k1[4], k1[5]
};

// blackholes/src/kerr.hpp:122-157. Returns the scaled error; on return `o` holds (yout, k7).
template <bool TIME>
__device__ __forceinline__ double dp54_step(const TraceParams& P, const RayConst& c, const State& s, double h,
                                            State& o) {
    // partial sums of stages 3..6, of the 5th-order increment (O) and of the error (E), per component
    // (0: r, 1: r', 2: u, 3: u'); k_i component 0 is stage i's r', component 2 is stage i's u'.
    const double ha21 = h * a21;
    double q0 = s.y1, q1 = s.k1, q2 = s.y3, q3 = s.k3;   // k1 components 0..3
    double S3_0 = a31 * q0, S3_1 = a31 * q1, S3_2 = a31 * q2, S3_3 = a31 * q3;
    double S4_0 = a41 * q0, S4_1 = a41 * q1, S4_2 = a41 * q2, S4_3 = a41 * q3;
    double S5_0 = a51 * q0, S5_1 = a51 * q1, S5_2 = a51 * q2, S5_3 = a51 * q3;
    double S6_0 = a61 * q0, S6_1 = a61 * q1, S6_2 = a61 * q2, S6_3 = a61 * q3;
    double O0 = b1 * q0, O1 = b1 * q1, O2 = b1 * q2, O3 = b1 * q3, O4 = b1 * s.k4, O5 = TIME ? b1 * s.k5 : 0.0;
    double E0 = e1 * q0, E1 = e1 * q1, E2 = e1 * q2, E3 = e1 * q3, E4 = e1 * s.k4;
    // stage 2
    double t0 = s.y0 + ha21 * q0, t1 = s.y1 + ha21 * q1, t2 = s.y2 + ha21 * q2, t3 = s.y3 + ha21 * q3;
    Rhs k = rhs<TIME>(P, c, t0, t2);
    q0 = t1; q1 = k.d1; q2 = t3; q3 = k.d3;
    S3_0 = S3_0 + a32 * q0; S3_1 = S3_1 + a32 * q1; S3_2 = S3_2 + a32 * q2; S3_3 = S3_3 + a32 * q3;
    S4_0 = S4_0 + a42 * q0; S4_1 = S4_1 + a42 * q1; S4_2 = S4_2 + a42 * q2; S4_3 = S4_3 + a42 * q3;
    S5_0 = S5_0 + a52 * q0; S5_1 = S5_1 + a52 * q1; S5_2 = S5_2 + a52 * q2; S5_3 = S5_3 + a52 * q3;
    S6_0 = S6_0 + a62 * q0; S6_1 = S6_1 + a62 * q1; S6_2 = S6_2 + a62 * q2; S6_3 = S6_3 + a62 * q3;
    // stage 3
    t0 = s.y0 + h * S3_0; t1 = s.y1 + h * S3_1; t2 = s.y2 + h * S3_2; t3 = s.y3 + h * S3_3;
    k = rhs<TIME>(P, c, t0, t2);
    q0 = t1; q1 = k.d1; q2 = t3; q3 = k.d3;
    S4_0 = S4_0 + a43 * q0; S4_1 = S4_1 + a43 * q1; S4_2 = S4_2 + a43 * q2; S4_3 = S4_3 + a43 * q3;
    S5_0 = S5_0 + a53 * q0; S5_1 = S5_1 + a53 * q1; S5_2 = S5_2 + a53 * q2; S5_3 = S5_3 + a53 * q3;
    S6_0 = S6_0 + a63 * q0; S6_1 = S6_1 + a63 * q1; S6_2 = S6_2 + a63 * q2; S6_3 = S6_3 + a63 * q3;
    O0 = O0 + b3 * q0; O1 = O1 + b3 * q1; O2 = O2 + b3 * q2; O3 = O3 + b3 * q3; O4 = O4 + b3 * k.d4;
    if (TIME) O5 = O5 + b3 * k.d5;
    E0 = E0 + e3 * q0; E1 = E1 + e3 * q1; E2 = E2 + e3 * q2; E3 = E3 + e3 * q3; E4 = E4 + e3 * k.d4;
    // stage 4
    t0 = s.y0 + h * S4_0; t1 = s.y1 + h * S4_1; t2 = s.y2 + h * S4_2; t3 = s.y3 + h * S4_3;
    k = rhs<TIME>(P, c, t0, t2);
    q0 = t1; q1 = k.d1; q2 = t3; q3 = k.d3;
    S5_0 = S5_0 + a54 * q0; S5_1 = S5_1 + a54 * q1; S5_2 = S5_2 + a54 * q2; S5_3 = S5_3 + a54 * q3;
    S6_0 = S6_0 + a64 * q0; S6_1 = S6_1 + a64 * q1; S6_2 = S6_2 + a64 * q2; S6_3 = S6_3 + a64 * q3;
    O0 = O0 + b4 * q0; O1 = O1 + b4 * q1; O2 = O2 + b4 * q2; O3 = O3 + b4 * q3; O4 = O4 + b4 * k.d4;
    if (TIME) O5 = O5 + b4 * k.d5;
    E0 = E0 + e4 * q0; E1 = E1 + e4 * q1; E2 = E2 + e4 * q2; E3 = E3 + e4 * q3; E4 = E4 + e4 * k.d4;
    // stage 5
    t0 = s.y0 + h * S5_0; t1 = s.y1 + h * S5_1; t2 = s.y2 + h * S5_2; t3 = s.y3 + h * S5_3;
    k = rhs<TIME>(P, c, t0, t2);
    q0 = t1; q1 = k.d1; q2 = t3; q3 = k.d3;
    S6_0 = S6_0 + a65 * q0; S6_1 = S6_1 + a65 * q1; S6_2 = S6_2 + a65 * q2; S6_3 = S6_3 + a65 * q3;
    O0 = O0 + b5 * q0; O1 = O1 + b5 * q1; O2 = O2 + b5 * q2; O3 = O3 + b5 * q3; O4 = O4 + b5 * k.d4;
    if (TIME) O5 = O5 + b5 * k.d5;
    E0 = E0 + e5 * q0; E1 = E1 + e5 * q1; E2 = E2 + e5 * q2; E3 = E3 + e5 * q3; E4 = E4 + e5 * k.d4;
    // stage 6
    t0 = s.y0 + h * S6_0; t1 = s.y1 + h * S6_1; t2 = s.y2 + h * S6_2; t3 = s.y3 + h * S6_3;
    k = rhs<TIME>(P, c, t0, t2);
    q0 = t1; q1 = k.d1; q2 = t3; q3 = k.d3;
    O0 = O0 + b6 * q0; O1 = O1 + b6 * q1; O2 = O2 + b6 * q2; O3 = O3 + b6 * q3; O4 = O4 + b6 * k.d4;
    if (TIME) O5 = O5 + b6 * k.d5;
    E0 = E0 + e6 * q0; E1 = E1 + e6 * q1; E2 = E2 + e6 * q2; E3 = E3 + e6 * q3; E4 = E4 + e6 * k.d4;
    // 5th-order solution and its derivative (FSAL)
    o.y0 = s.y0 + h * O0; o.y1 = s.y1 + h * O1; o.y2 = s.y2 + h * O2; o.y3 = s.y3 + h * O3;
    o.y4 = s.y4 + h * O4; o.y5 = TIME ? s.y5 + h * O5 : s.y5;
    k = rhs<TIME>(P, c, o.y0, o.y2);
    o.k1 = k.d1; o.k3 = k.d3; o.k4 = k.d4; o.k5 = TIME ? k.d5 : s.k5;
    E0 = E0 + e7 * o.y1; E1 = E1 + e7 * k.d1; E2 = E2 + e7 * o.y3; E3 = E3 + e7 * k.d3; E4 = E4 + e7 * k.d4;
    // scaled max-norm over r, r', u, u', phi (kerr.hpp:145-155): max_i |h E_i| / sc_i with sc = tol
    // for u and 4 tol for phi. Rounding is monotone and the factor 4 exact, so those two quotients are
    // the one of their larger numerator.
    const double x0 = fabs(h * E0), x1 = fabs(h * E1), x3 = fabs(h * E3);
    const double x2 = fmax(fabs(h * E2), 0.25 * fabs(h * E4));
    const double sc0 = P.tol * (1e-6 + fmax(fabs(s.y0), fabs(o.y0)));
    const double sc1 = P.tol * (1e-6 + fmax(fmax(fabs(s.y1), fabs(o.y1)), s.y0 * s.y0));
    const double sc3 = P.tol * fmax(1.0, fmax(fabs(s.y3), fabs(o.y3)));
    double m = fmax(0.0, bhm::quot_(x0, sc0));
    m = fmax(m, bhm::quot_(x1, sc1));
    m = fmax(m, bhm::quot_(x2, bhm::Recip{P.tol, P.inv_tol}));
    m = fmax(m, bhm::quot_(x3, sc3));
    // A diverged step (an error beyond 1e200 tol, an infinity) is rejected without its quotients, which
    // could overflow: the controller's factor is 0.2 for every error above 2e3. A NaN is no error, as
    // in the maximum above and in the reference's.
    return fmax(fmax(x0, x1), fmax(x2, x3)) > P.err_big ? 1e300 : m;
}

// The controller's factor min(5, max(0.2, 0.9 err^-0.2)) (trace.cuh:88,146) with the correctly rounded
// power of bhm::pow_m02. Errors outside [1e-6, 1e6] give the limits, so the argument is clamped there
// and the seed comes from the hardware's FP32 base-2 units (3e-7 relative) instead of the FP64 log and
// exp: two plain Newton steps on x y^5 = 1 (3e-13, then rounding), then pow_m02's last step, whose
// residual is formed in double-double. One evaluation serves both outcomes of a step (a rejected
// step's factor is below 0.9): 46 operations for 100, and lanes that disagree share them.
__device__ __forceinline__ double step_factor(double err) {
    const double x = fmin(fmax(err, 1e-6), 1e6);
    const float l2 = __builtin_amdgcn_logf((float)x);
    double y = (double)__builtin_amdgcn_exp2f(-0.2f * l2);
    for (int i = 0; i < 2; ++i) {
        const double y2 = y * y;
        y = fma(y * 0.2, fma(-x, y2 * y2 * y, 1.0), y);
    }
    const double p2 = y * y, e2 = fma(y, y, -p2);
    const double p4 = p2 * p2, e4 = fma(2.0 * p2, e2, fma(p2, p2, -p4));
    const double p5 = p4 * y, e5 = fma(e4, y, fma(p4, y, -p5));
    const double p6 = p5 * x, e6 = fma(e5, x, fma(p5, x, -p6));
    const double r = (1.0 - p6) - e6;
    // the double nearest 0.2 is 2^-56 * 4/5 above it: x^-0.2 = x^(-1/5) (1 - that * ln x)
    const double off = (double)(l2 * (0x1.999999999999ap-57f * 0.6931471805599453f));
    return fmin(5.0, fmax(0.2, 0.9 * fma(y, fma(r, 0.2, -off), y)));
}
// blackholes/src/kerr.hpp:166-173
__device__ __forceinline__ void project_radial(const TraceParams& P, const RayConst& c, State& s) {
    double r = s.y0;
    double Pp = r * r + P.a2 - c.alam, D = r * r - 2.0 * r + P.a2;
    double R = Pp * Pp - D * c.K;
    if (R > 0.25 * r * r * r * r) {
        double v = bhm::sqrt_pos_(R);
        s.y1 = s.y1 < 0.0 ? -v : v;
    }
}

// blackholes/src/device_util.cuh:74-80
__device__ __forceinline__ float table_lerp(const float* __restrict__ t, int n, float x0, float dx, float x) {
    float f = (x - x0) / dx;
    f = fminf(fmaxf(f, 0.f), (float)(n - 2) + 0.9999f);
    int i = (int)f;
    f -= i;
    float t0 = t[i], t1 = t[i + 1];
    return t0 + (t1 - t0) * f;
}

// The same with 1 / dx (correctly rounded) at hand: the quotient by its residual, as bhm::quot_.
__device__ __forceinline__ float table_lerp(const float* __restrict__ t, int n, float x0, float dx, float inv_dx,
                                            float x) {
    const float a = x - x0, q = a * inv_dx;
    float f = fmaf(fmaf(-dx, q, a), inv_dx, q);
    f = fminf(fmaxf(f, 0.f), (float)(n - 2) + 0.9999f);
    int i = (int)f;
    f -= i;
    float t0 = t[i], t1 = t[i + 1];
    return t0 + (t1 - t0) * f;
}

// Trilinear density factor on the Cartesian grid (slice pointer g), same order as the oracle.
__device__ __forceinline__ double grid_trilinear(const TraceParams& P, const float* __restrict__ G, double px,
                                                 double py, double pz) {
    const int n = P.turb_n;
    double gx = (px + P.turb_half) * P.turb_inv_dx - 0.5;
    double gy = (py + P.turb_half) * P.turb_inv_dx - 0.5;
    double gz = (pz + P.turb_half) * P.turb_inv_dx - 0.5;
    const double hi = (double)(n - 1);
    gx = fmin(fmax(gx, 0.0), hi);
    gy = fmin(fmax(gy, 0.0), hi);
    gz = fmin(fmax(gz, 0.0), hi);
    int ix = (int)gx, iy = (int)gy, iz = (int)gz;
    ix = ix > n - 2 ? n - 2 : ix;
    iy = iy > n - 2 ? n - 2 : iy;
    iz = iz > n - 2 ? n - 2 : iz;
    double fx = gx - (double)ix, fy = gy - (double)iy, fz = gz - (double)iz;
    const size_t sy = (size_t)n, sz = (size_t)n * n;
    const float* b = G + ((size_t)iz * sz + (size_t)iy * sy + (size_t)ix);
    double v000 = b[0], v100 = b[1], v010 = b[sy], v110 = b[sy + 1];
    double v001 = b[sz], v101 = b[sz + 1], v011 = b[sz + sy], v111 = b[sz + sy + 1];
    double c00 = v000 + (v100 - v000) * fx;
    double c10 = v010 + (v110 - v010) * fx;
    double c01 = v001 + (v101 - v001) * fx;
    double c11 = v011 + (v111 - v011) * fx;
    double c0 = c00 + (c10 - c00) * fy;
    double c1 = c01 + (c11 - c01) * fy;
    return c0 + (c1 - c0) * fz;
}

__device__ __forceinline__ double turb_factor(const TraceParams& P, double r, double R, double u, double sp,
                                              double cp, double t) {
    double px = R * cp, py = R * sp, pz = r * u;
    if (P.turb_nt <= 1) return grid_trilinear(P, P.turb, px, py, pz);
    // time slices: linear in coordinate time, clamped to the first/last slice
    double st = (t - P.turb_t0) * P.turb_inv_dt;
    st = fmin(fmax(st, 0.0), (double)(P.turb_nt - 1));
    int k = (int)st;
    k = k > P.turb_nt - 2 ? P.turb_nt - 2 : k;
    double f = st - (double)k;
    const size_t slice = (size_t)P.turb_n * P.turb_n * P.turb_n;
    double A = grid_trilinear(P, P.turb + (size_t)k * slice, px, py, pz);
    double B = grid_trilinear(P, P.turb + (size_t)(k + 1) * slice, px, py, pz);
    return A + (B - A) * f;
}

// a / b for a constant b of the physics
__device__ __forceinline__ double quot_const(double a, double b, double inv_b) {
    return bhm::quot_(a, bhm::Recip{b, inv_b});
}

// blackholes/src/emission.cuh:99-175 (exact thermal-synchrotron coefficients). w = 1 - u^2, sn =
// sqrt(max(w, 0)) and the azimuth's sine and cosine are those of the swept angle: the flow and the
// turbulence lookup read the same values. Quotients whose operands a scene or a sample can make zero
// or infinite keep the IEEE fix-up; j / B_nu keeps the operator (j falls to the denormals).
template <int RADIO>
__device__ __forceinline__ void flow_step(const TraceParams& P, double r, double u, double w, double sn, double phi,
                                          double sv, double cv, double t, double lam, double Ecam, double h, double* dI,
                                          double* dtau) {
    using bhm::quot_;
    using bhm::quot_ieee_;
    using bhm::sqrt_pos_;
    *dI = 0.0;
    *dtau = 0.0;
    const double a = P.a;
    const double s2 = fmax(w, 1e-12), s = w >= 1e-12 ? sn : __builtin_sqrt(1e-12);
    double R = r * s, z = r * u;
    if (r > P.r_flow_max || R < 1e-3) return;
    double zh = quot_ieee_(z, P.h_r * R);
    double vert = bhm::exp(-0.5 * zh * zh);
    if (vert < 1e-7) return;
    double lr = bhm::log(r);
    double ne = P.n0 * bhm::exp(-P.n_index * lr) * vert;
    if (P.turb_on) {
        if constexpr (RADIO == RADIO_SHEARED) ne *= (double)sheared_factor(P, r, R, z, phi, t);
        else ne *= turb_factor(P, r, R, u, sv, cv, t);
    }
    ne *= 1.0 - bhm::exp(-(r - P.rh) * (r - P.rh) / 0.25);
    if (ne < 1e-30) return;
    double Th = P.theta0 * bhm::exp(-P.theta_index * lr);
    double B = sqrt_pos_(quot_ieee_(8.0 * PI * ne * C_MP * C_C * C_C, 6.0 * r * P.beta_p));
    double r2 = r * r, a2 = P.a2;
    double Sigma = r2 + a2 * u * u, Delta = r2 - 2.0 * r + a2;
    double A = (r2 + a2) * (r2 + a2) - a2 * Delta * s2;
    const bhm::Recip iS = bhm::recip_(Sigma), iA = bhm::recip_(A);
    double g_tt = -(1.0 - quot_(2.0 * r, iS)), g_tph = quot_(-2.0 * a * r * s2, iS), g_phph = quot_(A * s2, iS);
    double omz = quot_(2.0 * a * r, iA);
    double Rk = fmax(R, P.r_isco);
    double Om = P.flow_kep * quot_(1.0, Rk * sqrt_pos_(Rk) + a);
    double vmax = quot_(bhm::sqrt_nn_(quot_(Sigma * Delta, iA)), sqrt_pos_(g_phph)) * 0.999;
    Om = omz + fmax(-vmax, fmin(vmax, Om - omz));
    double norm = -(g_tt + 2.0 * g_tph * Om + g_phph * Om * Om);
    if (norm <= 0.0) return;
    double ut = quot_(1.0, sqrt_pos_(norm));
    double kdotu = ut * (1.0 - Om * lam);
    double nu_f = P.nu_obs * Ecam * kdotu;
    double g = quot_ieee_(P.nu_obs, nu_f);
    double u_ph = ut * (g_tph + g_phph * Om);
    double kb = lam - kdotu * u_ph;
    double bb = g_phph + u_ph * u_ph;
    double cosb = quot_ieee_(kb, kdotu * sqrt_pos_(bb));
    double sinb = sqrt_pos_(fmax(1.0 - cosb * cosb, 1e-6));
    constexpr double NUC = 2.0 * PI * C_ME * C_C, CC2 = C_C * C_C;
    double nuc = quot_const(C_QE * B, NUC, 1.0 / NUC);
    double nus = 2.0 / 9.0 * nuc * Th * Th * sinb;
    double X = quot_ieee_(nu_f, nus);
    double x3 = bhm::cbrt(X);
    double k2 = bhm::exp((double)table_lerp(P.k2, P.k2_n, P.k2_l0, P.k2_dl, P.k2_inv_dl, (float)bhm::log(Th)));
    double brk = bhm::sqrt_nn_(X) + 1.887748625363387 * bhm::sqrt_nn_(x3);
    double j = quot_ieee_(ne * 1.4142135623730951 * PI * C_QE * C_QE * nus, 3.0 * k2 * C_C) * brk * brk * bhm::exp(-x3);
    double Te = quot_const(Th * C_ME * C_C * C_C, C_KB, 1.0 / C_KB);
    double hnu = quot_ieee_(C_H * nu_f, C_KB * Te);
    double Bnu = quot_ieee_(quot_const(2.0 * C_H * nu_f * nu_f * nu_f, CC2, 1.0 / CC2), bhm::expm1(hnu));
    double alpha = j / Bnu;
    double dl = kdotu * Sigma * h * P.rg_cm;
    double tau = alpha * dl;
    *dtau = tau;
    *dI = g * g * g * Bnu * (-bhm::expm1(-tau));
}

// atan2(y, x) for y >= 0 and a vector of length about 1 (the angle between two directions): the
// operations of bhm::atan2 with one quotient for both octant orders
__device__ __forceinline__ double angle_pos(double y, double x) {
    const double ax = fabs(x);
    const bool steep = !(y <= ax);
    double a = bhm::atan_unit(bhm::quot_(steep ? ax : y, steep ? y : ax));
    a = steep ? bhm::PI_2 - a : a;
    return x < 0.0 ? bhm::PI_ - a : a;
}

// blackholes/src/kerr.hpp:63-92 (+ trace.cuh:64 direction): initial state and constants
__device__ __forceinline__ void camera_photon(const TraceParams& P, double x, double yv, RayConst& c, State& s) {
    double ox = P.cx + x, oy = P.cy + yv;
    double vx = P.F[0] + P.R[0] * ox + P.U[0] * oy;
    double vy = P.F[1] + P.R[1] * ox + P.U[1] * oy;
    double vz = P.F[2] + P.R[2] * ox + P.U[2] * oy;
    double inv = 1.0 / sqrt(vx * vx + vy * vy + vz * vz);
    double kx = -(vx * inv), ky = -(vy * inv), kz = -(vz * inv);
    double k0 = 1.0;
    double b2 = P.beta[0] * P.beta[0] + P.beta[1] * P.beta[1] + P.beta[2] * P.beta[2];
    if (b2 > 0.0) {
        double b = sqrt(b2), g = 1.0 / sqrt(1.0 - b2);
        double ib = 1.0 / b;
        double bx = P.beta[0] * ib, by = P.beta[1] * ib, bz = P.beta[2] * ib;
        double kpar = kx * bx + ky * by + kz * bz;
        double k0z = g * (k0 + b * kpar);
        double f = (g - 1.0) * kpar + g * b * k0;
        kx = kx + bx * f;
        ky = ky + by * f;
        kz = kz + bz * f;
        k0 = k0z;
    }
    const double kr = P.kp[0], ks = P.kp[1], kc = P.kp[2], omega = P.kp[6], e_nu = P.kp[7], e_psi = P.kp[8];
    double L = e_psi * kz;
    double E = e_nu * k0 + omega * L;
    double pth = P.kp[9] * ky;
    double Q = pth * pth + kc * kc * (L * L / (ks * ks) - P.a2 * E * E);
    c.lam = L / E;
    c.eta = Q / (E * E);
    c.E = E;
    c.K = c.eta + (c.lam - P.a) * (c.lam - P.a);
    c.lam2 = c.lam * c.lam;
    c.alam = P.a * c.lam;
    double dr = P.kp[10] * kx / E;
    double dth = pth / E;
    s.y0 = kr;
    s.y1 = -dr;
    s.y2 = kc;
    s.y3 = ks * dth;
    s.y4 = P.ph0;
    s.y5 = P.t0;
}

// blackholes/src/kerr.hpp:175-178
__device__ __forceinline__ double initial_step(const State& s) {
    return 0.02 * fmin(s.y0 / (fabs(s.y1) + 1e-12), 1.0 / (fabs(s.y3) + 1e-3));
}

// Per-ray integration state of trace_ray (trace.cuh:62-80), kept in registers between steps.
struct RayState {
    RayConst c;
    State s;
    double h, acc0, acc1, acc2, acc3, trans, psi;
    double sn, ppx, ppy;   // radio: sin theta of the state and its direction's x and y (z is u = s.y2)
    int ncross, accepted, flow_steps, it, fate;
    bool done;
};

// blackholes/src/trace.cuh:62-80: initial state of the ray through image-plane offset (x, yv)
template <int RADIO>
__device__ __forceinline__ void ray_init(const TraceParams& P, double x, double yv, RayState& R) {
    camera_photon(P, x, yv, R.c, R.s);
    {
        Rhs k = rhs<true>(P, R.c, R.s.y0, R.s.y2);
        R.s.k1 = k.d1; R.s.k3 = k.d3; R.s.k4 = k.d4; R.s.k5 = k.d5;
    }
    R.h = initial_step(R.s);
    R.acc0 = R.acc1 = R.acc2 = R.acc3 = 0.0;
    R.trans = 1.0;
    R.psi = 0.0;
    R.ncross = R.accepted = R.flow_steps = R.it = R.fate = 0;
    R.sn = R.ppx = R.ppy = 0.0;
    if (RADIO) {
        double sv, cv;
        R.sn = bhm::sqrt_nn_(fmax(1.0 - R.s.y2 * R.s.y2, 0.0));
        bhm::sincos(R.s.y4, &sv, &cv);
        R.ppx = R.sn * cv;
        R.ppy = R.sn * sv;
    }
    R.done = P.max_steps <= 0;
}

// One DP54 attempt from R (trace.cuh:81-97): n is the accepted state; false when the attempt is rejected.
// ray_step spells the same out: through this function the persistent kernels take 11 more registers, and the
// 1024^2 frame 21.2 ms for 20.0.
template <int RADIO, bool TIME>
__device__ __forceinline__ bool ray_attempt(const TraceParams& P, RayState& R, State& n, double& hc) {
    hc = R.h;
    if (RADIO && P.flow_on && R.s.y0 < P.r_flow_max) {
        double cap = P.step_frac * fmin(bhm::quot_(R.s.y0, fabs(R.s.y1) + 1e-30),
                                        bhm::quot_(fmax(R.sn, 0.05), fabs(R.s.y3) + 1e-30));
        hc = fmin(hc, cap);
    }
    const double err = dp54_step<TIME>(P, R.c, R.s, hc, n);
    ++R.it;
    R.h = hc * step_factor(err);
    if (!(err <= 1.0)) {
        if (R.it >= P.max_steps) R.done = true;
        return false;
    }
    ++R.accepted;
    return true;
}

// The accepted state becomes the ray's; sets R.done when the ray stops there (trace.cuh:146-163).
__device__ __forceinline__ void ray_settle(const TraceParams& P, RayState& R, const State& n) {
    R.s = n;
    project_radial(P, R.c, R.s);
    if (R.s.y0 < P.r_stop) {
        R.fate = -1;
        R.done = true;
        return;
    }
    if (R.s.y0 > P.r_escape && R.s.y1 > 0.0) {
        R.fate = 1;   // escape angles are taken from the final state in ray_result
        R.done = true;
        return;
    }
    if (R.it >= P.max_steps) R.done = true;
}

// Angle between the directions p (of z component ppz) and q of two consecutive accepted states.
__device__ __forceinline__ double ring_angle(double ppx, double ppy, double ppz, double pnx, double pny, double pnz) {
    double cx = ppy * pnz - ppz * pny, cy = ppz * pnx - ppx * pnz, cz = ppx * pny - ppy * pnx;
    double cl = bhm::sqrt_nn_(cx * cx + cy * cy + cz * cz);
    double dt = ppx * pnx + ppy * pny + ppz * pnz;
    return angle_pos(cl, dt);
}

// Adds a flow sample's emission dI and transmission e; true when the ray is opaque from here on.
template <class RayS>
__device__ __forceinline__ bool ray_absorb(RayS& R, int ord, double dI, double e) {
    double cI = R.trans * dI;
    R.acc0 += cI;
    // value selects, not a branch chain: the chain becomes a dynamically indexed stack array
    R.acc1 += ord == 1 ? cI : 0.0;
    R.acc2 += ord == 2 ? cI : 0.0;
    R.acc3 += ord >= 3 ? cI : 0.0;
    R.trans *= e;
    return R.trans < 1e-5;
}

// One iteration of trace.cuh:81-163 (one DP54 attempt); sets R.done when the ray stops.
// P is what every attempt reads, F the same frame for what only a sample of the flow reads.
template <int RADIO, bool TIME>
__device__ __forceinline__ void ray_step(const TraceParams& P, const TraceParams& F, RayState& R) {
    State n;
    double hc = R.h;
    if (RADIO && P.flow_on && R.s.y0 < P.r_flow_max) {
        double cap = P.step_frac * fmin(bhm::quot_(R.s.y0, fabs(R.s.y1) + 1e-30),
                                        bhm::quot_(fmax(R.sn, 0.05), fabs(R.s.y3) + 1e-30));
        hc = fmin(hc, cap);
    }
    const double err = dp54_step<TIME>(P, R.c, R.s, hc, n);
    ++R.it;
    R.h = hc * step_factor(err);
    if (!(err <= 1.0)) {
        if (R.it >= P.max_steps) R.done = true;
        return;
    }
    ++R.accepted;
    double w = 0.0, sv = 0.0, cv = 1.0;
    if (RADIO) {
        w = 1.0 - n.y2 * n.y2;
        const double sn = bhm::sqrt_nn_(fmax(w, 0.0));
        bhm::sincos(n.y4, &sv, &cv);
        const double pnx = sn * cv, pny = sn * sv;
        R.psi += ring_angle(R.ppx, R.ppy, R.s.y2, pnx, pny, n.y2);
        R.ppx = pnx;
        R.ppy = pny;
        R.sn = sn;
    }
    if ((R.s.y2 > 0.0) != (n.y2 > 0.0)) ++R.ncross;
    if (RADIO && P.flow_on && n.y0 < P.r_flow_max) {
        double dI, dtau;
        ++R.flow_steps;
        flow_step<RADIO>(F, n.y0, n.y2, w, R.sn, n.y4, sv, cv, n.y5, R.c.lam, R.c.E, hc, &dI, &dtau);
        if (ray_absorb(R, (int)(R.psi * (1.0 / PI)), dI, bhm::exp(-dtau))) {
            R.fate = -1;
            R.done = true;
            return;
        }
    }
    ray_settle(P, R, n);
}

// What an accepted step leaves for another wave to evaluate: the new state and its step, the direction
// before it, and whether the new state lies in the flow.
struct StepSample {
    double r, u, phi, t, h, u0, phi0;
    bool flow;
};

// The attempt of ray_step without the ring angle and the flow: true when a step was accepted. SETTLE false
// leaves the ray where it was, as ray_step does when the step's sample makes it opaque. R.ppx and R.ppy are
// not kept up.
template <int RADIO, bool TIME, bool SETTLE>
__device__ __forceinline__ bool ray_move(const TraceParams& P, RayState& R, StepSample& q) {
    State n;
    if (!ray_attempt<RADIO, TIME>(P, R, n, q.h)) return false;
    R.sn = bhm::sqrt_nn_(fmax(1.0 - n.y2 * n.y2, 0.0));
    if ((R.s.y2 > 0.0) != (n.y2 > 0.0)) ++R.ncross;
    q.r = n.y0;
    q.u = n.y2;
    q.phi = n.y4;
    q.t = n.y5;
    q.u0 = R.s.y2;
    q.phi0 = R.s.y4;
    q.flow = P.flow_on && n.y0 < P.r_flow_max;
    if (q.flow) ++R.flow_steps;
    if (SETTLE) ray_settle(P, R, n);
    return true;
}

// The direction of a state as ray_step carries it
struct Direction {
    double x, y, z;
};
__device__ __forceinline__ Direction direction_of(double u, double phi) {
    double sv, cv;
    const double sn = bhm::sqrt_nn_(fmax(1.0 - u * u, 0.0));
    bhm::sincos(phi, &sv, &cv);
    return Direction{sn * cv, sn * sv, u};
}

// The ring angle, emission and transmission of a sample left by ray_move, as ray_step forms them; d is the
// direction before the step, and after it on return.
template <int RADIO>
__device__ __forceinline__ void sample_eval(const TraceParams& F, double lam, double E, const StepSample& q, Direction& d,
                                            double* ang, double* dI, double* e) {
    double sv, cv;
    const double w = 1.0 - q.u * q.u, sn = bhm::sqrt_nn_(fmax(w, 0.0));
    bhm::sincos(q.phi, &sv, &cv);
    const Direction n{sn * cv, sn * sv, q.u};
    *ang = ring_angle(d.x, d.y, d.z, n.x, n.y, n.z);
    d = n;
    if (!q.flow) return;
    double dtau;
    flow_step<RADIO>(F, q.r, q.u, w, sn, q.phi, sv, cv, q.t, lam, E, q.h, dI, &dtau);
    *e = bhm::exp(-dtau);
}

// blackholes/src/trace.cuh:25-33: galactic texture coordinates of the escape direction (th, ph),
// the direction rotated by sky_rot (black-hole frame -> galactic) and taken to (longitude, latitude)
__device__ __forceinline__ void sky_uv(const TraceParams& P, double th, double ph, float* u, float* v) {
    double st, ct, sp, cp;
    bhm::sincos(th, &st, &ct);
    bhm::sincos(ph, &sp, &cp);
    const double dx = st * cp, dy = st * sp, dz = ct;
    const double gx = P.sky_rot[0] * dx + P.sky_rot[1] * dy + P.sky_rot[2] * dz;
    const double gy = P.sky_rot[3] * dx + P.sky_rot[4] * dy + P.sky_rot[5] * dz;
    const double gz = P.sky_rot[6] * dx + P.sky_rot[7] * dy + P.sky_rot[8] * dz;
    const double l = bhm::atan2(gy, gx), b = bhm::asin(fmax(-1.0, fmin(1.0, gz)));
    float uu = (float)(0.5 - l * (0.5 / PI));
    uu -= floorf(uu);
    *u = uu;
    *v = (float)(0.5 - b / PI);
}

// Radiance of the procedural sky at (u, v): sky_nu x sky_nv squares, bright sky_scale, dark 0.1 of it
// (the reference samples its star-map texture here, trace.cuh:35-45)
__device__ __forceinline__ float sky_checker(const TraceParams& P, float u, float v) {
    const int iu = min(max((int)(u * (float)P.sky_nu), 0), P.sky_nu - 1);
    const int iv = min(max((int)(v * (float)P.sky_nv), 0), P.sky_nv - 1);
    return ((iu + iv) & 1) ? P.sky_scale : 0.1f * P.sky_scale;
}

// Visible mode, escaped ray (trace.cuh:154-160): sky coordinates and, with the sky on, its radiance
// in the first three channels (the reference's X, Y, Z), weighted by the transmission
__device__ __forceinline__ void sky_result(const TraceParams& P, double trans, RayResult& out) {
    out.sky_u = 0.f;
    out.sky_v = 0.f;
    if (P.mode != MODE_VISIBLE || out.fate != 1) return;
    sky_uv(P, out.th_inf, out.ph_inf, &out.sky_u, &out.sky_v);
    if (P.sky_on) {
        const double s = (double)sky_checker(P, out.sky_u, out.sky_v);
        out.I[0] += trans * s;
        out.I[1] += trans * s;
        out.I[2] += trans * s;
    }
}

__device__ __forceinline__ void ray_result(const TraceParams& P, const RayState& R, RayResult& out) {
    out.y[0] = R.s.y0; out.y[1] = R.s.y1; out.y[2] = R.s.y2; out.y[3] = R.s.y3; out.y[4] = R.s.y4;
    out.y[5] = R.s.y5;
    out.th_inf = 0.0;
    out.ph_inf = 0.0;
    if (R.fate == 1) {
        // blackholes/src/trace.cuh:49-55 (k1[4] is the phi derivative of the final state)
        double sq = sqrt(fmax(1.0 - R.s.y2 * R.s.y2, 1e-30));
        double tq = bhm::acos(fmax(-1.0, fmin(1.0, R.s.y2)));
        double dthdr = (-R.s.y3 / sq) / R.s.y1, dphdr = R.s.k4 / R.s.y1;
        out.th_inf = tq + R.s.y0 * dthdr;
        out.ph_inf = R.s.y4 + R.s.y0 * dphdr;
    }
    out.I[0] = R.acc0; out.I[1] = R.acc1; out.I[2] = R.acc2; out.I[3] = R.acc3;
    out.trans = R.trans;
    out.psi = R.psi;
    out.fate = R.fate;
    out.ncross = R.ncross;
    out.order = (int)(R.psi * (1.0 / PI));
    out.steps = R.it;
    out.accepted = R.accepted;
    out.flow_steps = R.flow_steps;
    sky_result(P, R.trans, out);
}

// blackholes/src/trace.cuh:62-165 (disk branch out of scope, procedural sky), FP64 intensity.
template <int RADIO, bool TIME>
__device__ __forceinline__ void trace_ray_fp64(const TraceParams& P, double x, double yv, RayResult& out) {
    RayState R;
    ray_init<RADIO>(P, x, yv, R);
    while (!R.done) ray_step<RADIO, TIME>(P, P, R);
    ray_result(P, R, out);
}

// blackholes/src/kerr.hpp:184-203 for one photon (lam, eta, E, y[6])
__device__ __forceinline__ int vacuum_fate(const TraceParams& P, const double* ph, double tol, double r_escape,
                                           int max_steps) {
    RayConst c;
    c.lam = ph[0];
    c.eta = ph[1];
    c.E = ph[2];
    c.K = c.eta + (c.lam - P.a) * (c.lam - P.a);
    c.lam2 = c.lam * c.lam;
    c.alam = P.a * c.lam;
    State s, n;
    s.y0 = ph[3]; s.y1 = ph[4]; s.y2 = ph[5]; s.y3 = ph[6]; s.y4 = ph[7]; s.y5 = ph[8];
    Rhs k = rhs<false>(P, c, s.y0, s.y2);   // the fate reads no coordinate time
    s.k1 = k.d1; s.k3 = k.d3; s.k4 = k.d4; s.k5 = k.d5;
    double h = initial_step(s);
    const double rcap = P.rh * 1.0001 + 1e-3;
    for (int it = 0; it < max_steps; ++it) {
        const double err = dp54_step<false>(P, c, s, h, n);
        h *= step_factor(err);
        if (err > 1.0) continue;
        s = n;
        project_radial(P, c, s);
        if (s.y0 < rcap) return -1;
        if (s.y0 > r_escape && s.y1 > 0.0) return 1;
    }
    return 0;
}

}  // namespace bhd

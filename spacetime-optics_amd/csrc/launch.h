/* launch.h - the shape of a persistent launch: kernel, workgroups, queue order (host code, no device types).
   Every rule is a function of the load below; the figures beside them are MI355X times of the launch in ms. */
#pragma once
#include <cmath>

#include "../../include/bhrt.h"

namespace launch {

struct Load {
    int precision = BH_PREC_FP64;
    int radio = 0;          // the tracer's flow variant (0: vacuum)
    double w = 0.0;         // waves of rays per compute unit (a CU holds 12 waves of these kernels, 3 per SIMD)
    double reach = 0.0;     // mixed radio: of them, those whose rays reach the emitting region
    bool opaque = false;    // mixed radio: the flow is opaque as far out as the longest rays circle
};

// Share of the region's rays (x0, y0, w, h of a W x H frame, pixel angle pix, image centre off by cx, cy) that
// pass within r of the hole, from 16 x 16 of them; r_cam is the camera's distance.
inline double share_within(double r, double r_cam, double cx, double cy, double pix, int W, int H, int x0, int y0, int w,
                           int h) {
    constexpr int N = 16;
    int in = 0;
    for (int j = 0; j < N; ++j)
        for (int i = 0; i < N; ++i) {
            const double x = cx + (x0 + (i + 0.5) / N * w - 0.5 * W) * pix;
            const double y = cy + (0.5 * H - (y0 + (j + 0.5) / N * h)) * pix;
            in += std::sqrt(x * x + y * y) * r_cam <= r;
        }
    return (double)in / (N * N);
}

/* Whether a radio launch takes two waves per 64 rays (k_pair, 4 workgroups per CU). It halves the chain of
   the longest rays, but the two waves wait for each other, so it does less work per time: it pays until the
   launch's work, not its longest ray, sets its end. One wave per 64 rays (8 waves per CU) -> two:
   - FP64 (every ray samples the whole flow): 64^2 3.9 -> 2.9, 256^2 5.6 -> 4.4, 352^2 (w = 7.6) 5.2 -> 4.7, 384^2
     (9) 4.8 -> 4.1 to 4.9 -> 5.2 by field, 408^2 (10.2) 5.1 -> 5.6; thicker flows cross between 7 and 10.
   - Mixed: the work is in the rays that reach the emitting region. 40 M wide, the 0.6 Jy flow: 384^2 1.82 ->
     1.37, 640^2 (w = 25, reach 11) 1.91 -> 1.43, 808^2 (40, 17) 2.10 -> 2.05; with the full flow (reach = w)
     512^2 2.12 -> 1.66, 608^2 (22.6) 2.08 -> 1.80, 640^2 (25) 1.81 -> 1.97, 768^2 (36) 2.18 -> 2.79.
   - An opaque flow ends the longest rays early, and the work sets the end sooner: 30 times the density, 24 M
     wide, 384^2 (9) 1.36 -> 1.36, 448^2 (12.2) 1.48 -> 1.66, 640^2 (25) 2.44 -> 3.05; 100 times, 60 M wide, 448^2
     1.04 -> 0.94, 512^2 (16) 1.10 -> 1.18. */
constexpr double PAIR_W_FP64 = 10.0, PAIR_W_MIXED = 40.0, PAIR_REACH = 24.0, PAIR_REACH_OPAQUE = 12.0;

inline bool pairs(const Load& l) {
    if (l.radio == 0) return false;
    if (l.precision == BH_PREC_FP64) return l.w <= PAIR_W_FP64;
    return l.w <= PAIR_W_MIXED && l.reach <= (l.opaque ? PAIR_REACH_OPAQUE : PAIR_REACH);
}

}  // namespace launch

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

constexpr int PAIR_RAYS = 64, PAIR_PER_CU = 4;   // the shape of such a launch: rays of a workgroup, workgroups of a CU

// Whether a resolved configuration asks for it where the load does: by its shape (interval, refill_min and order
// hold for both kernels, prio_age for the other one only)
inline bool pair_shape(const bh_batch_cfg& g) { return g.block == PAIR_RAYS && g.grid_per_cu == PAIR_PER_CU && g.waves == 3; }

/* Defaults. Measured on frames of 32^2 to 2048^2:
   - A SIMD issues one wave's instructions at half its rate, so 2 waves fill it and a third covers the
     stalls; but the longest rays set the end of a launch, and each of their instructions waits for the
     SIMD's other waves. Few rays are therefore spread thinly - and evenly: the waves that find no ray
     exit, and with 3 resident waves per SIMD which SIMD they leave idle is chance. FP64 vacuum, at most one
     wave per SIMD to w = 7 (16 M wide, 8 -> 4 waves per CU: 272^2 (w = 4.5) 2.4 -> 1.9, 336^2 (6.9) 2.6 -> 2.4;
     360^2 (7.9) and 448^2 (12) within 5 % either way); 512^2 radio, FP64: 8.7 with 12, 6.0 with 8; 1024^2: 18.3
     with 12. Mixed radio: 1400^2 4.82 with 8, 4.17 with 12; zoom 768^2: 13.5 with 8, 11.9 with 12 (every ray
     is long: throughput, from 8 waves of rays per CU on).
   - Longest rays first (critical order) where several generations of rays share the launch, but not so
     many that its tail no longer counts: FP64 vacuum 280^2 (w = 4.8, 3 waves per CU in rows -> 4, sorted) 2.8 ->
     2.1 at 16 M wide, 2.7 -> 2.0 at 30 M, 2.1 -> 1.8 at 40 M; radio 280^2 (two waves per 64 rays) 4.7 -> 4.3, 384^2
     6.0 -> 4.8, 768^2 11.3 -> 11.1, 1024^2 18.3 -> 18.9, 1500^2 37.6 -> 39.9. Up to w = 4 at most a quarter of the
     rays waits for a place, short ones finish soon enough for them in most fields, and rows with 3 waves per CU
     are ahead: 256^2 records 40 M wide, 3 rows / 3 sorted / 4 rows / 4 sorted: 3.20 / 3.28 / 3.40 / 3.41, 240^2 2.53 /
     2.39 / 2.49 / 2.49, 224 x 288 2.69 / 2.73 / 2.79 / 2.88 (16 M wide, where most rays are long, 256^2 2.6 / 2.0 /
     2.0 / 2.0). The mixed tracer's rays differ by over 10x in length: always.
   - Workgroups of one wave where they are few, so that the dispatcher can place each on its own. */
inline bh_batch_cfg defaults(const Load& l) {
    bh_batch_cfg d{};
    const bool mixed = l.precision == BH_PREC_MIXED;
    d.use_graph = 1;
    d.waves = 3;
    d.interval = 64;
    d.refill_min = mixed ? 32 : 48;
    d.prio_age = mixed ? 128 : 256;
    d.order = mixed || (l.w > 4.0 && l.w <= 48.0) ? BH_ORDER_CRITICAL : BH_ORDER_ROWS;
    if (pairs(l)) {
        d.block = PAIR_RAYS;
        d.grid_per_cu = PAIR_PER_CU;
    } else if (mixed) {
        d.block = 256;
        d.grid_per_cu = l.radio == 0 ? (l.w <= 8.0 ? 1 : 3) : (l.w <= 48.0 ? 2 : 3);
    } else {
        d.block = l.w <= 20.0 ? 64 : 256;
        d.grid_per_cu = l.w <= 4.0 ? 3 : (l.w <= 7.0 ? 4 : (l.w <= 20.0 ? 8 : 3));
    }
    return d;
}

/* A tuned configuration stands in for the defaults it was tuned from, and for no others: what is best for 1024^2
   rays is not for 64^2 (FP64, tuned at 64^2, then 1024^2: 36.1 for 19.7; mixed, the other way round: 1.35 for
   1.02). */
struct Tuned {
    bool ok = false;
    int radio = 0;
    bh_batch_cfg from{}, cfg{};
};

inline const bh_batch_cfg& choose(const Tuned& t, const Load& l, const bh_batch_cfg& dflt) {
    const bh_batch_cfg &a = t.from, &b = dflt;
    const bool same = t.ok && (t.radio != 0) == (l.radio != 0) && a.block == b.block && a.grid_per_cu == b.grid_per_cu &&
                      a.interval == b.interval && a.refill_min == b.refill_min && a.waves == b.waves &&
                      a.order == b.order && a.prio_age == b.prio_age;
    return same ? t.cfg : dflt;
}

}  // namespace launch

/* Answers the lines of standard input, one each:
   - "precision radio w reach opaque": launch::pairs
   - "share r r_cam cx cy pix W H x0 y0 w h": launch::share_within
   - "defaults precision radio w reach opaque": block grid_per_cu order, and whether the launch is paired
   - "tuned <load> <load> block grid_per_cu interval": a tuning for the first load that found these; the second
     load's block grid_per_cu interval, and whether it is paired */
#include <cstdio>
#include <cstring>

#include "../../spacetime-optics_amd/csrc/launch.h"

static bool load(const char* s, launch::Load* l, int* used) {
    int opaque;
    if (std::sscanf(s, "%d %d %lf %lf %d%n", &l->precision, &l->radio, &l->w, &l->reach, &opaque, used) != 5) return false;
    l->opaque = opaque != 0;
    return true;
}

static int paired(const launch::Load& l, const bh_batch_cfg& g) { return launch::pairs(l) && launch::pair_shape(g); }

int main() {
    char line[256];
    while (std::fgets(line, sizeof line, stdin)) {
        double r, rc, cx, cy, pix;
        int W, H, x0, y0, w, h, used, used2;
        launch::Load l, l2;
        if (std::sscanf(line, "share %lf %lf %lf %lf %lf %d %d %d %d %d %d", &r, &rc, &cx, &cy, &pix, &W, &H, &x0, &y0, &w,
                        &h) == 11)
            std::printf("%.17g\n", launch::share_within(r, rc, cx, cy, pix, W, H, x0, y0, w, h));
        else if (std::strncmp(line, "defaults ", 9) == 0 && load(line + 9, &l, &used)) {
            const bh_batch_cfg d = launch::defaults(l);
            std::printf("%d %d %d %d\n", d.block, d.grid_per_cu, d.order, paired(l, d));
        } else if (std::strncmp(line, "tuned ", 6) == 0 && load(line + 6, &l, &used) && load(line + 6 + used, &l2, &used2)) {
            launch::Tuned t{true, l.radio, launch::defaults(l), launch::defaults(l)};
            std::sscanf(line + 6 + used + used2, "%d %d %d", &t.cfg.block, &t.cfg.grid_per_cu, &t.cfg.interval);
            const bh_batch_cfg g = launch::choose(t, l2, launch::defaults(l2));
            std::printf("%d %d %d %d\n", g.block, g.grid_per_cu, g.interval, paired(l2, g));
        } else if (load(line, &l, &used))
            std::printf("%d\n", (int)launch::pairs(l));
    }
}

/* Prints launch::pairs for lines "precision radio w reach opaque" and launch::share_within for lines
   "share r r_cam cx cy pix W H x0 y0 w h" of standard input. */
#include <cstdio>
#include <cstring>

#include "../../spacetime-optics_amd/csrc/launch.h"

int main() {
    char line[256];
    while (std::fgets(line, sizeof line, stdin)) {
        double r, rc, cx, cy, pix;
        int W, H, x0, y0, w, h, opaque;
        launch::Load l;
        if (std::sscanf(line, "share %lf %lf %lf %lf %lf %d %d %d %d %d %d", &r, &rc, &cx, &cy, &pix, &W, &H, &x0, &y0, &w,
                        &h) == 11)
            std::printf("%.17g\n", launch::share_within(r, rc, cx, cy, pix, W, H, x0, y0, w, h));
        else if (std::sscanf(line, "%d %d %lf %lf %d", &l.precision, &l.radio, &l.w, &l.reach, &opaque) == 5) {
            l.opaque = opaque != 0;
            std::printf("%d\n", (int)launch::pairs(l));
        }
    }
}

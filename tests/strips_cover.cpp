// The start net's strips (csrc/trl_strips.h) on the CPU: for each "nimg h w"
// on the command line prints the weight-gradient strips' pixels that are not
// covered exactly once, the most pixels and rows any wave has, the pixels that
// the convolutions' strips of 8, 4 and 2 rows do not cover exactly once, their
// neighbours that are not the image's, and the convolutions' waves of 8 rows.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

#define __host__
#define __device__

#include "trl_strips.h"

int main(int argc, char **argv)
{
    for (int a = 1; a + 2 < argc; a += 3) {
        Geo g = geo_of(std::atoi(argv[a]), std::atoi(argv[a + 1]), std::atoi(argv[a + 2]), kRows);
        std::vector<int> seen(g.np, 0);
        const long nt = dw_tasks(g);
        const long nw = std::min<long>(kDwBlocks, (nt + 3) / 4) * 4;
        long most = 0, rows = 0;
        for (long w = 0; w < nw; ++w) {
            long px = 0, rw = 0;
            for (long t = w; t < nt; t += nw) {
                const DwStrip s = dw_strip(g, t);
                if (s.x1 - s.x0 > kDwW || s.x1 > g.w || s.y1 > g.h) std::abort();
                for (int y = s.y0; y < s.y1; ++y)
                    for (int x = s.x0; x < s.x1; ++x, ++px) ++seen[s.base + (long)y * g.w + x];
                rw += s.y1 - s.y0;
            }
            most = std::max(most, px);
            rows = std::max(rows, rw);
        }
        long bad = 0;
        for (int c : seen) bad += c != 1;
        long cbad = 0, nbad = 0, waves = 0;
        for (int r = kRows; r >= 2; r /= 2) {
            g = geo_of(g.nimg, g.h, g.w, r);
            if (r == kRows) waves = g.tasks;
            std::fill(seen.begin(), seen.end(), 0);
            Strip s;
            for (long t = 0; t < g.tasks; ++t)
                for (int lane = 0; lane < kStrip; ++lane) {
                    if (!strip_of(g, t, lane, s)) std::abort();
                    const long hw = (long)g.h * g.w, img = (s.base + s.x) / hw, x = (s.base + s.x) % hw;
                    nbad += s.base % hw != 0 || s.base < 0 || img >= g.nimg || x >= g.w || s.y1 > g.h;
                    for (int d = 0; d < 3; ++d) nbad += s.base + s.xc[d] != img * hw + (x + d - 1 + g.w) % g.w;
                    if (s.ok)
                        for (int y = s.y0; y < s.y1; ++y) ++seen[s.base + (long)y * g.w + s.x];
                }
            if (strip_of(g, g.tasks, 0, s)) std::abort();
            for (int c : seen) cbad += c != 1;
        }
        std::printf("%ld %ld %ld %ld %ld %ld\n", bad, most, rows, cbad, nbad, waves);
    }
    return 0;
}

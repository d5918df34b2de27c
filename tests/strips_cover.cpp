// The start net's strips (csrc/trl_strips.h) on the CPU: for each "nimg h w"
// on the command line prints the weight-gradient strips' pixels that are not
// covered exactly once, and the most pixels and the rows any wave has.
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
        Geo g{std::atoi(argv[a]), std::atoi(argv[a + 1]), std::atoi(argv[a + 2]), 0, 0, 0};
        g.np = (long)g.nimg * g.h * g.w;
        g.dwr = dw_rows(g.nimg, g.h, g.w);
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
        std::printf("%ld %ld %ld\n", bad, most, rows);
    }
    return 0;
}

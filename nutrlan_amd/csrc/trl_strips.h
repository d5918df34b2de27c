// trl_strips.h -- how the start net's kernels divide images among waves
// (included by trlnet.hip; a CPU test includes it too).
#ifndef TRL_STRIPS_H
#define TRL_STRIPS_H

struct Geo {
    int nimg, h, w;
    long np;   // pixels
    int rows;  // rows a wave of a convolution walks (conv_rows)
    int dwr;   // rows of a weight-gradient strip (dw_rows)
};

// Weight gradients: strips of at most kDwW columns, equally wide, and dwr <=
// kDwRows rows, dealt to the waves of at most kDwBlocks blocks in turn.
constexpr int kDwW = 32, kDwRows = 8;
constexpr int kDwBlocks = 256, kDwWaves = 4 * kDwBlocks;

__host__ __device__ inline int dw_strips(int w) { return (w + kDwW - 1) / kDwW; }
__host__ __device__ inline int dw_width(int w) { return (w + dw_strips(w) - 1) / dw_strips(w); }
__host__ __device__ inline int dw_segs(int h, int dwr) { return (h + dwr - 1) / dwr; }
__host__ __device__ inline long dw_tasks(const Geo &g)
{
    return (long)g.nimg * dw_strips(g.w) * dw_segs(g.h, g.dwr);
}

// Strip height.  A strip of r rows loads r + 2 rows of inputs, but a wave's
// FP32 sums are to run over no more pixels than an even split gives them (32
// up to 1,024 strips of one row), but for an eighth: of the heights that keep
// to that, the one with the fewest rows to load for the busiest wave.  Forward
// and backward of 1, 8 and 32 images of 64 x 64 with 8-row strips throughout:
// 211, 200 and 256 us, so 174, 171 and 240 (more waves).
__host__ __device__ inline long dw_wave_strips(int nimg, int h, int w, int r)
{
    return ((long)nimg * dw_strips(w) * dw_segs(h, r) + kDwWaves - 1) / kDwWaves;
}
inline int dw_rows(int nimg, int h, int w)
{
    const long even = dw_wave_strips(nimg, h, w, 1);
    int best = 1;
    long least = 3 * even;
    for (int r = 2; r <= kDwRows && r <= h; ++r) {
        const long n = dw_wave_strips(nimg, h, w, r);
        if (n * r <= even + even / 8 && n * (r + 2) < least) {
            least = n * (r + 2);
            best = r;
        }
    }
    return best;
}

struct DwStrip {
    long base;           // its image's first pixel
    int x0, x1, y0, y1;  // columns [x0, x1), rows [y0, y1)
};

__host__ __device__ inline DwStrip dw_strip(const Geo &g, long task)
{
    const int ns = dw_strips(g.w), sw = dw_width(g.w), per = ns * dw_segs(g.h, g.dwr);
    const int img = (int)(task / per), r = (int)(task - (long)img * per);
    const int seg = r / ns;
    DwStrip s;
    s.base = (long)img * g.h * g.w;
    s.x0 = (r - seg * ns) * sw;
    s.x1 = s.x0 + sw < g.w ? s.x0 + sw : g.w;
    s.y0 = seg * g.dwr;
    s.y1 = s.y0 + g.dwr < g.h ? s.y0 + g.dwr : g.h;
    return s;
}

#endif

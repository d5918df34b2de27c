// trl_strips.h -- how the start net's kernels divide images among waves
// (included by trlnet.hip; a CPU test includes it too).
#ifndef TRL_STRIPS_H
#define TRL_STRIPS_H

struct Geo {
    int nimg, h, w;
    long np;   // pixels
    // a convolution's wave: the rows it walks (conv_rows), the images side by
    // side (strip_images); strips across, waves for these images, all waves.
    // Formed on the host: divisions in the kernels' first microsecond show at
    // a few images
    int rows, ni, ns, per;
    long tasks;
    unsigned recip;  // a lane's image is lane * recip >> 16
    int dwr;   // rows of a weight-gradient strip (dw_rows)
};

// Convolutions: a wave takes strips of kStrip columns of an image, or, where
// an image has at most half as many, of as many images side by side as fit,
// and walks down up to kRows rows of them.  With one 3 x 3 image to a strip 13
// of 16 lanes have no pixel: the forward pass of 20,000 such images, host to
// host, took 218 us (174 with 16 consecutive pixels to a wave), now 140; 64
// images of 400 x 3 107 (95), now 90.
constexpr int kStrip = 16, kRows = 8;

__host__ __device__ inline int strips_of(int w) { return (w + kStrip - 1) / kStrip; }
__host__ __device__ inline int segs_of(int h, int rows) { return (h + rows - 1) / rows; }
inline int strip_images(int h, int w)
{
    return 2 * w <= kStrip && h <= 65536 ? kStrip / w : 1;  // the images' offset is an int
}
inline long conv_tasks(int nimg, int h, int w, int rows)
{
    const int ni = strip_images(h, w);
    return (long)((nimg + ni - 1) / ni) * strips_of(w) * segs_of(h, rows);
}

// task / per, in 32 bits where it fits.
__host__ __device__ inline int group_of_task(long task, int per)
{
    return task <= 0x7fffffffL ? (int)task / per : (int)(task / per);
}

// A lane's part of a wave's strip: pixel (y, its column) is base + y w + x,
// its neighbours' columns (periodic) are xc.  Its image's offset from the
// wave's first is part of x and xc, so that base stays the wave's.
struct Strip {
    long base;
    int x, xc[3], y0, y1;  // rows [y0, y1)
    bool ok;               // it has a pixel (others repeat one)
};

__host__ __device__ inline bool strip_of(const Geo &g, long task, int lane, Strip &s)
{
    if (task >= g.tasks) return false;
    const int ns = g.ns, ni = g.ni;
    const int grp = group_of_task(task, g.per), r = (int)(task - (long)grp * g.per);
    const int seg = r / ns, strip = r - seg * ns;
    int x = strip * kStrip + lane, off = 0;
    s.ok = x < g.w;
    if (ni > 1) {
        const int i = (int)(lane * g.recip >> 16), last = g.nimg - 1 - grp * ni;
        x = lane - i * g.w;
        s.ok = i < ni && i <= last;
        off = (i < last ? i : last) * g.h * g.w;
    }
    x = x < g.w ? x : g.w - 1;
    s.x = off + x;
    s.xc[0] = off + (x == 0 ? g.w - 1 : x - 1);
    s.xc[1] = s.x;
    s.xc[2] = off + (x == g.w - 1 ? 0 : x + 1);
    s.base = (long)grp * ni * g.h * g.w;
    s.y0 = seg * g.rows;
    s.y1 = s.y0 + g.rows < g.h ? s.y0 + g.rows : g.h;
    return true;
}

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
// up to 1,024 strips of one row), but for a quarter: of the heights that keep
// to that, the one with the fewest rows to load for the busiest wave.  Forward
// and backward of 1, 8 and 32 images of 64 x 64 with 8-row strips throughout:
// 211, 200 and 256 us, so 175, 168 and 236 (more waves).
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
        if (n * r <= even + even / 4 && n * (r + 2) < least) {
            least = n * (r + 2);
            best = r;
        }
    }
    return best;
}

inline Geo geo_of(int nimg, int h, int w, int rows)
{
    const int ns = strips_of(w);
    return Geo{nimg, h, w, (long)nimg * h * w, rows, strip_images(h, w), ns, ns * segs_of(h, rows),
               conv_tasks(nimg, h, w, rows), 65536u / (unsigned)w + 1u, dw_rows(nimg, h, w)};
}

struct DwStrip {
    long base;           // its image's first pixel
    int x0, x1, y0, y1;  // columns [x0, x1), rows [y0, y1)
};

__host__ __device__ inline DwStrip dw_strip(const Geo &g, long task)
{
    const int ns = dw_strips(g.w), sw = dw_width(g.w), per = ns * dw_segs(g.h, g.dwr);
    const int img = group_of_task(task, per), r = (int)(task - (long)img * per);
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

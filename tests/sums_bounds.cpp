// The wide update's column sums (csrc/trl_sums.h) on the CPU, every load
// checked against the columns a caller owns: m columns of leading dimension
// ld whose last one ends at row n.  Prints the loads out of range and the
// sums that differ from a plain loop in the same order.  With an argument the
// rows are read as whole quads, which must be seen to leave the range.
#include <cstdio>
#include <vector>

#define __device__
#define __forceinline__ inline

static const char *lo, *hi;
static long out_of_range;

template <typename VS>
static double ld1(const VS *p)
{
    const char *c = reinterpret_cast<const char *>(p);
    if (c < lo || c + sizeof(VS) > hi) {
        ++out_of_range;
        return 0.0;
    }
    return (double)*p;
}
template <typename VS>
static void ld4(const VS *p, double v[4])
{
    for (int j = 0; j < 4; ++j) v[j] = ld1(p + j);
}
template <typename VS>
static void ld4u(const VS *p, double v[4])
{
    ld4(p, v);
}

#include "trl_sums.h"

template <typename VS>
static long run(bool whole)
{
    long wrong = 0;
    for (int n = 1; n <= 13; ++n)
        for (int m : {1, 3, 7, 8, 9, 15, 16, 17, 24, 31, 40})
            for (long ld = (n + 3) & ~3; ld <= ((n + 3) & ~3) + 4; ld += 4) {
                std::vector<VS> V((size_t)(m - 1) * ld + n);
                std::vector<double> h(m);
                for (size_t i = 0; i < V.size(); ++i) V[i] = (VS)((double)((i * 37) % 101) / 101 - 0.5);
                for (int i = 0; i < m; ++i) h[i] = (double)((i * 13) % 29) / 29 - 0.4;
                lo = reinterpret_cast<const char *>(V.data());
                hi = lo + V.size() * sizeof(VS);
                for (int row = 0; row < n; row += 4)
                    for (int k = 0; k < 4; ++k) {
                        double s[4];
                        if (whole)
                            group_sums(V.data() + row, ld, m, h.data(), k, s);
                        else
                            quad_sums(n, row, V.data(), ld, m, h.data(), k, s);
                        for (int j = 0; j < 4 && row + j < n; ++j) {
                            double t = 0.0;
                            for (int c = 0; c < m; ++c)
                                if (c < (m & ~7) ? c % 4 == k : k == 0) t += (double)V[c * ld + row + j] * h[c];
                            wrong += t != s[j];
                        }
                    }
            }
    return wrong;
}

int main(int argc, char **)
{
    const long wrong = run<float>(argc > 1) + run<double>(argc > 1);
    std::printf("%ld %ld\n", out_of_range, wrong);
    return 0;
}

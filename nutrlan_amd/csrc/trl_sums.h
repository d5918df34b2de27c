// trl_sums.h -- the wide update's sums over basis columns (included by
// trlhip.hip, which defines the loads ld4, ld4u and ld1).
//
// A column group k takes the columns of one running sum of update_rows4: c
// mod 4 = k within the full groups of 8, the columns after them all to group
// 0, so its sums are update_rows4's bit for bit.
#ifndef TRL_SUMS_H
#define TRL_SUMS_H

#include <cstddef>

// Column group k's running sums over columns [0, m) for four rows (Vc: the
// first row in column 0).  With ZERO the sums start at 0; else they go on
// from column c, the first one not in s yet (a multiple of 16; past the full
// groups only the tail is left).  LD: whole quads, aligned (ld4) or at any
// row (ld4u), or only the first nr rows (ld1).
enum { LD_QUAD, LD_ANY, LD_ROWS };
template <typename VS, bool ZERO = true, int LD = LD_QUAD>
__device__ __forceinline__ void group_sums(const VS *Vc, long ld, int m, const double *hs, int k, double s[4],
                                           int c = 0, int nr = 4)
{
    auto rows = [&](int col, double v[4]) {
        const VS *p = Vc + (size_t)col * ld;
        if constexpr (LD == LD_ROWS) {
            for (int j = 0; j < 4; ++j) v[j] = j < nr ? ld1(p + j) : 0.0;
        } else if constexpr (LD == LD_ANY) {
            ld4u(p, v);
        } else {
            ld4(p, v);
        }
    };
    if (ZERO) s[0] = s[1] = s[2] = s[3] = 0.0;
    const int full = m & ~7;
    for (; c + 16 <= full; c += 16) {
        double v[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i) rows(c + 4 * i + k, v[i]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] += v[i][j] * hs[c + 4 * i + k];
    }
    for (; c < full; c += 8) {
        double v[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i) rows(c + 4 * i + k, v[i]);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] += v[i][j] * hs[c + 4 * i + k];
    }
    if (k == 0) {
        for (c = ZERO ? c : full; c < m; ++c) {
            double v[4];
            rows(c, v);
#pragma unroll
            for (int j = 0; j < 4; ++j) s[j] += v[j] * hs[c];
        }
    }
}

// The same for rows [row, row + 4) of a basis of n rows: no row past n is
// read, as a caller's last column may end there (its columns are only known
// to be 16-byte aligned, so even the second half of an FP64 quad may lie in
// memory that is not the caller's).  The thread of a ragged end reads the
// last four rows with everyone else's loads and keeps the sums of its own:
// reading them row by row, after the others, costs 1 us of the 39 a pass of
// 28,561 rows takes.
template <typename VS>
__device__ __forceinline__ void quad_sums(int n, int row, const VS *V, long ld, int m, const double *hs, int k,
                                          double s[4])
{
    if (n < 4) {
        group_sums<VS, true, LD_ROWS>(V + row, ld, m, hs, k, s, 0, n - row);
        return;
    }
    const int q = row + 3 < n ? row : n - 4;
    group_sums<VS, true, LD_ANY>(V + q, ld, m, hs, k, s);
    const int d = row - q;
    if (d) {
        s[0] = d == 1 ? s[1] : d == 2 ? s[2] : s[3];
        s[1] = d == 1 ? s[2] : s[3];
        s[2] = s[3];
    }
}

#endif

// trl_chain.h -- a chain of Lanczos steps of one real solve in one kernel
// (included by trlhip.hip after the single-step kernels it agrees with).
//
// What bounds a small solve (n up to some 10^5 rows): a step is five short
// kernels and a round trip to the host, about 40 us at n = 10^4, of which
// the memory traffic is under 2 us.  Here the rows stay with their
// workgroups for a whole chain of steps: workgroup b owns rows [R b, R b +
// R), R = 256 RW, and the step's three reductions (alpha, h = V^T r, the two
// norms) cross workgroups through global partials and a flag barrier
// (1.4-2.4 us at up to 64 workgroups on eight XCDs, measured) instead of
// kernel boundaries.  After each step every workgroup makes the solver's
// decision for it (chain_go) from the same sums, so the next step starts
// without the host.
//
// Every sum is formed in the order of the single-step kernels (256-row alpha
// partials, 1024-row partials of the projection and the norms, the four
// interleaved column sums of update_rows4), so results are theirs bit for
// bit.  A wave holds 256 rows (4 consecutive rows a lane); the four column
// groups of waves split the columns of the update by c mod 4 -- its four
// running sums -- and the projection's columns in chunks.  With RW < 4 a
// workgroup covers only RW of the four waves whose totals make up a 1024-row
// partial, so the partials cross workgroups as wave totals and the reader
// adds the four in order.
//
// Lanes load four rows at once up to the padding of a context's columns (ld
// is n rounded up to 64; the padding holds zeros).
//
// Visibility: what another workgroup reads (partials, the new vector's rows,
// y of a CSR operator) is stored and loaded with agent-scope atomics, which
// go to the device's point of coherence; before a workgroup raises its flag
// all of its waves have waited for their stores (chain_barrier).  Basis
// columns are read and written by their owner only.  The CSR kinds gather the
// new vector with ordinary loads after an agent-scope acquire.
//
// Termination: a chain's workgroups first meet at a gate (chain_gate).
// Either all of them are running and the chain starts, or -- the device is
// filled by other work -- the gate closes after a while, nothing has been
// written and the host runs the step's ordinary kernels (chain_shut).  Past
// the gate every workgroup is resident, so each barrier ends; its wait is
// bounded all the same.
#ifndef TRL_CHAIN_H
#define TRL_CHAIN_H

// ticks of 10 ns: a single solve gives up soon, a batch's chains also wait for each other
constexpr unsigned long long kGateTicks = 200000, kBatchGateTicks = 20000000;  // 2 ms, 200 ms
constexpr unsigned long long kBarrierTicks = 6000000000ull;  // 60 s

struct ChainArgs {
    int n, g, steps, first, qa, qb, rcol, jnd, kept, ntot;
    int kind, nb, L;        // SpMV kind as spmv_kind (-3, -2, -1, 0)
    long ld;
    double beta_prev, eps, xscale, off;
    const double *x;        // the first step's SpMV input; x * xscale is q_a
    int store_q;            // q_a is stored (a deferred scale-copy)
    double *V, *scratch;
    float *V32;             // FP32 shadow (mixed precision) or null
    const double *dg, *val, *tab;
    const int *rb, *rp, *ci;
    const uint32_t *pk;
    double *part_alpha, *part_recur, *part_update, *part_proj;
    const double *coef;     // first step: its jnd - 1 coefficients
    double *hm;             // host-coherent: step 0's results, status at 6
    double *hchain;         // followers' results, 7 each
    unsigned *sync;         // a flag per workgroup
    unsigned base;          // flag value before this launch
    unsigned *gate;         // this launch's gate word (zero)
    unsigned *gate_next;    // the next launch's, cleared at the end, or null
    unsigned long long gate_ticks;
    unsigned *shut;         // a batch's launch: set once one of its gates has closed, else null
};

__device__ __forceinline__ double ld_agent(const double *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(double *p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// This wave's vector stores have reached the point of coherence.
__device__ __forceinline__ void stores_done()
{
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

// Waits until every workgroup's flag reaches `want`; wave 0 of a workgroup
// calls it.  False when the wait ran out.
__device__ __forceinline__ bool chain_poll(const unsigned *flags, int g, unsigned want)
{
    const int lane = threadIdx.x & 63;
    unsigned long long t0 = 0;
    for (unsigned spin = 0;; ++spin) {
        bool in = true;
        for (int i = lane; i < g; i += 64) {
            const unsigned f = __hip_atomic_load(flags + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            in = in && (int)(f - want) >= 0;
        }
        if (__all(in)) return true;
        if ((spin & 255u) == 255u) {
            const unsigned long long t = wall_clock64();
            if (!t0)
                t0 = t;
            else if (t - t0 > kBarrierTicks)
                return false;
        }
    }
}

// All workgroups have passed this point and their agent-scope stores are
// visible to agent-scope loads.  *ok_s: the workgroup's flag in LDS.
// ACQ: visible to ordinary loads too.
template <bool ACQ = false>
__device__ __forceinline__ bool chain_barrier(const ChainArgs &q, int b, unsigned want, int *ok_s)
{
    stores_done();
    __syncthreads();
    if (q.g > 1) {
        if (threadIdx.x < 64) {
            if (threadIdx.x == 0)
                __hip_atomic_store(q.sync + b, want, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool ok = chain_poll(q.sync, q.g, want);
            if (threadIdx.x == 0 && !ok) *ok_s = 0;
            if constexpr (ACQ) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        __syncthreads();
    }
    return *ok_s != 0;
}

// The gate: true in every workgroup when all g are running, false in every
// workgroup when one of them gave up waiting first (the gate word is set
// once: 1 open, 2 closed).  Once a chain of a batch's launch has waited in
// vain the others do not wait: where few workgroups find a place, each chain
// would spend the whole time anew.
__device__ __forceinline__ bool chain_gate(const ChainArgs &q, int b, int *ok_s)
{
    if (q.g == 1) return true;
    unsigned *gate = q.gate;
    const unsigned want = q.base + 1;
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        if (lane == 0)
            __hip_atomic_store(q.sync + b, want, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long t0 = wall_clock64();
        unsigned st = 0;
        while (!st) {
            bool in = true;
            for (int i = lane; i < q.g; i += 64) {
                const unsigned f = __hip_atomic_load(q.sync + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                in = in && (int)(f - want) >= 0;
            }
            const bool all = __all(in) && q.gate_ticks;  // a gate of no ticks never opens
            if (lane == 0) {
                const bool late =
                    wall_clock64() - t0 > q.gate_ticks ||
                    (q.shut && __hip_atomic_load(q.shut, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                if (all || late) {
                    unsigned seen = 0;
                    if (__hip_atomic_compare_exchange_strong(gate, &seen, all ? 1u : 2u, __ATOMIC_RELAXED,
                                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                        seen = all ? 1u : 2u;
                    st = seen;
                    if (st == 2 && q.shut)
                        __hip_atomic_store(q.shut, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                } else {
                    st = __hip_atomic_load(gate, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            st = __shfl(st, 0);
        }
        if (lane == 0) *ok_s = st == 1;
    }
    __syncthreads();
    return *ok_s != 0;
}

// strided_sum over partials other workgroups stored.
__device__ __forceinline__ double strided_sum_agent(const double *part, int nb, int b0, int step)
{
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int b = b0;
    for (; b + 3 * step < nb; b += 4 * step) {
        s0 += ld_agent(part + b);
        s1 += ld_agent(part + b + step);
        s2 += ld_agent(part + b + 2 * step);
        s3 += ld_agent(part + b + 3 * step);
    }
    for (; b < nb; b += step) s0 += ld_agent(part + b);
    return (s0 + s1) + (s2 + s3);
}

// The partial of 1024-row block rb (0 past the last): stored whole (RW = 4),
// or as the totals of its four waves (nw of them in all), added in wave
// order.  Clamped loads and selects, no branches, so that a wave's loads of
// several coefficients are in flight together.
template <int RW>
__device__ __forceinline__ double row_partial(const double *p, int nrb, int nw, int rb)
{
    if constexpr (RW == 4) {
        const double v = ld_agent(p + min(rb, nrb - 1));
        return rb < nrb ? v : 0.0;
    } else {
        double t = 0.0;
        double v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = ld_agent(p + min(4 * rb + i, nw - 1));
#pragma unroll
        for (int i = 0; i < 4; ++i) t += 4 * rb + i < nw ? v[i] : 0.0;
        return t;
    }
}

// ordered_sum of nrb <= 256 row partials by one wave: the four 64-lane
// totals a block's waves would form, added in order.
template <int RW>
__device__ __forceinline__ double wave_ordered_sum(const double *p, int nrb, int nw)
{
    const int lane = threadIdx.x & 63;
    double t = 0.0;
    for (int v = 0; v < kBlock / 64 && v * 64 < nrb; ++v) t += wave_sum(row_partial<RW>(p, nrb, nw, v * 64 + lane));
    return t;
}

// One thread's part of a row block of a CSR operator (at most kNnzBlk
// nonzeros, NZT a thread): the nonzeros tg, tg + 256, ... of the block and
// the thread's row.  Past the end: value 0 in column 0, no row.
constexpr int NZT = kNnzBlk / 256;
template <int KIND>
struct CsrPart {
    int r0, nr, ka, kb;
    int c[NZT];
    double v[NZT];
    __device__ __forceinline__ void load(const ChainArgs &q, int blk, int tg)
    {
        nr = ka = kb = r0 = 0;
        int k0 = 0, nz = 0;
        if (blk < q.nb) {
            r0 = q.rb[blk];
            nr = q.rb[blk + 1] - r0;
            k0 = q.rp[r0];
            nz = q.rp[r0 + nr] - k0;
            if (tg < nr) {
                ka = q.rp[r0 + tg] - k0;
                kb = q.rp[r0 + tg + 1] - k0;
            }
        }
#pragma unroll
        for (int u = 0; u < NZT; ++u) {
            const int k = tg + 256 * u;
            c[u] = 0;
            v[u] = 0.0;
            if (k < nz) {
                if constexpr (KIND == -1) {
                    const uint32_t wd = q.pk[k0 + k];
                    c[u] = r0 + ((int)(wd << 8) >> 8);
                    const uint32_t vi = wd >> 24;
                    v[u] = vi == 255u ? q.dg[c[u]] : q.tab[vi];
                } else {
                    c[u] = q.ci[k0 + k];
                    v[u] = q.val[k0 + k];
                }
            }
        }
    }
};

// Squares of the four rows [row, row + 4): as update_rows4 sums them, or
// for a ragged end as update_body's row-by-row tail does.
__device__ __forceinline__ double norm4(const double r[4], int row, int n)
{
    if (row + 3 < n) return sumsq4(r);
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (row + j < n) acc = fma(r[j], r[j], acc);
    return acc;
}

// Four rows of a column as stored.
__device__ __forceinline__ void res4(const float *p, float v[4])
{
    const f32x4 t = *reinterpret_cast<const f32x4 *>(p);
    v[0] = t.x;
    v[1] = t.y;
    v[2] = t.z;
    v[3] = t.w;
}
__device__ __forceinline__ void res4(const double *p, double v[4]) { load4(p, v); }

// KIND as spmv_kind: -3 / -2 periodic stencils, -1 packed CSR, 0 CSR.  VS =
// what the Gram-Schmidt pass reads (float: the FP32 shadow).  NRES = columns
// per group (c mod 4 = k, c < 4 NRES) that stay in registers for the chain.
template <int RW, int KIND, typename VS, int NRES = 0>
__device__ __forceinline__ void chain_body(const ChainArgs &q, const int b)
{
    constexpr int R = 256 * RW, NT = 256 * RW, NWAVE = 4 * RW;
    constexpr bool kStencil = KIND <= -2;
    constexpr int D = KIND == -3 ? 3 : 2;
    constexpr int K = 2 * D + 1;
    static_assert(RW == 2 || (RW == 4 && kStencil), "workgroup shapes");
    constexpr int CH = RW == 4 ? 4 : 8;  // columns per projection chunk (16 waves: 128 registers each)
    constexpr int HC = 4;                // coefficients a wave sums at once
    // LDS: y then r, q_a, q_b, the new vector's rows; the update's sums of
    // column groups 1..3, or the CSR products
    constexpr int kPool = kStencil ? 3 * R : (3 * R > RW * kNnzBlk ? 3 * R : RW * kNnzBlk);
    __shared__ double ys[R], qas[R], qbs[R], ss[R];
    __shared__ double pool[kPool];
    __shared__ double hs[kChainMaxCols], psum[RW == 4 ? 4 * kChainMaxCols : 1];
    __shared__ double wsum[2 * NWAVE], bc[8];
    __shared__ int ok_s;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int rw = w % RW, k = w / RW;  // row wave, column group
    const int n = q.n, g = q.g;
    const int R0 = b * R;
    const int row = R0 + rw * 256 + 4 * lane;  // first of this lane's four rows
    const int vrow = row < n ? row : 0;        // the row it loads (a lane past n: unused)
    const int lrow = rw * 256 + 4 * lane;
    const int nw = (n + 255) / 256, nrb = (n + 1023) / 1024;
    const int gw = b * RW + rw;                // this wave's row wave among nw
    const VS *VG;
    if constexpr (std::is_same<VS, float>::value)
        VG = q.V32 + vrow;
    else
        VG = q.V + vrow;
    if (t == 0) ok_s = 1;
    __syncthreads();
    if (!chain_gate(q, b, &ok_s)) {
        if (b == 0 && t == 0) {
            q.hm[6] = 2.0;
            if (q.gate_next) *q.gate_next = 0;
        }
        return;
    }
    unsigned want = q.base + 1;
    const double *x = q.x;
    double xs = q.xscale, bprev = q.beta_prev;
    int qa = q.qa, rcol = q.rcol, jnd = q.jnd;
    const int srow = R0 + t;  // SpMV: one row per thread (stencils), row-wise stores
    int cols[K];
    double dv = 0.0;
    if constexpr (kStencil) {
        if (srow < n) {
            stencil_cols<D>(srow, q.L, cols);
            dv = q.dg[srow];
        }
    }
    // CSR: the row block at hand and how many a group walks
    const int niter = kStencil ? 0 : (q.nb + g * RW - 1) / (g * RW);
    CsrPart<KIND> cur;
    if constexpr (!kStencil) cur.load(q, b * RW + (t >> 8), t & 255);
    VS vres[NRES > 0 ? NRES : 1][4];
#pragma unroll
    for (int i = 0; i < NRES; ++i) {
        const int c = 4 * i + k;
#pragma unroll
        for (int j = 0; j < 4; ++j) vres[i][j] = 0;
        if (c < jnd - 1) res4(VG + (size_t)c * q.ld, vres[i]);
    }
    // q_b of the first step
    if (!q.first && q.qb >= 0)
        qbs[t] = srow < n ? q.V[(size_t)q.qb * q.ld + srow] : 0.0;
    else
        qbs[t] = 0.0;
    int status = 1;
    for (int step = 0;; ++step) {
        // ---- y = A q_a, alpha partials, q_a stored
        {
            double xr = 0.0;
            if (srow < n) xr = (double)((kStencil ? ld_agent(x + srow) : x[srow]) * xs);
            if constexpr (kStencil) {
                double acc = 0.0, y = 0.0;
                if (srow < n) {
                    double xv[K];
#pragma unroll
                    for (int i = 0; i < K; ++i) xv[i] = ld_agent(x + cols[i]);
#pragma unroll
                    for (int i = 0; i < K; ++i)
                        y = add_prod(y, cols[i] == srow ? dv : q.off, (double)(xv[i] * xs));
                    acc = add_prod(0.0, xr, y);
                }
                ys[t] = y;
                acc = wave_sum(acc);
                if (lane == 0) wsum[w] = acc;
                __syncthreads();
                if (t < RW && (b * RW + t) < q.nb) {
                    double s = 0.0;
#pragma unroll
                    for (int i = 0; i < 4; ++i) s += wsum[4 * t + i];
                    st_agent(q.part_alpha + b * RW + t, s);
                }
            } else {
                // CSR-stream: each group of 256 threads takes row blocks; the
                // next one's nonzeros (after the last, the first one's for the
                // next step) are loaded while this one's products are summed
                const int grp = t >> 8, tg = t & 255;
                double *prod = pool + grp * kNnzBlk;
                double *yc = q.V + (size_t)rcol * q.ld;
                for (int it = 0; it < niter; ++it) {
                    const int blk = (it * g + b) * RW + grp;
                    double xv[NZT];
#pragma unroll
                    for (int u = 0; u < NZT; ++u) xv[u] = x[cur.c[u]];
                    const int r0 = cur.r0, nr = cur.nr, ka = cur.ka, kb = cur.kb;
                    double xo = 0.0;
                    if (tg < nr) xo = (double)(x[r0 + tg] * xs);
#pragma unroll
                    for (int u = 0; u < NZT; ++u) prod[tg + 256 * u] = cur.v[u] * (double)(xv[u] * xs);
                    cur.load(q, it + 1 < niter ? blk + g * RW : b * RW + grp, tg);
                    __syncthreads();
                    double acc = 0.0;
                    if (tg < nr) {
                        double s = 0.0;
                        for (int i = ka; i < kb; i += 4) {
                            double p[4];
#pragma unroll
                            for (int u = 0; u < 4; ++u) p[u] = prod[min(i + u, kNnzBlk - 1)];
#pragma unroll
                            for (int u = 0; u < 4; ++u) s = i + u < kb ? s + p[u] : s;
                        }
                        st_agent(yc + r0 + tg, s);
                        acc = add_prod(acc, xo, s);
                    }
                    acc = wave_sum(acc);
                    if (lane == 0) wsum[w] = acc;
                    __syncthreads();
                    if (tg == 0 && blk < q.nb) {
                        double s = 0.0;
#pragma unroll
                        for (int i = 0; i < 4; ++i) s += wsum[4 * grp + i];
                        st_agent(q.part_alpha + blk, s);
                    }
                }
            }
            qas[t] = xr;
            if (srow < n && (step > 0 || q.store_q)) {
                q.V[(size_t)qa * q.ld + srow] = xr;
                if (q.V32) q.V32[(size_t)qa * q.ld + srow] = (float)xr;
            }
        }
        if (!chain_barrier(q, b, ++want, &ok_s)) break;
        // ---- alpha; r = y - beta q_b - alpha q_a (or the restart's columns)
        if (t < 256) {
            const double v = wave_sum(strided_sum_agent(q.part_alpha, q.nb, t, 256));
            if (lane == 0) wsum[w] = v;
        }
        if constexpr (!kStencil) ys[t] = srow < n ? ld_agent(q.V + (size_t)rcol * q.ld + srow) : 0.0;
        const int rm = q.first && step == 0 ? jnd : 0;
        if (rm)
            for (int i = t; i < rm - 1; i += NT) hs[i] = q.coef[i];
        __syncthreads();
        double alpha = 0.0;
#pragma unroll
        for (int i = 0; i < 4; ++i) alpha += wsum[i];
        if (rm && t == 0) hs[rm - 1] = alpha;
        double r4[4];
        if (rm) {
            // the restart's first step: V(:, 0:rm) h over the FP64 basis,
            // the columns split over the groups as in the update
            __syncthreads();
            double s[4] = {0.0, 0.0, 0.0, 0.0};
            group_sums(q.V + vrow, q.ld, rm, hs, k, s);
            if (k > 0)
#pragma unroll
                for (int j = 0; j < 4; ++j) pool[(k - 1) * R + lrow + j] = s[j];
            __syncthreads();
            if (k == 0) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    r4[j] = ys[lrow + j] - ((s[j] + pool[lrow + j]) + (pool[R + lrow + j] + pool[2 * R + lrow + j]));
                    ys[lrow + j] = row + j < n ? r4[j] : 0.0;
                }
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < 4; ++j) r4[j] = ys[lrow + j];
        } else {
            const bool two = step > 0 || q.qb >= 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                double s = 0.0;
                if (two) s += qbs[lrow + j] * bprev;
                s += qas[lrow + j] * alpha;
                r4[j] = ys[lrow + j] - ((s + 0.0) + (0.0 + 0.0));
            }
        }
        if (row >= n) {
#pragma unroll
            for (int j = 0; j < 4; ++j) r4[j] = 0.0;
        }
        // ||r||^2 partial: wave totals of the first column group
        if (k == 0) {
            const double a = wave_sum(row < n ? norm4(r4, row, n) : 0.0);
            if (lane == 0) {
                if constexpr (RW == 4)
                    wsum[NWAVE + rw] = a;
                else if (gw < nw)
                    st_agent(q.part_recur + gw, a);
            }
        }
        // ---- projection partials: the resident columns, then chunks of CH
        // columns over the groups
        if constexpr (NRES > 0) {
            double p[NRES];
#pragma unroll
            for (int i = 0; i < NRES; ++i) {
                if (qa == 4 * i + k)  // q_a joins the resident columns
#pragma unroll
                    for (int j = 0; j < 4; ++j) vres[i][j] = (VS)qas[lrow + j];
                p[i] = 0.0;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < NRES; ++i) p[i] += (double)vres[i][j] * r4[j];
            const double tot = wave_transpose_sum<NRES>(p, lane);
            const int c = 4 * (lane / (64 / NRES)) + k;
            if (lane % (64 / NRES) == 0 && c < jnd && gw < nw) st_agent(q.part_proj + (size_t)c * nw + gw, tot);
        }
        for (int cb = 4 * NRES + CH * k; cb < jnd; cb += 4 * CH) {
            double p[CH];
            double v[CH][4];
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                p[c] = 0.0;
                ld4(VG + (size_t)min(cb + c, jnd - 1) * q.ld, v[c]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < CH; ++c) p[c] += v[c][j] * r4[j];
            const double tot = wave_transpose_sum<CH>(p, lane);
            const int c = cb + lane / (64 / CH);
            if (lane % (64 / CH) == 0 && c < jnd) {
                if constexpr (RW == 4)
                    psum[4 * c + rw] = tot;
                else if (gw < nw)
                    st_agent(q.part_proj + (size_t)c * nw + gw, tot);
            }
        }
        __syncthreads();  // also: q_a, q_b and y of this step have been read
        if constexpr (RW == 4) {
            for (int c = t; c < jnd; c += NT) {
                double s = 0.0;
#pragma unroll
                for (int i = 0; i < 4; ++i) s += psum[4 * c + i];
                st_agent(q.part_proj + (size_t)c * nrb + b, s);
            }
            if (t == NT - 1) {
                double s = 0.0;
#pragma unroll
                for (int i = 0; i < 4; ++i) s += wsum[NWAVE + i];
                st_agent(q.part_recur + b, s);
            }
        }
        if (k == 0)
#pragma unroll
            for (int j = 0; j < 4; ++j) ys[lrow + j] = r4[j];
        if (!chain_barrier(q, b, ++want, &ok_s)) break;
        // ---- h, then s = r - V h and its norm
        {
            const int np = RW == 4 ? nrb : nw;
            if (nrb <= 64) {  // one virtual wave of partials: HC columns in flight
                for (int c0 = w; c0 < jnd; c0 += HC * NWAVE) {
                    double v[HC];
#pragma unroll
                    for (int i = 0; i < HC; ++i) {
                        const int c = min(c0 + i * NWAVE, jnd - 1);
                        v[i] = row_partial<RW>(q.part_proj + (size_t)c * np, nrb, nw, lane);
                    }
#pragma unroll
                    for (int i = 0; i < HC; ++i) {
                        const double h = 0.0 + wave_sum(v[i]);
                        if (lane == 0 && c0 + i * NWAVE < jnd) hs[c0 + i * NWAVE] = h;
                    }
                }
            } else {
                for (int c = w; c < jnd; c += NWAVE) {
                    const double h = wave_ordered_sum<RW>(q.part_proj + (size_t)c * np, nrb, nw);
                    if (lane == 0) hs[c] = h;
                }
            }
        }
        __syncthreads();
        {
            double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int i = 0; i < NRES; ++i)
                if (4 * i < (jnd & ~7))
#pragma unroll
                    for (int j = 0; j < 4; ++j) s[j] += (double)vres[i][j] * hs[4 * i + k];
            group_sums<VS, NRES == 0>(VG, q.ld, jnd, hs, k, s, 4 * NRES);
            if (k > 0)
#pragma unroll
                for (int j = 0; j < 4; ++j) pool[(k - 1) * R + lrow + j] = s[j];
            if (t == NT - 1) {
                double hh = 0.0;
                for (int i = 0; i < jnd; ++i) hh += hs[i] * hs[i];
                bc[0] = hh;
            }
            __syncthreads();
            if (k == 0) {
                double ro[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    ro[j] = r4[j] - ((s[j] + pool[lrow + j]) + (pool[R + lrow + j] + pool[2 * R + lrow + j]));
                    ss[lrow + j] = ro[j];
                }
                const double a = wave_sum(row < n ? norm4(ro, row, n) : 0.0);
                if (lane == 0) {
                    if constexpr (RW == 4)
                        wsum[rw] = a;
                    else if (gw < nw)
                        st_agent(q.part_update + gw, a);
                }
            }
        }
        __syncthreads();
        if (srow < n) st_agent(q.scratch + srow, ss[t]);
        if constexpr (RW == 4) {
            if (t == 0) {
                double s = 0.0;
#pragma unroll
                for (int i = 0; i < 4; ++i) s += wsum[i];
                st_agent(q.part_update + b, s);
            }
        }
        if (!chain_barrier<!kStencil>(q, b, ++want, &ok_s)) break;
        // ---- the norms, the step's results, the decision for the next step
        if (w < 2) {
            const double v = wave_ordered_sum<RW>(w == 0 ? q.part_recur : q.part_update, nrb, nw);
            if (lane == 0) bc[1 + w] = v;
        }
        __syncthreads();
        const double rr2 = bc[1], rr2b = bc[2], hh = bc[0];
        const bool more = step + 1 < q.steps;
        const bool go = more && chain_go(alpha, rr2, hh, rr2b, bprev, jnd, q.kept, q.ntot, q.eps);
        const double beta = go ? sqrt(rr2b) : 0.0;
        const double inv = go ? 1.0 / beta : 0.0;
        if (b == 0 && t == 0) {
            double *o = step == 0 ? q.hm : q.hchain + 7 * (step - 1);
            o[S_ALPHA] = alpha;
            o[S_RR2] = rr2;
            o[S_HH] = hh;
            o[S_RR2B] = rr2b;
            if (more) {
                double *f = q.hchain + 7 * step;
                f[4] = go ? 1.0 : 0.0;
                f[5] = inv;
                f[6] = beta;
            }
        }
        if (!go) {
            // r of the step the chain ends with, for the solver to go on from
            if (srow < n) q.V[(size_t)rcol * q.ld + srow] = ys[t];
            status = 0;
            break;
        }
        qbs[t] = qas[t];
        x = q.scratch;
        xs = inv;
        bprev = beta;
        qa = rcol;
        ++rcol;
        ++jnd;
        __syncthreads();  // bc and wsum have been read
    }
    if (b == 0 && t == 0) {
        q.hm[6] = status == 0 ? 1.0 : 3.0;
        if (q.gate_next) *q.gate_next = 0;
    }
}

// 8 waves of a stencil in FP64 leave 64 registers free: the first 32 columns
// are read once a chain and not twice a step (2-D lattice, n = 10^4: a solve
// of 268 steps 6.15 -> 5.71 ms).  Elsewhere it costs more than it gives:
// 16 waves and the batch's kernel spill, the CSR products need the
// registers, and the conversion of FP32 columns is kept as doubles
// (n = 181^2, mixed: 9.84 -> 10.48 ms with 32 columns).
template <int RW, int KIND, typename VS>
__global__ __launch_bounds__(256 * RW) void k_chain(ChainArgs q)
{
    chain_body<RW, KIND, VS, RW == 2 && KIND <= -2 && std::is_same<VS, double>::value ? 8 : 0>(q, blockIdx.x);
}

// The chains of many solves in one launch.  At most one workgroup per CU is
// launched; each takes pieces (one workgroup's share of one chain, pieces of
// a chain consecutive) by ticket until none are left, so the pieces taken
// are always the first ones.  A chain waits at its gate for pieces that
// workgroups free of earlier chains take next; with at most a quarter of the
// CUs' workgroups per chain that holds also when other lanes' launches or
// other work take part of the device, and should the device be taken
// altogether the gate closes and the host runs that chain's step otherwise.
// (A workgroup per piece does not do: workgroups go to the XCDs round-robin,
// so the last ones may all belong to one XCD and wait for each other's
// place there.)  Flags, gate words and ticket start at zero: they are copied
// with the launch's records.
template <int RW, int KIND, typename VS>
__global__ __launch_bounds__(256 * RW) void kb_chain(const ChainArgs *__restrict__ d,
                                                     const int *__restrict__ pre, int nreq,
                                                     unsigned *__restrict__ ticket)
{
    __shared__ int mine;
    const int total = pre[nreq];
    for (;;) {
        if (threadIdx.x == 0)
            mine = (int)__hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const int i = __builtin_amdgcn_readfirstlane(mine);
        if (i >= total) return;
        const int p = __builtin_amdgcn_readfirstlane(batch_find(pre, nreq, i));
        const ChainArgs q = d[p];
        chain_body<RW, KIND, VS>(q, i - pre[p]);
        __syncthreads();  // the LDS of this piece has been read
    }
}

#endif

"""Chains of steps in one kernel (real solves on stencil or CSR-stream
operators, alone and in small batches) against the kernels that run a step
phase by phase: the same eigenvalues, vectors, residual estimates and
counters bit for bit, at sizes around the kernels' edges (256 rows a wave,
512 and 1024 a workgroup, 64 row blocks a reduction wave, ragged ends), and
with several solves on the device at once.

A batch too large for chains runs phase by phase, so each solve is compared
with itself in a batch beside operators that fill it up; the kernel statistics
say which kernels ran."""
import ctypes
import threading

import numpy as np
import pytest

from nutrlan_amd import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("stat", "nec", "matvec", "nloop", "north", "nrand", "locked")


def same(a, b):
    assert [a[k] for k in KEYS] == [b[k] for k in KEYS]
    for k in ("eval", "evec", "resid"):
        assert np.array_equal(a[k], b[k]), k


_fill = []


def filler(T):
    if not _fill:
        _fill.append((T.Csr(*W.anderson2d_csr(255, 6.0, seed=255)[0]), W.start_vector(255 * 255, seed=1)))
    return _fill[0]


def counted(T, solve):
    """solve() and the kernel launches of it by class."""
    T.stats_enable(True)
    r = solve()
    st = T.stats_get()
    T.stats_enable(False)
    return r, {k: v[0] for k, v in st.items()}


def both(T, csr, mixed, lohi, ned, maxlan, tol=1e-8, maxmv=4000, seed=3, dense=False):
    """dense: a CSR operator with more nonzeros than chains take."""
    n = len(csr[0]) - 1
    A = T.Csr(*csr, mixed=mixed)
    args = (lohi, ned, maxlan, tol, 1, maxmv, ned)
    x0 = W.start_vector(n, seed=seed)
    print(f"n={n} mixed={mixed} stencil={A.stencil} packed={A.packed}", flush=True)
    one, k1 = counted(T, lambda: T.solve_csr(A, *args, x0))
    (rc, small, _), k2 = counted(T, lambda: T.solve_batch([(A,) + args + (x0,)]))
    assert rc == 0
    # 2 x 11 fillers of 65,025 rows that stop after the same number of steps:
    # each of the batch's two lanes holds over 600,000 rows
    F, fx = filler(T)
    fill = [(F, -1, 8, maxlan, 1e-14, 1, one["matvec"] + maxlan, 8, fx)] * 11
    (rc, large, _), k3 = counted(T, lambda: T.solve_batch([(A,) + args + (x0,)] + [fill[0]] + fill + fill[:9]))
    stencil = A.stencil[0] > 0
    A.close()
    assert rc == 0
    assert (k1["chain"] > 0) == (not dense and n <= (262144 if stencil else 131072)), k1
    assert (k2["b_chain"] > 0) == (not dense and n <= (65536 if stencil else 32768)), k2
    # fillers past a chain's columns are not among the rows that keep the
    # batch from chains, so the last steps of such a cycle may be one
    assert 10 * k3["b_chain"] <= (k2["b_chain"] if maxlan > 192 else 0) and k3["b_update"] > 0, k3
    same(one, small[0])
    same(one, large[0])


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("L", [16, 23, 32, 33, 45, 181, 182, 362, 363, 512, 513])
def test_chain_lattice2d(gpu_lib, L, mixed):
    both(gpu_lib, W.anderson2d_csr(L, 6.0, seed=L)[0], mixed, -1, 6, 24, maxmv=120 if L > 200 else 4000)


@pytest.mark.parametrize("mixed,L", [(True, 256), (True, 257), (False, 257), (False, 361)])
def test_chain_lattice2d_row_waves(gpu_lib, L, mixed):
    """Either side of the line between workgroups of 2 and of 4 row waves."""
    both(gpu_lib, W.anderson2d_csr(L, 6.0, seed=L)[0], mixed, -1, 6, 24, maxmv=120)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("L", [8, 11, 32, 33, 64])
def test_chain_lattice3d(gpu_lib, L, mixed):
    both(gpu_lib, W.laplace3d_csr(L, seed=L), mixed, 1, 8, 40, maxmv=150)


@pytest.mark.parametrize("n", [257, 511, 513, 1022, 1025, 2050])
def test_chain_packed(gpu_lib, n):
    """A diagonal operator: packed CSR, one nonzero a row."""
    both(gpu_lib, W.diag_csr(n), False, 1, 5, 30)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("n,degree", [(300, 16.0), (1023, 3.0), (4099, 16.0), (20001, 40.0), (131072, 4.0),
                                      (131073, 4.0)])
def test_chain_random_rows(gpu_lib, n, degree, mixed):
    both(gpu_lib, W.random_sym_csr(n, degree=degree, seed=n), mixed, 1, 10, 60, maxmv=130, dense=degree == 40.0)


def test_chain_wide_basis(gpu_lib):
    """More basis columns than a chain kernel takes: its last steps of a
    cycle run as ordinary kernels."""
    both(gpu_lib, W.random_sym_csr(3001, seed=9), False, 1, 6, 200, maxmv=450)


def test_chain_batch_mixed_kinds(gpu_lib):
    """A small batch of stencils, packed and random operators in both
    precisions: several chain groups in a launch, each solve as alone."""
    T = gpu_lib
    spec = [(W.anderson2d_csr(L, 4.0, seed=L)[0], m, -1, 6, 24) for L, m in ((40, 0), (41, 1), (90, 0), (200, 1), (250, 0))]
    spec += [(W.laplace3d_csr(L, seed=L), m, 1, 6, 30) for L, m in ((9, 0), (20, 1))]
    spec += [(W.diag_csr(900), 0, 1, 5, 30), (W.random_sym_csr(2500, seed=2), 0, 1, 8, 40),
             (W.random_sym_csr(30001, seed=3), 1, 1, 8, 40)]
    probs = []
    for i, (csr, m, lohi, ned, maxlan) in enumerate(spec):
        probs.append((T.Csr(*csr, mixed=bool(m)), lohi, ned, maxlan, 1e-8, 1, 400, ned,
                      W.start_vector(len(csr[0]) - 1, seed=i)))
    alone = [T.solve_csr(*p) for p in probs]
    rc, got, _ = T.solve_batch(probs)
    assert rc == 0
    for p, a, b in zip(probs, alone, got):
        p[0].close()
        same(a, b)


def test_chain_concurrent_solves(gpu_lib):
    """Solves from several threads, together more workgroups than the device
    holds at once: each equals the solve alone."""
    T = gpu_lib
    probs = [(W.anderson2d_csr(L, 5.0, seed=L)[0], W.start_vector(L * L, seed=L)) for L in (500, 505, 510, 300, 64, 40)]
    ops = [T.Csr(*csr) for csr, _ in probs]

    def solve(i):
        return T.solve_csr(ops[i], -1, 6, 24, 1e-8, 1, 100, 6, probs[i][1])

    alone = [solve(i) for i in range(len(probs))]
    got = [None] * len(probs)

    def work(i):
        got[i] = solve(i)

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(probs))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    steps, wgs = ctypes.c_int(-1), ctypes.c_int(-1)
    assert T.lib().trlhip_device_load(0, ctypes.byref(steps), ctypes.byref(wgs)) == 0
    assert (steps.value, wgs.value) == (0, 0)  # what they had taken is given back
    for A in ops:
        A.close()
    for a, b in zip(alone, got):
        same(a, b)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("kind,size", [("2d", 32), ("2d", 45), ("3d", 11), ("diag", 700), ("random", 3001)])
def test_step_any_column(gpu_lib, kind, size, mixed):
    """trlhip_step_cgs with q_a any column and r any column past the basis,
    against NumPy in FP64.  Columns are FP32 values, so a mixed context's
    shadow holds them exactly.  Bound: every result is a sum of at most n +
    jnd products of O(1) magnitude after its factors' own sums, 8 (n + jnd)
    eps of the magnitudes' sum."""
    T = gpu_lib
    csr = {"2d": lambda: W.anderson2d_csr(size, 6.0, seed=size)[0], "3d": lambda: W.laplace3d_csr(size, seed=size),
           "diag": lambda: W.diag_csr(size), "random": lambda: W.random_sym_csr(size, seed=size)}[kind]()
    n = len(csr[0]) - 1
    mv = W.csr_matvec(*csr)
    A = T.Csr(*csr, mixed=mixed)
    ncols = 40
    c = T.Ctx(n, ncols, mixed=mixed)
    rng = np.random.default_rng(size)
    V = (rng.standard_normal((ncols, n)) / np.sqrt(n)).astype(np.float32).astype(np.float64)
    for j in range(ncols):
        c.set(j, V[j])
    for jnd in (1, 2, 5, 8, 9, 16, 31, 32, 33):
        for qa, qb, rcol in ((0, -1, jnd), (jnd // 2, jnd // 2 - 1, jnd), (jnd - 1, jnd - 2, jnd + 2),
                             (jnd + 1, -1, jnd), (jnd - 1, jnd - 2, jnd)):
            print(f"{kind} n={n} mixed={mixed} jnd={jnd} qa={qa} qb={qb} rcol={rcol}", flush=True)
            out = c.step_cgs(A, 0, qa, qb, 0.25, None, jnd, rcol)
            y = np.asarray(mv(V[qa])).ravel()
            alpha = V[qa] @ y
            r = y - alpha * V[qa] - (0.25 * V[qb] if qb >= 0 else 0.0)
            h = V[:jnd] @ r
            s = r - h @ V[:jnd]
            tol = 8 * (n + jnd) * np.finfo(float).eps
            scale = np.abs(y).max() * 2 + np.linalg.norm(y) * (1 + np.abs(h).max())
            got_r = c.get(rcol)
            c.scale_copy(rcol, ncols, 1.0)
            got_s = c.get(rcol)
            c.set(rcol, V[rcol])
            assert np.abs(got_r - r).max() <= tol * scale
            assert np.abs(got_s - s).max() <= tol * scale * jnd
            want = np.array([alpha, r @ r, h @ h, s @ s])
            assert (np.abs(out - want) <= tol * jnd * (1 + scale) ** 2).all(), (out, want)
    c.close()
    A.close()


@pytest.mark.parametrize("maxlan", [194, 200, 210])
def test_chain_past_its_columns_after_phases(gpu_lib, maxlan):
    """A batch that starts phase by phase and, its larger solves done, goes on
    in chains, past the columns a chain takes: the steps cut off must not run
    on what the phase kernels left."""
    T = gpu_lib
    n = 3001
    A = T.Csr(*W.random_sym_csr(n, seed=9))
    args = (1, 6, maxlan, 1e-8, 1, 450, 6)
    x0 = W.start_vector(n, seed=3)
    one = T.solve_csr(A, *args, x0)
    F, fx = filler(T)
    fill = [(F, -1, 2, 24, 1e-14, 1, 60, 2, fx)] * 22
    print(f"n={n} maxlan={maxlan}", flush=True)
    (rc, got, _), k = counted(T, lambda: T.solve_batch([(A,) + args + (x0,)] + fill))
    A.close()
    assert rc == 0 and k["b_chain"] > 0 and k["b_update"] > 0
    same(one, got[0])


@pytest.mark.parametrize("mixed", [False, True])
def test_chain_statistics(gpu_lib, mixed):
    """Chain kernels are a class of their own, with the bytes of the steps
    that ran: a chain over columns that are not orthogonal stops after one."""
    T = gpu_lib
    L, ncols = 40, 30
    n = L * L
    A = T.Csr(*W.anderson2d_csr(L, 6.0, seed=1)[0], mixed=mixed)
    c = T.Ctx(n, ncols, mixed=mixed)
    rng = np.random.default_rng(1)
    for j in range(ncols):
        c.set(j, rng.standard_normal(n) / np.sqrt(n))

    def step(steps, jnd):
        T.stats_enable(True)
        if steps > 1:
            c.step_chain(steps, 0, n)
        c.step_cgs(A, 0, jnd - 1, -1, 0.0, None, jnd, jnd)
        st = T.stats_get()
        T.stats_enable(False)
        assert {k for k, s in st.items() if s[0]} == {"chain"} and st["chain"][0] == 1
        return st["chain"][2]

    one = step(1, 8)
    assert one > 0 and step(8, 8) == one
    # a column more: read twice as stored
    assert step(1, 9) - one == 2 * (4 if mixed else 8) * n
    c.close()
    # a solve: every step in a chain, none as ordinary kernels
    args = (A, -1, 6, 24, 1e-8, 1, 500, 6, W.start_vector(n, seed=3))
    st, bst = counted(T, lambda: T.solve_csr(*args))[1], counted(T, lambda: T.solve_batch([args]))[1]
    A.close()
    assert st["chain"] > 10 and st["b_chain"] == 0 and st["recur"] == 0
    assert bst["b_chain"] > 10 and bst["chain"] == 0 and bst["b_update"] == 0

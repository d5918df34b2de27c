"""Chains whose gate closes because the device is full: the step runs as
ordinary kernels with the same bits, followers are recorded again, and later
steps are chains again.  A gate that waits for no time never opens (every
workgroup leaves), so the busy device is set from the host.  Contexts are
driven step by step as the solver drives them, alone and in a batch of one
whose yield runs what was recorded."""
import ctypes
import time

import numpy as np
import pytest

from nutrlan_amd import workloads as W

pytestmark = pytest.mark.gpu

YIELD = ctypes.CFUNCTYPE(None, ctypes.c_void_p)


class Batch:
    """A batch whose contexts are driven by one thread: what a context waits
    for runs at once, with whatever `before` records first."""

    before = None

    def __init__(self, T, n, ncols, mixed):
        L, P = T.lib(), ctypes.c_void_p
        for name, args in [("trlhip_batch_create", [P]), ("trlhip_batch_set_yield", [P, YIELD, P]),
                           ("trlhip_batch_flush", [P]), ("trlhip_batch_destroy", [P]),
                           ("trlhip_ctx_create_batched", [P, ctypes.c_int, ctypes.c_int, ctypes.c_int, P])]:
            getattr(L, name).argtypes = args
        self.L, self.b = L, P()
        assert L.trlhip_batch_create(ctypes.byref(self.b)) == 0

        def run(_):
            f, self.before = self.before, None
            if f:
                f()
            L.trlhip_batch_flush(self.b)

        self.cb = YIELD(run)
        L.trlhip_batch_set_yield(self.b, self.cb, None)
        self.T, self.all = T, []
        self.ctx = self.add(n, ncols, mixed)

    def add(self, n, ncols, mixed):
        c = self.T.Ctx(1, 1)  # its bound functions, with the batch's handle
        c.close()
        h = ctypes.c_void_p()
        vt = self.T.TRLHIP_R32 if mixed else self.T.TRLHIP_R64
        assert self.L.trlhip_ctx_create_batched(ctypes.byref(h), n, ncols, vt, self.b) == 0
        c.h, c.n, c.ncols = h, n, ncols
        self.all.append(c)
        return c

    def close(self):
        for c in self.all:
            c.close()
        self.L.trlhip_batch_destroy(self.b)


def gate(T, c, ticks, hold=0):
    f = T.lib().trlhip_ctx_chain_gate
    f.argtypes = [ctypes.c_void_p, ctypes.c_ulonglong, ctypes.c_ulonglong]
    assert f(c.h, ticks, hold) == 0


def counts(T, c):
    f = T.lib().trlhip_ctx_chain_counts
    f.argtypes = [ctypes.c_void_p] * 3
    ran, closed = ctypes.c_long(), ctypes.c_long()
    assert f(c.h, ctypes.byref(ran), ctypes.byref(closed)) == 0
    return ran.value, closed.value


def lanczos(c, A, n, m, chain, x0, coef):
    """m steps of which the first starts a cycle, then a restart's first step
    on the columns so far and a few more; the results of all steps and the
    columns, the last one's r and s among them."""
    res = []
    c.set(0, x0)
    prev = 0.0
    for jnd in range(1, m + 6):
        first = jnd in (1, m + 1)
        if not first:
            left = m - jnd + 1 if jnd <= m else m + 6 - jnd
            c.step_chain(min(chain, left), 0 if jnd <= m else m, n)
        beta = coef[:jnd - 1] if first else None
        out = c.step_cgs(A, int(first), jnd - 1, jnd - 2 if not first else -1, 0.0 if first else prev, beta, jnd, jnd)
        res.append(out.copy())
        prev = np.sqrt(out[3])
        if jnd < m + 5:
            c.scale_copy(jnd, c.ncols, 1.0 / prev)  # pending until the next step
    last = m + 5
    cols = [c.get(j) for j in range(last + 1)]
    c.scale_copy(last, c.ncols, 1.0)
    cols.append(c.get(last))
    return np.array(res), np.array(cols)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("kind,size", [("2d", 45), ("3d", 12), ("diag", 2000), ("random", 3001)])
@pytest.mark.parametrize("batch", [False, True])
def test_closed_gate(gpu_lib, batch, kind, size, mixed):
    T = gpu_lib
    csr = {"2d": lambda: W.anderson2d_csr(size, 6.0, seed=size)[0], "3d": lambda: W.laplace3d_csr(size, seed=size),
           "diag": lambda: W.diag_csr(size), "random": lambda: W.random_sym_csr(size, seed=size)}[kind]()
    n = len(csr[0]) - 1
    A = T.Csr(*csr, mixed=mixed)
    x0 = W.start_vector(n, seed=1)
    x0 /= np.linalg.norm(x0)
    m = 17
    coef = np.random.default_rng(2).standard_normal(m) * 0.1

    def run(ticks):
        print(f"{kind} n={n} mixed={mixed} batch={batch} ticks={ticks}", flush=True)
        b = Batch(T, n, m + 8, mixed) if batch else None
        c = b.ctx if b else T.Ctx(n, m + 8, mixed=mixed)
        if ticks is not None:
            gate(T, c, ticks)
        got = lanczos(c, A, n, m, 6, x0, coef)
        cnt = counts(T, c)
        again = None
        if ticks == 0:  # the device is free again: the next step is a chain
            gate(T, c, 200000)
            c.set(0, x0)
            c.step_cgs(A, 1, 0, -1, 0.0, coef[:0], 1, 1)
            again = counts(T, c)
        (b or c).close()
        return got, cnt, again

    (res, cols), (ran, closed), _ = run(None)
    assert ran >= 5 and closed == 0
    (res0, cols0), (ran0, closed0), again = run(0)
    assert ran0 == 0 and closed0 >= 5  # every chain was tried, and none ran
    assert again == (1, closed0)
    A.close()
    assert np.array_equal(res, res0)
    assert np.array_equal(cols, cols0)


def test_gate_closed_for_a_while(gpu_lib):
    """After a gate has closed the ordinary kernels run for the time set,
    without another try, then chains again."""
    T = gpu_lib
    n = 2000
    A = T.Csr(*W.diag_csr(n))
    c = T.Ctx(n, 8)
    x0 = W.start_vector(n, seed=1)
    c.set(0, x0 / np.linalg.norm(x0))

    def step():
        return c.step_cgs(A, 1, 0, -1, 0.0, np.zeros(0), 1, 1)

    gate(T, c, 0, 20000000)  # 0.2 s
    want = step()
    t0 = time.perf_counter()
    for _ in range(20):
        assert np.array_equal(step(), want)
    if time.perf_counter() - t0 < 0.15:
        assert counts(T, c) == (0, 1)
    gate(T, c, 200000)
    time.sleep(0.25)
    assert np.array_equal(step(), want)
    assert counts(T, c)[0] == 1
    c.close()
    A.close()


@pytest.mark.parametrize("closed", [0, 1])
def test_closed_gate_beside_others(gpu_lib, closed):
    """One of two chains of a launch has a gate that never opens: once it has
    closed the other need not wait for its own, and either way both steps have
    the bits they have alone."""
    T = gpu_lib
    sizes = (45, 60)
    ops = [T.Csr(*W.anderson2d_csr(L, 6.0, seed=L)[0]) for L in sizes]
    x0 = [W.start_vector(L * L, seed=L) for L in sizes]
    x0 = [x / np.linalg.norm(x) for x in x0]
    want = []
    for A, x in zip(ops, x0):
        c = T.Ctx(len(x), 6)
        c.set(0, x)
        want.append((c.step_cgs(A, 1, 0, -1, 0.0, np.zeros(0), 1, 1), c.get(1)))
        c.close()
    b = Batch(T, len(x0[0]), 6, False)
    c = [b.ctx, b.add(len(x0[1]), 6, False)]
    for k in (0, 1):
        c[k].set(0, x0[k])
    gate(T, c[closed], 0, 100000000)
    print(f"closed={closed}", flush=True)
    got = [None, None]

    def step(k):
        got[k] = c[k].step_cgs(ops[k], 1, 0, -1, 0.0, np.zeros(0), 1, 1)

    b.before = lambda: step(1)  # recorded beside the first one's step
    step(0)
    assert counts(T, c[closed]) == (0, 1)
    assert sum(counts(T, c[1 - closed])) == 1
    for k in (0, 1):
        assert np.array_equal(got[k], want[k][0]) and np.array_equal(c[k].get(1), want[k][1])
    b.close()
    for A in ops:
        A.close()


@pytest.mark.parametrize("size,complex_", [(12, True), (31, True), (65, True), (66, False)])
def test_queued_steps(gpu_lib, size, complex_):
    """Complex and larger solves queue their steps phase by phase: the bits of
    the same steps taken one at a time."""
    T = gpu_lib
    csr = W.anderson3d_csr(size, seed=size) if complex_ else W.laplace3d_csr(size, seed=size)
    n = len(csr[0]) - 1
    A = T.Csr(*csr, complex_=complex_)
    x0 = W.start_vector(n, seed=1, complex_=complex_)
    m = 17
    coef = np.random.default_rng(2).standard_normal(m) * 0.1
    got = []
    for steps in (1, 6):
        print(f"n={n} complex={complex_} steps={steps}", flush=True)
        c = T.Ctx(n, m + 8, complex_=complex_)
        got.append(lanczos(c, A, n, m, steps, x0 / np.linalg.norm(x0), coef))
        assert counts(T, c) == (0, 0)
        c.close()
    A.close()
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("lpr", [2, 4, 8, 16, 32])
def test_queued_steps_vector_csr(gpu_lib, lpr, mixed):
    """The same for operators set to the vector-CSR kernel, which no chain
    takes."""
    T = gpu_lib
    n, m = 3001, 17
    A = T.Csr(*W.random_sym_csr(n, seed=n), mixed=mixed)
    A.set_spmv(lpr)
    x0 = W.start_vector(n, seed=1)
    coef = np.random.default_rng(2).standard_normal(m) * 0.1
    got = []
    for steps in (1, 6):
        print(f"lpr={lpr} mixed={mixed} steps={steps}", flush=True)
        c = T.Ctx(n, m + 8, mixed=mixed)
        got.append(lanczos(c, A, n, m, steps, x0 / np.linalg.norm(x0), coef))
        assert counts(T, c) == (0, 0)
        c.close()
    A.close()
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1])

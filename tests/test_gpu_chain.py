"""Chains of steps in one kernel (a single real solve on a stencil or
CSR-stream operator) against the batched kernels, which run every step as
kernels of their own: the same eigenvalues, vectors, residual estimates and
counters bit for bit, at sizes around the kernels' edges (256 rows a wave,
512 and 1024 a workgroup, 64 row blocks a reduction wave, ragged ends), and
with several solves on the device at once."""
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


def both(T, csr, mixed, lohi, ned, maxlan, tol=1e-8, maxmv=4000, seed=3):
    n = len(csr[0]) - 1
    A = T.Csr(*csr, mixed=mixed)
    args = (lohi, ned, maxlan, tol, 1, maxmv, ned)
    x0 = W.start_vector(n, seed=seed)
    print(f"n={n} mixed={mixed} stencil={A.stencil} packed={A.packed}", flush=True)
    one = T.solve_csr(A, *args, x0)
    rc, many, _ = T.solve_batch([(A,) + args + (x0,)])
    A.close()
    assert rc == 0
    same(one, many[0])


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("L", [16, 23, 32, 33, 45, 181, 182, 362, 363, 512, 513])
def test_chain_lattice2d(gpu_lib, L, mixed):
    both(gpu_lib, W.anderson2d_csr(L, 6.0, seed=L)[0], mixed, -1, 6, 24, maxmv=120 if L > 200 else 4000)


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
    both(gpu_lib, W.random_sym_csr(n, degree=degree, seed=n), mixed, 1, 10, 60, maxmv=130)


def test_chain_wide_basis(gpu_lib):
    """More basis columns than a chain kernel takes: its last steps of a
    cycle run as ordinary kernels."""
    both(gpu_lib, W.random_sym_csr(3001, seed=9), False, 1, 6, 200, maxmv=450)


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
    for A in ops:
        A.close()
    for a, b in zip(alone, got):
        same(a, b)

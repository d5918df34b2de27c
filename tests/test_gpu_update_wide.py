"""The Gram-Schmidt update with 1024 threads a block (cgs_pass, up to 262,144
rows) against the 256-thread update (trlhip_update with the same
coefficients), at ragged row counts and every remainder of the column groups:
the same vector and norm bit for bit for real bases.  The complex products of
the two kernels may be contracted differently (which of two products is
rounded first), so complex results agree to the rounding of m products and
sums a row: 2 (m + 2) eps of the row's magnitude, (n + 2) eps of the norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("complex_", [False, True])
@pytest.mark.parametrize("n", [1, 3, 255, 1023, 1025, 2050, 9003, 262144, 262145])
def test_wide_update_matches(gpu_lib, n, complex_):
    T = gpu_lib
    rng = np.random.default_rng(n)
    for m in ((1, 3, 4, 7, 8, 9, 14, 16, 23, 40) if n < 10000 else (9, 24)):
        print(f"n={n} m={m} complex={complex_}", flush=True)
        c = T.Ctx(n, m + 2, complex_=complex_)
        for j in range(m):
            v = rng.standard_normal(n) + (1j * rng.standard_normal(n) if complex_ else 0)
            c.set(j, v / np.sqrt(n))
        r = rng.standard_normal(n) + (1j * rng.standard_normal(n) if complex_ else 0)
        c.set(m, r)
        c.set(m + 1, r)
        h = c.proj(0, m, m)
        hh, rr2, h2 = c.cgs_pass(0, m, m)
        ref2 = c.update(0, m, h, m + 1)
        assert np.array_equal(h, h2)
        a, b = c.get(m), c.get(m + 1)
        if complex_:
            eps = np.finfo(float).eps
            V = np.stack([np.abs(c.get(j)) for j in range(m)], 1)
            assert (np.abs(a - b) <= 2 * (m + 2) * eps * (np.abs(r) + V @ np.abs(h))).all()
            assert abs(rr2 - ref2) <= (2 * (m + 2) + n) * eps * ref2
        else:
            assert rr2 == ref2
            assert np.array_equal(a, b)
        c.close()


@pytest.mark.parametrize("complex_,m", [(False, 4096), (False, 4097), (False, 6000), (False, 17500), (True, 2048),
                                        (True, 2049), (True, 8700)])
def test_update_long_basis(gpu_lib, complex_, m):
    """Coefficients up to and past what the wide update's LDS takes, up to
    those that fit the 256-thread update alone.  Bounds as above."""
    T = gpu_lib
    n = 130
    rng = np.random.default_rng(m)
    print(f"n={n} m={m} complex={complex_}", flush=True)
    V = rng.standard_normal((3, n)) + (1j * rng.standard_normal((3, n)) if complex_ else 0)
    r = rng.standard_normal(n) + (1j * rng.standard_normal(n) if complex_ else 0)
    c = T.Ctx(n, m + 1, complex_=complex_)
    cols = (0, m // 2, m - 1)  # the others stay zero
    for j, v in zip(cols, V):
        c.set(j, v / np.sqrt(n))
    c.set(m, r)
    hh, rr2, h = c.cgs_pass(0, m, m)
    got = c.get(m)
    c.close()
    Vn = V / np.sqrt(n)
    href = Vn.conj() @ r
    want = r - href @ Vn
    tol = 8 * (n + 8) * np.finfo(float).eps * np.abs(r).max() * 4
    assert np.count_nonzero(h) == 3
    assert np.abs(h[list(cols)] - href).max() <= tol * np.sqrt(n)
    assert np.abs(got - want).max() <= tol * np.sqrt(n)
    assert abs(hh - np.vdot(href, href).real) <= tol * np.sqrt(n) * 8 and abs(rr2 - np.vdot(want, want).real) <= tol * n * 4

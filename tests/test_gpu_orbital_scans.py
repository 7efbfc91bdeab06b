"""The scan forms of the Crank-Nicolson half step and the register
Gram-Schmidt where their shapes change: one to eight points per thread, the
first and last grid of each block width (256, 512, 1024 threads), zero and
periodic bounds, one to nine orbitals.  Crank-Nicolson (reference
split_linear_orbitals.c:335-373) against a sparse LU solve of the same system,
Gram-Schmidt against the oracle (reference calculus.c:170-191).

Bounds: the Crank-Nicolson matrix has condition number below 10 at the dt and
dx used, and either solve rounds a few times per row: 1e-12.  (The oracle's
periodic solve follows the reference's split gamma = b_0, whose zero first
pivot makes it divide by the off-diagonal entry twice; on these grids that
entry is 3e-4 to 0.1 of the diagonal and costs it up to 7 digits, 5e-11 on 6
points, so it does not bound this test.)  Gram-Schmidt
of nearly orthonormal functions: sums of up to 4097 terms at 1.1e-16, 1e-12."""
import numpy as np
import pytest

import gpu_util as gu
import inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import mctdhb_amd

    mctdhb_amd.lib()
    return mctdhb_amd


def _orb(M, x, periodic):
    orb = inputs.hermite_gauss(M, x, seed=5, noise=1e-2)
    if periodic:
        orb[:, -1] = orb[:, 0]
    return np.ascontiguousarray(orb.ravel())


GRIDS = [6, 65, 256, 257, 258, 512, 513, 768, 769, 1024, 1025, 1536, 1537, 2049, 2050, 3072, 3073, 4097]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("bounds", [1000, 1001])
@pytest.mark.parametrize("imagtime", [False, True])
def test_crank_nicolson_matches_oracle(amd, orc, grid, bounds, imagtime):
    import scipy.sparse as sp
    from scipy.sparse.linalg import splu

    M, dt, d1, d2 = 3, 0.004, 0.3j, -0.5
    x = np.linspace(-8, 8, grid)
    dx = (x[-1] - x[0]) / (grid - 1)
    periodic = bounds == 1001
    orb = _orb(M, x, periodic)
    # (1 + i p/2 T) new = (1 - i p/2 T) old, T = d2 D2 + d1 D1, p half the (imaginary-time) step
    m = grid - 1 if periodic else grid
    up, lo = d2 / dx ** 2 + d1 / (2 * dx), d2 / dx ** 2 - d1 / (2 * dx)
    T = sp.diags([np.full(m, -2 * d2 / dx ** 2), np.full(m - 1, up), np.full(m - 1, lo)], [0, 1, -1],
                 dtype=complex).tolil()
    if periodic:
        T[0, m - 1] += lo
        T[m - 1, 0] += up
    p = 0.5 * dt * dx * (-1j if imagtime else 1.0)
    one = sp.identity(m, dtype=complex)
    solve = splu((one + 0.5j * p * T).tocsc()).solve
    ref = orb.reshape(M, grid)[:, :m].T
    w = amd.DeviceOrbital(M, grid, x[0], x[-1], dt * dx, 1.0, 0.5 * x ** 2, imagtime=imagtime, bounds=bounds,
                          d1coef=d1)
    d = gu.dev(orb)
    for _ in range(2):
        ref = solve((one - 0.5j * p * T) @ ref)
        w.linear_cn(d)
    got = gu.host(d).reshape(M, grid)
    assert gu.rel_err(got[:, :m], ref.T) < 1e-12
    if periodic:
        assert np.array_equal(got[:, -1], got[:, 0])


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 9])
def test_gram_schmidt_matches_oracle(amd, orc, grid, M):
    if grid < 65 and M > 4:
        pytest.skip("more functions than the grid resolves")
    x = np.linspace(-8, 8, grid)
    w = amd.DeviceOrbital(M, grid, x[0], x[-1], 0.004, 1.0, 0.5 * x ** 2)
    ref = _orb(M, x, False)
    d = gu.dev(ref)
    orc.lib().orc_orthonormalize(grid, x[1] - x[0], M, ref)
    w.orthonormalize(d)
    assert gu.rel_err(gu.host(d), ref) < 1e-12

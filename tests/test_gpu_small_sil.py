"""The one-workgroup SIL step where it can go wrong: N = 1 (no pairs) and
N = 2 (one configuration of N - 2 particles), fewer chunks of configurations
than waves and just past whole ones, rows around the 512 and 1024 threads,
every place its vectors can be (all in LDS, psi in LDS, neither: by size and
by the number of vectors), 2 and 15 vectors, and the largest spaces it takes.

Bound: the step's recurrences and sums are FP64; at these sizes (sums of at
most 8192 terms, exp of a matrix of norm below 1) two orders of summation
agree to 1e-10."""
import math

import pytest

import gpu_util as gu
import inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd():
    import mctdhb_amd

    mctdhb_amd.lib()
    return mctdhb_amd


SIZES = [(1, 2, 2), (1, 5, 3), (1, 7, 4), (2, 2, 2), (2, 7, 6), (3, 6, 15), (511, 2, 5), (512, 2, 15), (1024, 2, 4),
         (4000, 2, 3), (30, 3, 4), (31, 3, 4), (43, 3, 5), (60, 3, 15), (126, 3, 3), (12, 4, 6), (13, 4, 6), (18, 4, 2),
         (34, 4, 4), (7, 5, 5), (8, 5, 15), (12, 5, 4), (18, 5, 3), (6, 6, 5), (9, 6, 4), (11, 6, 3), (5, 7, 5),
         (8, 7, 3), (9, 7, 3)]


@pytest.mark.parametrize("npar,norb,lm", SIZES)
@pytest.mark.parametrize("imag", [False, True])
def test_step_matches_oracle(amd, orc, npar, norb, lm, imag):
    dim = math.comb(npar + norb - 1, norb - 1)
    print(f"one workgroup N={npar} M={norb} NC={dim} lm={lm} imag={imag}", flush=True)
    assert dim <= 8192
    c, h, g = inputs.coefficients(dim, 3), inputs.onebody(norb, 3), inputs.twobody(norb, 3, 0.3)
    dt = 0.1 / npar ** 2 * (-1j if imag else 1.0)
    _, ref = orc.Space(npar, norb).sil_step(c, h, g, lm, dt, imag)
    D = amd.DeviceSpace(npar, norb, tables=False)
    sil = amd.DeviceSil(D, lm, prec=amd.FP64, index=amd.INDEX_FLY)
    dc = gu.dev(c)
    sil.step(dc, gu.dev(h), gu.dev(g), dt, imag)
    assert gu.rel_err(gu.host(dc), ref) < 1e-10
    sil.close()
    D.close()

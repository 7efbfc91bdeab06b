"""The multi-kernel SIL step on both sides of the block count up to which the
kernel behind the H.C adds its sums (512 blocks of 256 rows), on spaces of one
block, with one and two vectors before the last, and past the 15 vectors of
the register kernels.

Bounds: FP64 sums of at most 135,000 terms in two orders agree to 1e-10 after
the step; complex64 vectors carry 6e-8 each, below 2e-5 after it."""
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


# NC 130,816 (511 blocks), 131,328 (513), 129,766 (507), 134,044 (524; 491 of
# the last iteration's sums), 5, 330, 496
@pytest.mark.parametrize("npar,norb,lm", [(510, 3, 2), (511, 3, 3), (90, 4, 3), (91, 4, 3), (1, 5, 3), (4, 8, 4),
                                          (30, 3, 15), (30, 3, 18)])
@pytest.mark.parametrize("imag", [False, True])
@pytest.mark.parametrize("prec", [0, 1])
def test_step_matches_oracle(amd, orc, npar, norb, lm, imag, prec):
    if norb > 7 and prec == amd.MIXED:
        pytest.skip("more than seven orbitals are FP64")
    dim = math.comb(npar + norb - 1, norb - 1)
    print(f"sums N={npar} M={norb} NC={dim} lm={lm} imag={imag} prec={prec}", flush=True)
    c, h, g = inputs.coefficients(dim, 3), inputs.onebody(norb, 3), inputs.twobody(norb, 3, 0.3)
    dt = 0.1 / npar ** 2 * (-1j if imag else 1.0)
    _, ref = orc.Space(npar, norb).sil_step(c, h, g, lm, dt, imag)
    D = amd.DeviceSpace(npar, norb, tables=norb > 7)
    sil = amd.DeviceSil(D, lm, prec=prec, index=amd.INDEX_TABLES if norb > 7 else amd.INDEX_FLY)
    sil.set_small(False)
    dc = gu.dev(c)
    sil.step(dc, gu.dev(h), gu.dev(g), dt, imag)
    assert gu.rel_err(gu.host(dc), ref) < (1e-10 if prec == amd.FP64 else 2e-5)
    sil.close()
    D.close()

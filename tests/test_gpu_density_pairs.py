"""The pair-sum density kernel (2 <= M <= 7) where its plan changes: N = 1
(no pairs) and N = 2 (one configuration of N - 2 particles), one block and
the first size of two (1024 configurations of N - 2 particles), the last size
one block finishes and the first of the grid-wide finish (64 blocks of 512),
root table and computed roots (N + 3 > 2048), remainders of a pass in every
orbital count, and a rho1 that needs the regularisation.  Against the FP64
oracle (reference density_matrices.c:8-443, synchronize.c:41-56).

Bounds: FP64 sums of at most 6e4 products, rounded at 1.1e-16 each and
pairwise over lanes, waves and blocks, stay below 1e-13 of the largest
element; complex64 input is rounded at 6e-8 per coefficient, products and sums
are FP64, so the relative error of an element is below 2 x 6e-8 times the ratio
of the absolute sum to the sum, here at most 5: 1e-6.  rho1 is well conditioned
for random coefficients (largest over smallest occupation below 10 from
NC = 10 on)."""
import math

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


def _run(amd, npar, norb, c, prec, sync=True):
    D = amd.DeviceSpace(npar, norb, tables=False)
    r1, r2, ri = gu.empty(norb ** 2), gu.empty(norb ** 4), gu.empty(norb ** 2)
    src = gu.dev(c) if prec == amd.FP64 else gu.dev(c, np.complex64)
    for _ in range(2):  # the arrival count of the grid-wide finish is cleared
        r1.zero_(), r2.zero_(), ri.zero_()
        if sync:
            amd.density_sync(D, src, r1, r2, ri, prec=prec)
        else:
            D.density(src, r1, r2, prec=prec)
    out = gu.host(r1).reshape(norb, norb), gu.host(r2), gu.host(ri).reshape(norb, norb)
    D.close()
    return out


SHAPES = [(1, 2), (1, 7), (2, 2), (2, 5), (2, 7), (3, 6), (9, 4), (45, 3), (46, 3), (65, 2), (58, 4), (59, 4),
          (11, 6), (9, 7), (2045, 2), (2046, 2), (2100, 2)]


@pytest.mark.parametrize("npar,norb", SHAPES)
def test_pair_sums_match_oracle(amd, orc, npar, norb):
    dim = math.comb(npar + norb - 1, norb - 1)
    print(f"pair sums N={npar} M={norb} dim={dim}", flush=True)
    S = orc.Space(npar, norb)
    c = inputs.coefficients(dim, 29)
    ref1, ref2 = S.onebody_dm(c), S.twobody_dm(c)
    for prec, tol in ((amd.FP64, 1e-13), (amd.MIXED, 1e-6)):
        r1, r2, ri = _run(amd, npar, norb, c, prec, sync=dim >= 10)  # rho1 is singular at N = 1
        assert gu.rel_err(r1, ref1) < tol
        if npar > 1:
            assert gu.rel_err(r2, ref2) < tol
        else:
            assert not r2.any()
        if dim >= 10:
            assert np.max(np.abs(ri @ r1 - np.eye(norb))) < 1e-13


@pytest.mark.parametrize("npar,norb", [(6, 3), (50, 3), (60, 4), (4, 7)])
def test_singular_rho1_is_regularised(amd, orc, npar, norb):
    """One configuration: rho1 has empty natural orbitals, the inverse without
    regularisation does not exist and the eigenvalue path runs."""
    print(f"singular rho1 N={npar} M={norb}", flush=True)
    S = orc.Space(npar, norb)
    c = np.zeros(S.dim, complex)
    c[0] = 1
    ref1, ref2, refi = S.sync_density(c)
    r1, r2, ri = _run(amd, npar, norb, c, amd.FP64)
    assert gu.rel_err(r1, np.asarray(ref1).reshape(norb, norb)) < 1e-13
    assert gu.rel_err(r2, ref2) < 1e-13
    assert gu.rel_err(ri, np.asarray(refi).reshape(norb, norb)) < 1e-10


def test_overlapped_calls_leave_no_trace(amd):
    """Calls that overlap on one space share its sums, so their own results
    are not defined; a call after them counts from zero all the same."""
    import torch

    npar, norb = 18, 7  # 146 blocks: the grid-wide finish, in 406 blocks
    D = amd.DeviceSpace(npar, norb, tables=False)
    src, other = gu.dev(inputs.coefficients(D.dim, 31)), gu.dev(inputs.coefficients(D.dim, 37))
    r1, r2 = gu.empty(norb ** 2), gu.empty(norb ** 4)
    want = {}
    for c in (src, other):
        D.density(c, r1, r2)
        want[c] = gu.host(r1), gu.host(r2)
    # chains of calls on several streams, as graphs: launched close enough to overlap
    streams = [torch.cuda.Stream() for _ in range(4)]
    graphs, outs = [], []
    for _ in streams:
        a, b = gu.empty(norb ** 2), gu.empty(norb ** 4)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for _ in range(100):
                D.density(src, a, b, stream=torch.cuda.current_stream())
        graphs.append(g)
        outs.append((a, b))
    torch.cuda.synchronize()
    for _ in range(5):
        for st, g in zip(streams, graphs):
            with torch.cuda.stream(st):
                g.replay()
    torch.cuda.synchronize()
    for c in (other, src, other):
        r1.zero_(), r2.zero_()
        D.density(c, r1, r2)
        assert np.array_equal(gu.host(r1), want[c][0]) and np.array_equal(gu.host(r2), want[c][1])
    D.close()

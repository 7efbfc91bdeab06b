"""The two-stage H.C (M = 6, 7) where it can go wrong: N = 1 (no pairs: the
one-stage kernel), N = 2 (one configuration of N - 2 particles), sizes around
its 256-thread blocks, every call that takes it (product, prebuilt
coefficients), products on several streams and threads at once, which share
the space's scratch and keep their form, the one-stage form of a capturing
stream, and h and g
without the usual symmetries, where it must read the same entries as the
one-stage kernel.  The last Lanczos iteration's pair form of <w, H w> is
covered for every orbital count.

Bounds: FP64 sums of at most 504 products agree to 1e-12 of the largest
element.  In the mixed form psi and the result are complex64 (6e-8 each, some
30 values summed in FP64), below 1e-6 of the largest element."""
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


def _problem(npar, norb, symmetric=True):
    dim = math.comb(npar + norb - 1, norb - 1)
    if symmetric:
        return inputs.coefficients(dim, 3), inputs.onebody(norb, 3), inputs.twobody(norb, 3, 0.3)
    r = np.random.default_rng(8)
    z = lambda *s: r.standard_normal(s) + 1j * r.standard_normal(s)
    return inputs.coefficients(dim, 3), z(norb, norb), z(norb ** 4)


# NC' = C(N + M - 3, M - 1): 252 and 462 (M = 6), 210 and 462 (M = 7)
@pytest.mark.parametrize("npar,norb", [(1, 6), (1, 7), (2, 6), (2, 7), (3, 7), (7, 6), (8, 6), (6, 7), (7, 7)])
def test_product_matches_oracle(amd, orc, npar, norb):
    print(f"two-stage N={npar} M={norb}", flush=True)
    c, h, g = _problem(npar, norb)
    ref = orc.Space(npar, norb).apply_hamiltonian(c, h, g)
    D = amd.DeviceSpace(npar, norb, tables=False)
    dh, dg = gu.dev(h), gu.dev(g)
    for prec, dt, tol in ((amd.FP64, np.complex128, 1e-12), (amd.MIXED, np.complex64, 1e-6)):
        out = gu.empty(D.dim, np.dtype(dt).name)
        D.apply_hamiltonian(gu.dev(c, dt), dh, dg, out, prec=prec)
        assert gu.rel_err(gu.host(out), ref) < tol
        cf = gu.empty(D.coef_bytes(prec) // 8 + 1, "float64")
        D.hc_coefficients(dh, dg, cf, prec=prec)
        out2 = gu.empty(D.dim, np.dtype(dt).name)
        D.apply_hamiltonian_cf(gu.dev(c, dt), cf, out2, prec=prec)
        assert np.array_equal(gu.host(out2), gu.host(out))
    D.close()


@pytest.mark.parametrize("npar,norb", [(1, 6), (5, 6), (4, 7), (8, 5)])
def test_mixed_block_serves_fp64_products(amd, npar, norb):
    c, h, g = _problem(npar, norb)
    D = amd.DeviceSpace(npar, norb, tables=False)
    dc, dh, dg = gu.dev(c), gu.dev(h), gu.dev(g)
    outs = []
    for built in (amd.FP64, amd.MIXED):
        cf = gu.empty(D.coef_bytes(built) // 8 + 1, "float64")
        D.hc_coefficients(dh, dg, cf, prec=built)
        outs.append(gu.empty(D.dim))
        D.apply_hamiltonian_cf(dc, cf, outs[-1], prec=amd.FP64)
    assert np.array_equal(gu.host(outs[0]), gu.host(outs[1]))
    D.close()


@pytest.mark.parametrize("npar,norb", [(5, 6), (4, 7), (9, 6)])
def test_same_entries_of_h_and_g_as_the_one_stage_kernel(amd, npar, norb):
    c, h, g = _problem(npar, norb, symmetric=False)
    D = amd.DeviceSpace(npar, norb, tables=False)
    a, b = gu.empty(D.dim), gu.empty(D.dim)
    D.apply_hamiltonian(gu.dev(c), gu.dev(h), gu.dev(g), a)
    D.apply_hamiltonian_noalloc(gu.dev(c), gu.dev(h), gu.dev(g), b)  # one stage
    assert not np.array_equal(gu.host(a), gu.host(b))  # two kernels
    assert gu.rel_err(gu.host(a), gu.host(b)) < 1e-12
    D.close()


def test_products_on_two_streams_do_not_share_scratch(amd, orc):
    import torch

    npar, norb = 12, 6
    dim = math.comb(npar + norb - 1, norb - 1)
    h, g = inputs.onebody(norb, 3), inputs.twobody(norb, 3, 0.3)
    D = amd.DeviceSpace(npar, norb, tables=False)
    dh, dg = gu.dev(h), gu.dev(g)
    cs = [gu.dev(inputs.coefficients(dim, 20 + i)) for i in range(6)]
    ref = []
    for c in cs:
        o = gu.empty(dim)
        D.apply_hamiltonian(c, dh, dg, o)
        ref.append(gu.host(o))
    st = [torch.cuda.Stream() for _ in range(6)]  # more than the blocks kept
    outs = [gu.empty(dim) for _ in cs]
    torch.cuda.synchronize()
    for _ in range(20):
        for c, o, s in zip(cs, outs, st):
            D.apply_hamiltonian(c, dh, dg, o, stream=s)
    torch.cuda.synchronize()
    for o, r in zip(outs, ref):
        assert np.array_equal(gu.host(o), r)
    D.close()


@pytest.mark.parametrize("npar,norb", [(9, 2), (6, 5), (5, 6), (4, 7)])
@pytest.mark.parametrize("prec", [0, 1])
def test_coefficient_blocks_take_one_launch(amd, npar, norb, prec):
    """Kernels counted as the nodes of a captured graph: a block is built by
    one, a product on the fixed scratch is two (block and rows)."""
    import ctypes

    import torch

    c, h, g = _problem(npar, norb)
    D = amd.DeviceSpace(npar, norb, tables=False)
    src = gu.dev(c, np.complex128 if prec == amd.FP64 else np.complex64)
    dh, dg, out = gu.dev(h), gu.dev(g), torch.zeros_like(src)
    cf = gu.empty(D.coef_bytes(prec) // 8 + 1, "float64")

    def kernels(call):
        call(torch.cuda.current_stream())
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph):
            call(torch.cuda.current_stream())
        n = ctypes.c_size_t()
        assert gu.hip().hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(n)) == 0
        return n.value

    assert kernels(lambda st: D.hc_coefficients(dh, dg, cf, prec=prec, stream=st)) == 1
    assert kernels(lambda st: D.apply_hamiltonian_noalloc(src, dh, dg, out, prec=prec, stream=st)) == 2
    D.close()


def _reference_bits(amd, npar, norb, cs, dh, dg, prec):
    """Products one at a time on a space of their own, and one-stage ones,
    whose bits differ."""
    D = amd.DeviceSpace(npar, norb, tables=False)
    out = []
    for c in cs:
        a, b = gu.empty(D.dim, str(c.dtype)[6:]), gu.empty(D.dim, str(c.dtype)[6:])
        D.apply_hamiltonian(c, dh, dg, a, prec=prec)
        D.apply_hamiltonian_noalloc(c, dh, dg, b, prec=prec)
        assert not np.array_equal(gu.host(a), gu.host(b))
        out.append(gu.host(a))
    D.close()
    return out


def test_form_does_not_depend_on_the_scratch_in_use(amd):
    """Blocks of the mixed form, as many as a space keeps and all in flight,
    do not keep FP64 products (larger blocks) off the two-stage form."""
    import torch

    npar, norb = 12, 6
    h, g = inputs.onebody(norb, 3), inputs.twobody(norb, 3, 0.3)
    dh, dg = gu.dev(h), gu.dev(g)
    c = gu.dev(inputs.coefficients(math.comb(npar + norb - 1, norb - 1), 20))
    c32 = c.to(torch.complex64)
    ref, = _reference_bits(amd, npar, norb, [c], dh, dg, amd.FP64)
    ref32, = _reference_bits(amd, npar, norb, [c32], dh, dg, amd.MIXED)
    D = amd.DeviceSpace(npar, norb, tables=False)
    st = [torch.cuda.Stream() for _ in range(6)]
    small, full = [torch.zeros_like(c32) for _ in st], [torch.zeros_like(c) for _ in st]
    torch.cuda.synchronize()
    for prec, src, outs in ((amd.MIXED, c32, small), (amd.FP64, c, full), (amd.MIXED, c32, small)):
        for s, o in zip(st, outs):
            with torch.cuda.stream(s):
                torch.cuda._sleep(50_000_000)  # some 20 ms: the block stays in flight
            D.apply_hamiltonian(src, dh, dg, o, prec=prec, stream=s)
    torch.cuda.synchronize()
    for o in full:
        assert np.array_equal(gu.host(o), ref)
    for o in small:
        assert np.array_equal(gu.host(o), ref32)
    D.close()


def test_form_does_not_depend_on_other_threads(amd):
    import threading

    import torch

    npar, norb, threads, rounds = 9, 7, 8, 40
    h, g = inputs.onebody(norb, 3), inputs.twobody(norb, 3, 0.3)
    dh, dg = gu.dev(h), gu.dev(g)
    dim = math.comb(npar + norb - 1, norb - 1)
    cs = [gu.dev(inputs.coefficients(dim, 40 + i)) for i in range(threads)]
    ref = _reference_bits(amd, npar, norb, cs, dh, dg, amd.FP64)
    D = amd.DeviceSpace(npar, norb, tables=False)
    st = [torch.cuda.Stream() for _ in range(threads)]
    outs = [[torch.zeros_like(cs[0]) for _ in range(rounds)] for _ in range(threads)]
    torch.cuda.synchronize()
    go, failed = threading.Barrier(threads), []

    def work(i):
        try:
            for r in range(rounds):
                go.wait(60)
                D.apply_hamiltonian(cs[i], dh, dg, outs[i][r], stream=st[i])
        except Exception as e:  # noqa: BLE001
            failed.append(e)
            go.abort()

    pool = [threading.Thread(target=work, args=(i,)) for i in range(threads)]
    for t in pool:
        t.start()
    for t in pool:
        t.join()
    assert not failed
    torch.cuda.synchronize()
    for i in range(threads):
        for o in outs[i]:
            assert np.array_equal(gu.host(o), ref[i])
    D.close()


def test_captured_product_matches_oracle(amd, orc):
    """A capturing stream takes the one-stage kernels: its graph keeps no
    scratch of the space."""
    import torch

    npar, norb = 8, 6
    c, h, g = _problem(npar, norb)
    D = amd.DeviceSpace(npar, norb, tables=False)
    dc, dh, dg, out, cf = gu.dev(c), gu.dev(h), gu.dev(g), gu.empty(D.dim), gu.empty(D.coef_bytes(amd.FP64) // 8, "float64")
    D.hc_coefficients(dh, dg, cf)
    D.apply_hamiltonian_cf(dc, cf, out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        D.apply_hamiltonian_cf(dc, cf, out, stream=torch.cuda.current_stream())
    S = orc.Space(npar, norb)
    for seed in (3, 4, 5):
        dc.copy_(gu.dev(inputs.coefficients(D.dim, seed)))
        eager = gu.empty(D.dim)
        D.apply_hamiltonian_cf(dc, cf, eager)  # eager work between the replays
        out.zero_()
        graph.replay()
        ref = S.apply_hamiltonian(inputs.coefficients(D.dim, seed), h, g)
        assert gu.rel_err(gu.host(out), ref) < 1e-12 and gu.rel_err(gu.host(eager), ref) < 1e-12
    del graph
    D.close()


@pytest.mark.parametrize("npar,norb,lm", [(2, 2, 3), (9, 2, 5), (12, 3, 6), (10, 4, 5), (9, 5, 4), (7, 6, 6),
                                          (5, 7, 5), (1, 6, 4)])
@pytest.mark.parametrize("imag", [False, True])
@pytest.mark.parametrize("prec", [0, 1])
def test_sil_step_matches_oracle(amd, orc, npar, norb, lm, imag, prec):
    print(f"two-stage sil N={npar} M={norb} lm={lm} imag={imag} prec={prec}", flush=True)
    c, h, g = _problem(npar, norb)
    dt = -0.01j if imag else 0.01
    _, ref = orc.Space(npar, norb).sil_step(c, h, g, lm, dt, imag)
    D = amd.DeviceSpace(npar, norb, tables=False)
    sil = amd.DeviceSil(D, lm, prec=prec, index=amd.INDEX_FLY)
    sil.set_small(False)
    dc = gu.dev(c)
    sil.step(dc, gu.dev(h), gu.dev(g), dt, imag)
    assert gu.rel_err(gu.host(dc), ref) < (1e-10 if prec == amd.FP64 else 2e-5)
    sil.close()
    D.close()


def test_tiling_names_the_form(amd):
    D6, D5 = amd.DeviceSpace(6, 6, tables=False), amd.DeviceSpace(6, 5, tables=False)
    assert D6.hc_tiling(3) == 3 and D6.hc_tiling(0) == 0
    with pytest.raises(amd.MctdhbError):
        D5.hc_tiling(3)
    D6.close()
    D5.close()


def test_open_workspace_keeps_its_form_when_the_tiling_changes(amd, orc):
    npar, norb, lm = 9, 6, 5
    c, h, g = _problem(npar, norb)
    _, ref = orc.Space(npar, norb).sil_step(c, h, g, lm, 0.01, False)
    D = amd.DeviceSpace(npar, norb, tables=False)
    for made, later in ((3, 1), (3, 0), (1, 3), (0, 1)):
        D.hc_tiling(made)
        sil = amd.DeviceSil(D, lm, prec=amd.MIXED, index=amd.INDEX_FLY)
        D.hc_tiling(later)
        dc = gu.dev(c)
        sil.step(dc, gu.dev(h), gu.dev(g), 0.01, False)
        assert gu.rel_err(gu.host(dc), ref) < 2e-5, (made, later)
        sil.close()
    D.close()

"""GPU tests of the single-vector solvers (the reference's single-mode operators, the Ritz bounds) and of
the batched multi-shift CG against the oracle, at the sizes where their launches can go wrong: fewer
sites than half a wavefront, a last wavefront and a last workgroup that are partly filled, uneven
extents, one and several modes.

Tolerances: the stencil sums 6 x 2 x Nc products per component, so its rounding stays within 1e-13 of
the largest entry; the CG stops at ||r|| <= 1e-8 and the Ritz values are Rayleigh quotients whose error
is the square of the vector's, both 1e-9."""
import numpy as np
import pytest

import orc
from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu

SHAPES = [(2, (3, 3, 3)), (3, (3, 4, 3)), (2, (5, 7, 3)), (3, (4, 4, 4)), (2, (8, 8, 5)), (3, (11, 3, 9))]


def rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def problem(nc, n, seed, M):
    g = cf.rng(seed)
    links = cf.su2_links(n, 0.3, g) if nc == 2 else cf.su3_links(n, 0.25, g)
    phi = cf.spinors(n, nc, 1, g)[0]
    L = orc.lat(nc, n, 1.0, 0.1, M)
    return L, links, orc.links_to_ucc(L, links, orc.u1_phases(n, 1, 1.0)), phi


@pytest.mark.parametrize("nc,n", SHAPES)
def test_single_mode_operators(gpu, nc, n):
    print(f"[case] single-mode operators nc={nc} n={n}", flush=True)
    L, _, ucc, phi = problem(nc, n, 500 + nc + n[0], 1.0)
    with ovl.Context(nc, n, 1, m_fermion=0.1, m_dw=1.0) as ctx:
        for _ in range(2):  # the second call finds the work buffers as the first left them
            assert rel(ctx.wilson_evo_compute(ucc, phi), orc.wilson_evo(L, ucc, phi)) <= 1e-13
            out = ctx.overlap_operator_compute(ucc, phi, 0.2, 30.0)
            assert rel(out, orc.overlap_evo_zolo(L, ucc, phi, 0.2, 30.0)[0]) <= 1e-9
        zero = ctx.overlap_operator_compute(ucc, 0 * phi, 0.2, 30.0)
        assert not np.any(zero)


@pytest.mark.parametrize("nc,n", SHAPES)
def test_ritz_bounds(gpu, nc, n):
    print(f"[case] Ritz nc={nc} n={n}", flush=True)
    L, links, ucc, _ = problem(nc, n, 600 + nc + n[0], 1.0)
    start = cf.rng(7).uniform(size=int(np.prod(n)) * 4 * nc).astype(complex)
    start /= np.linalg.norm(start)
    with ovl.Context(nc, n, 1, m_fermion=0.1, m_dw=1.0) as ctx:
        ctx.set_links(links)
        ctx.set_u1_flux(1, 1.0)
        # 40 iterations are within the convergence of both; restarts at odd and even iterations, an
        # iteration cap inside a batch of launches, a single iteration
        for sign, nrestart, nitlz in ((1.0, 100, 2000), (-1.0, 100, 300), (1.0, 7, 400)):
            want = orc.ritz(L, ucc, start, sign=sign, nrestart=nrestart, nitlz=nitlz)
            got = ctx.ritz(start, sign, nitlz=nitlz, nrestart=nrestart)
            assert abs(got - want) <= 1e-9 * max(abs(want), 1.0), (sign, nrestart, nitlz, got, want)
        for nitlz in (1, 5):
            want = orc.ritz(L, ucc, start, sign=1.0, nrestart=3, nitlz=nitlz)
            got = ctx.ritz(start, 1.0, nitlz=nitlz, nrestart=3)
            assert abs(got - want) <= 1e-9 * max(abs(want), 1.0), (nitlz, got, want)


@pytest.mark.parametrize("nc,n,nm,mb", [(2, (3, 3, 3), 1, 16), (3, (3, 5, 4), 33, 32), (2, (4, 3, 5), 70, 64)])
def test_batched_zolotarev(gpu, nc, n, nm, mb):
    # one mode in a block, a partly filled second block, and a zero mode that has nothing to solve
    print(f"[case] batched zolotarev nc={nc} n={n} modes={nm} mb={mb}", flush=True)
    L, links, ucc, _ = problem(nc, n, 700 + nm, 1.0)
    psi = cf.spinors(n, nc, nm, cf.rng(9))
    psi[nm // 2] *= 0.0 if nm > 1 else 1.0
    with ovl.Context(nc, n, nm, m_fermion=0.1, m_dw=1.0, mode_block=mb) as ctx:
        ctx.set_links(links)
        ctx.set_u1_flux(1, 1.0)
        ctx.set_modes(ovl.PSI, psi)
        ctx.apply_overlap(ovl.PSI, ovl.PSIMID, ovl.sign_opts(method=ovl.SIGN_ZOLOTAREV, lmin=0.2, lmax=30.0))
        out = ctx.get_modes(ovl.PSIMID)
    for k in range(nm):
        if np.any(psi[k]):
            assert rel(out[k], orc.overlap_evo_zolo(L, ucc, psi[k], 0.2, 30.0)[0]) <= 1e-9, k
        else:
            assert not np.any(out[k])

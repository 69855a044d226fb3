"""GPU tests of the Zolotarev sign with its own spectral interval (lmin = lmax = 0): both Ritz bounds advance in the
same launches, their iterations replayed as a graph that the context keeps.  The same call with the interval
from two single solves of the oracle has to give the same result, on the links at hand: the context is used again
after its links changed, and for leapfrog steps that move them.

Tolerances: the bounds are 1.05 and 0.95 times Rayleigh quotients that agree to 1e-9; the sign hardly depends on
its interval (a wider or narrower one moves the 25 poles by as much, the approximation stays within 1e-8 in it)
and the CG stops at ||r|| <= 1e-8, so the results agree to 1e-8."""
import numpy as np
import pytest

import orc
from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu


def start_vector(n, nc):
    """The library's fixed start: xorshift64 uniforms, normalised (re, im of flat entry m = s + V (spin + 4 colour))."""
    st, out, mask = 0x9E3779B97F4A7C15, [], (1 << 64) - 1
    for _ in range(2 * int(np.prod(n)) * 4 * nc):
        st = (st ^ (st << 13)) & mask
        st ^= st >> 7
        st = (st ^ (st << 17)) & mask
        out.append((st >> 11) * 2.0 ** -53)
    v = np.array(out).view(complex)
    return v / np.linalg.norm(v)


def interval(L, ucc, v):
    lmax = -1.05 * orc.ritz(L, ucc, v, sign=-1.0, nrestart=100, nitlz=2000)
    return 0.95 * orc.ritz(L, ucc, v, sign=1.0, nrestart=100, nitlz=2000), lmax


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("nc,n,nm", [(2, (4, 4, 4), 3), (2, (5, 7, 3), 17), (3, (4, 4, 6), 5), (3, (3, 5, 4), 1)])
def test_own_interval(gpu, nc, n, nm):
    print(f"[case] Ritz interval nc={nc} n={n} modes={nm}", flush=True)
    L = orc.lat(nc, n, 1.0, 0.1, 1.0)
    v = start_vector(n, nc)
    phases = orc.u1_phases(n, 1, 1.0)
    own = ovl.sign_opts(method=ovl.SIGN_ZOLOTAREV, lmin=0.0, lmax=0.0)
    with ovl.Context(nc, n, nm, m_fermion=0.1, m_dw=1.0) as ctx:
        ctx.set_u1_flux(1, 1.0)
        for k in range(3):  # new links each time: the kept graph and start vector hold nothing of the last ones
            g = cf.rng(900 + 10 * nc + n[0] + k)
            links = cf.su2_links(n, 0.2 + 0.15 * k, g) if nc == 2 else cf.su3_links(n, 0.2 + 0.15 * k, g)
            psi = cf.spinors(n, nc, nm, g)
            ctx.set_links(links)
            ctx.set_modes(ovl.PSI, psi)
            ctx.apply_overlap(ovl.PSI, ovl.PSIMID, own)
            out = ctx.get_modes(ovl.PSIMID)
            ucc = orc.links_to_ucc(L, links, phases)
            lmin, lmax = interval(L, ucc, v)
            given = ovl.sign_opts(method=ovl.SIGN_ZOLOTAREV, lmin=lmin, lmax=lmax)
            ctx.apply_overlap(ovl.PSI, ovl.PSIMID, given)
            assert rel(out, ctx.get_modes(ovl.PSIMID)) <= 1e-8, k
            assert rel(out[0], orc.overlap_evo_zolo(L, ucc, psi[0], lmin, lmax)[0]) <= 1e-8, k


@pytest.mark.parametrize("nc,n,nm", [(2, (4, 5, 4), 4), (3, (4, 3, 4), 2)])
def test_leapfrog_with_own_interval(gpu, nc, n, nm):
    print(f"[case] leapfrog with Ritz intervals nc={nc} n={n} modes={nm}", flush=True)
    L = orc.lat(nc, n, 1.0, 0.1, 1.0)
    g = cf.rng(950 + nc)
    links = cf.su2_links(n, 0.3, g) if nc == 2 else cf.su3_links(n, 0.3, g)
    e, psi, mid = cf.efield(n, nc, 0.3, g), cf.spinors(n, nc, nm, g), cf.spinors(n, nc, nm, g)
    dt = 0.05
    with ovl.Context(nc, n, nm, m_fermion=0.1, m_dw=1.0) as ctx:
        ctx.set_links(links)
        ctx.set_efield(e)
        ctx.set_modes(ovl.PSI, psi)
        ctx.set_modes(ovl.PSIMID, mid)
        own = ovl.sign_opts(method=ovl.SIGN_ZOLOTAREV, lmin=0.0, lmax=0.0)
        ctx.fermion_update(ovl.StepOpts(kind=ovl.OVERLAP, dt=dt, gauge=ovl.GAUGE_LINKS, sign=own), 2)
        got = [ctx.get_modes(ovl.PSI), ctx.get_modes(ovl.PSIMID), ctx.get_links()]
    v = start_vector(n, nc)
    u, a, b = links, psi.copy(), mid.copy()
    for _ in range(2):
        for src, tgt in ((b, a), (a, b)):
            ucc = orc.links_to_ucc(L, u)
            lmin, lmax = interval(L, ucc, v)
            for k in range(nm):
                tgt[k] += dt * orc.overlap_evo_zolo(L, ucc, src[k], lmin, lmax)[0]
            u = orc.update_links(L, u, e, dt / 2)
    for x, want in zip(got, (a, b, u)):
        assert rel(x, want) <= 1e-8

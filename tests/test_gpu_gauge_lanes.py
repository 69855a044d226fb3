"""GPU tests of the link and E-field updates on both sides of the lattice sizes where a link changes from four lanes
to one: against the oracle, and the leapfrog's half steps (their own launches, and the launches that
they share with the stencil) against the single updates.

Tolerance: matrix products of numbers of order one, 1e-13; the leapfrog's updates do the same arithmetic as the
single ones in launches of their own, so they may differ by the last bits only."""
import numpy as np
import pytest

import orc
from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu

# 3 V links: SU(2) E fields turn at 16384, SU(3) links at 90000, with the stencil links at 200000
CASES = [(2, (15, 14, 26)), (2, (15, 14, 27)), (2, (31, 33, 17)), (3, (30, 31, 32)), (3, (31, 31, 32)), (3, (40, 41, 41))]


@pytest.mark.parametrize("nc,n", CASES)
def test_updates(gpu, nc, n):
    print(f"[case] gauge updates nc={nc} n={n}", flush=True)
    g = cf.rng(820 + nc + sum(n))
    links = cf.su2_links(n, 0.5, g) if nc == 2 else cf.su3_links(n, 0.5, g)
    e = cf.efield(n, nc, 0.3, g)
    L = orc.lat(nc, n)
    dt = 0.06
    with ovl.Context(nc, n, 1, m_fermion=0.1, reunitarize=0) as ctx:
        for step in (0.03, 2.0):  # without and with squarings of the exponential
            ctx.set_links(links)
            ctx.set_efield(e)
            ctx.update_links(step)
            want = orc.update_links(L, links, e, step)
            assert np.abs(ctx.get_links() - want).max() <= 1e-13 * np.abs(want).max()
        ctx.set_links(links)
        ctx.update_efield(dt / 2)
        e1 = ctx.get_efield()
        assert np.abs(e1 - orc.efield_update(L, links, e, dt / 2)).max() <= 1e-13
        # one leapfrog step: E, U, E, U by dt / 2 each
        ctx.update_links(dt / 2)
        ctx.update_efield(dt / 2)
        ctx.update_links(dt / 2)
        u2, e2 = ctx.get_links(), ctx.get_efield()
        for kind in (ovl.WILSON, ovl.OVERLAP):
            ctx.set_links(links)
            ctx.set_efield(e)
            o = ovl.StepOpts(kind=kind, dt=dt, gauge=ovl.GAUGE_FULL, sign=ovl.sign_opts(degree=2, cut=0.5))
            ctx.fermion_update(o, 1)
            assert np.abs(ctx.get_links() - u2).max() <= 1e-14 * np.abs(u2).max()
            assert np.abs(ctx.get_efield() - e2).max() <= 1e-14


def test_reunitarised_links_in_one_lane(gpu):
    n = (31, 31, 32)
    g = cf.rng(83)
    links, e = cf.su3_links(n, 0.5, g), cf.efield(n, 3, 0.3, g)
    L = orc.lat(3, n)
    with ovl.Context(3, n, 1, reunitarize=1) as ctx:
        ctx.set_links(links * (1.0 + 1e-9))
        ctx.set_efield(e)
        ctx.update_links(0.03)
        assert ctx.unitarity_violation()[0] <= 1e-13
        want = orc.update_links(L, links, e, 0.03)
        assert np.abs(ctx.get_links() - want).max() <= 1e-13 * np.abs(want).max()

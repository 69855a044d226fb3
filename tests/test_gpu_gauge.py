"""GPU tests of the gauge kernels against the oracle at the shapes where their lanes can go wrong: extents
of 3 (two-site paths that wrap on both sides), fewer pairs than a wavefront holds, a last workgroup that
is partly filled, more pairs than one pass of the grid, and links off the group (the loops multiply
every link they pass, also back and forth).

Tolerances: a value of a site is a sum of at most a few hundred products of entries of size one, each
within 2e-16, so 1e-13 per site for the sums over sites and 1e-13 of the largest entry for fields."""
import numpy as np
import pytest

import orc
from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 3), (3, 4, 5), (7, 3, 4), (8, 8, 8), (5, 11, 6), (32, 24, 20)]


@pytest.mark.parametrize("nc", [2, 3])
@pytest.mark.parametrize("n", SHAPES)
def test_observables_and_updates(gpu, nc, n):
    print(f"[case] gauge kernels nc={nc} n={n}", flush=True)
    g = cf.rng(800 + nc + sum(n))
    V = int(np.prod(n))
    links = cf.su2_links(n, 0.5, g) if nc == 2 else cf.su3_links(n, 0.5, g)
    per = 4 if nc == 2 else 18
    off = (links.reshape(-1, per) * (1.0 + g.normal(0, 1e-2, size=(3 * V, 1)))).reshape(-1)
    e = cf.efield(n, nc, 0.3, g)
    L = orc.lat(nc, n)
    with ovl.Context(nc, n, 1) as ctx:
        for u in (links, off):
            ctx.set_links(u)
            ctx.set_efield(e)
            o = ctx.system_observables(0)
            el, mag = orc.plaquette_energy(L, u, e)
            assert abs(o["e_el"] - el) <= 1e-13 * V and abs(o["e_mag"] - mag) <= 1e-13 * 3 * V
            gmax, grms = orc.gauss_violation(L, u, e)
            assert abs(o["gauss_max"] - gmax) <= 1e-13 and abs(o["gauss_rms"] - grms) <= 1e-13
            umax, urms = orc.unitarity_violation(L, u)
            assert abs(o["unit_max"] - umax) <= 1e-13 and abs(o["unit_rms"] - urms) <= 1e-13
            assert abs(o["ncs_dot"] * 8 * np.pi ** 2 - orc.edotb(L, u, e)) <= 1e-13 * 3 * V
            # the calls that ask for some of them run the same sums
            assert ctx.energy() == (o["e_el"], o["e_mag"]) and ctx.ncs_dot() == o["ncs_dot"]
            assert ctx.gauss_violation() == (o["gauss_max"], o["gauss_rms"])
            assert ctx.unitarity_violation() == (o["unit_max"], o["unit_rms"])
            for dt in (0.03, 2.0):  # without and with squarings of the exponential
                ctx.set_links(u)
                ctx.update_links(dt)
                want = orc.update_links(L, u, e, dt)
                assert np.abs(ctx.get_links() - want).max() <= 1e-13 * np.abs(want).max()
            ctx.set_links(u)
            ctx.update_efield(0.03)
            assert np.abs(ctx.get_efield() - orc.efield_update(L, u, e, 0.03)).max() <= 1e-13


@pytest.mark.parametrize("nc", [2, 3])
def test_half_step_writes_the_stencil_links(gpu, nc):
    # the leapfrog's link update also writes the stencil links with their phases: the Wilson operator after a
    # step equals the one of a context that derives them from the moved links
    n = (5, 3, 7)
    g = cf.rng(77 + nc)
    links = cf.su2_links(n, 0.4, g) if nc == 2 else cf.su3_links(n, 0.4, g)
    e, psi = cf.efield(n, nc, 0.2, g), cf.spinors(n, nc, 5, g)
    outs = []
    with ovl.Context(nc, n, 5, m_fermion=0.1) as a, ovl.Context(nc, n, 5, m_fermion=0.1) as b:
        for nb in (2, 0):
            a.set_links(links)
            a.set_efield(e)
            a.set_u1_flux(nb, 1.0)
            for f in (ovl.PSI, ovl.PSIMID):
                a.set_modes(f, psi)
            a.fermion_update(ovl.StepOpts(kind=ovl.WILSON, dt=0.05, gauge=ovl.GAUGE_FULL, sign=ovl.sign_opts()), 3)
            b.set_links(a.get_links())
            b.set_u1_flux(nb, 1.0)
            for c in (a, b):
                c.set_modes(ovl.PSI, psi)
                c.apply_wilson(ovl.PSI, ovl.SCRATCH)
            outs = [c.get_modes(ovl.SCRATCH) for c in (a, b)]
            assert np.array_equal(outs[0], outs[1])

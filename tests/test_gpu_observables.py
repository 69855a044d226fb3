"""GPU tests of the observables where their launches change: the sites of one, of all and of more shares than
the local pass has (64 sites each, 1024 shares at most, taken by 256 workgroups in the launch for all), against the
oracle, and the calls for one quantity against the call for all.

Tolerances: sums of V terms of order one, 1e-13 a term; largest values 1e-13."""
import numpy as np
import pytest

import orc
from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc", [2, 3])
@pytest.mark.parametrize("n", [(4, 4, 4), (5, 13, 3), (24, 24, 29), (40, 34, 48), (31, 46, 47)])
def test_one_quantity_and_all(gpu, nc, n):
    print(f"[case] observables nc={nc} n={n}", flush=True)
    g = cf.rng(810 + nc + sum(n))
    V = int(np.prod(n))
    links = cf.su2_links(n, 0.5, g) if nc == 2 else cf.su3_links(n, 0.5, g)
    per = 4 if nc == 2 else 18
    links = (links.reshape(-1, per) * (1.0 + g.normal(0, 1e-2, size=(3 * V, 1)))).reshape(-1)
    e = cf.efield(n, nc, 0.3, g)
    L = orc.lat(nc, n)
    with ovl.Context(nc, n, 1) as ctx:
        ctx.set_links(links)
        ctx.set_efield(e)
        o = ctx.system_observables(0)
        el, mag = orc.plaquette_energy(L, links, e)
        assert abs(o["e_el"] - el) <= 1e-13 * V and abs(o["e_mag"] - mag) <= 1e-13 * 3 * V
        gmax, grms = orc.gauss_violation(L, links, e)
        assert abs(o["gauss_max"] - gmax) <= 1e-13 and abs(o["gauss_rms"] - grms) <= 1e-13
        umax, urms = orc.unitarity_violation(L, links)
        assert abs(o["unit_max"] - umax) <= 1e-13 and abs(o["unit_rms"] - urms) <= 1e-13
        assert abs(o["ncs_dot"] * 8 * np.pi ** 2 - orc.edotb(L, links, e)) <= 1e-13 * 3 * V
        for _ in range(2):
            assert ctx.energy() == (o["e_el"], o["e_mag"]) and ctx.ncs_dot() == o["ncs_dot"]
            assert ctx.gauss_violation() == (o["gauss_max"], o["gauss_rms"])
            assert ctx.unitarity_violation() == (o["unit_max"], o["unit_rms"])
            assert ctx.system_observables(0) == o

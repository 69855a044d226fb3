"""GPU test of the stencil's lane orders on lattices that do not split evenly: site counts that are odd, not a
multiple of a workgroup or of the eight XCDs, fewer workgroups than XCDs, boxes whose lanes end inside a
workgroup.  A lane order only moves work, so the results are those of the lexicographic order bit for
bit, and the first mode agrees with the oracle (FP64 stencil rounding, 1e-13)."""
import numpy as np
import pytest

import orc
from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,n,nm,mb", [(2, (3, 3, 3), 1, 16), (3, (5, 7, 3), 33, 0), (2, (4, 4, 4), 5, 16),
                                        (3, (15, 12, 10), 24, 0), (2, (13, 11, 9), 20, 16), (3, (6, 10, 14), 70, 64),
                                        (3, (11, 14, 9), 40, 32), (2, (2 * 8, 3, 5), 64, 64)])
def test_lane_orders_on_ragged_lattices(gpu, nc, n, nm, mb):
    print(f"[case] lane orders nc={nc} n={n} modes={nm} mb={mb}", flush=True)
    g = cf.rng(1200 + sum(n) + nm)
    links = cf.su2_links(n, 0.4, g) if nc == 2 else cf.su3_links(n, 0.4, g)
    e, psi = cf.efield(n, nc, 0.2, g), cf.spinors(n, nc, nm, g)
    outs = []
    for trav in (1, 0, 2, 3):
        with ovl.Context(nc, n, nm, m_fermion=0.1, m_dw=1.2, mode_block=mb, traversal=trav) as ctx:
            ctx.set_links(links)
            ctx.set_efield(e)
            ctx.set_modes(ovl.PSI, psi)
            ctx.set_modes(ovl.PSIMID, psi)
            ctx.apply_wilson(ovl.PSI, ovl.SCRATCH)
            res = [ctx.get_modes(ovl.SCRATCH)]
            ctx.apply_sign(ovl.PSI, ovl.SCRATCH,
                           ovl.sign_opts(degree=24, cut=0.1, precision=ovl.PREC_MIXED, head=8, head16=16, guard=0))
            res.append(ctx.get_modes(ovl.SCRATCH))
            for prec in (ovl.PREC_FP64, ovl.PREC_FP32):
                for gauge in (ovl.GAUGE_FROZEN, ovl.GAUGE_LINKS, ovl.GAUGE_FULL):
                    ctx.fermion_update(ovl.StepOpts(kind=ovl.WILSON, dt=0.04, gauge=gauge,
                                                    sign=ovl.sign_opts(precision=prec), use_graph=1), 2)
                    res += [ctx.get_modes(ovl.PSI), ctx.get_modes(ovl.PSIMID), ctx.get_links(), ctx.get_efield()]
            outs.append(res)
    for res in outs[1:]:
        for a, b in zip(res, outs[0]):
            assert np.array_equal(a, b)
    L = orc.lat(nc, n, 1.0, 0.1, 1.2)
    want = orc.wilson_evo(L, orc.links_to_ucc(L, links), psi[0])
    assert np.abs(outs[0][0][0] - want).max() <= 1e-13 * np.abs(want).max()

"""GPU test of the XCD boxes on lattices of small extents, where the split avoids boxes thinner than three sites (from
512 workgroups on) or cannot: a box order only moves work, so the results are those of the lexicographic order bit for bit."""
import numpy as np
import pytest

from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc,n,nm", [(2, (8, 8, 8), 70), (2, (8, 8, 8), 256), (3, (8, 8, 16), 128), (3, (8, 8, 16), 16), (2, (8, 16, 8), 40), (2, (16, 8, 8), 5),
                                     (3, (4, 4, 4), 20), (2, (4, 8, 3), 64), (3, (3, 4, 8), 33), (2, (12, 12, 12), 20),
                                     (3, (6, 6, 6), 64)])
def test_boxes_keep_the_bits(gpu, nc, n, nm):
    print(f"[case] boxes nc={nc} n={n} modes={nm}", flush=True)
    g = cf.rng(1300 + sum(n) + nm)
    links = cf.su2_links(n, 0.4, g) if nc == 2 else cf.su3_links(n, 0.4, g)
    psi = cf.spinors(n, nc, nm, g)
    outs = []
    for trav, slabs in ((1, 1), (2, 1), (2, 2)):
        with ovl.Context(nc, n, nm, m_fermion=0.1, m_dw=1.2) as ctx:
            for p in range(4):
                t = ctx.get_tuning(p)
                ctx.set_tuning(p, trav, slabs, t.nt_store, t.waves_per_eu)
                assert ctx.get_tuning(p).traversal == trav
            ctx.set_links(links)
            ctx.set_modes(ovl.PSI, psi)
            ctx.apply_wilson(ovl.PSI, ovl.SCRATCH)
            res = [ctx.get_modes(ovl.SCRATCH)]
            for o in (ovl.sign_opts(degree=24, cut=0.1, precision=ovl.PREC_MIXED, head=12, head48=6, head16=18, guard=0),
                      ovl.sign_opts(degree=8, cut=0.1, precision=ovl.PREC_FP32)):
                ctx.apply_sign(ovl.PSI, ovl.SCRATCH, o)
                res.append(ctx.get_modes(ovl.SCRATCH))
            outs.append(res)
    for res in outs[1:]:
        for a, b in zip(res, outs[0]):
            assert np.array_equal(a, b)

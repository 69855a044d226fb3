"""GPU test of the output stores that a new context starts with: which FP64 lattices stream them, and that neither
kind of store changes a bit."""
import numpy as np
import pytest

from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu


# vectors of SU(2) in 64-mode blocks: 18.9, 20.8, 138.2 and 144.0 MB; then FP64 lattices outside the rule
@pytest.mark.parametrize("nc,n,nm,stream", [(2, (12, 12, 8), 128, 1), (2, (13, 13, 15), 64, 0), (2, (27, 25, 25), 64, 0),
                                            (2, (26, 26, 26), 64, 1), (2, (16, 16, 16), 32, 1), (3, (12, 12, 12), 64, 1),
                                            (2, (4, 4, 4), 64, 1)])
def test_stores_of_a_new_context(gpu, nc, n, nm, stream):
    check_stores(nc, n, nm, stream)


# vectors of both groups around 12 and 17.5 MB: 11.9, 12.0, 16.9 and 17.6; 11.9, 12.0, 17.3 and 17.5
@pytest.mark.parametrize("nc,n,nm,stream", [(2, (12, 11, 11), 64, 1), (2, (7, 14, 15), 64, 0), (2, (17, 11, 11), 33, 0),
                                            (2, (13, 11, 15), 64, 1), (3, (11, 11, 8), 64, 1), (3, (10, 7, 14), 64, 0),
                                            (3, (9, 12, 13), 40, 0), (3, (12, 7, 17), 64, 1)])
def test_stores_of_vectors_that_pair_in_the_caches(gpu, nc, n, nm, stream):
    check_stores(nc, n, nm, stream)


def check_stores(nc, n, nm, stream):
    print(f"[case] stores nc={nc} n={n} modes={nm}", flush=True)
    links = np.zeros((int(np.prod(n)) * 3, 4 if nc == 2 else 18))
    links[:, [3] if nc == 2 else [0, 8, 16]] = 1.0
    psi = cf.spinors(n, nc, 2, cf.rng(5))
    with ovl.Context(nc, n, nm, m_fermion=0.1, m_dw=1.2) as ctx:
        ctx.set_links(links.reshape(-1))
        ctx.set_modes(ovl.PSI, psi)
        t = ctx.get_tuning(ovl.PREC_FP64)
        assert t.nt_store == stream and ctx.get_tuning(1).nt_store == 0
        outs = []
        for nt in (t.nt_store, 1 - t.nt_store):
            ctx.set_tuning(ovl.PREC_FP64, t.traversal, t.slabs, nt, t.waves_per_eu)
            ctx.apply_sign(ovl.PSI, ovl.SCRATCH, ovl.sign_opts(degree=4, cut=0.3))
            outs.append(ctx.get_modes(ovl.SCRATCH, 0, 2))
        assert np.array_equal(outs[0], outs[1])

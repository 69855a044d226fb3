"""GPU tests of what ovl_get_timing counts: the stencil launches of a call, their algorithmic bytes and, with profiling
on, their event times, in total and per variant."""
import numpy as np
import pytest

from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu


def consistent(t):
    assert sum(t.var_launches) == t.hop_launches
    assert abs(sum(t.var_bytes) - t.hop_bytes) <= 1e-9 * t.hop_bytes
    assert abs(sum(t.var_ms) - t.hop_ms) <= 1e-9 * max(t.hop_ms, 1.0)


@pytest.mark.parametrize("nc,n,nm", [(2, (4, 4, 4), 3), (3, (5, 3, 4), 17)])
def test_ritz_bounds_are_counted(gpu, nc, n, nm):
    print(f"[case] timing of the Ritz bounds nc={nc} n={n}", flush=True)
    V = int(np.prod(n))
    g = cf.rng(960 + nc)
    links = cf.su2_links(n, 0.3, g) if nc == 2 else cf.su3_links(n, 0.3, g)
    psi = cf.spinors(n, nc, nm, g)
    own = ovl.sign_opts(method=ovl.SIGN_ZOLOTAREV, lmin=0.0, lmax=0.0)
    given = ovl.sign_opts(method=ovl.SIGN_ZOLOTAREV, lmin=0.01, lmax=40.0)
    with ovl.Context(nc, n, nm, m_fermion=0.1, m_dw=1.0) as ctx:
        ctx.set_links(links)
        ctx.set_modes(ovl.PSI, psi)
        ts, outs = {}, {}
        for profiling in (False, True):
            ctx.set_profiling(profiling)
            for name, o in (("own", own), ("given", given)):
                ctx.apply_overlap(ovl.PSI, ovl.PSIMID, o)
                t = ctx.timing()
                consistent(t)
                assert (t.hop_ms > 0) == profiling
                ts[name, profiling] = t
                outs[name, profiling] = ctx.get_modes(ovl.PSIMID)
        # profiling changes neither the results nor the counts (the timed iterations are the graph's)
        assert np.array_equal(outs["own", True], outs["own", False])
        for name in ("own", "given"):
            a, b = ts[name, False], ts[name, True]
            assert a.hop_launches == b.hop_launches and a.hop_bytes == b.hop_bytes
        # an iteration of a solve moves six vectors in its two launches, a restart five
        own_t = ts["own", False]
        assert own_t.hop_launches >= 40 and own_t.hop_bytes >= 40 * 2 * V * 4 * nc * 16


@pytest.mark.parametrize("nc,flux", [(2, 0), (2, 1), (3, 0), (3, 2)])
@pytest.mark.parametrize("prec", [ovl.PREC_FP64, ovl.PREC_FP32])
def test_shared_launches_count_both(gpu, nc, flux, prec):
    print(f"[case] timing of shared launches nc={nc} flux={flux} prec={prec}", flush=True)
    n, nm, steps = (4, 5, 6), 3, 2
    V = int(np.prod(n))
    links_b, e_b, nn = 8 * (4 if nc == 2 else 18), 8 * (nc * nc - 1), nc * nc
    g = cf.rng(970 + nc)
    with ovl.Context(nc, n, nm, m_fermion=0.1) as ctx:
        ctx.set_links(cf.su2_links(n, 0.3, g) if nc == 2 else cf.su3_links(n, 0.3, g))
        ctx.set_efield(cf.efield(n, nc, 0.2, g))
        ctx.set_u1_flux(flux, 1.0)
        t = {}
        for gauge in (ovl.GAUGE_FROZEN, ovl.GAUGE_LINKS, ovl.GAUGE_FULL):
            for graph in (0, 1):
                ctx.fermion_update(ovl.StepOpts(kind=ovl.WILSON, dt=0.01, gauge=gauge, sign=ovl.sign_opts(precision=prec),
                                                use_graph=graph), steps)
                t[gauge, graph] = ctx.timing()
                consistent(t[gauge, graph])
        for graph in (0, 1):
            frozen = t[ovl.GAUGE_FROZEN, graph]
            assert frozen.hop_launches == 2 * steps
            # links: read, written, E read, stencil links (24 bytes an entry) written, phases read
            half = 3 * V * (2 * links_b + e_b + 24 * nn + (16 if flux else 0))
            moved = t[ovl.GAUGE_LINKS, graph]
            assert moved.hop_launches == 2 * steps
            assert abs(moved.hop_bytes - frozen.hop_bytes - 2 * steps * half) <= 1e-9 * moved.hop_bytes
            # with E moving its half step shares the launch: links read, E read and written
            full = t[ovl.GAUGE_FULL, graph]
            assert full.hop_launches == 2 * steps
            assert abs(full.hop_bytes - frozen.hop_bytes - 2 * steps * 3 * V * (links_b + 2 * e_b)) <= 1e-9 * full.hop_bytes

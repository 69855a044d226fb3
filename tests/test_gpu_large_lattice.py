"""GPU test of the observables of a lattice whose SU(3) links pass 2^31 doubles (54 a site): a small periodic
configuration repeated over it.  Energies and dN_CS/dt are sums over sites and scale with the number of
copies; the largest violations are those of one copy, and so are the root mean squares.

Tolerances: a partial sum adds about 1e4 terms, so the positive sums hold 1e-10 of themselves; the
terms of E.B have either sign and are bounded by the two energies' geometric mean.  The largest violations
come from the same arithmetic on the same numbers and agree bit for bit."""
import math

import numpy as np
import pytest
import torch

from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu


def observables(nc, n, links, e):
    out = torch.zeros(len(ovl.OBS_NAMES), dtype=torch.float64, device="cuda")
    ovl.observables_noalloc(nc, n, links.data_ptr(), e.data_ptr(), out.data_ptr(),
                            torch.cuda.current_stream().cuda_stream)
    return dict(zip(ovl.OBS_NAMES, out.cpu().tolist()))


@pytest.mark.parametrize("copies", [(43, 43, 43)])
def test_links_beyond_32_bit_offsets(gpu, copies):
    n = (8, 8, 8)
    big = tuple(a * b for a, b in zip(n, copies))
    print(f"[case] observables of SU(3) {big}", flush=True)
    assert 54 * math.prod(big) > 2**31 and math.prod(big) <= 2**26
    g = cf.rng(90)
    links = torch.from_numpy(cf.su3_links(n, 0.4, g) * (1.0 + g.normal(0, 1e-3, size=512 * 54))).cuda()
    e = torch.from_numpy(cf.efield(n, 3, 0.5, g)).cuda()
    small = observables(3, n, links, e)

    def tiled(a, width):  # [z][y][x][width]
        return a.reshape(8, 8, 8, width).repeat(copies[2], copies[1], copies[0], 1)

    L, E = tiled(links, 54), tiled(e, 24)
    got = observables(3, big, L, E)
    del L, E
    torch.cuda.empty_cache()
    times = math.prod(copies)
    for k in ("e_el", "e_mag"):
        assert abs(got[k] - times * small[k]) <= 1e-10 * times * small[k], k
    for k in ("gauss_max", "unit_max"):
        assert got[k] == small[k], k
    for k in ("gauss_rms", "unit_rms"):
        assert abs(got[k] - small[k]) <= 1e-10 * small[k], k
    assert abs(got["ncs_dot"] - times * small["ncs_dot"]) <= 1e-10 * times * math.sqrt(small["e_el"] * small["e_mag"])

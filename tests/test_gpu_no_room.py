"""GPU tests of calls that find no device memory for a buffer they only use to be faster: they give the results they
give with it.  Each case runs in a process of its own, whose hipMalloc refuses the buffer's size."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

pytestmark = pytest.mark.gpu

PRELUDE = """
import sys
sys.path[:0] = [{root!r}, {here!r}]
import alloc_shim
shim = alloc_shim.install(sys.argv[1])
import numpy as np
from overlap_amd import configs as cf
from overlap_amd import ovl
"""


def run(script, folder):
    text = PRELUDE.format(root=os.path.dirname(HERE), here=HERE) + script
    r = subprocess.run([sys.executable, "-c", text, str(folder)], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0


@pytest.mark.parametrize("refuse", [16, 8])  # the FP64 or the FP32 links of the second set
def test_wilson_steps_without_a_second_set_of_stencil_links(gpu, tmp_path, refuse):
    print(f"[case] Wilson steps, second stencil links of {refuse} bytes an entry refused", flush=True)
    run(f"""
n, nm = (5, 6, 7), 7
g = cf.rng(61)
links, e, psi = cf.su3_links(n, 0.4, g), cf.efield(n, 3, 0.2, g), cf.spinors(n, 3, nm, g)
outs = []
for refused in (0, {refuse} * 3 * 210 * 9):
    with ovl.Context(3, n, nm, m_fermion=0.1) as ctx:
        ctx.set_links(links)
        ctx.set_efield(e)
        for f in (ovl.PSI, ovl.PSIMID):
            ctx.set_modes(f, psi)
        ctx.apply_wilson(ovl.PSI, ovl.SCRATCH)
        shim.shim_refuse(0, refused)
        before = shim.shim_refusals()
        for graph in (0, 1):
            ctx.fermion_update(ovl.StepOpts(kind=ovl.WILSON, dt=0.05, gauge=ovl.GAUGE_LINKS, sign=ovl.sign_opts(),
                                            use_graph=graph), 3)
        assert (shim.shim_refusals() > before) == (refused > 0)
        shim.shim_refuse(0, 0)
        outs.append([ctx.get_modes(ovl.PSI), ctx.get_modes(ovl.PSIMID), ctx.get_links()])
for a, b in zip(*outs):
    assert np.array_equal(a, b)
""", tmp_path)


def test_link_upload_without_a_staging_buffer(gpu, tmp_path):
    print("[case] upload of 2.9 MB of links, staging refused", flush=True)
    run("""
n = (18, 20, 19)
g = cf.rng(62)
links = cf.su3_links(n, 0.4, g)
e = cf.efield(n, 3, 0.2, g)
bad = links.copy()
bad[-2] = np.nan
with ovl.Context(3, n, 1) as ctx:
    shim.shim_refuse(0, links.nbytes)
    ctx.set_links(links)
    assert shim.shim_refusals() >= 1
    ctx.set_efield(e)  # small enough for the host's scan: no staging
    try:
        ctx.set_links(bad)
        raise SystemExit("non-finite links were taken")
    except ovl.OvlError as err:
        assert err.code == ovl.E_ARG
    assert np.array_equal(ctx.get_links(), links) and np.array_equal(ctx.get_efield(), e)
    ctx.apply_wilson(ovl.PSI, ovl.SCRATCH)
""", tmp_path)

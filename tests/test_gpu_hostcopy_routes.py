"""GPU tests of the way a result takes to the host: which arrays go through the ring of pinned buffers and
which are copied directly.  The results are the same bytes either way."""
import ctypes as C

import numpy as np
import pytest
import torch

from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu

N = (16, 16, 32)  # SU(2): one mode is 1 MiB
MIB = 1 << 20


def ring_copies():
    f = ovl.lib().ovl_hostcopy_ring_copies
    f.restype = C.c_long
    return f()


def read_modes(ctx, address, count):
    rc = ovl.lib().ovl_get_modes(ctx.h, ovl.PSI, C.cast(C.c_void_p(address), C.POINTER(C.c_double)), 0, count)
    assert rc == ovl.OK, rc


def context(count):
    g = cf.rng(70 + count)
    psi = g.normal(size=(count, int(np.prod(N)) * 8)) + 1j * g.normal(size=(count, int(np.prod(N)) * 8))
    assert psi.nbytes == count * MIB
    ctx = ovl.Context(2, N, count)
    ctx.set_modes(ovl.PSI, psi)
    return ctx, psi


@pytest.mark.parametrize("count", [1, 8, 40])
@pytest.mark.parametrize("touched", [False, True])
def test_pinned_arrays_are_copied_directly(gpu, count, touched):
    print(f"[case] pinned read-back {count} MiB touched={touched}", flush=True)
    ctx, psi = context(count)
    with ctx:
        out = torch.empty(psi.shape, dtype=torch.complex128, pin_memory=True)
        if touched:
            out.zero_()
        before = ring_copies()
        read_modes(ctx, out.data_ptr(), count)
        assert ring_copies() == before
        assert np.array_equal(out.numpy(), psi)

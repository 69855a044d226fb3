"""GPU tests of the way a result takes to the host: which arrays go through the ring of pinned buffers and
which are copied directly.  The results are the same bytes either way."""
import ctypes as C
import mmap

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


# fresh anonymous pages: below the line, at it, one ring of 16 chunks, a chunk more, several rings
@pytest.mark.parametrize("count,rings", [(1, 0), (2, 1), (16, 1), (17, 1), (40, 1)])
def test_fresh_arrays_take_the_ring(gpu, count, rings):
    print(f"[case] fresh read-back {count} MiB", flush=True)
    ctx, psi = context(count)
    with ctx:
        fresh = mmap.mmap(-1, count * MIB)
        buf = (C.c_char * (count * MIB)).from_buffer(fresh)
        before = ring_copies()
        read_modes(ctx, C.addressof(buf), count)
        assert ring_copies() == before + rings
        assert bytes(buf) == psi.tobytes()
        read_modes(ctx, C.addressof(buf), count)  # the pages exist now
        assert ring_copies() == before + rings
        assert bytes(buf) == psi.tobytes()


@pytest.mark.parametrize("n", [(24, 32, 40), (31, 33, 47)])  # links in 96 bytes a site: broken last chunks
def test_broken_last_chunk(gpu, n):
    print(f"[case] fresh read-back of links {n}", flush=True)
    links = cf.su2_links(n, 0.3, cf.rng(n[2]))
    assert links.nbytes > 2 * MIB and links.nbytes % MIB
    with ovl.Context(2, n, 1) as ctx:
        ctx.set_links(links)
        fresh = mmap.mmap(-1, links.nbytes)
        buf = (C.c_char * links.nbytes).from_buffer(fresh)
        before = ring_copies()
        rc = ovl.lib().ovl_get_links(ctx.h, C.cast(C.c_void_p(C.addressof(buf)), C.POINTER(C.c_double)))
        assert rc == ovl.OK, rc
        assert ring_copies() == before + 1
        assert bytes(buf) == links.tobytes()

"""GPU tests of the copies between host arrays and the device: bit-exact round trips at the sizes where
the chunked form starts, ends a chunk and wraps its ring of pinned buffers, from one thread and from
several at once, and rejected uploads that leave the device untouched."""
import threading

import numpy as np
import pytest

from overlap_amd import configs as cf
from overlap_amd import ovl

pytestmark = pytest.mark.gpu

# SU(2) E field: 72 bytes a site.  Just below and above 1 MiB, whole and broken chunks, more than the 16 MiB
# of the ring
SHAPES = [(24, 24, 25), (24, 32, 19), (32, 32, 32), (31, 33, 32), (64, 64, 60)]


def round_trip(n, seed):
    g = cf.rng(seed)
    e = cf.efield(n, 2, 0.5, g)
    bad = e.copy()
    bad[-1] = np.nan
    with ovl.Context(2, n, 1) as ctx:
        ctx.set_efield(e)
        assert np.array_equal(ctx.get_efield(), e)
        with pytest.raises(ovl.OvlError):
            ctx.set_efield(bad)
        assert np.array_equal(ctx.get_efield(), e)
        psi = g.normal(size=(1, int(np.prod(n)) * 8)) + 1j * g.normal(size=(1, int(np.prod(n)) * 8))
        ctx.set_modes(ovl.PSI, psi)
        worse = psi.copy()
        worse[0, 3] = np.inf
        with pytest.raises(ovl.OvlError):
            ctx.set_modes(ovl.PSI, worse)
        assert np.array_equal(ctx.get_modes(ovl.PSI), psi)


@pytest.mark.parametrize("n", SHAPES)
def test_round_trips(gpu, n):
    print(f"[case] host copies n={n}", flush=True)
    for k in range(2):  # with the ring made anew, and given back in between
        round_trip(n, 40 + k)


def test_round_trips_from_several_threads(gpu):
    errors = []

    def work(k):
        try:
            for j in range(3):
                round_trip(SHAPES[(k + j) % 4], 100 * k + j)
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors

"""The pinned staging of the host transfers: one for all members of an
ensemble, made by the first transfer, grown for a larger member, and taken in
turn by threads that move different members at the same time."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from mhd3d.desc import Descriptor
from mhd3d.ensemble import Ensemble
from mhd3d.initial import periodic_fill, stratified_config

pytestmark = pytest.mark.gpu

NAMES = ("RU", "RV", "RW", "RO", "TT", "BX", "BY", "BZ")


def _random(desc, seed):
    rng = np.random.default_rng(seed)
    return {k: periodic_fill(rng.uniform(0.5, 2.0, size=desc.shape)) for k in NAMES[:8 if desc.cfg.lMag else 5]}


def _same(a, b):
    return all(np.array_equal(a[k].view(np.int64), b[k].view(np.int64)) for k in a)


def _mapped():
    """Bytes of the process's mappings of GPU buffers, pinned host memory included."""
    total = 0
    with open("/proc/self/maps") as f:
        for line in f:
            if "/dev/dri/" in line and line.split()[1].startswith("rw"):
                lo, hi = line.split()[0].split("-")
                total += int(hi, 16) - int(lo, 16)
    return total


def test_members_share_one_staging():
    """What an ensemble maps is its members' registers, one staging of at most
    a member's state and (generously) 16 allocations of 2 MB a member."""
    n, shape = 8, (96, 96, 96)
    descs = [Descriptor(stratified_config(*shape, lMag=True)) for _ in range(n)]
    # as many members set up the device's queues, whose scratch memory is mapped too
    small = Ensemble([Descriptor(stratified_config(8, 8, 8, lMag=True)) for _ in range(n)])
    before = _mapped()
    ens = Ensemble(descs)
    st = _random(descs[0], 1)
    for i in range(n):
        ens.set_state(i, st)
    for i in range(n):
        assert _same(st, ens.state(i)), i
    grown = _mapped() - before
    state = sum(a.nbytes for a in st.values())
    assert grown <= n * 3 * state + state + n * (32 << 20), (grown >> 20, state >> 20)
    ens.close()
    small.close()


def test_members_of_different_sizes_from_several_threads():
    shapes = [(20, 16, 12), (130, 67, 41), (8, 8, 8), (101, 75, 37), (24, 200, 30)]
    descs = [Descriptor(stratified_config(*s, lMag=k % 2 == 1)) for k, s in enumerate(shapes)]
    ens = Ensemble(descs)

    def turns(i):
        for r in range(6):
            st = _random(descs[i], 10 * i + r)
            ens.set_state(i, st)
            if not _same(st, ens.state(i)):
                return False
        return True

    with ThreadPoolExecutor(len(shapes)) as ex:
        assert all(ex.map(turns, range(len(shapes))))
    ens.close()

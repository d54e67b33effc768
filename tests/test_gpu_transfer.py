"""Host transfers of the state and of the fluxes: what goes in comes back, bit
for bit, with the x and y ghosts periodic, for states of one chunk, of several
chunks, with planes split over fields and more chunks than slabs for large
ones; z ghost planes included."""
import numpy as np
import pytest

from mhd3d import _lib as L
from mhd3d.desc import Descriptor
from mhd3d.domain import Domain
from mhd3d.initial import periodic_fill, stratified_config

pytestmark = pytest.mark.gpu

SIZES = [(1, 9, 5), (5, 3, 6), (32, 32, 32), (101, 75, 37), (130, 67, 41), (200, 190, 70), (700, 700, 9)]


def _random(desc, seed):
    rng = np.random.default_rng(seed)
    names = ["RU", "RV", "RW", "RO", "TT"] + (["BX", "BY", "BZ"] if desc.cfg.lMag else [])
    return {k: periodic_fill(rng.uniform(0.5, 2.0, size=desc.shape)) for k in names}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("n", SIZES)
def test_round_trip(n, mag, precision):
    print(f"round trip {n} mag={mag} precision={precision}", flush=True)
    desc = Descriptor(stratified_config(*n, lMag=mag, precision=precision))
    with Domain(desc) as dom:
        for seed in (1, 2):   # the second through staging that has been used
            st = _random(desc, seed)
            dom.set_state(st)
            got = dom.state()
            for k, a in st.items():
                assert np.array_equal(a.view(np.int64), got[k].view(np.int64)), (k, seed)


def test_state_after_steps_keeps_z_ghosts():
    """Both registers take the z ghost planes, whichever holds the state."""
    desc = Descriptor(stratified_config(24, 20, 12, lMag=True))
    st = _random(desc, 3)
    with Domain(desc) as dom:
        for steps in (1, 2):
            dom.set_state(st)
            dom.step(steps, dt=1e-7)
            got = dom.state()
            for k in st:
                assert np.array_equal(got[k][0], st[k][0]) and np.array_equal(got[k][-1], st[k][-1]), (k, steps)


@pytest.mark.parametrize("n", [(9, 7, 6), (130, 67, 41)])
def test_flux_ghosts_are_zero(n):
    desc = Descriptor(stratified_config(*n, lMag=True))
    with Domain(desc) as dom:
        dom.set_state(_random(desc, 4))
        for a in dom.fluxes().values():
            inner = a[1:-1, 1:-1, 1:-1]
            assert np.isfinite(inner).all() and np.count_nonzero(a) == np.count_nonzero(inner)


@pytest.mark.parametrize("n", [(60, 50, 40), (200, 190, 70)])
def test_transfers_take_no_device_memory(n):
    """A served run's device bytes are its registers, whatever is fetched: the
    transfers allocate nothing on the device, also where the state fills the
    ring of slabs several times (its chunks then straddle fields)."""
    print(f"no device memory {n}", flush=True)
    desc = Descriptor(stratified_config(*n, lMag=True))
    with Domain(desc) as dom:
        before = L.lib().mhd3d_device_bytes(dom.h)
        for seed in (5, 6):
            st = _random(desc, seed)
            dom.set_state(st)
            got = dom.state()
            assert all(np.array_equal(st[k].view(np.int64), got[k].view(np.int64)) for k in st)
        assert L.lib().mhd3d_device_bytes(dom.h) == before

"""Every wall condition on the GPU against the oracle, bit for bit: iTCon 3,
whose top wall keeps the temperature its own flux gives, next to the
conditions that replace it, with a vertical field on the walls at the start;
and an ensemble that mixes them."""
import dataclasses

import numpy as np
import pytest

from gpu_common import bit_identical_fraction
from mhd3d.desc import Descriptor
from mhd3d.domain import Domain
from mhd3d.ensemble import Ensemble
from mhd3d.initial import stratified_config, stratified_state
from oracle import oracle as om

pytestmark = pytest.mark.gpu


def _desc(n, mag, iz, it, precision=0):
    cfg = stratified_config(*n, lMag=mag, lRot=True, precision=precision)
    return Descriptor(dataclasses.replace(cfg, izCon=iz, iTCon=it))


def _state(desc, seed):
    st = stratified_state(desc, seed=seed)
    if desc.cfg.lMag:
        st["BZ"] = st["BX"].copy()   # nonzero on the walls
    return st


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("iz,it", [(0, 0), (0, 1), (1, 1), (0, 3), (1, 3), (0, 4)])
def test_wall_conditions(mag, iz, it):
    print(f"walls izCon={iz} iTCon={it} mag={mag}", flush=True)
    desc = _desc((21, 13, 10), mag, iz, it)
    st = _state(desc, 5)
    orc = om.Oracle(desc)
    orc.set_state(st)
    orc.communicate()
    dts = [orc.step() for _ in range(3)]
    with Domain(desc) as dom:
        dom.set_state(st)
        assert dom.step(3) == dts[-1]
        for name, g in dom.state().items():
            assert bit_identical_fraction(g, orc.get(name)) == 1.0, name


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("its", [(0, 3), (0, 1)])
def test_ensemble_of_wall_conditions(precision, its):
    print(f"ensemble walls {its} precision={precision}", flush=True)
    descs = [_desc(n, mag, 0, it, precision) for n, mag, it in
             [((20, 12, 9), True, its[0]), ((16, 16, 12), False, its[1]), ((33, 9, 7), True, its[1])]]
    ens = Ensemble(descs)
    for i, d in enumerate(descs):
        ens.set_state(i, _state(d, 7 + i))
    ens.step(3)
    for i, d in enumerate(descs):
        with Domain(d) as dom:
            dom.set_state(_state(d, 7 + i))
            dom.step(3)
            alone, mixed = dom.state(), ens.state(i)
        for k in alone:
            assert np.array_equal(alone[k].view(np.int64), mixed[k].view(np.int64)), (i, k)
    ens.close()

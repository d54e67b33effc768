"""The z split of a launch on the GPU against the oracle, bit for bit: depths
that divide unevenly into chunks, chunks of one plane, more chunks than one
round of blocks and a single chunk."""
import numpy as np
import pytest

from gpu_common import bit_identical_fraction, make_pair
from mhd3d.domain import Domain
from mhd3d.desc import Descriptor
from mhd3d.initial import stratified_config, stratified_state

pytestmark = pytest.mark.gpu

# (nx, ny, nz): 1-plane chunks; 5 + 4 planes; 17 tiles on 65 planes; partial
# tiles in x and y; a depth of the fewest planes; 300 tiles (two rounds)
SIZES = [(32, 8, 12), (96, 96, 64), (33, 65, 67), (101, 75, 37), (16, 16, 5), (640, 120, 24)]


@pytest.mark.parametrize("case", ["hydro", "mhd_rot"])
@pytest.mark.parametrize("n", SIZES)
def test_two_steps(n, case):
    print(f"z split {n} {case}", flush=True)
    desc, dom, orc, _ = make_pair(n, case)
    dts = [orc.step() for _ in range(2)]
    assert dom.step(2) == dts[-1]
    for name, g in dom.state().items():
        assert bit_identical_fraction(g, orc.get(name)) == 1.0, (n, case, name)
    dom.close()


def test_mixed_split_changes_nothing(monkeypatch):
    """The mixed form's points do not depend on the chunk a plane falls in."""
    desc = Descriptor(stratified_config(70, 44, 31, lMag=True, lRot=True, precision=1))
    st = stratified_state(desc, seed=3)
    out = []
    for target in (None, "1"):
        if target:
            monkeypatch.setenv("MHD3D_TARGET_BLOCKS", target)
        with Domain(desc) as dom:
            dom.set_state(st)
            dom.step(4)
            out.append(dom.state())
    for k in out[0]:
        assert np.array_equal(out[0][k].view(np.int64), out[1][k].view(np.int64)), k


@pytest.mark.parametrize("mag", [False, True])
@pytest.mark.parametrize("n", [(64, 16, 150), (64, 64, 160), (64, 64, 200), (96, 96, 32), (128, 128, 20), (160, 160, 24)])
def test_mixed_walls_in_the_stage_or_apart(monkeypatch, n, mag):
    """The mixed form on both sides of the line that puts the walls into the
    stage launch (chunks and planes a chunk), against a variant that launches
    its walls apart: the same bits."""
    print(f"mixed walls {n} mag={mag}", flush=True)
    desc = Descriptor(stratified_config(*n, lMag=mag, lRot=True, precision=1))
    st = stratified_state(desc, seed=4)
    out = []
    for variant in (None, "1,0"):
        if variant:
            monkeypatch.setenv("MHD3D_TUNE_MIXED_MHD" if mag else "MHD3D_TUNE_MIXED_HYDRO", variant)
        with Domain(desc) as dom:
            dom.set_state(st)
            out.append((dom.step(3), dom.state()))
    assert out[0][0] == out[1][0]
    for k in out[0][1]:
        assert np.array_equal(out[0][1][k].view(np.int64), out[1][1][k].view(np.int64)), k

"""A new context is ready when it is returned: the clearing of its registers
is not still running, on a stream its own does not wait for, when the first
state is set."""
import pytest
import torch

from mhd3d.desc import Descriptor
from mhd3d.domain import Domain
from mhd3d.ensemble import Ensemble
from mhd3d.initial import stratified_config, stratified_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [(24, 16, 9), (512, 512, 160)])
def test_nothing_is_pending_after_create(n, precision):
    print(f"create {n} precision={precision}", flush=True)
    desc = Descriptor(stratified_config(*n, lMag=True, precision=precision))
    torch.cuda.synchronize()
    with Domain(desc):
        assert torch.cuda.default_stream().query()


def test_nothing_is_pending_after_an_ensemble_is_set():
    """Its tables and its members' scalars are on the device as well."""
    descs = [Descriptor(stratified_config(*n, lMag=True)) for n in [(24, 16, 9), (160, 128, 96)]]
    torch.cuda.synchronize()
    ens = Ensemble(descs)
    assert torch.cuda.default_stream().query()
    for i, d in enumerate(descs):
        ens.set_state(i, stratified_state(d, seed=i))
        assert torch.cuda.default_stream().query(), i
    ens.close()

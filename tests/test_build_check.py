"""The build's check of the stage kernels with the wall points: one whose values
do not fit the vector registers is refused."""
import importlib.util
import os

import pytest

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rast-3dmhd-cpp_amd")


@pytest.fixture(scope="module")
def build():
    spec = importlib.util.spec_from_file_location("mhd3d_build_check", os.path.join(PKG, "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _report(walls, agprs=0, scratch=0, spill=0):
    name = f"_ZN3mhd19stage_stream_kernelIdLb1ELb1ELi3ELi1ELb0ELb1ELb0ELi191ELb0ELb{walls}EEEvNS_9StageArgsEiiiiiNS_8StepEndsE"
    at, end = "csrc/kernels_stream.hpp:647:0: remark: ", " [-Rpass-analysis=kernel-resource-usage]\n"
    lines = [f"Function Name: {name}", "    TotalSGPRs: 108", "    VGPRs: 251", f"    AGPRs: {agprs}",
             f"    ScratchSize [bytes/lane]: {scratch}", "    Dynamic Stack: False", "    Occupancy [waves/SIMD]: 2",
             "    SGPRs Spill: 152", f"    VGPRs Spill: {spill}", "    LDS Size [bytes/block]: 76160"]
    return "".join(at + line + end for line in lines)


def test_kernels_that_fit_pass(build):
    assert build.check_walls(build.kernel_usage("In file included from a.hip:1:\n" + _report(1))) == 1


@pytest.mark.parametrize("over", [dict(agprs=3), dict(scratch=8), dict(spill=2)])
def test_kernels_that_do_not_fit_are_refused(build, over):
    with pytest.raises(RuntimeError):
        build.check_walls(build.kernel_usage(_report(1, **over)))


def test_kernels_without_walls_may_use_them(build):
    assert build.check_walls(build.kernel_usage(_report(0, agprs=80, scratch=16))) == 0

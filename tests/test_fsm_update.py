"""Accurate_FSM's cell update on the CPU: the short form the sweeps run against
the form of the method's code, both built for the host from the kernels' own
header (tests/fsm_update_host.cpp says which neighbourhoods are tried).
"""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "seismic_tomography_3d_amd", "csrc")


@pytest.fixture(scope="module")
def compare(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("fsm") / "fsm_update_host")
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O2", "-ffp-contract=off",
                    "-I" + CSRC, os.path.join(HERE, "fsm_update_host.cpp"), "-o", exe], check=True)

    def run(form, draws, per, seed):
        r = subprocess.run([exe, form, str(draws), str(per), str(seed)], capture_output=True,
                           text=True, timeout=300)
        assert r.returncode == 0, r.stdout
    return run


@pytest.mark.parametrize("draws,per", [(0, 10000), (400, 4000)])   # ordinary units, the whole range
def test_walk_equals_general_form(compare, draws, per):
    compare("walk", draws, per, 1)


@pytest.mark.parametrize("draws,per", [(0, 10000), (400, 4000)])
def test_test_lowers_what_the_general_form_lowers(compare, draws, per):
    compare("test", draws, per, 2)


def test_roots_next_to_zero(compare):
    compare("roots", 2000, 2000, 3)

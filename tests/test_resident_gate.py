"""Turns of resident launches of several handles, on the CPU with streams of
the test's own."""
import ctypes
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CUS, ENGINES = 256, 32


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    so = tmp_path_factory.mktemp("gate") / "gate.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-pthread", f"-I{ROOT / 'cvfbulkwater_amd/csrc'}",
                    str(ROOT / "tests/native/cvf_gate_probe.cpp"), "-o", str(so)], check=True)
    return ctypes.CDLL(str(so))


# one-plane handles of L = 48 and 64, a workgroup per CU, run together while
# there are CUs for all their workgroups; whole-card plans never do; small
# workgroups may share CUs, up to half of the room
@pytest.mark.parametrize("groups,per_cu,together", [(48, 1, 4), (64, 1, 4), (33, 1, 4), (32, 1, 8), (12, 8, 32),
                                                    (32, 2, 8), (32, 4, 16), (129, 1, 1), (128, 1, 2), (256, 1, 1), (512, 2, 1)])
def test_handles_that_fit_run_together(probe, groups, per_cu, together):
    assert probe.probe_together(40, groups, per_cu, CUS) == together
    # they fit on every engine of workgroups: as many CUs, or half of the room
    busiest = -(-groups // ENGINES) * together
    assert busiest <= CUS // ENGINES or busiest <= per_cu * CUS // ENGINES // 2 or together == 1


def test_handles_get_in_as_they_came(probe):
    """A handle that launches on and on does not keep another one out."""
    assert probe.probe_order()

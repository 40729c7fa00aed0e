import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

GOLDEN = os.path.join(ROOT, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the libmdk C ABI)")


# a test that holds a wrong value -> why; it stays as it is and is expected to fail
WRONG_VALUE = {
    "test_gpu_companion_edges.py::test_far_poses_score_zero[nan]":
        "expects a pose that is not a number to score 0; it is not a number (test_gpu_companion_nan.py)",
}


def pytest_collection_modifyitems(items):
    for item in items:
        for name, why in WRONG_VALUE.items():
            if item.nodeid.endswith(name):
                item.add_marker(pytest.mark.xfail(reason=why, strict=True))


@pytest.fixture(scope="session")
def golden_dir():
    return GOLDEN


@pytest.fixture(scope="session")
def synth_pair(tmp_path_factory):
    """Small synthetic receptor/ligand pair (PDB files) from the project generator."""
    from megadock_amd import synth
    d = tmp_path_factory.mktemp("synth")
    rec = str(d / "rec.pdb")
    lig = str(d / "lig.pdb")
    synth.write_pdb(rec, 120, seed=11)
    synth.write_pdb(lig, 40, seed=12)
    return rec, lig

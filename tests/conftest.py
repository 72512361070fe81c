import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "ib3d-gpu_amd"))
sys.path.insert(0, os.path.join(ROOT, "oracle"))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs on the GPU box)")


def pytest_collection_modifyitems(config, items):
    """An empty /root/reference counts as "not mounted", as a missing one
    does: the tests that read the reference's files are skipped there."""
    ref = "/root/reference"
    if not os.path.isdir(ref) or os.listdir(ref):
        return
    skip = pytest.mark.skip(reason="/root/reference is empty: the reference is not mounted")
    for it in items:
        if it.path.name == "test_dropin_reference_tree.py" or it.name == "test_reads_the_reference_shipped_case":
            it.add_marker(skip)


@pytest.fixture(scope="session")
def case_dir(tmp_path_factory):
    """Generated case directories, one per configuration name."""
    from ib3d_amd import cases
    made = {}

    def get(name):
        if name not in made:
            d = tmp_path_factory.mktemp("case_" + name)
            cases.write_case(cases.CONFIGS[name], str(d))
            made[name] = str(d)
        return made[name]
    return get

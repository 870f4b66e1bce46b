import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built HIP library")
    config.addinivalue_line("markers", "slow: long-running (full BASELINE sizes)")


@pytest.fixture(scope="session")
def host_rules(tmp_path_factory):
    """The runtime's host decisions, built for the CPU."""
    import ctypes
    import subprocess
    out = str(tmp_path_factory.mktemp("rules") / "libhost_rules.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(ROOT, "tests", "native", "host_rules.cpp"), "-o", out], check=True)
    return ctypes.CDLL(out)


@pytest.fixture(scope="session")
def orc():
    from oracle import oracle
    return oracle

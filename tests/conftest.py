import glob
import importlib
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "oracle")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def moon():
    """The product package (its directory name is not a Python identifier)."""
    return importlib.import_module("moondream-zig_amd")


@pytest.fixture(scope="session")
def O():
    """The CPU oracle (test infrastructure)."""
    return importlib.import_module("moon_oracle")


@pytest.fixture(scope="session")
def ctx(moon):
    c = moon.Context(0)
    yield c
    c.close()


# parity bar: relative Frobenius error against the oracle's f32-accumulated, f16-rounded result
TOL = 1e-3


def compute_units():
    """Of the machine's GPUs, as the kernel driver lists them."""
    units = set()
    for path in glob.glob("/sys/class/kfd/kfd/topology/nodes/*/properties"):
        with open(path) as f:
            node = dict(line.split() for line in f)
        if int(node["simd_count"]):
            units.add(int(node["simd_count"]) // int(node["simd_per_cu"]))
    assert len(units) == 1, units
    return units.pop()

import os
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "quickpic-opensource_amd")
for p in (REPO, PKG):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device)")
    config.addinivalue_line("markers", "slow: longer CPU test")


def pytest_collection_modifyitems(items):
    """The tests against the reference's own kernels are skipped where those are not
    built, also the ones that load a copy of their own."""
    from oracle import refharness
    if refharness.available():
        return
    skip = pytest.mark.skip(reason="reference kernels not built (oracle/_ref needs /root/reference)")
    for item in items:
        if item.path.name == "test_oracle_vs_ref.py":
            item.add_marker(skip)


@pytest.fixture(scope="session")
def ref():
    from oracle import refharness
    if not refharness.available():
        pytest.skip("reference kernels not built (oracle/_ref needs /root/reference)")
    return refharness.Ref()

import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device) to run")
    config.addinivalue_line("markers", "slow: takes more than a few seconds on the CPU")


def pytest_collection_modifyitems(items):
    # the drop-in tests need a harness built from the reference's sources and
    # fail where it was not: they run last, so that a run that ends at its first
    # failure has run all others
    items.sort(key=lambda i: "test_gpu_dropin" in i.nodeid)

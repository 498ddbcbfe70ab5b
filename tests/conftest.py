"""pytest configuration: import paths and the ``gpu`` marker.

Tests marked ``gpu`` need a visible AMD GPU and the built libplutomx.so;
everything else runs on the CPU (oracle, golden fixtures, host logic,
library exports)."""
import pathlib
import sys

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
for p in (ROOT / "pluto-sirocco_amd", ROOT):
    if str(p) not in sys.path:
        sys.path.insert(0, str(p))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an AMD GPU (MI355X) and libplutomx.so")


def pytest_collection_modifyitems(items):
    """The drop-in tests run PLUTO's own driver, compiled from the reference
    sources (oracle/ref/Makefile, GLUE=1): skipped where it is not built, as
    the other tests that run the reference are, so that a run that stops at
    its first failure goes on to the rest."""
    from oracle import refrun
    if any(refrun.REF_DIR.glob("glue_*/pluto")):
        return
    skip = pytest.mark.skip(reason="the reference's driver with the drop-in is not built")
    for item in items:
        if item.path.name == "test_gpu_dropin.py":
            item.add_marker(skip)

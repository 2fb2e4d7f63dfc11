import os
import sys

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, REPO)
sys.path.insert(0, os.path.join(REPO, "oracle"))
sys.path.insert(0, os.path.join(REPO, "tests"))


ARTIFACTS = [os.path.join(REPO, "ggems_amd", "lib", "libggems_engine.so"),
             os.path.join(REPO, "ggems_amd", "lib", "libggems.so"),
             os.path.join(REPO, "oracle", "_build", "libggems_oracle.so")]
# extracted from a GGEMS source tree by the build, where there is one
PHYSICS_DATA = os.path.join(REPO, "ggems_amd", "data", "_gen", "ggems_physics.bin")
NO_DATA = ("cannot load physics data blob", "cannot open physics data", "cannot open the material database",
           "data/_gen/materials.txt")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP engine)")
    # a fresh checkout: build the libraries, the data blob and the oracle once
    sys.path.insert(0, os.path.join(REPO, "ggems_amd", "data"))
    import extract_physics_data
    missing = not all(os.path.exists(p) for p in ARTIFACTS)
    if missing or (not os.path.exists(PHYSICS_DATA) and extract_physics_data.available()):
        from ggems_amd import build
        build.build_all(oracle=True)


def pytest_runtest_setup(item):
    # flush the case name before any GPU step so a lost box still names it
    if "gpu" in item.keywords:
        print("\n[gpu-test] %s" % item.nodeid, flush=True)


@pytest.hookimpl(hookwrapper=True)
def pytest_runtest_makereport(item, call):
    """Without a GGEMS source tree there is no physics data, and what reads it
    cannot run: such a test is skipped, and says so."""
    outcome = yield
    if call.excinfo is None or os.path.exists(PHYSICS_DATA):
        return
    text = str(call.excinfo.value)
    if any(t in text for t in NO_DATA):
        report = outcome.get_result()
        report.outcome = "skipped"
        report.longrepr = (str(item.path), 0, "Skipped: no physics data (built from a GGEMS source tree)")

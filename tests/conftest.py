import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (gfx950) device")


# The programs linked with the reference's own sources (a test file or a test -> its program), and one of the
# sources they are compiled from where the reference is checked out.
REFERENCE_PROGRAMS = {"test_walker_end_to_end_gpu.py": "walker_end_to_end",
                      "test_reference_paged_kv_storage_runs_on_the_hip_library": "paged_kv_roundtrip"}
REFERENCE_SOURCE = "/root/reference/compiler/runtime/paged_kv.cpp"


def why_skipped(file_name, test_name, root=ROOT, source=REFERENCE_SOURCE):
    """Tests of those programs are skipped where the program is missing because there is nothing to build it from;
    where the sources are at hand a missing program is a failed build, and its tests run and fail."""
    program = REFERENCE_PROGRAMS.get(file_name) or REFERENCE_PROGRAMS.get(test_name)
    if not program or os.path.exists(source) or os.path.exists(os.path.join(root, "oracle", "_ref", "integration", program)):
        return None
    return f"{program} is not built and there is no reference checkout to build it from"


def pytest_collection_modifyitems(items):
    for item in items:
        reason = why_skipped(item.path.name, item.name)
        if reason:
            item.add_marker(pytest.mark.skip(reason=reason))


@pytest.fixture(scope="session")
def exe():
    """The HIP executor.  GPU tests fail (not skip) when the native library or the
    device is missing: a silent fallback would void every parity claim."""
    from mlcompiler_amd import HipExecutor

    e = HipExecutor.Instance()
    assert e.isAvailable(), "gfx950 device / native library unavailable: " + e.lastError()
    return e

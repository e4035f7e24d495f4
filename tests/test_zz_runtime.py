"""At the end of a GPU run the process still has one HIP runtime, and no torch."""
import sys

import pytest

pytestmark = pytest.mark.gpu


def test_one_runtime_is_mapped(amps):
    with open("/proc/self/maps") as f:
        paths = {line.split()[-1] for line in f if "libamdhip64" in line or "libhsa-runtime64" in line}
    assert sum("libamdhip64" in p for p in paths) == 1 and sum("libhsa-runtime64" in p for p in paths) == 1, paths
    assert "torch" not in sys.modules and all("/torch/" not in p for p in paths), paths

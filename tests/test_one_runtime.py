"""The GPU tests' process uses one HIP runtime, the one libamps.so is built
against, and starts no program itself once that is loaded (tests/conftest.py)."""
import json
import os
import subprocess
import sys

import pytest

from tests.launcher import Launcher

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

COLLECT = """
import json, sys
import pytest
class Look:
    def pytest_collection_finish(self, session):
        self.items = len(session.items)
look = Look()
rc = pytest.main(["--collect-only", "-q", "-p", "no:cacheprovider", "-m", "gpu", "tests"], plugins=[look])
torch = "torch" in sys.modules
import w3914777_amd
w3914777_amd.lib()
maps = sorted({l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l or "libhsa-runtime64" in l})
print("RESULT " + json.dumps([int(rc), look.items, torch, maps]))
"""


def test_collection_leaves_the_runtime_to_the_library():
    r = subprocess.run([sys.executable, "-c", COLLECT], cwd=ROOT, capture_output=True, text=True, timeout=300)
    line = [l for l in r.stdout.splitlines() if l.startswith("RESULT ")]
    assert line, r.stdout + r.stderr
    rc, items, torch, maps = json.loads(line[0][len("RESULT "):])
    assert rc == 0 and items > 300
    assert not torch
    assert sum("libamdhip64" in m for m in maps) == 1 and sum("libhsa-runtime64" in m for m in maps) == 1, maps
    assert all("/torch/" not in m for m in maps), maps


def test_launcher_runs_programs_like_subprocess(tmp_path):
    launcher = Launcher()
    try:
        script = "import os, sys; print(os.getcwd(), os.getppid()); print('e', file=sys.stderr); sys.exit(3)"
        r = launcher.run([sys.executable, "-c", script], cwd=tmp_path, capture_output=True, text=True, timeout=60)
        cwd, parent = r.stdout.split()
        assert r.returncode == 3 and r.stderr == "e\n" and os.path.samefile(cwd, tmp_path)
        assert int(parent) != os.getpid()
        with pytest.raises(subprocess.TimeoutExpired):
            launcher.run([sys.executable, "-c", "import time; time.sleep(30)"], timeout=0.5)
        with pytest.raises(OSError):
            launcher.run([str(tmp_path / "missing")])
        assert launcher.run([sys.executable, "-c", "pass"]).returncode == 0
    finally:
        launcher.close()
    assert launcher._p.returncode == 0

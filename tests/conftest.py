import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

from tests.launcher import Launcher  # noqa: E402

# The first library that brings a HIP runtime into a process decides which one
# libamps.so uses: torch carries its own, of another release than the one the
# library is built against.  What needs torch runs in a process of its own, so
# that every other test has the library's runtime and no second one beside it:
# files that import torch when they are collected and pass its streams and
# memory to the library (on torch's runtime), and single tests that import it.
TORCH_FIRST = {"test_gpu_noalloc_streams.py"}
TORCH_TESTS = {"test_gpu_adjoint.py::test_torch_autograd_binding"}

_launcher = None


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP engine)")


def _alone(config, names):
    """Only these files or tests were asked for: this is their own process."""
    args = [os.path.basename(str(a)) for a in config.args]
    return bool(args) and all(a.split("::")[0] in names or a in names for a in args)


def _run_alone(nodeid):
    r = _launcher.run([sys.executable, "-u", "-m", "pytest", "-x", "-q", "-p", "no:cacheprovider", "-m", "gpu", nodeid],
                      cwd=ROOT, timeout=600)  # the first import of torch can take minutes
    if r.returncode != 0:
        pytest.fail(r.stdout + r.stderr, pytrace=False)


@pytest.hookimpl(tryfirst=True)
def pytest_pycollect_makemodule(module_path, parent):
    if module_path.name in TORCH_FIRST and not _alone(parent.config, TORCH_FIRST):
        return OwnProcessFile.from_parent(parent, path=module_path)


class OwnProcessFile(pytest.File):
    def collect(self):
        item = OwnProcessItem.from_parent(self, name="own_process")
        item.add_marker("gpu")
        yield item


class OwnProcessItem(pytest.Item):
    def runtest(self):
        _run_alone(str(self.path))

    def reportinfo(self):
        return self.path, 0, self.name


def _torch_test(item):
    return os.path.basename(item.nodeid) in TORCH_TESTS and not _alone(item.config, TORCH_TESTS)


@pytest.hookimpl(tryfirst=True)
def pytest_pyfunc_call(pyfuncitem):
    if _torch_test(pyfuncitem):
        _run_alone(os.path.join(ROOT, "tests", os.path.basename(pyfuncitem.nodeid)))
        return True


def pytest_collection_finish(session):
    """Start the launcher before a test loads the HIP runtime."""
    global _launcher
    if session.config.option.collectonly or _launcher is not None:
        return
    if any(isinstance(i, OwnProcessItem) or _torch_test(i) or _starts_programs(i) for i in session.items):
        _launcher = Launcher()


def pytest_unconfigure(config):
    if _launcher is not None:
        _launcher.close()


def _starts_programs(item):
    return item.get_closest_marker("gpu") is not None and hasattr(getattr(item, "module", None), "subprocess")


@pytest.fixture(autouse=True)
def _programs_by_launcher(request, monkeypatch):
    """The GPU tests' subprocess.run is the launcher's."""
    if _launcher is not None and _starts_programs(request.node):
        monkeypatch.setattr(request.module, "subprocess", _launcher)


@pytest.fixture(scope="session")
def O():
    """The CPU oracle (built on first use)."""
    from oracle import oracle as mod
    mod.lib()
    return mod


@pytest.fixture(scope="session")
def amps():
    """The engine; on a GPU test this must load libamps.so (no fallback)."""
    import w3914777_amd as mod
    mod.lib()
    return mod

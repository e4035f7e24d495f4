"""Which kernels a call launches, and the device memory it takes: the host code
on a HIP runtime without a GPU (tests/hip_stub.c)."""
import pytest

from tests import stub_runtime


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = stub_runtime.build(str(tmp_path_factory.mktemp("stub")))
    return lambda script: stub_runtime.run(lib, script)


def test_workgroups_per_cu_select_the_single_step_sweeps(run):
    """wg_per_cu sizes the sweeps of PURE_FP64 grain growth and sintering; the
    launches of several steps have no such size, so they need wg_per_cu = 0.
    The snowflake's FP64 sweep ignores it."""
    out = run("""
for name, model, q in (("gg2", amps.GRAINGROWTH, 2), ("gg5", amps.GRAINGROWTH, 5), ("sn", amps.SINTERING, 2),
                       ("sf", amps.SNOWFLAKE, 2)):
    for wg in (0, 1, 4):
        for tile in (16, 32):
            cfg = amps.Config.default(model)
            cfg.nx, cfg.ny, cfg.q, cfg.tile, cfg.wg_per_cu = 256, 192, q, tile, wg
            with amps.Context(cfg) as c:
                c.init()
                stub.clear()
                c.step(16)
                log = [k for k in stub.log() if "advance" not in k]
                out[f"{name} {wg} {tile}"] = [sum("multi" in k for k in log), len(log)]
""")
    for key, (multi, n) in out.items():
        name, wg, _ = key.split()
        if wg == "0" or name == "sf":
            assert multi and n < 16, key
        else:
            assert (multi, n) == (0, 16), key

"""Short calls, each after the host has waited, replay graphs of few steps once
a context has taken 100; calls that follow without a wait enqueue their steps
one by one.  The same bits as without graphs, over monitor periods and call
lengths that leave remainders, with single steps, reads and unwaited calls
between the replays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (steps, wait after the call)
CALLS = [(60, 1), (39, 1), (1, 1), (10, 1), (10, 0), (10, 1), (30, 1), (1, 1), (25, 1), (20, 0), (14, 1), (39, 1), (28, 1), (10, 1)]


@pytest.mark.parametrize("model", ["SNOWFLAKE", "GRAINGROWTH", "SINTERING"])
@pytest.mark.parametrize("every", [0, 1, 7, 10])
def test_short_calls_equal_single_steps(amps, monkeypatch, model, every):
    cfg = amps.Config.default(getattr(amps, model))
    cfg.nx, cfg.ny, cfg.tile, cfg.mode = 96, 64, 16, amps.ADAPTIVE if every else amps.PURE_HALF2
    if every:
        cfg.monitor_every = every
    runs = []
    for no_graph in ("1", "0"):
        monkeypatch.setenv("AMPS_NO_GRAPH", no_graph)
        with amps.Context(cfg) as ctx:
            states = []
            for again in range(2):  # the second with graphs from its first waited call
                ctx.init()
                for n, wait in CALLS:
                    ctx.step(n)
                    if wait:
                        ctx.sync()
                        states += [ctx.get_field(f) for f in range(cfg.nfields())]
            info = ctx.info()
            runs.append((states, info.steps_done, info.monitor_passes, info.hi_frac_mean, info.fp64_tile_updates))
    assert runs[0][1:] == runs[1][1:]
    assert all(np.array_equal(a, b) for a, b in zip(runs[0][0], runs[1][0]))

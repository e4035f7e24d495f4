"""Steps replayed as graphs (a context takes 400 steps one by one first, and
graphs of at least 40 steps after that) against the same steps enqueued one by
one: the same bits after several replays from either buffer, with calls that
leave a remainder, a synchronisation and a field read between them, over
monitor periods that are odd, short and longer than a graph's 40 steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CALLS = [411, 40, 3, 130, 7, 97, 250]   # odd starts too; replays in the fourth, sixth and last


def config(amps, model, every):
    c = amps.Config.default(getattr(amps, model))
    c.nx, c.ny, c.tile, c.mode = 96, 64, 16, amps.ADAPTIVE if every else amps.PURE_HALF2
    if every:
        c.monitor_every = every
    return c


@pytest.mark.parametrize("model", ["SNOWFLAKE", "GRAINGROWTH", "SINTERING"])
@pytest.mark.parametrize("every", [0, 1, 7, 10, 50])
def test_replays_equal_single_steps(amps, monkeypatch, model, every):
    runs = []
    for no_graph in ("1", "0"):
        monkeypatch.setenv("AMPS_NO_GRAPH", no_graph)
        with amps.Context(config(amps, model, every)) as ctx:
            nf = 3 if model == "SINTERING" else 2
            states = []
            for again in range(2):          # the second from a new initial state, with graphs from its first step
                ctx.init()
                for n in CALLS:
                    ctx.step(n)
                    ctx.sync()
                    states.append([ctx.get_field(f) for f in range(nf)])
            info = ctx.info()
            runs.append((states, info.steps_done, info.monitor_passes, info.hi_frac_mean, info.fp64_tile_updates))
    assert runs[0][1:] == runs[1][1:]
    for a, b in zip(runs[0][0], runs[1][0]):
        for x, y in zip(a, b):
            np.testing.assert_array_equal(x, y)

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


@pytest.mark.parametrize("ckpt", [1, 3, 8, 20])
@pytest.mark.parametrize("model", ["SNOWFLAKE", "SINTERING"])
def test_adjoint_fits_the_memory_of_its_states(run, model, ckpt):
    """A taped run and its adjoint fit a device that holds the context, the
    checkpoints, the states between two of them and two cotangents, whatever
    the number of checkpoints (blocks of them are allocated ahead)."""
    out = run(f"""
cfg = amps.Config.default(amps.{model})
cfg.nx, cfg.ny, cfg.tile = 64, 64, 16
ids = [amps.GRAD_SF["DELTA"]] if cfg.model == amps.SNOWFLAKE else [amps.GRAD_SN["KC"]]
import numpy as np
F = cfg.nfields()
for ckpts in (1, 2, 3, 4, 5, 8, 9, 16, 17):
    with amps.Context(cfg) as c:
        c.init()
        base = stub.live()
        state = F * (64 * 64 + 1056) * 8
        steps = {ckpt} * (ckpts - 1) + ({ckpt} - 1 if {ckpt} > 1 else 0)
        stub.limit(base + (ckpts + {ckpt} - 1 + 2) * state + 65536)
        try:
            c.tape_begin({ckpt})
            c.step(steps)
            c.adjoint([np.zeros((F, 64, 64))], ids, want_du0=True)
            out[str(ckpts)] = "fits"
        except amps.AmpsError as e:
            out[str(ckpts)] = str(e)
        stub.limit(2 ** 63)
""")
    assert set(out.values()) == {"fits"}, out


def test_short_calls_replay_graphs_on_an_idle_stream(run):
    """Calls of 10 to 39 steps replay graphs once the context has taken 100
    steps, if the host waited for the stream before the call; without a wait
    their steps are enqueued one by one, and calls of 40 and more replay the
    long graphs after 400 steps either way."""
    out = run("""
def graphs(every, calls, wait):
    cfg = amps.Config.default(amps.SINTERING)
    cfg.nx = cfg.ny = 64
    if every:
        cfg.mode, cfg.monitor_every = amps.ADAPTIVE, every
    else:
        cfg.mode = amps.PURE_HALF2
    res = []
    with amps.Context(cfg) as c:
        c.init()
        for n in calls:
            stub.clear()
            c.step(n)
            res.append(stub.log().count("graph"))
            if wait == "sync": c.sync()
            if wait == "get": c.get_field(0)
    return res
calls = [10] * 12 + [25, 39, 9]
for every in (0, 1, 7, 10, 20, 50):
    for wait in ("sync", "get", "none"):
        out[f"{every} {wait}"] = graphs(every, calls, wait)
out["long"] = graphs(10, [400, 40, 10, 80, 10], "none")
out["long after short"] = graphs(10, [10] * 40 + [40], "sync")[-1]
""")
    for key, got in out.items():
        if key == "long":
            assert got == [0, 1, 0, 2, 0]
        elif key == "long after short":
            assert got == 1
        elif key.split()[1] == "none" or key.startswith("50"):
            assert got == [0] * 15, key
        else:
            # graphs hold whole monitor periods and start on a monitor step
            every = int(key.split()[0])
            if every in (0, 1, 10):
                assert got == [0] * 10 + [1, 1, 2, 3, 0], (key, got)
            else:
                assert max(got) >= 1 and got[:10] == [0] * 10, (key, got)


def test_block_tables_only_for_batches(run):
    """The map from blocks to instances of the launches of several steps exists
    for batches only: one grid takes the same memory without such launches."""
    out = run("""
def live(model, n, wg):
    cfgs = []
    for k in range(n):
        cfg = amps.Config.default(model)
        cfg.nx, cfg.ny, cfg.wg_per_cu = 512, 512 + 32 * k, wg
        cfgs.append(cfg)
    with amps.Context(cfgs) as c:
        c.init()
        stub.clear()
        c.step(12)
        return stub.live(), any("multi" in k for k in stub.log())
for name, model in (("gg", amps.GRAINGROWTH), ("sn", amps.SINTERING)):
    for n in (1, 3):
        out[f"{name} {n}"] = [live(model, n, 0), live(model, n, 1)]
""")
    for key, ((with_multi, used), (without, unused)) in out.items():
        assert used and not unused, key
        assert (with_multi > without) == (key[-1] == "3"), key


def test_info_and_init_take_few_runtime_calls(run):
    """amps_get_info of an adaptive context is one kernel that writes the sums
    to host memory (a copy of the spread counters took twice as long); amps_init
    clears all counters with one memset."""
    out = run("""
for name, model in (("sf", amps.SNOWFLAKE), ("gg", amps.GRAINGROWTH), ("sn", amps.SINTERING)):
    cfg = amps.Config.default(model)
    cfg.nx = cfg.ny = 64
    cfg.mode = amps.ADAPTIVE
    with amps.Context(cfg) as c:
        c.init()
        stub.clear(); c.init()
        init = [k for k in stub.log() if k in ("copy", "memset")]
        c.step(1); c.info()
        stub.clear(); c.info()
        out[name] = [len(init), stub.log()]
""")
    for name, (init, info) in out.items():
        assert init <= (8 if name == "gg" else 6), (name, init)  # gg: two zero masks
        assert len(info) == 1 and "counters" in info[0], (name, info)


@pytest.mark.parametrize("n", [64, 512])
def test_memory_is_freed_after_the_commands_are_retired(run, n):
    """Between the last command of a stream and the first free of 2 MiB or more
    after it stands a host function: what is freed before the runtime has retired
    the commands is released later, on a thread that slows the next calls.
    Smaller memory needs none."""
    out = run(f"""
import numpy as np
n = {n}
cfg = amps.Config.default(amps.SNOWFLAKE)
cfg.nx = cfg.ny = n
def log(name, f):
    stub.clear(); f(); out[name] = stub.log()
c = amps.Context(cfg)
c.init()
log("close untaped", lambda: (c.step(5), c.close()))
c = amps.Context(cfg)
c.init(); c.tape_begin(2); c.step(5)
log("adjoint", lambda: c.adjoint([np.zeros((2, n, n))], [1], want_du0=True))
log("set_field", lambda: c.set_field(0, np.zeros((n, n))))
c.tape_begin(2); c.step(5)
log("tape_begin", lambda: (c.step(1), c.tape_begin(1)))
log("init", lambda: (c.step(1), c.init()))
c.tape_begin(2)
log("close", lambda: (c.step(5), c.close()))
""")
    assert set(out) == {"close untaped", "adjoint", "set_field", "tape_begin", "init", "close"}
    for name, log in out.items():
        assert "free" in log, name
        if n == 64:
            assert "host" not in log, name
            continue
        retired = False
        for what in log:
            assert what != "free" or retired, (name, log)
            if what != "free":
                retired = what == "host"

"""The adjoint's recomputed states: with checkpoints several steps apart it
runs launches of several steps that store each step's state, in memory that
lies partly in the tape's unused checkpoints.  Gradients and dJ/du_0 have the
bits of the run that keeps every state (checkpoints one step apart), which
recomputes nothing: both sides run the same reverse steps on states that
single and joined forward steps produce alike.

Grids by plan (block edge, steps a launch), for 256 compute units.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STEPS = 23
CKPTS = [5, 8, 11, 40]  # the segment ends inside, at and past whole launches; 40: one segment

SF_GRIDS = {"16x4": [(64, 48)], "16x3": [(16 * 23, 16 * 24)], "32x3": [(512, 480)], "16x2": [(16 * 25, 16 * 24)],
            "batch": [(64, 48), (48, 80), (32, 32)], "single": [(1024, 1024)]}
SN_GRIDS = {"16x4": [(64, 48)], "32x3": [(384, 384)], "16x2": [(16 * 25, 16 * 24)], "32x2": [(1024, 800)],
            "batch": [(64, 48), (48, 80), (32, 32)]}


def gradients(amps, cfgs, ids, u0, ckpt, W):
    with amps.Context(cfgs) as ctx:
        ctx.init()
        for i, fields in enumerate(u0):
            for f, a in enumerate(fields):
                ctx.set_field(f, a, inst=i)
        ctx.tape_begin(ckpt)
        ctx.step(STEPS)
        return ctx.adjoint(W, ids, want_du0=True)


def check(amps, cfgs, ids, nf):
    rng = np.random.default_rng(len(cfgs) + cfgs[0].nx)
    u0, W = [], []
    for c in cfgs:
        y, x = np.mgrid[0:c.ny, 0:c.nx]
        u0.append([np.ascontiguousarray(0.5 + 0.3 * np.sin(rng.uniform(0.1, 0.5) * x + f) * np.cos(rng.uniform(0.1, 0.5) * y))
                   for f in range(nf)])
        W.append(rng.uniform(0.5, 1.5, (nf, c.ny, c.nx)))
    g1, du1 = gradients(amps, cfgs, ids, u0, 1, W)
    assert np.all(np.isfinite(g1)) and np.all(g1 != 0.0)
    for ckpt in CKPTS:
        g, du = gradients(amps, cfgs, ids, u0, ckpt, W)
        assert np.array_equal(g, g1), ckpt
        assert all(np.array_equal(a, b) for a, b in zip(du, du1)), ckpt


@pytest.mark.parametrize("plan", sorted(SF_GRIDS))
@pytest.mark.parametrize("bc", [0, 1])
def test_snowflake_recomputed_states(amps, plan, bc):
    cfgs = []
    for k, (ny, nx) in enumerate(SF_GRIDS[plan]):
        c = amps.Config.default(amps.SNOWFLAKE)
        c.nx, c.ny, c.bc, c.stencil, c.seed = nx, ny, bc, (k + bc) % 2, 5 + k
        c.params[amps.SF["NOISE"]] = 0.01
        cfgs.append(c)
    check(amps, cfgs, list(amps.GRAD_SF.values()), 2)


@pytest.mark.parametrize("plan", sorted(SN_GRIDS))
@pytest.mark.parametrize("bc", [0, 1])
def test_sintering_recomputed_states(amps, plan, bc):
    cfgs = []
    for ny, nx in SN_GRIDS[plan]:
        c = amps.Config.default(amps.SINTERING)
        c.nx, c.ny, c.bc = nx, ny, bc
        cfgs.append(c)
    check(amps, cfgs, list(amps.GRAD_SN.values()), 3)

"""PURE_FP64 runs that advance several steps a launch against the same run one
step a call (a call of one step never takes such a launch): bit for bit, at
grids that take each block edge and step count, with sides that are no
multiple of 32, one-block and ragged rectangular grids, both boundaries and
Laplacians, noise on and off, step counts that leave remainders, and batches
of uneven grids.  The single step itself is held to the oracle elsewhere.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def fields(ny, nx, k, seed):
    """k random fields in (0, 1) with structure at every cell, plus flat patches."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(k):
        f = rng.uniform(0.0, 1.0, (ny, nx))
        f[: ny // 3, : nx // 2] = 0.0
        f[-ny // 4:, -nx // 3:] = 1.0
        out.append(f)
    return out


def run(amps, cfgs, u0, calls):
    with amps.Context(cfgs) as ctx:
        ctx.init()
        for i, u in enumerate(u0):
            for f, v in enumerate(u):
                ctx.set_field(f, v, inst=i)
        for n in calls:
            ctx.step(n)
        ctx.sync()
        assert ctx.info().steps_done == sum(calls)
        return [[ctx.get_field(f, inst=i) for f in range(c.nfields())] for i, c in enumerate(ctx.cfgs)]


def check(amps, cfgs, total, seed):
    u0 = [fields(c.ny, c.nx, c.nfields(), seed + i) for i, c in enumerate(cfgs)]
    one = run(amps, cfgs, u0, [1] * total)
    many = run(amps, cfgs, u0, [total])
    split = run(amps, cfgs, u0, [total - 4, 1, 3])
    for a, b, c in zip(one, many, split):
        for x, y, z in zip(a, b, c):
            assert np.array_equal(x, y) and np.array_equal(x, z)


def sf(amps, ny, nx, tile, bc, stencil, aniso, noise):
    c = amps.Config.default(amps.SNOWFLAKE)
    c.nx, c.ny, c.tile, c.bc, c.stencil, c.seed = nx, ny, tile, bc, stencil, 7 + nx
    c.params[amps.SF["ANISO"]] = aniso
    c.params[amps.SF["NOISE"]] = noise
    c.params[amps.SF["THETA0"]] = 0.3
    return c


# ny, nx: one block, ragged strips (K = 4), 306 to 576 blocks of 16^2 (K = 4, 3), 32^2 blocks, K = 2 with and
# without sides divisible by 32, and a grid past the last plan
@pytest.mark.parametrize("ny,nx,tile", [(16, 16, 16), (48, 16, 16), (32, 96, 32), (272, 288, 16), (336, 304, 16),
                                        (384, 384, 32), (512, 416, 32), (528, 336, 16), (640, 512, 32),
                                        (784, 784, 16)])
@pytest.mark.parametrize("bc,stencil,aniso,noise", [(0, 0, 4, 0.0), (1, 0, 4, 0.01), (1, 1, 6, 0.01), (0, 1, 3, 0.01)])
def test_snowflake_steps_per_launch_bitwise(amps, ny, nx, tile, bc, stencil, aniso, noise):
    check(amps, [sf(amps, ny, nx, tile, bc, stencil, aniso, noise)], 11, 1)


@pytest.mark.parametrize("sides", [((16, 48), (64, 16), (32, 32)), ((256, 256), (128, 384), (64, 64)),
                                   ((400, 400), (96, 208))])
def test_snowflake_batches_bitwise(amps, sides):
    cfgs = [sf(amps, ny, nx, 16, i % 2, (i + 1) % 2, (4, 6, 5)[i % 3], 0.01 * (i % 2)) for i, (ny, nx) in enumerate(sides)]
    check(amps, cfgs, 10, 3)


def gg(amps, ny, nx, tile, bc, stencil, q):
    c = amps.Config.default(amps.GRAINGROWTH)
    c.nx, c.ny, c.tile, c.bc, c.stencil, c.q = nx, ny, tile, bc, stencil, q
    return c


# every (edge, K, q) of the plan: one block, up to 1.25 blocks of 16^2 per CU, sides that divide by 32 or not
@pytest.mark.parametrize("ny,nx,tile", [(16, 16, 16), (96, 48, 16), (256, 320, 32), (272, 336, 16), (416, 256, 32),
                                        (608, 512, 32), (752, 400, 16)])
@pytest.mark.parametrize("q,bc,stencil", [(2, 0, 0), (2, 1, 1), (3, 1, 0), (4, 0, 1), (5, 1, 0), (6, 0, 0), (7, 1, 1)])
def test_graingrowth_steps_per_launch_bitwise(amps, ny, nx, tile, q, bc, stencil):
    check(amps, [gg(amps, ny, nx, tile, bc, stencil, q)], 17, 5)


@pytest.mark.parametrize("q", [2, 4])
def test_graingrowth_batches_bitwise(amps, q):
    cfgs = [gg(amps, ny, nx, 16, i % 2, (i + 1) % 2, q) for i, (ny, nx) in enumerate(((16, 48), (320, 336), (64, 64)))]
    check(amps, cfgs, 13, 9)


def sn(amps, ny, nx, tile, bc, flags):
    c = amps.Config.default(amps.SINTERING)
    c.nx, c.ny, c.tile, c.bc, c.flags = nx, ny, tile, bc, flags
    return c


# one block, 16^2 blocks with K = 4 and K = 2, 32^2 blocks with K = 3 and K = 2
@pytest.mark.parametrize("ny,nx,tile", [(16, 16, 16), (48, 96, 16), (256, 320, 32), (288, 384, 32), (400, 336, 16),
                                        (800, 1056, 32)])
@pytest.mark.parametrize("bc,flags", [(0, 0), (1, 0), (0, 2), (1, 2)])
def test_sintering_steps_per_launch_bitwise(amps, ny, nx, tile, bc, flags):
    check(amps, [sn(amps, ny, nx, tile, bc, flags)], 11, 6)


def test_sintering_batch_bitwise(amps):
    cfgs = [sn(amps, ny, nx, 16, i % 2, 0) for i, (ny, nx) in enumerate(((16, 48), (320, 336), (64, 64)))]
    check(amps, cfgs, 9, 8)

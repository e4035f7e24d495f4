"""The snowflake's one-launch low-precision step (grids of at most 4096 tiles of
16^2, 2048 of 32^2) against the two launches, which sweep timing keeps: the
same bits, tile types and tile counts, over modes, NO_SKIP, both stencils,
several instances, states in which tiles hold, are flat or do neither, and
with the timing switched in the middle of a run."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIDES = {16: [(16, 16), (80, 48), (1024, 1024), (1024, 1040)],   # 1, 15, 4096 and 4160 tiles
         32: [(32, 32), (96, 64), (512, 1024), (1024, 544), (1024, 2048), (1024, 2080)]}  # 1, 6, 512, 544, 2048, 2080


def config(amps, nx, ny, tile, mode, flags, stencil):
    c = amps.Config.default(amps.SNOWFLAKE)
    c.nx, c.ny, c.tile, c.mode, c.flags, c.stencil = nx, ny, tile, mode, flags, stencil
    c.params[amps.SF["CX"]], c.params[amps.SF["CY"]], c.params[amps.SF["R2"]] = nx // 2, ny // 2, 36
    c.params[amps.SF["ANISO"]] = 6 if stencil == amps.STENCIL_REF else 4
    return c


def state(ctx, n):
    i = ctx.info()
    out = [ctx.get_field(f, inst=j) for f in range(2) for j in range(n)] + [ctx.get_tile_types(j) for j in range(n)]
    return out, (i.fp64_tile_updates, i.low_full_tile_updates, i.low_listed_tile_updates, i.hi_frac_mean,
                 i.hi_frac_last)


@pytest.mark.parametrize("busy", [False, True])
@pytest.mark.parametrize("mode,flags", [("ADAPTIVE", 0), ("ADAPTIVE", 1), ("PURE_HALF2", 0), ("PURE_HALF2", 1)])
@pytest.mark.parametrize("tile", [16, 32])
def test_one_launch_equals_two(amps, tile, mode, flags, busy):
    small = SIDES[tile][:2]
    batches = [[s] for s in SIDES[tile]] + [small + [(10 * tile, 3 * tile)]]
    for k, sides in enumerate(batches):
        st = amps.STENCIL_REF if k % 2 else amps.STENCIL_LAP5
        cfgs = [config(amps, nx, ny, tile, getattr(amps, mode), flags, st) for nx, ny in sides]
        runs = []
        for timed in ((0, 1), (), (0,), (1,)):  # the 23-step parts, of two, with sweep timing (two launches)
            with amps.Context(cfgs) as ctx:
                ctx.init()
                if busy:
                    for j, (nx, ny) in enumerate(sides):
                        y, x = np.mgrid[0:ny, 0:nx]
                        p = 0.5 + 0.45 * np.sin(x / 9.0) * np.sin(y / 7.0)
                        ctx.set_field(0, np.where(x < nx // 2, p, 0.0), inst=j)
                for part in range(2):
                    ctx.set_kernel_timing(part in timed)
                    ctx.step(23)
                runs.append(state(ctx, len(sides)))
        for got, info in runs[1:]:
            assert info == runs[0][1]
            for g, r in zip(got, runs[0][0]):
                np.testing.assert_array_equal(g, r)

"""Classification and work-lists: the tile types of a monitor pass equal the
rule applied on the host to the pass's own monitor values, for dilations below,
at and above one round of eight neighbour loads; and the two-launch step's lists
hold every tile once where the tile count is no multiple of four."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def config(amps, nx, ny, tile, **kw):
    c = amps.Config.default(amps.SNOWFLAKE)
    c.nx, c.ny, c.tile, c.mode, c.monitor = nx, ny, tile, amps.ADAPTIVE, amps.MON_GRADIENT
    c.params[amps.SF["CX"]], c.params[amps.SF["CY"]], c.params[amps.SF["R2"]] = nx // 2, ny // 2, 25
    for k, v in kw.items():
        setattr(c, k, v)
    return c


@pytest.mark.parametrize("dilate", [0, 1, 3, 4, 9])
def test_types_follow_the_rule(amps, dilate):
    cfgs = [config(amps, 16 * tx, 16 * ty, 16, threshold=0.05, dilate=dilate)
            for tx, ty in ((1, 1), (17, 9), (40, 23))]
    with amps.Context(cfgs) as ctx:
        ctx.init()
        ctx.step(10)
        ctx.monitor_now()
        for j in range(len(cfgs)):
            md = ctx.get_monitor_values(j)
            ty, tx = md.shape
            m = np.full((ty + 2, tx + 2), -np.inf)
            m[1:-1, 1:-1] = md
            m = np.max([m[1:-1, 1:-1], m[:-2, 1:-1], m[2:, 1:-1], m[1:-1, :-2], m[1:-1, 2:]], axis=0)
            hit = np.zeros((ty, tx), bool)
            for y in range(ty):
                for x in range(tx):
                    box = md[max(y - dilate, 0):y + dilate + 1, max(x - dilate, 0):x + dilate + 1]
                    hit[y, x] = max(m[y, x], box.max()) >= 0.05
            np.testing.assert_array_equal(ctx.get_tile_types(j), np.where(hit, 2, 1))


@pytest.mark.parametrize("tile,tx,ty", [(16, 65, 65), (16, 83, 51), (32, 33, 63)])  # 4225, 4233 and 2079 tiles
def test_lists_hold_every_tile_once(amps, tile, tx, ty):
    c = config(amps, tile * tx, tile * ty, tile, flags=amps.FLAG_NO_SKIP, monitor_every=1000)
    rng = np.random.default_rng(tx)
    with amps.Context(c) as ctx:
        ctx.init()
        ctx.step(1)
        a = ctx.info()
        t = np.where(rng.random((ty, tx)) < 0.3, 2, 1).astype(np.int32)
        t[-1, -5:] = [2, 1, 1, 2, 1]
        ctx.set_tile_types(t)
        ctx.step(3)
        b = ctx.info()
        assert b.fp64_tile_updates - a.fp64_tile_updates == 3 * int((t == 2).sum())
        assert b.low_full_tile_updates - a.low_full_tile_updates == 3 * int((t == 1).sum())

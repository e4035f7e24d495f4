"""The adaptive sintering sweep's 512-thread workgroups (up to 256 tiles of
32^2) against the 256-thread ones that more tiles take: a grid of at most 256
tiles alone, and in a batch whose tiles exceed 256, ends in the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def config(amps, nx, ny, mode, flags):
    c = amps.Config.default(amps.SINTERING)
    c.nx, c.ny, c.tile, c.mode, c.flags = nx, ny, 32, mode, flags
    c.params[amps.SN["X1"]], c.params[amps.SN["X2"]] = nx * 0.4, nx * 0.6
    c.params[amps.SN["Y1"]] = c.params[amps.SN["Y2"]] = ny * 0.5
    c.params[amps.SN["R1"]] = c.params[amps.SN["R2"]] = min(nx, ny) * 0.11
    return c


@pytest.mark.parametrize("flags", [0, 2])
@pytest.mark.parametrize("mode", ["ADAPTIVE", "PURE_HALF2"])
@pytest.mark.parametrize("nx,ny", [(32, 32), (96, 64), (256, 1024)])   # 1, 6 and 256 tiles
def test_same_bits_alone_and_in_a_large_batch(amps, nx, ny, mode, flags):
    mode = getattr(amps, mode)
    cfg = config(amps, nx, ny, mode, flags)
    out = []
    for batch in ([cfg], [cfg, config(amps, 736, 736, mode, flags)]):  # the second: 529 tiles more
        with amps.Context(batch) as ctx:
            ctx.init()
            if mode == amps.ADAPTIVE and min(nx, ny) > 32:             # neighbours of both types
                t = np.arange((nx // 32) * (ny // 32)) % 3 == 0
                ctx.set_tile_types(np.where(t, 2, 1).astype(np.int32).reshape(ny // 32, nx // 32))
            ctx.step(13)
            out.append([ctx.get_field(f) for f in range(3)] + [ctx.get_tile_types()])
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)

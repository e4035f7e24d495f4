"""Grain growth's sum-of-squares pass after a monitor pass, on more and on
fewer tiles than it takes one by one (4,096): the next step of every FP64 tile
agrees with the update restated in numpy from the decoded fields, to the FP64 bar
of 1e-12 (a stale sum differs by 1e-5 and more, the fp16 rounding of a field)."""
import numpy as np
import pytest

from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,q,tile", [(1040, 3, 16), (1040, 20, 16), (2080, 2, 32), (1024, 3, 16), (96, 5, 32)])
def test_sums_follow_the_conversions(amps, n, q, tile):
    c = amps.Config.default(amps.GRAINGROWTH)
    c.nx = c.ny = n
    c.q, c.tile, c.mode, c.monitor, c.monitor_field, c.threshold = q, tile, amps.ADAPTIVE, amps.MON_SPATIAL, -1, 0.9
    c.monitor_every = 1000
    nt = n // tile
    rng = np.random.default_rng(n + q)
    base = rng.uniform(0.0, 1.0, (n, n))
    p = np.array(c.params[:12])
    with amps.Context(c) as ctx:
        ctx.init()
        ctx.step(1)  # step 0's own monitor pass
        for rnd in range(2):  # most tiles become low, then some change either way
            for f in range(q):
                share = 0.3 if rnd == 0 else 0.4
                amp = np.repeat(np.repeat(rng.uniform(0.3, 1.2, (nt, nt)) * (rng.random((nt, nt)) < share) + 0.2, tile, 0), tile, 1)
                ctx.set_field(f, np.ascontiguousarray(np.roll(base, (7 * f, 5 * f), (0, 1)) * amp))
            ctx.monitor_now()
            types = ctx.get_tile_types()
            assert 0 < (types == 2).sum() < types.size
            fields = [ctx.get_field(f) for f in range(q)]
            s2 = sum(f * f for f in fields)
            ctx.step(1)
            for f in (0, q // 2, q - 1):
                e = fields[f]
                row = np.roll(e, 1, 1) + e + np.roll(e, -1, 1)
                lap = (row + np.roll(row, 1, 0) + np.roll(row, -1, 0) - 9 * e) / (p[0] * p[1])
                df = 2 * p[7] * e * (s2 - e * e) + p[6] * e ** 3 - p[5] * e
                want = e - p[2] * p[3] * (df - p[4] * lap)
                hi = np.repeat(np.repeat(types[f] == 2, tile, 0), tile, 1)
                if hi.any():
                    assert rel_err(ctx.get_field(f)[hi], want[hi]) <= 1e-12, (rnd, f)

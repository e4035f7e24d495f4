"""A monitor pass whose (group, tile) items outnumber one round of the
classification's workgroups (2,048 of 64 items): 36 fields of 4,225 tiles, and
the smaller passes beside it.  The types follow the rule applied on the host to
the pass's own monitor values; tiles that become low hold exactly the
round-to-nearest-even encoding of their values, all others are untouched; the
FP64 fractions are those of the types.  A second pass on new values converts in
both directions."""
import numpy as np
import pytest

from tests.test_gpu_convert_grid import encode_decode

pytestmark = pytest.mark.gpu


def rule(md, thr):
    q, ty, tx = md.shape
    m = np.full((q, ty + 2, tx + 2), -np.inf)
    m[:, 1:-1, 1:-1] = md
    m = np.max([m[:, 1:-1, 1:-1], m[:, :-2, 1:-1], m[:, 2:, 1:-1], m[:, 1:-1, :-2], m[:, 1:-1, 2:]], axis=0)
    return np.where(m >= thr, 2, 1)


@pytest.mark.parametrize("n,q,tile", [(1040, 36, 16), (128, 5, 32), (64, 2, 16)])
def test_pass_beyond_one_round(amps, n, q, tile):
    c = amps.Config.default(amps.GRAINGROWTH)
    c.nx = c.ny = n
    c.q, c.tile, c.mode, c.monitor, c.monitor_field, c.threshold = q, tile, amps.ADAPTIVE, amps.MON_SPATIAL, -1, 0.9
    nt = n // tile
    rng = np.random.default_rng(n)
    base = rng.uniform(0.0, 1.0, (n, n))
    with amps.Context(c) as ctx:
        ctx.init()
        types = np.full((q, nt, nt), 2)
        fractions = []
        for rnd in range(2):
            fields = []
            for f in range(q):
                amp = np.repeat(np.repeat(rng.uniform(0.3, 1.2, (nt, nt)) * (rng.random((nt, nt)) < 0.3) + 0.2, tile, 0), tile, 1)
                ctx.set_field(f, np.ascontiguousarray(np.roll(base, (7 * f, 5 * f), (0, 1)) * amp))
                fields.append(ctx.get_field(f))  # low tiles as stored
            ctx.monitor_now()
            new = rule(ctx.get_monitor_values(), 0.9)
            got = ctx.get_tile_types()
            assert np.array_equal(got, new) and 0 < (new == 1).sum() < new.size
            fractions.append((new == 2).mean())
            for f in range(q):
                enc = np.repeat(np.repeat((types[f] == 2) & (new[f] == 1), tile, 0), tile, 1)
                want = np.where(enc, encode_decode(fields[f], tile), fields[f])
                assert np.array_equal(ctx.get_field(f), want), (rnd, f)
            if rnd:
                assert ((types == 1) & (new == 2)).any() and ((types == 2) & (new == 1)).any()
            types = new
        info = ctx.info()
        assert info.monitor_passes == 2
        assert abs(info.hi_frac_last - fractions[1]) <= 1e-12
        assert abs(info.hi_frac_mean - 0.5 * sum(fractions)) <= 1e-12

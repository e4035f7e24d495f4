"""Conversion and grain-growth aux passes whose items outnumber their
workgroups: 36 x 4225 (field, tile) items go round the conversion's workgroups
and their 64 items more than once, 4225 tiles round the aux pass's.

Conversion: every low field-tile decodes to exactly the IEEE
round-to-nearest-even encoding of its values (numpy's float64 -> float16 of
values scaled by the tile's power of two), every FP64 one is untouched.  Aux:
one FP64 step from the fields agrees with the oracle's, to the FP64 bar of
1e-12 relative (its per-cell sum of squares is the aux pass's).
"""
import numpy as np
import pytest

from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


def encode_decode(f, tile):
    """Per-tile fp16 round trip of a field (offset = mid-range, power-of-two scale)."""
    ny, nx = f.shape
    v = f.reshape(ny // tile, tile, nx // tile, tile)
    mn, mx = v.min(axis=(1, 3), keepdims=True), v.max(axis=(1, 3), keepdims=True)
    off, hw = 0.5 * (mn + mx), 0.5 * (mx - mn)
    ex = np.where(hw > 0, np.frexp(hw)[1], -100).clip(-100, 100)
    h = np.ldexp(v - off, 14 - ex).astype(np.float16).astype(np.float64)
    return (off + np.ldexp(h, ex - 14)).reshape(ny, nx)


@pytest.mark.parametrize("n,q,tile", [(1040, 36, 16), (64, 3, 16), (96, 2, 32)])
def test_conversion_and_aux_cover_every_item(amps, O, n, q, tile):
    c = amps.Config.default(amps.GRAINGROWTH)
    c.nx = c.ny = n
    c.q, c.tile, c.mode = q, tile, amps.STATIC_MAP
    rng = np.random.default_rng(n)
    base = rng.uniform(-0.2, 1.0, (n, n))
    fields = [np.ascontiguousarray(np.roll(base, (17 * f, 5 * f), (0, 1)) * (0.3 + 0.02 * f)) for f in range(q)]
    nt = n // tile
    types = rng.integers(1, 3, (q, nt, nt)).astype(np.int32)
    with amps.Context(c) as ctx:
        ctx.init()
        for f in range(q):
            ctx.set_field(f, fields[f])
        ctx.step(1)
        p = np.array(c.params[:12])
        if q <= 3:
            ref = O.gg_step(np.stack(fields), p, stencil=c.stencil, bc=c.bc)
        else:  # the sum over 36 fields in numpy, one field's update at a time
            ref = None
            s2 = sum(f * f for f in fields)
        for f in (0, q - 1):
            got = ctx.get_field(f)
            if ref is not None:
                want = ref[f]
            else:
                e = fields[f]
                row = np.roll(e, 1, 1) + e + np.roll(e, -1, 1)
                lap = (row + np.roll(row, 1, 0) + np.roll(row, -1, 0) - 9 * e) / (p[0] * p[1])
                df = 2 * p[7] * e * (s2 - e * e) + p[6] * e ** 3 - p[5] * e
                want = e - p[2] * p[3] * (df - p[4] * lap)
            assert rel_err(got, want) <= 1e-12, f
        for f in range(q):
            ctx.set_field(f, fields[f])
        ctx.set_tile_types(types)
        low = np.repeat(np.repeat(types, tile, 1), tile, 2) == 1
        for f in range(q):
            want = np.where(low[f], encode_decode(fields[f], tile), fields[f])
            assert np.array_equal(ctx.get_field(f), want), f

"""amps_get_field's check for non-finite values, made on the device: a NaN or
an infinity in any cell (first, last, inside) of a decoded or a plain field
fails the read with AMPS_E_NONFINITE, after the values have been copied; the
next read of a finite field succeeds, and an untouched field of the same
context too.  Extreme finite values (largest, subnormal, -0) pass unchanged.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model,mode,tile", [(1, 0, 16), (1, 0, 32), (1, 1, 16), (1, 3, 32), (2, 1, 32), (3, 3, 16)])
@pytest.mark.parametrize("ny,nx", [(32, 32), (64, 96)])
def test_nonfinite_values_are_reported(amps, model, mode, tile, ny, nx):
    c = amps.Config.default(model)
    c.nx, c.ny, c.tile, c.mode = nx, ny, tile, mode
    base = np.random.default_rng(1).uniform(0.1, 0.9, (ny, nx))
    with amps.Context(c) as ctx:
        ctx.init()
        if mode == 3:  # a mix of FP64 and low tiles
            ctx.set_tile_types(np.random.default_rng(2).integers(1, 3, (ny // tile, nx // tile)).astype(np.int32))
        ctx.set_field(0, base)
        ctx.set_field(1, base)
        for cell in ((0, 0), (ny - 1, nx - 1), (ny // 2, 5)):
            for v in (np.nan, np.inf, -np.inf):
                a = base.copy()
                a[cell] = v
                ctx.set_field(0, a)
                out = np.zeros((ny, nx))
                rc = amps.lib().amps_get_field(ctx._h, 0, 0, out.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), out.size)
                assert rc == -5
                assert not np.isfinite(out[cell])
                assert np.all(np.isfinite(ctx.get_field(1)))
        ctx.set_field(0, base)
        assert np.all(np.isfinite(ctx.get_field(0)))


def test_extreme_finite_values_pass(amps):
    c = amps.Config.default(amps.SNOWFLAKE)
    c.nx = c.ny = 32
    a = np.zeros((32, 32))
    a[0, :4] = [np.finfo(float).max, -np.finfo(float).max, 5e-324, -0.0]
    with amps.Context(c) as ctx:
        ctx.init()
        ctx.set_field(0, a)
        got = ctx.get_field(0)
        assert np.array_equal(got, a) and np.array_equal(np.signbit(got), np.signbit(a))

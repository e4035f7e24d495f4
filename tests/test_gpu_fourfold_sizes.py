"""The single FP64 snowflake step at both sides of the sizes where it drops the
branch-free four-fold path: with sweep timing on a context takes single steps,
whose fields and those of the no-allocation step are bitwise alike, and each
step agrees with the oracle's from the same state to the FP64 bar."""
import numpy as np
import pytest

from tests.helpers import rel_err, smooth_fields
from tests.test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


SMALL = [(t, s, b, 1024, nx) for t, s, b in ((16, 0, 0), (32, 0, 1), (16, 1, 1), (32, 1, 0)) for nx in (1024, 1056)]
LARGE = [(t, s, 1, n, n) for t, s in ((32, 0), (16, 1)) for n in (2880, 2912)]


@pytest.mark.parametrize("tile,stencil,bc,ny,nx", SMALL + LARGE)
def test_same_bits_on_both_sides(amps, O, tile, stencil, bc, ny, nx):
    c = amps.Config.default(amps.SNOWFLAKE)
    c.nx, c.ny, c.tile, c.stencil, c.bc, c.seed = nx, ny, tile, stencil, bc, 3
    c.params[amps.SF["NOISE"]] = 0.01
    assert c.params[amps.SF["ANISO"]] == 4
    phi, T = smooth_fields(nx, ny, seed=tile, nbump=4)
    with amps.Context(c) as ctx:
        ctx.init()
        ctx.set_field(0, phi)
        ctx.set_field(1, T)
        ctx.set_kernel_timing(True)
        states = [np.stack([phi, T])]
        for _ in range(2):
            ctx.step(1)
            states.append(np.stack([ctx.get_field(0), ctx.get_field(1)]))
    ref = states[2]
    hip = Hip(amps)
    try:
        a, b = hip.alloc(ref.nbytes), hip.alloc(ref.nbytes)
        hip.upload(a, np.stack([phi, T]))
        amps.sf_step_fp64_noalloc(c, a, b, 0)
        amps.sf_step_fp64_noalloc(c, b, a, 1)
        hip.sync()
        assert np.array_equal(hip.download(a, ref.shape), ref)
    finally:
        hip.free()
    if ny == 1024:
        p = np.array(c.params[:17])
        for k in range(2):
            po, to = O.sf_step(states[k][0], states[k][1], p, stencil=stencil, bc=bc, seed=c.seed, step=k)
            assert rel_err(states[k + 1][0], po) <= 1e-12 and rel_err(states[k + 1][1], to) <= 1e-12, k

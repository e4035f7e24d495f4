"""The fused reverse step (one kernel per model and step) at the shapes where
its boxes can go wrong: grids of one tile (every halo cell is a wrapped or
mirrored cell of the tile itself), of one tile by two or three (a tile with
an edge on three sides), tile sizes 16 and 32, both boundaries and both
Laplacian reaches, and a batch that mixes the two reaches.

J = sum(W u_final) with seeded weights; dJ/du_0 by the dot-product identity
and every parameter gradient, against the oracle's forward-mode tangents.
Both sides are sums of at most 2e4 products of order 1 whose terms agree to
~1e-14 relative after 4 steps; with sums a hundredth of their absolute terms'
sum the rounding stays below 1e-10, and 1e-9 is the bar.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STEPS, CKPT = 4, 3
SHAPES = [(16, 16, 16), (16, 48, 16), (32, 16, 16), (32, 32, 32), (64, 32, 32), (32, 96, 32)]  # ny, nx, tile


def fields(ny, nx, k, seed):
    """k random smooth fields in (0.1, 0.9) with full variation up to the edges."""
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:ny, 0:nx]
    out = []
    for _ in range(k):
        a = rng.uniform(0.2, 0.6, 4)
        ph = rng.uniform(0, 6, 4)
        out.append(0.5 + 0.2 * np.sin(a[0] * x + ph[0]) * np.cos(a[1] * y + ph[1])
                   + 0.15 * np.sin(a[2] * x + a[3] * y + ph[2]))
    return [np.ascontiguousarray(f) for f in out]


def check(amps, O, cfg, ids, u0, tangent, seed):
    rng = np.random.default_rng(seed)
    W = [rng.uniform(0.5, 1.5, u0[0].shape) for _ in u0]
    v = [rng.uniform(0.5, 1.5, u0[0].shape) for _ in u0]
    with amps.Context(cfg) as ctx:
        ctx.init()
        for f, a in enumerate(u0):
            ctx.set_field(f, a)
        ctx.tape_begin(CKPT)
        ctx.step(STEPS)
        g, du0 = ctx.adjoint([np.stack(W)], ids, want_du0=True)
    for k, pid in enumerate(ids):
        ref = sum(float(np.sum(w * d)) for w, d in zip(W, tangent(pid, None)))
        assert abs(g[0, k] - ref) <= 1e-9 * abs(ref), (pid, g[0, k], ref)
    lhs = sum(float(np.sum(a * b)) for a, b in zip(du0[0], v))
    rhs = sum(float(np.sum(w * d)) for w, d in zip(W, tangent(0, v)))
    assert abs(lhs - rhs) <= 1e-9 * abs(rhs), (lhs, rhs)


@pytest.mark.parametrize("ny,nx,tile", SHAPES)
@pytest.mark.parametrize("stencil,bc", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_snowflake_reverse_step_edges(amps, O, ny, nx, tile, stencil, bc):
    cfg = amps.Config.default(amps.SNOWFLAKE)
    cfg.nx, cfg.ny, cfg.tile, cfg.stencil, cfg.bc = nx, ny, tile, stencil, bc
    cfg.params[amps.SF["NOISE"]] = 0.01
    p = np.array(cfg.params[:17])
    phi, T = fields(ny, nx, 2, seed=ny + nx)

    def tangent(pid, v):
        kw = {} if v is None else dict(dphi=v[0], dT=v[1])
        return O.sf_tangent(phi, T, p, STEPS, pid, stencil=stencil, bc=bc, seed=cfg.seed, **kw)[2:]

    check(amps, O, cfg, [O.GRAD_SF[k] for k in ("DELTA", "KAPPA", "EPSB", "TAU")], [phi, T], tangent, 7)


@pytest.mark.parametrize("ny,nx,tile", SHAPES)
@pytest.mark.parametrize("bc", [0, 1])
def test_sintering_reverse_step_edges(amps, O, ny, nx, tile, bc):
    cfg = amps.Config.default(amps.SINTERING)
    cfg.nx, cfg.ny, cfg.tile, cfg.bc = nx, ny, tile, bc
    p = np.array(cfg.params[:20])
    u0 = fields(ny, nx, 3, seed=ny * nx)

    def tangent(pid, v):
        kw = {} if v is None else dict(dc=v[0], de1=v[1], de2=v[2])
        return O.sn_tangent(*u0, p, STEPS, pid, bc=bc, **kw)[3:]

    check(amps, O, cfg, [O.GRAD_SN[k] for k in ("DSURF", "DGB", "KC", "KE", "L", "DVOL")], u0, tangent, 9)


def test_batch_mixing_laplacian_reaches(amps, O):
    cfgs = []
    for i, (n, stencil) in enumerate(((32, 0), (64, 1), (32, 1))):
        c = amps.Config.default(amps.SNOWFLAKE)
        c.nx = c.ny = n
        c.tile, c.stencil, c.bc, c.seed = 16, stencil, i % 2, 5 + i
        cfgs.append(c)
    u0 = [fields(c.ny, c.nx, 2, seed=c.nx + i) for i, c in enumerate(cfgs)]
    ids = [O.GRAD_SF["DELTA"], O.GRAD_SF["KAPPA"]]
    with amps.Context(cfgs) as ctx:
        ctx.init()
        for i, u in enumerate(u0):
            for f in range(2):
                ctx.set_field(f, u[f], inst=i)
        ctx.tape_begin(CKPT)
        ctx.step(STEPS)
        g, _ = ctx.adjoint([np.ones((2, c.ny, c.nx)) for c in cfgs], ids)
    for i, c in enumerate(cfgs):
        for k, pid in enumerate(ids):
            d = O.sf_tangent(*u0[i], np.array(c.params[:17]), STEPS, pid, stencil=c.stencil, bc=c.bc, seed=c.seed)[2:]
            ref = float(np.sum(d[0]) + np.sum(d[1]))
            assert abs(g[i, k] - ref) <= 1e-9 * abs(ref), (i, pid, g[i, k], ref)

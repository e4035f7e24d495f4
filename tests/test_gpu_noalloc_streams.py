"""amps_sf_step_fp64_noalloc keeps nothing on the device between calls: calls
of two configurations interleaved on two streams, with no synchronisation
between them, give the bits that each gives alone; and a call recorded into a
HIP graph gives the same on every replay, with eager calls of another
configuration between the replays.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def setup(amps, n, tile, stencil, bc, aniso, seed):
    c = amps.Config.default(amps.SNOWFLAKE)
    c.nx, c.ny, c.tile, c.stencil, c.bc, c.seed = n, n + tile, tile, stencil, bc, seed
    c.params[amps.SF["ANISO"]] = aniso
    c.params[amps.SF["NOISE"]] = 0.01
    g = torch.Generator().manual_seed(seed)
    x = torch.rand(2, c.ny, c.nx, generator=g, dtype=torch.float64).cuda()
    return c, x


def chain(amps, c, x, steps, stream):
    a, b = x.clone(), torch.empty_like(x)
    for k in range(steps):
        amps.sf_step_fp64_noalloc(c, a.data_ptr(), b.data_ptr(), k, stream.cuda_stream)
        a, b = b, a
        yield a


@pytest.mark.parametrize("tile", [16, 32])
def test_interleaved_streams_and_graph_replays(amps, tile):
    c1, x1 = setup(amps, 64, tile, 0, 0, 4, 3)
    c2, x2 = setup(amps, 160, tile, 1, 1, 6, 4)
    main = torch.cuda.current_stream()
    ref1, ref2 = list(chain(amps, c1, x1, 6, main))[-1].clone(), list(chain(amps, c2, x2, 6, main))[-1].clone()
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s1):
        g1 = chain(amps, c1, x1, 6, s1)
        r1 = next(g1)
    with torch.cuda.stream(s2):
        g2 = chain(amps, c2, x2, 6, s2)
        r2 = next(g2)
    for r1, r2 in zip(g1, g2):
        pass
    torch.cuda.synchronize()
    assert torch.equal(r1, ref1) and torch.equal(r2, ref2)

    out = torch.empty_like(x1)
    want = torch.empty_like(x1)
    amps.sf_step_fp64_noalloc(c1, x1.data_ptr(), want.data_ptr(), 5, main.cuda_stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        amps.sf_step_fp64_noalloc(c1, x1.data_ptr(), out.data_ptr(), 5, torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        out.zero_()
        graph.replay()
        other = list(chain(amps, c2, x2, 6, main))[-1]
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(other, ref2)

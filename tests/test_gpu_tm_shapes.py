"""The strip shapes the plan chooses by a grid's cells -- both sides of each
change, wide and tall grids -- against another strip shape, bit for bit."""
import numpy as np
import pytest
import torch

from conftest import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,depth,rows", [
    (1640, 1651, 8, 8), (9000, 600, 8, 16), (500, 11200, 10, 16), (2569, 2570, 10, 28),
    (9001, 1210, 10, 47), (3320, 3320, 11, 47), (1100, 17000, 11, 80),
])
def test_default_strips(gpu, nx, ny, depth, rows):
    from simulation_amd import fd2d
    print(f"[tm shapes] {nx}x{ny}", flush=True)
    f = torch.randn((nx, ny), generator=torch.Generator(gpu).manual_seed(nx), device=gpu)
    out = []
    for kw in ({}, dict(depth=5, rows=37)):
        cfg = fd2d.TMConfig(nx=nx, ny=ny, ns=44, npml=8, sources=[(nx // 2, 20, 20, 6.0)],
                            cylinders=[(nx / 2, ny / 2, 90, 4.0, 0.02)], probes=[(9, ny - 9)], **kw)
        s = fd2d.build_solver(cfg, gpu)
        if not kw:
            p = s.plan(2 * depth)
            assert (p["depth"], p["rows"]) == (depth, rows)
        s.dz.copy_(f)
        s.run(2 * depth)
        s.run(44 - 2 * depth)
        out.append(s)
    a, b = out
    for k in fd2d.STATE:
        assert torch.equal(getattr(a, k).view(torch.int32), getattr(b, k).view(torch.int32)), k
    assert same_bits(np.asarray(a.probe_traces()), np.asarray(b.probe_traces()))

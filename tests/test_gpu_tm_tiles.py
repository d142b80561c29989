"""The register tiles small TM grids run (fd2d_rt.hip) against the oracle and
against the strip form, bit for bit: one tile, the first cuts, the tile shapes
the plan chooses between, sources and probes on grid edges and tile cuts, call
lengths from two steps on; plane wave and running DFT against the strips."""
import numpy as np
import pytest
import torch

from conftest import same_bits
from test_gpu_tm_bodies import run_both

pytestmark = pytest.mark.gpu


# sides: one tile (32 x 64), one cell more, 2 cells; depth 14 (60, 130), 12
# (300) and 8 (380) at 8 waves, 12 waves (490), 16 waves at depth 12, 10 and 8
# (600, 700, 740), 8 waves at depth 8 past that (800, 1200); cuts at depth 14: rows 18, 22, .., columns 50, 86, ..
@pytest.mark.parametrize("nx,ny,npml,lossy,src,probes,chunks", [
    (2, 2, -1, False, [], [(1, 1)], (2, 3)),
    (5, 3, -1, True, [(0, 0), (4, 2)], [(4, 2)], (17,)),
    (32, 64, 6, True, [(16, 31)], [(0, 0), (31, 63)], (2, 16, 33)),
    (33, 65, 8, True, [(17, 49), (18, 50)], [(17, 50), (32, 64)], (28, 29, 5)),
    (60, 60, 8, False, [(18, 50)], [(17, 50), (18, 49), (59, 59), (1, 1)], (200,)),
    (63, 62, -1, True, [(22, 10)], [(5, 61)], (70,)),
    (130, 131, 20, True, [(21, 49), (22, 86), (22, 86)], [(22, 86), (129, 130)], (57, 2)),
    (300, 301, 8, False, [(150, 150)], [(20, 52), (299, 0)], (48,)),
    (300, 70, -1, False, [(0, 0), (299, 69)], [(299, 69)], (31,)),
    (40, 700, 8, True, [(20, 350)], [(20, 351)], (33,)),
    (380, 377, 8, True, [(1, 1)], [(24, 56)], (33,)),
    (490, 501, 8, True, [(245, 250)], [(36, 52)], (26,)),
    (600, 607, 100, True, [(300, 300)], [(40, 56)], (17,)),
    (700, 703, 8, True, [(350, 350)], [(54, 54)], (21,)),
    (740, 737, 8, False, [(370, 370)], [(56, 56)], (17,)),
    (800, 797, 8, True, [(400, 400)], [(40, 56)], (18,)),
    (1200, 1203, 8, True, [(600, 600)], [(25, 57)], (15,)),
])
def test_tiles(gpu, oracle, nx, ny, npml, lossy, src, probes, chunks):
    print(f"[tm tiles] {nx}x{ny} npml={npml} lossy={lossy}", flush=True)
    run_both(gpu, oracle, nx, ny, npml, lossy, src, probes, chunks)


def test_tiles_general_body(gpu, oracle):
    """Without a promised band every wave runs the general body."""
    from simulation_amd import fd2d
    print("[tm tiles] no band", flush=True)
    band = fd2d.TMSolver.default_band
    try:
        fd2d.TMSolver.default_band = lambda self: ((0, 0), (0, 0))
        run_both(gpu, oracle, 150, 170, 8, True, [(75, 85)], [(76, 85)], (40,))
    finally:
        fd2d.TMSolver.default_band = band


@pytest.mark.parametrize("nx,ny,npml,nf,lossy,steps", [
    (40, 30, 8, 1, True, 70), (97, 131, 20, 3, True, 130), (150, 140, 8, 0, False, 64),
    (211, 190, 32, 2, False, 67), (400, 397, 20, 3, True, 96), (90, 64, 2, 3, True, 65),
    (650, 640, 20, 3, True, 40), (800, 811, 20, 1, True, 33),
])
def test_plane_wave_tiles_match_strips(gpu, nx, ny, npml, nf, lossy, steps):
    from simulation_amd import fd2d
    print(f"[tm tiles] plane wave {nx}x{ny} npml={npml} nf={nf}", flush=True)
    dt = fd2d.time_step()
    pml = fd2d.new_pmlayer(nx, ny, gpu)
    fd2d.pmlparam(nx, ny, npml, pml)
    md = fd2d.dielectric(nx, ny, npml, 0, dt, 1.0, 0.0, gpu,
                         cylinders=[(nx / 2, ny / 2, min(nx, ny) / 6, 4.0, 0.02)])
    if not lossy:
        md = fd2d.medium(md.naz, None)
    rng = np.random.default_rng(5)
    f = torch.from_numpy(rng.standard_normal((nx, ny)).astype(np.float32)).to(gpu)
    out = []
    for kw in ({}, dict(depth=4, rows=7)):
        s = fd2d.PlaneWaveSolver(nx, ny, npml, pml, md, 2 * steps, freq=(5e7, 3e8, 7e8)[:nf], dt=dt,
                                 probes=[(nx // 2, ny // 2), (npml, npml)], device=gpu, **kw)
        s.tm.dz.copy_(f)
        s.run(steps)
        s.run(9)
        out.append(s)
    a, b = out
    for k in fd2d.STATE:
        if getattr(a.tm, k) is not None:
            assert same_bits(getattr(a.tm, k).cpu().numpy(), getattr(b.tm, k).cpu().numpy()), k
    for k in ("ezi", "hxi", "bc"):
        assert same_bits(getattr(a, k).cpu().numpy(), getattr(b, k).cpu().numpy()), k
    if nf:
        for k, v in a.ft._asdict().items():
            assert same_bits(v.cpu().numpy(), getattr(b.ft, k).cpu().numpy()), k
    assert same_bits(a.tm.probe_traces(), b.tm.probe_traces())


def test_tiles_in_a_replayed_graph(gpu):
    """A captured run, replayed with eager work in between, against eager runs."""
    from simulation_amd import fd2d
    print("[tm tiles] graph", flush=True)
    cfg = fd2d.TMConfig(nx=100, ny=90, ns=400, npml=8, sources=[(50, 45, 20, 6.0)],
                        cylinders=[(50, 45, 12, 4.0, 0.02)], probes=[(50, 50)])
    a, b = fd2d.build_solver(cfg, gpu), fd2d.build_solver(cfg, gpu)
    a.run(40)
    b.run(40)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        a.run(40)
    for _ in range(3):
        g.replay()                       # steps 41 .. 80 again
        b.t = 40
        b.run(40)
        torch.cuda.synchronize()
        for k in fd2d.STATE:
            assert same_bits(getattr(a, k).cpu().numpy(), getattr(b, k).cpu().numpy()), k

"""A register-tile shape given back -- the reported one, others, one step, a
plane wave, a batch, the learned boundary -- against strips, bit for bit."""
import numpy as np
import pytest
import torch

from conftest import same_bits

pytestmark = pytest.mark.gpu

TILE = 64


def _same(a, b, names):
    for k in names:
        if getattr(a, k) is not None:
            assert same_bits(getattr(a, k).cpu().numpy(), getattr(b, k).cpu().numpy()), k


@pytest.mark.parametrize("nx,ny,shape", [
    (60, 60, None), (33, 65, None), (700, 703, None),
    (60, 60, (16, 36)), (61, 130, (1, 4)), (97, 211, (9, 20)), (150, 170, (16, 64)), (2, 2, (3, 12)),
    (1700, 1650, (8, 32)),
])
def test_tm_shape_given_back(gpu, nx, ny, shape):
    from simulation_amd import fd2d
    print(f"[plan given back] {nx}x{ny} {shape}", flush=True)
    npml = 8 if min(nx, ny) > 32 else -1
    out = []
    for tiles in (True, False):
        cfg = fd2d.TMConfig(nx=nx, ny=ny, ns=110, npml=npml, sources=[(nx // 2, ny // 2, 20, 6.0)],
                            cylinders=[], probes=[(nx - 1, ny // 2)])
        s = fd2d.build_solver(cfg, gpu)
        if tiles:
            p = s.plan(50)
            s.depth, s.rows, s.cols = (p["depth"], p["rows"], p["cols"]) if shape is None else (*shape, TILE)
            assert s.cols == TILE
            if shape is None:
                assert s.plan(50) == p
        else:
            s.depth, s.rows = 5, 7
        s.dz.copy_(torch.randn((nx, ny), generator=torch.Generator(gpu).manual_seed(nx), device=gpu))
        for n in (50, 1, 57, 2):
            s.run(n)
        out.append(s)
    _same(*out, fd2d.STATE)
    assert same_bits(np.asarray(out[0].probe_traces()), np.asarray(out[1].probe_traces()))


@pytest.mark.parametrize("nf", [0, 3])
def test_plane_wave_shape_given_back(gpu, nf):
    from simulation_amd import fd2d
    print(f"[plan given back] plane wave nf={nf}", flush=True)
    nx, ny, npml = 131, 97, 20
    pml = fd2d.new_pmlayer(nx, ny, gpu)
    fd2d.pmlparam(nx, ny, npml, pml)
    md = fd2d.dielectric(nx, ny, npml, 10, fd2d.time_step(), 4.0, 0.02, gpu)
    out = []
    for kw in (dict(depth=10, rows=24, cols=TILE), dict(depth=4, rows=7)):
        s = fd2d.PlaneWaveSolver(nx, ny, npml, pml, md, 200, freq=(5e7, 3e8, 7e8)[:nf],
                                 probes=[(60, 50)], device=gpu, **kw)
        for n in (65, 1, 30):
            s.run(n)
        out.append(s)
    a, b = out
    _same(a.tm, b.tm, fd2d.STATE)
    _same(a, b, ("ezi", "hxi", "bc"))
    for x, y in zip(a.ft or (), b.ft or ()):
        assert same_bits(x.cpu().numpy(), y.cpu().numpy())


def test_batch_shape_given_back(gpu):
    from simulation_amd.batch import BatchSolver, c3_specs
    print("[plan given back] batch", flush=True)
    specs = c3_specs(3, count=5, lo=96, hi=300)
    a, b = (BatchSolver(specs, 60, device=gpu) for _ in range(2))
    d = a.desc
    assert d.cols == TILE
    b.plan(d.depth, d.rows, d.cols, d.waves)
    assert [getattr(b.desc, k) for k in ("depth", "rows", "cols", "waves", "nunits")] == \
           [getattr(d, k) for k in ("depth", "rows", "cols", "waves", "nunits")]
    c = BatchSolver(specs, 60, depth=5, rows=20, cols=TILE, device=gpu)
    e = BatchSolver(specs, 60, depth=4, rows=30, device=gpu)
    for s in (a, b, c, e):
        s.run(37)
    for k in range(len(specs)):
        want = e.grid_state(k)
        for s in (a, b, c):
            got = s.grid_state(k)
            for f in want:
                assert same_bits(got[f], want[f]), (k, f)


def test_learned_boundary_takes_a_tile_shape(gpu):
    from simulation_amd import fd2d, learned
    print("[plan given back] learned", flush=True)
    md = fd2d.dielectric(150, 140, 0, 12, fd2d.time_step(), 4.0, 0.02, gpu)
    out = []
    for tiles in (True, False):
        s = learned.LearnedTMSolver(150, 140, learned.load(device=gpu), md, nsteps_max=40, device=gpu)
        if tiles:
            p = s.tm.plan(40)
            s.tm.depth, s.tm.rows, s.tm.cols = p["depth"], p["rows"], p["cols"]
        s.tm.dz[75, 70] = 1.0
        s.run(40)
        out.append(s.tm)
    _same(*out, ("dz", "iz", "ez", "hx", "hy"))

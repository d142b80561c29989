"""Batches in the library's own launch shapes -- register tiles or strips, one
workgroup a unit, depth and rows by the cells of all grids -- and in persistent
waves against single-grid runs, bit for bit: fewer units than XCDs, unit counts
that 8 does not divide, grids of edge units only, row blocks cut short, row-,
column-only and corner units, both sides of each change of shape."""
import pytest

from conftest import same_bits

pytestmark = pytest.mark.gpu


def _specs(sides):
    from simulation_amd.batch import GridSpec
    out = []
    for k, (nx, ny) in enumerate(sides):
        cyl = [(nx / 2, ny / 2, min(nx, ny) / 7, 3.0, 0.02)] if min(nx, ny) > 60 else []
        src = (nx // 3, ny // 2, 20, 6.0) if k % 3 != 1 else None
        prb = (nx // 3 + 3, ny // 2) if k % 3 != 2 else None
        out.append(GridSpec(nx, ny, 8, cyl, src, prb))
    return out


@pytest.mark.parametrize("sides,depth,rows,steps,waves", [
    # register tiles: one tile, tiles of one grid cut and another not, 14 to 8
    # steps a launch, past two tiles a CU, fewer workgroups than tiles
    ([(20, 30)], 14, 32, 13, 0),
    ([(32, 64), (33, 65), (64, 48), (25, 130)], 14, 32, 29, 0),
    ([(150, 170), (97, 211)], 14, 32, 50, 0),
    ([(150, 170), (97, 211), (300, 49), (211, 64)], 12, 32, 50, 0),
    ([(200, 210)] * 4 + [(250, 140)] * 3, 12, 48, 31, 0),
    ([(260, 310)] * 7 + [(100, 640)], 10, 48, 25, 0),
    ([(260, 310)] * 9 + [(100, 640)], 8, 48, 25, 0),
    ([(700, 900), (1500, 600), (1200, 1100)], 8, 48, 17, 0),
    ([(150, 170), (97, 211), (300, 49)], 12, 32, 30, 7),
    # strips: 5.0, 8.0 and 30 million cells
    ([(2200, 2200), (150, 1200)], 8, 24, 17, 0),
    ([(2700, 2960), (61, 333)], 10, 32, 21, 0),
    ([(5300, 5650), (700, 90)], 10, 48, 20, 0),
])
def test_default_shapes_match_single_grids(gpu, sides, depth, rows, steps, waves):
    from simulation_amd.batch import BatchSolver, single_solver
    print(f"[batch units] {sides} waves={waves}", flush=True)
    specs = _specs(sides)
    b = BatchSolver(specs, 2 * steps, waves=waves, device=gpu)
    assert (b.desc.depth, b.desc.rows) == (depth, rows)
    assert b.desc.waves == (waves or b.desc.nunits)
    b.run(steps)
    b.run(steps)
    for k, sp in enumerate(specs):
        s = single_solver(sp, 2 * steps, gpu, depth=5, rows=37)
        s.run(steps)
        s.run(steps)
        a, r = b.grid_state(k), s.state()
        for f in ("dz", "iz", "ez", "hx", "hy", "ihx", "ihy"):
            assert same_bits(a[f], r[f]), (k, f)
        if sp.probe is not None:
            assert same_bits(b.probe_trace(k), s.probe_traces()[0]), k


@pytest.mark.parametrize("depth,rows,steps,waves", [(6, 12, 26, 0), (6, 12, 26, 7), (8, 24, 21, 3)])
def test_strip_units_match_single_grids(gpu, depth, rows, steps, waves):
    from simulation_amd.batch import BatchSolver, single_solver
    print(f"[batch units] strips {depth}/{rows} waves={waves}", flush=True)
    specs = _specs([(40, 33), (150, 170), (97, 211), (300, 49), (25, 130)])
    b = BatchSolver(specs, steps, depth=depth, rows=rows, waves=waves, device=gpu)
    b.run(steps)
    for k, sp in enumerate(specs):
        s = single_solver(sp, steps, gpu, depth=5, rows=37)
        s.run(steps)
        a, r = b.grid_state(k), s.state()
        for f in ("dz", "iz", "ez", "hx", "hy", "ihx", "ihy"):
            assert same_bits(a[f], r[f]), (k, f)


def test_tile_batch_replayed_as_a_graph(gpu):
    """A captured tile batch replayed three times, eager work in between,
    against eager runs."""
    import torch
    from simulation_amd.batch import BatchSolver
    print("[batch units] graph", flush=True)
    specs = _specs([(150, 170), (97, 211), (64, 48)])
    with torch.cuda.stream(torch.cuda.Stream()):
        a, b = BatchSolver(specs, 60, device=gpu), BatchSolver(specs, 60, device=gpu)
        for _ in range(3):
            a.t = b.t = 0                        # steps 1 .. 30 again
            a.run_graph(30)
            b.run(30)
            torch.cuda.synchronize()
            for k in range(len(specs)):
                x, y = a.grid_state(k), b.grid_state(k)
                for f in x:
                    assert same_bits(x[f], y[f]), (k, f)
        a.close()


@pytest.mark.parametrize("sides,shape,runs,waves", [
    # more than two tiles a CU: launches shallower than the list cut their own
    # tiles; flat grids: tiles no taller than they are
    ([(30, 3000)] * 13 + [(20, 30), (3, 500), (32, 64)], (8, 32), (2, 3, 7, 16, 21), 0),
    ([(20, 2500)] * 14, (8, 20), (2, 9, 34), 0),
    ([(20, 2500)] * 14, (8, 20), (2, 9, 34), 150),
    ([(33, 1700), (1500, 40), (61, 60)] * 9 + [(700, 700)], (8, 48), (2, 5, 11), 0),
    ([(30, 700)] * 3, (14, 32), (2, 3, 5), 0),
    ([(30, 1000)] * 20, (12, 32), (3, 24), 0),
])
def test_shallow_launches_match_single_grids(gpu, sides, shape, runs, waves):
    from simulation_amd.batch import BatchSolver, GridSpec, single_solver
    print(f"[batch units] shallow {sides[:3]} waves={waves}", flush=True)
    specs = [GridSpec(nx, ny, 8 if nx > 16 and ny > 16 else 1, [],
                      (nx // 3, ny // 2, 20, 6.0) if k % 3 != 1 else None,
                      (nx // 3 + 1, ny // 2) if k % 3 != 2 else None) for k, (nx, ny) in enumerate(sides)]
    b = BatchSolver(specs, sum(runs), waves=waves, device=gpu)
    assert (b.desc.depth, b.desc.rows, b.desc.cols) == (*shape, 64)
    for n in runs:
        b.run(n)
    for k, sp in list(enumerate(specs))[:4] + list(enumerate(specs))[-3:]:
        s = single_solver(sp, sum(runs), gpu, depth=5, rows=37)
        for n in runs:
            s.run(n)
        a, r = b.grid_state(k), s.state()
        for f in ("dz", "iz", "ez", "hx", "hy", "ihx", "ihy"):
            assert same_bits(a[f], r[f]), (k, f)
        if sp.probe is not None:
            assert same_bits(b.probe_trace(k), s.probe_traces()[0]), k


@pytest.mark.parametrize("depth,rows,cols", [(4, 4, 1), (8, 4, 1), (11, 4, 1), (12, 4, 1), (8, 4, 2)])
def test_persistent_waves_at_most_those_held_at_once(gpu, depth, rows, cols):
    """Waves past those resident together, each with a share of the units,
    would run as a second, partial round; as many as the units: one each."""
    from simulation_amd.batch import BatchSolver, single_solver
    print(f"[batch units] resident {depth}/{rows}/{cols}", flush=True)
    specs = _specs([(700, 900), (1500, 600), (1201, 1100)])
    b = BatchSolver(specs, 30, depth=depth, rows=rows, cols=cols, waves=4096, device=gpu)
    per_simd = 4 if depth <= 7 else 3 if depth <= 11 else 2
    assert b.desc.nunits > 4096
    assert 1024 <= b.desc.waves <= 4096 and (cols > 1 or b.desc.waves == 1024 * per_simd)
    b.run(30)
    n = b.desc.nunits
    c = BatchSolver(specs, 30, depth=depth, rows=rows, cols=cols, waves=n, device=gpu)
    assert c.desc.waves == n
    c.run(30)
    for k, sp in enumerate(specs):
        s = single_solver(sp, 30, gpu, depth=5, rows=37)
        s.run(30)
        r = s.state()
        for x in (b.grid_state(k), c.grid_state(k)):
            for f in r:
                assert same_bits(x[f], r[f]), (k, f)

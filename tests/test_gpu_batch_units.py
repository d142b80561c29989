"""Batches in the library's own launch shapes -- one workgroup a unit, depth and
rows by the cells of all grids -- and in persistent waves against single-grid
runs, bit for bit: fewer units than XCDs, unit counts that 8 does not divide,
grids of edge units only, row blocks cut short, row-, column-only and corner
units, both sides of each change of shape."""
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
    ([(20, 30)], 6, 12, 13, 0),
    ([(40, 33), (64, 48), (25, 130)], 6, 12, 26, 0),
    ([(150, 170), (97, 211), (300, 49), (211, 64)], 6, 12, 50, 0),
    ([(2200, 2200), (150, 1200)], 8, 24, 17, 0),             # 5.0 million cells
    ([(2700, 2960), (61, 333)], 10, 32, 21, 0),              # 8.0 million
    ([(5300, 5650), (700, 90)], 10, 48, 20, 0),              # 30 million
    ([(150, 170), (97, 211), (300, 49)], 6, 12, 26, 7),      # persistent waves
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

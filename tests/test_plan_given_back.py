"""A reported launch shape given back plans the same launches (host only)."""
import ctypes as C

import pytest


def _desc(L, nx, ny):
    fake = C.cast(0x1000, C.POINTER(C.c_float))
    d = L.Fd2dTmDesc()
    d.nx, d.ny = nx, ny
    for k in ("dz", "ez", "hx", "hy"):
        setattr(d, k, fake)
    d.md.naz = fake
    return d


def _plan(L, d, ns):
    out = [C.c_int() for _ in range(4)]
    rc = L.lib().fd2d_tm_plan(C.byref(d), ns, *[C.byref(o) for o in out])
    assert rc == 0, L.lib().fdtd_last_error()
    return [o.value for o in out]


@pytest.mark.parametrize("nx,ny", [(2, 2), (60, 60), (210, 211), (300, 300), (500, 480), (650, 600),
                                   (1024, 1024), (1640, 1640), (1700, 1600), (2048, 2048),
                                   (3000, 3000), (40, 60000), (8192, 8192)])
@pytest.mark.parametrize("ns", [0, 1, 2, 3, 13, 28, 29, 200, 1000])
def test_plan_given_back(nx, ny, ns):
    from simulation_amd import _lib as L
    d = _desc(L, nx, ny)
    want = _plan(L, d, ns)
    d.depth, d.rows, d.cols = want[1:]
    assert _plan(L, d, ns) == want
    # the form is part of the shape: tiles keep no free-space tiles
    tiles = want[3] == L.TILE_COLS
    assert tiles == (nx * ny <= 2700000 and ns >= 2)
    assert (L.lib().fd2d_tm_tile_elems(C.byref(d), ns) == 0) == tiles
    # at another length it stays what it is
    assert _plan(L, d, ns + 77)[2:] == want[2:]


@pytest.mark.parametrize("nx,ny,depth,rows,cols,form", [
    (60, 60, 16, 32, 64, 0), (60, 60, 0, 32, 64, 0), (60, 60, 8, 0, 64, 0), (60, 60, 8, 30, 64, 0),
    (60, 60, 8, 68, 64, 0), (60, 60, 17, 64, 64, 0), (60, 60, -1, 32, 64, 0), (60, 60, 8, 32, 63, 0),
    (60, 60, 8, 32, 64, 1), (60, 60, 8, 32, 64, 2), (4200, 4200, 8, 32, 64, 0), (60, 60, 13, 32, 1, 0),
])
def test_no_such_shape(nx, ny, depth, rows, cols, form):
    from simulation_amd import _lib as L
    d = _desc(L, nx, ny)
    d.depth, d.rows, d.cols, d.form = depth, rows, cols, form
    for ns in (0, 1, 2, 50):
        assert L.lib().fd2d_tm_plan(C.byref(d), ns, None, None, None, None) == L.FDTD_EINVAL
    grids = (L.Fd2dGrid * 1)()
    grids[0].nx, grids[0].ny = nx, ny
    n = C.c_int()
    if form == 0:
        assert L.lib().fd2d_batch_units(grids, 1, depth, rows, cols, C.byref(n)) == L.FDTD_EINVAL


@pytest.mark.parametrize("sides,shape", [([(60, 60)], (14, 32)), ([(300, 300)] * 4, (8, 48)),
                                         ([(700, 900), (1500, 600)], (8, 48))])
def test_batch_shape_given_back(sides, shape):
    from simulation_amd import _lib as L
    grids = (L.Fd2dGrid * len(sides))()
    for g, (nx, ny) in zip(grids, sides):
        g.nx, g.ny = nx, ny
    a, b = C.c_int(), C.c_int()
    assert L.lib().fd2d_batch_units(grids, len(sides), 0, 0, 0, C.byref(a)) == 0
    assert L.lib().fd2d_batch_units(grids, len(sides), *shape, L.TILE_COLS, C.byref(b)) == 0
    assert a.value == b.value


@pytest.mark.parametrize("depth,rows,cols,vec", [(0, 32, 64, 0), (0, 0, 64, 0), (0, 32, 64, 2), (0, 32, 1, 2),
                                                 (16, 32, 64, 0), (8, 30, 64, 0), (13, 32, 1, 2)])
def test_batch_descriptor_without_a_shape(depth, rows, cols, vec):
    """An incomplete descriptor is an error, not a division by zero."""
    from simulation_amd import _lib as L
    d = L.Fd2dBatchDesc()
    d.grids_dev = d.units_dev = 0x1000
    d.nunits = d.waves = 1
    d.wave_len = d.probe_len = 100
    d.depth, d.rows, d.cols, d.vec = depth, rows, cols, vec
    assert L.lib().fd2d_batch_run(C.byref(d), 0, 4, 100, 100, None) == L.FDTD_EINVAL

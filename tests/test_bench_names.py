"""bench.py names kernels and traffic records by the plan's shape: register
tiles never share a strip's name."""
import ctypes as C

import pytest


@pytest.mark.parametrize("n,kernel", [(60, "tm_rt_kernel"), (1024, "tm_rt_kernel"), (1640, "tm_rt_kernel"),
                                      (2048, "tm_tb_kernel"), (8192, "tm_tb_kernel")])
def test_names_follow_the_plan(n, kernel):
    import bench
    from simulation_amd import _lib as L
    fake = C.cast(0x1000, C.POINTER(C.c_float))
    d = L.Fd2dTmDesc()
    d.nx = d.ny = n
    for k in ("dz", "ez", "hx", "hy"):
        setattr(d, k, fake)
    d.md.naz = fake
    _, depth, rows, cols = out = [C.c_int() for _ in range(4)]
    assert L.lib().fd2d_tm_plan(C.byref(d), 200, *[C.byref(o) for o in out]) == 0
    assert bench.TILE_COLS == L.TILE_COLS
    assert bench.tm_kernel(cols.value) == kernel
    shape = bench.tm_shape(depth.value, rows.value, cols.value)
    assert (shape == bench.tm_shape(depth.value, rows.value, 1)) == (kernel == "tm_tb_kernel")


def test_multiwave_names():
    import bench
    assert bench.tm_kernel(1, "multiwave") == "tm_mw_kernel"
    assert bench.tm_shape(8, 32, 1, "multiwave") == "d8_r32_c1_mw"

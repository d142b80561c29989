"""The pointer structs of the per-step calls: fields by name from any object
that has them (medium, pmlayer, ftrans), in the struct's own order."""
import ctypes as C
from types import SimpleNamespace

import pytest


@pytest.fixture
def ptrs(monkeypatch):
    from simulation_amd import _dev
    monkeypatch.setattr(_dev, "ptr", lambda t, dtype=None: t)


def _addr(s, k):
    return C.cast(getattr(s, k), C.c_void_p).value


def test_ftrans_fields_by_name(ptrs):
    from simulation_amd import fd1d, fd2d
    names = ("i_in", "r_in", "i_pt", "r_pt")                 # another order than the struct's
    want = {k: 4096 * (n + 1) for n, k in enumerate(names)}
    for make in (fd2d._ft_struct, fd1d._ft1):
        s = make(SimpleNamespace(**want, more=1))
        assert {k: _addr(s, k) for k in names} == want
    s = fd2d._ft_struct(fd2d.ftrans(4096, 8192, None, None))
    assert [_addr(s, k) for k in ("r_pt", "i_pt", "r_in", "i_in")] == [4096, 8192, None, None]


def test_profiles_and_media_by_name(ptrs):
    from simulation_amd import fd1d, fd2d
    want = {k: 4096 * (n + 1) for n, k in enumerate(reversed(fd2d.pmlayer._fields))}
    s = fd2d._pml_struct(SimpleNamespace(**want))._obj
    assert {k: _addr(s, k) for k in want} == want
    s = fd1d._md1(SimpleNamespace(ndx=4096, ncx=None, nbx=8192, nax=12288))
    assert [_addr(s, k) for k in ("nax", "nbx", "ncx", "ndx")] == [12288, 8192, None, 4096]

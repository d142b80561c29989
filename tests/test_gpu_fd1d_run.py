"""The C entries fd1d_run and fd1d_run_f64, called as a C program calls them,
against the oracle, bit for bit: the sizes where the launch changes (cells in
registers up to 592, with one wave up to 64, then fields in LDS) and the
largest."""
import ctypes as C

import numpy as np
import pytest
import torch

from conftest import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("nx,ns,form,mode,probes", [
    (3, 19, "free", 1, (0, 1, 2)),
    (64, 130, "abc", 2, (0, 63)),
    (592, 75, "coef", 1, (0, 299, 300, 591)),
    (593, 75, "coef", 1, (0, 299, 300, 592)),
    (593, 41, "abc", 2, ()),
    (0, 33, "coef", 2, tuple(range(0, 3200, 200))),          # 0: the largest
])
def test_fd1d_run_matches_oracle(gpu, oracle, dt, nx, ns, form, mode, probes):
    from simulation_amd import _lib
    from simulation_amd._dev import ptr, stream
    size = np.dtype(dt).itemsize
    nx = nx or _lib.lib().fd1d_run_max_nx(size)
    print(f"[fd1d_run] nx={nx} ns={ns} {form} {np.dtype(dt)}", flush=True)
    rng = np.random.default_rng(nx + ns)
    ex, hy, bc, wave = (rng.standard_normal(n).astype(dt) for n in (nx, nx, 4, ns))
    ca, cb = (rng.uniform(a, b, nx).astype(dt) for a, b in ((0.8, 1.0), (0.1, 0.5)))
    if form != "coef":
        ca = cb = None
    if form == "free":
        bc = None
    d = [None if a is None else torch.from_numpy(a.copy()).to(gpu) for a in (ca, cb, ex, hy, bc, wave)]
    out = torch.full((max(len(probes), 1), ns), -1.0, dtype=d[2].dtype, device=gpu)
    pk = (C.c_int * max(len(probes), 1))(*probes)
    p = [ptr(t, d[2].dtype) for t in d]
    _lib.call("fd1d_run_f64" if size == 8 else "fd1d_run", nx, 0, ns, p[0], p[1], p[2], p[3], p[4],
              mode, nx // 2, p[5], len(probes), pk if probes else None,
              out.data_ptr() if probes else None, stream())
    ref = oracle.fd1d_run(nx, 0, ns, ex, hy, bc, ca, cb, mode, nx // 2, wave, probes)
    assert same_bits(d[2].cpu().numpy(), ex) and same_bits(d[3].cpu().numpy(), hy)
    if bc is not None:
        assert same_bits(d[4].cpu().numpy(), bc)
    if probes:
        assert same_bits(out.cpu().numpy(), ref)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("nx", [592, 593, 1365, 2048, 4096])
def test_short_runs_match_oracle(gpu, oracle, dt, nx):
    """fd1d.run a few steps at a time: one launch in LDS while nx * steps is
    small, the blocked run past that."""
    from simulation_amd import _lib, fd1d
    print(f"[fd1d short] nx={nx} {np.dtype(dt)}", flush=True)
    rng = np.random.default_rng(nx)
    ex, hy, bc, wave = (rng.standard_normal(n).astype(dt) for n in (nx, nx, 4, 40))
    d = [torch.from_numpy(a.copy()).to(gpu) for a in (ex, hy, bc, wave)]
    probes, t = (0, nx // 2, nx - 1), 0
    for n in (1, 2, 3, 4, 6, 7, 12, 1):
        pr = fd1d.run(nx, n, d[0], d[1], d[2], None, None, 2, nx // 3, d[3][t:t + n], probes, t)
        ref = oracle.fd1d_run(nx, t, n, ex, hy, bc, None, None, 2, nx // 3,
                              np.ascontiguousarray(wave[t:t + n]), probes)
        assert same_bits(pr.cpu().numpy(), ref), n
        t += n
    assert fd1d.run(nx, 0, d[0], d[1], d[2]).shape == (0, 0)
    with pytest.raises(_lib.FdtdError, match="probe_out"):       # an empty trace has no address
        fd1d.run(nx, 0, d[0], d[1], d[2], probes=probes)
    for a, b in zip(d, (ex, hy, bc)):
        assert same_bits(a.cpu().numpy(), b)

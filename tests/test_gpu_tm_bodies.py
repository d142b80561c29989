"""The tile bodies of the temporally blocked TM launches against the oracle,
bit for bit: row blocks longer than the 64 rows whose profile values a wave
holds, row, column and corner tiles of the layer, sources and probes in the
first rows (whose levels run above the grid) and on tile cuts, probes without
any source."""
import numpy as np
import pytest
import torch

from conftest import same_bits

pytestmark = pytest.mark.gpu
STATE = ("dz", "iz", "ez", "hx", "hy", "ihx", "ihy")


def run_both(gpu, oracle, nx, ny, npml, lossy, src, probes, chunks, seed=3, **kw):
    """A TMSolver and the oracle from the same random fields through `chunks`."""
    from simulation_amd import fd2d
    rng = np.random.default_rng(seed)
    ns = sum(chunks)
    pml = pm = None
    if npml >= 0:
        pml = fd2d.new_pmlayer(nx, ny, gpu)
        fd2d.pmlparam(nx, ny, npml, pml)
        pm = {k: getattr(pml, k).cpu().numpy() for k in pml._fields}
    naz = np.ones((nx, ny), np.float32)
    nbz = np.zeros((nx, ny), np.float32)
    naz[nx // 3:nx // 2, ny // 4:] = rng.uniform(0.2, 1, (nx // 2 - nx // 3, ny - ny // 4))
    nbz[nx // 3:nx // 2, ny // 4:] = rng.uniform(0, 0.05, (nx // 2 - nx // 3, ny - ny // 4))
    t = lambda a: torch.from_numpy(a.copy()).to(gpu)  # noqa: E731
    wave = rng.standard_normal((len(src), ns)).astype(np.float32)
    s = fd2d.TMSolver(nx, ny, pml, fd2d.medium(t(naz), t(nbz) if lossy else None),
                      [(i, j, w) for (i, j), w in zip(src, wave)], probes, nsteps_max=ns,
                      device=gpu, **kw)
    ref = oracle.TMState(nx, ny)
    for k in STATE:
        a = rng.standard_normal((nx, ny)).astype(np.float32)
        if k == "iz":
            a[:] = 0
        setattr(ref, k, a)
        if getattr(s, k) is not None:
            getattr(s, k).copy_(t(a))
    for n in chunks:
        s.run(n)
    tr = oracle.fd2d_tm_run(ref, 0, ns, pm, naz, nbz if lossy else None, src,
                            wave if src else None, probes)
    for k in STATE:
        if getattr(s, k) is not None:
            assert same_bits(getattr(s, k).cpu().numpy(), getattr(ref, k)), k
    if probes:
        assert same_bits(s.probe_traces(), tr)


@pytest.mark.parametrize("nx,ny,npml,lossy,depth,rows,src,probes", [
    (300, 140, 16, True, 8, 150, [(1, 70), (70, 30), (299, 139)], [(0, 0), (149, 70), (150, 70)]),
    (260, 100, 70, False, 5, 130, [], [(0, 50), (3, 99), (129, 1)]),
    (150, 300, 8, True, 11, 40, [(39, 41), (40, 42)], [(1, 1), (5, 299)]),
    (90, 70, -1, True, 4, 90, [(2, 2)], [(0, 3), (89, 69)]),
])
def test_tile_bodies(gpu, oracle, nx, ny, npml, lossy, depth, rows, src, probes):
    print(f"[tm bodies] {nx}x{ny} npml={npml} depth={depth} rows={rows}", flush=True)
    run_both(gpu, oracle, nx, ny, npml, lossy, src, probes, (2 * depth, 7, 3 * depth + 1),
             depth=depth, rows=rows)

"""The incident grid of the fused plane-wave run (registers, 1 to 16 cells a
lane) against the per-step kernels, bit for bit: one wave, the first cuts
between waves, the last size of each width and the next, sources on ends and
cuts, chunks that end between two exchanges."""
import numpy as np
import pytest
import torch

from conftest import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ny,nf,inc_pos,steps", [
    (12, 3, 3, 70), (64, 1, 63, 130), (65, 3, 56, 65), (112, 0, 55, 9), (113, 2, 112, 72),
    (784, 3, 3, 96), (785, 3, 120, 66), (1808, 3, 1, 64), (1809, 1, 240, 73), (3856, 3, 3, 16),
    (3857, 3, 496, 40), (7952, 3, 0, 24), (7953, 2, 1008, 33), (16144, 3, 16143, 18),
    (16145, 3, 3, 18),
])
def test_incident_chunk(gpu, ny, nf, inc_pos, steps):
    from simulation_amd import fd2d
    print(f"[incident] ny={ny} nf={nf} inc_pos={inc_pos} steps={steps}", flush=True)
    nx, npml = 14, 3
    dt = fd2d.time_step()
    pml = fd2d.new_pmlayer(nx, ny, gpu)
    fd2d.pmlparam(nx, ny, npml, pml)
    md = fd2d.dielectric(nx, ny, npml, 0, dt, 1.0, 0.0, gpu, cylinders=np.zeros((0, 5)))
    rng = np.random.default_rng(ny)
    wave = rng.standard_normal(steps + 4).astype(np.float32)
    init = {k: rng.standard_normal(n).astype(np.float32) for k, n in
            (("ezi", ny), ("hxi", ny), ("bc", 4))}
    out = []
    for fused in (True, False):
        s = fd2d.PlaneWaveSolver(nx, ny, npml, pml, md, steps + 4, freq=(5e7, 3e8, 7e8)[:nf], dt=dt,
                                 inc_pos=inc_pos, inc_wave=wave, device=gpu, fused=fused)
        for k, v in init.items():
            getattr(s, k).copy_(torch.from_numpy(v))
        s.run(steps)
        s.run(4)
        out.append(s)
    a, b = out
    assert a.work is not None and b.work is None
    for k in ("ezi", "hxi", "bc"):
        assert same_bits(getattr(a, k).cpu().numpy(), getattr(b, k).cpu().numpy()), k
    if nf:
        for k, v in a.ft._asdict().items():
            assert same_bits(v.cpu().numpy(), getattr(b.ft, k).cpu().numpy()), k
    for k in fd2d.STATE:
        assert same_bits(getattr(a.tm, k).cpu().numpy(), getattr(b.tm, k).cpu().numpy()), k

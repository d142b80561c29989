"""The fused D/E-form run against the per-step kernels, bit for bit, at the
sizes where its segments change: one wave (64 cells), one workgroup (400
cells), several; launches of up to 112 steps, odd remainders, sources and
probes on segment cuts, every count of DFT frequencies."""
import numpy as np
import pytest
import torch

from conftest import same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,debye,nf,src_pos,chunks", [
    (11, True, 1, 5, (2, 117)),
    (63, False, 3, 62, (130,)),
    (64, True, 2, 1, (113, 2)),
    (65, True, 3, 64, (31, 9)),
    (112, False, 0, 56, (225,)),
    (400, True, 3, 399, (112, 113)),
    (401, True, 3, 200, (2, 3, 120)),
    (700, False, 2, -1, (338,)),
    (5001, True, 1, 2500, (337, 40)),
    (70000, True, 3, 35000, (201,)),
])
def test_fused_matches_per_step(gpu, nx, debye, nf, src_pos, chunks):
    from simulation_amd import fd1d
    dt = float(np.float32(np.float32(0.01) / np.float32(6e8)))
    rng = np.random.default_rng(nx)
    ns = sum(chunks)
    wave = rng.standard_normal(ns).astype(np.float32)
    init = {k: torch.from_numpy(rng.standard_normal(4 if k == "bc" else nx).astype(np.float32)).to(gpu)
            for k in ("dx", "ix", "sx", "ex", "hy", "bc")}
    probes = sorted({0, 1, 10, nx // 2, nx - 2, nx - 1, min(nx - 1, 64), min(nx - 1, 48)})
    print(f"[dform blocked] nx={nx} debye={debye} nf={nf} chunks={chunks}", flush=True)

    def make(fused):
        md = fd1d.dielectric_dform(nx, dt, 2.0, 0.001e-6, 2.0, 0.01, debye=debye, device=gpu)
        s = fd1d.DFormSolver(nx, md, ns, freq=(50e6, 200e6, 500e6)[:nf], dt=dt, src_pos=src_pos,
                             src_wave=wave, probes=probes, device=gpu, fused=fused)
        for k, v in init.items():
            if getattr(s, k) is not None:
                getattr(s, k).copy_(v)
        if nf:
            for v in s.ft:
                v.fill_(0.25)
        return s
    a, b = make(True), make(False)
    for n in chunks:
        a.run(n)
        b.run(n)
    for k in ("dx", "ix", "ex", "hy", "bc", "probe_out") + (("sx",) if debye else ()):
        assert same_bits(getattr(a, k).cpu().numpy(), getattr(b, k).cpu().numpy()), k
    if nf:
        for k in ("r_pt", "i_pt", "r_in", "i_in"):
            assert same_bits(getattr(a.ft, k).cpu().numpy(), getattr(b.ft, k).cpu().numpy()), k

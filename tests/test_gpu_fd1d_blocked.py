"""The blocked 1-D run against the oracle, bit for bit, at the sizes where its
segments change: one wavefront (up to 64 cells), one workgroup of overlapping
waves (to 416 and 592 cells), then several workgroups; launches of one step,
an even split and remainders; sources and probes on segment cuts and edge
cells."""
import numpy as np
import pytest
import torch

from conftest import same_bits

pytestmark = pytest.mark.gpu


def _fields(nx, dt, seed):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal(n).astype(dt) for n in (nx, nx, 4)]


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("nx,ns,form,mode,pos,probes", [
    (3, 40, "free", 1, 1, (0, 1, 2)),
    (63, 70, "abc", 2, 62, (0, 62)),
    (64, 129, "coef", 1, 0, (63,)),
    (65, 65, "abc", 1, 64, (1, 63, 64)),
    (96, 33, "free", 2, 95, ()),
    (97, 300, "coef", 2, 48, (0, 15, 16, 17, 47, 48, 96)),
    (416, 200, "abc", 2, 415, (414, 415)),
    (417, 64, "free", 0, 0, (400, 416)),
    (592, 77, "abc", 1, 32, (31, 32, 33, 591)),
    (593, 1, "abc", 2, 3, (0, 592)),
    (593, 2, "coef", 1, 591, (1,)),
    (593, 353, "abc", 1, 64, (63, 64, 592)),
    (700, 113, "cb", 2, 699, (698, 699)),
    (3001, 449, "coef", 2, 1499, tuple(range(0, 3001, 200))),
    (4096, 223, "free", 1, 4095, (0, 4095)),
])
def test_run_matches_oracle(gpu, oracle, dt, nx, ns, form, mode, pos, probes):
    from simulation_amd import fd1d
    print(f"[fd1d blocked] nx={nx} ns={ns} {form} {np.dtype(dt)}", flush=True)
    ex, hy, bc = _fields(nx, dt, nx + ns)
    rng = np.random.default_rng(ns)
    ca = cb = None
    if form in ("coef", "cb"):
        cb = rng.uniform(0.1, 0.5, nx).astype(dt)
    if form == "coef":
        ca = rng.uniform(0.8, 1.0, nx).astype(dt)
    if form == "free":
        bc = None
    wave = rng.standard_normal(ns).astype(dt)
    d = [None if a is None else torch.from_numpy(a.copy()).to(gpu) for a in (ex, hy, bc, ca, cb, wave)]
    pr = fd1d.run(nx, ns, d[0], d[1], d[2], d[3], d[4], mode, pos, d[5], probes)
    ref = oracle.fd1d_run(nx, 0, ns, ex, hy, bc, ca, cb, mode, pos, wave, probes)
    assert same_bits(d[0].cpu().numpy(), ex) and same_bits(d[1].cpu().numpy(), hy)
    if bc is not None:
        assert same_bits(d[2].cpu().numpy(), bc)
    if probes:
        assert same_bits(pr.cpu().numpy(), ref)


@pytest.mark.parametrize("dt,nx,probes", [
    (np.float32, 38001, (150, 38000)),
    (np.float64, 9001, (0, -1)),                       # counted from the end
    (np.float32, 8193, tuple(range(1, 8193, 455))),    # more than a launch records
    (np.float32, 250000, (125003,)),                   # more segments than SIMDs
])
def test_simulate_past_the_single_launch_limit(gpu, oracle, dt, nx, probes):
    from simulation_amd import fd1d
    print(f"[fd1d simulate] nx={nx} {np.dtype(dt)}", flush=True)
    cfg = fd1d.Fd1dConfig(nx=nx, ns=130, dtype=dt, epsr=3.0, sigma=0.02, probes=probes, snap_every=50)
    out = fd1d.simulate(cfg, gpu)
    ca, cb = (a.astype(dt) for a in oracle.fd1d_dielectric(nx, 0.01 / 6e8, 3.0, 0.02))
    ex, hy, bc = np.zeros(nx, dt), np.zeros(nx, dt), np.zeros(4, dt)
    w = oracle.waveform("gaussian", 0, 130, dt, center=40, spread=12.0)
    traces = []
    for t0, t1 in ((0, 50), (50, 100), (100, 130)):
        at = tuple(k % nx for k in probes)
        traces.append(np.concatenate([oracle.fd1d_run(nx, t0, t1 - t0, ex, hy, bc, ca, cb, 1, nx // 2,
                                                      w[t0:t1].copy(), at[:16])]) if len(at) <= 16 else None)
        if len(at) > 16:
            oracle.fd1d_run(nx, t0, t1 - t0, ex, hy, bc, ca, cb, 1, nx // 2, w[t0:t1].copy(), ())
            assert same_bits(out["probe"][:, t1 - 1], ex[list(at)])
        if t1 % 50 == 0:
            assert same_bits(out["snap_ex"][t1 // 50 - 1], ex)
            assert same_bits(out["snap_hy"][t1 // 50 - 1], hy)
    assert same_bits(out["ex"], ex) and same_bits(out["hy"], hy) and same_bits(out["bc"], bc)
    if len(probes) <= 16:
        assert same_bits(out["probe"], np.concatenate(traces, 1))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("nx,ns,mode,pos,probes", [
    (3, 70, 1, 1, (2, 0, 1, 1, 0, 2) * 2 + (1, 1, 0, 2)),
    (64, 131, 2, 30, tuple(range(20, 36))),
    (64, 9, 1, 63, (63, 0, 63, 5)),
    (592, 77, 2, 300, tuple(range(290, 306))),
    (1500, 300, 1, 40, tuple(range(33, 49))),
    (3001, 130, 2, 1499, (1499, 1500) * 8),
])
def test_many_probes_of_one_wave_match_oracle(gpu, oracle, dt, nx, ns, mode, pos, probes):
    from simulation_amd import fd1d
    print(f"[fd1d probes] nx={nx} ns={ns} {np.dtype(dt)}", flush=True)
    ex, hy, bc = _fields(nx, dt, nx + ns)
    wave = np.random.default_rng(ns).standard_normal(ns).astype(dt)
    d = [torch.from_numpy(a.copy()).to(gpu) for a in (ex, hy, bc, wave)]
    pr = fd1d.run(nx, ns, d[0], d[1], d[2], None, None, mode, pos, d[3], probes)
    ref = oracle.fd1d_run(nx, 0, ns, ex, hy, bc, None, None, mode, pos, wave, probes)
    assert same_bits(d[0].cpu().numpy(), ex) and same_bits(d[1].cpu().numpy(), hy)
    assert same_bits(pr.cpu().numpy(), ref)


def test_many_probes_of_one_wave_cost_no_loop(gpu):
    """16 probes in a wave: an exchange and a store a step (a loop over them
    took 16 times as long as one probe; the bar is half of that)."""
    from simulation_amd import fd1d
    print("[fd1d probes] time", flush=True)
    ex, hy = torch.zeros(64, device=gpu), torch.zeros(64, device=gpu)
    best = []
    for probes in ((20,), tuple(range(20, 36))):
        us = []
        for _ in range(12):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            fd1d.run(64, 4000, ex, hy, probes=probes)
            b.record()
            b.synchronize()
            us.append(a.elapsed_time(b) * 1e3)
        best.append(min(us))
    print(f"[fd1d probes] {best[0]:.0f} us, 16 probes {best[1]:.0f} us", flush=True)
    assert best[1] < 8 * best[0]

"""The learned boundary refuses a stream that is being captured, before it
launches or records anything, and runs on as before."""
import pytest
import torch

from conftest import same_bits

pytestmark = pytest.mark.gpu


def test_capture_is_an_error(gpu):
    from simulation_amd import _lib, fd2d, learned
    print("[lbc capture]", flush=True)
    md = fd2d.dielectric(100, 90, 0, 12, fd2d.time_step(), 4.0, 0.02, gpu)
    a, b = (learned.LearnedTMSolver(100, 90, learned.load(device=gpu), md, nsteps_max=40, device=gpu)
            for _ in range(2))
    for s in (a, b):
        s.tm.dz[50, 45] = 1.0
        s.run(20)
    torch.cuda.synchronize()
    x = torch.zeros(8, device=gpu)
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        x += 1                                       # the capture holds a node
        with pytest.raises(_lib.FdtdError, match="captured"):
            a.run(20)
    assert a.t == 20
    for s in (a, b):
        s.run(20)
    for k in ("dz", "iz", "ez", "hx", "hy"):
        assert same_bits(getattr(a.tm, k).cpu().numpy(), getattr(b.tm, k).cpu().numpy()), k

"""The resident reverse loop's accumulators as its stores leave them, at shapes whose kernels follow a
wide store closely with the next column's arithmetic: every output equals the step kernels', pass
after pass, and an adjoint without a source leaves no backward illumination at all."""
import numpy as np
import pytest

from helpers import integrated_sources
from swit_amd import workloads


@pytest.mark.gpu
@pytest.mark.parametrize("nz,npml", [(50, 10), (120, 20), (180, 20), (240, 20), (300, 20), (360, 30), (420, 30)])
@pytest.mark.parametrize("nx,ns", [(300, 8), (100, 3), (300, 30)])
def test_accumulators(nx, nz, npml, ns):
    import torch
    from swit_amd.engine import Plan
    w = workloads.small(seed=3, nx=nx, nz=nz, npml=npml, nt=60, ns=ns)
    src = torch.from_numpy(integrated_sources(w)).cuda()
    p = Plan(w.nx, w.nz, w.dx, w.dt, w.nt, w.npml, w.src_xz, w.rec_xz)
    p.set_model(torch.from_numpy(w.vp_init), torch.from_numpy(workloads.gardner(w.vp_init)))
    adj = (p.forward(src) * 1e-2).contiguous()
    p.set_option("resident", 0)
    want = [t.cpu().numpy() for t in p.adjoint(src, adj)]
    p.set_option("resident", 1)
    assert p.resident("backward")
    for _ in range(3):
        for a, b in zip(p.adjoint(src, adj), want):
            np.testing.assert_array_equal(a.cpu().numpy(), b)
        g, fw, bk = p.adjoint(src, torch.zeros_like(adj))
        assert not bk.any() and not g.any()
        np.testing.assert_array_equal(fw.cpu().numpy(), want[1])
    p.close()

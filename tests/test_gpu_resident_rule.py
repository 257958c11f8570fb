"""Which plans start with a resident reverse loop: those whose step kernels are not the faster.
Measured us per reverse step, resident against step kernels (rows per lane in brackets): 201x81 one
shot 5.1 / 7.5 (3); 100x206, 50 layers, one shot 7.5 / 7.1 (5), 4 shots 7.7 / 9.3; 220x259 one shot
8.2 / 7.3 (6), 8 shots 9.6 / 17.0; 100x330 two shots 10.1 / 7.4 (7), 20 shots 13.0 / 28.9; 100x400 one
shot 14.7 / 7.1 (8), 8 shots 20.4 / 16.2; 400x400 4 shots 23.1 / 17.9, 8 shots 27.2 / 31.1.  The
forward is faster resident at every one of them."""
import numpy as np
import pytest

from helpers import integrated_sources
from swit_amd import workloads


def _plan(w):
    from swit_amd.engine import Plan
    return Plan(w.nx, w.nz, w.dx, w.dt, w.nt, w.npml, w.src_xz, w.rec_xz)


@pytest.mark.gpu
@pytest.mark.parametrize("nx,nz,npml,ns,resident", [
    (201, 81, 40, 1, True), (100, 206, 50, 1, False), (100, 206, 50, 4, True), (220, 259, 50, 1, False),
    (220, 259, 50, 8, True), (100, 330, 50, 2, False), (100, 330, 50, 20, True), (400, 330, 50, 1, False),
    (400, 330, 50, 4, True), (100, 400, 50, 1, False), (100, 400, 50, 8, False), (400, 400, 50, 4, False),
    (400, 400, 50, 8, True)])
def test_route(nx, nz, npml, ns, resident):
    w = workloads.small(seed=1, nx=nx, nz=nz, npml=npml, nt=20, ns=ns)
    p = _plan(w)
    assert p.resident("forward") and p.resident("backward") == resident
    p.set_option("resident", 1)
    assert p.resident("backward")
    p.set_option("resident", 0)
    assert not p.resident("forward") and not p.resident("backward")
    p.close()


@pytest.mark.gpu
def test_resident_forward_with_step_kernels_backward():
    import torch
    w = workloads.small(seed=2, nx=60, nz=300, npml=20, nt=60, ns=1)
    src = torch.from_numpy(integrated_sources(w))
    out = []
    for resident in (None, 1, 0):
        p = _plan(w)
        p.set_model(torch.from_numpy(w.vp_init), torch.from_numpy(workloads.gardner(w.vp_init)))
        if resident is None:
            assert p.resident("forward") and not p.resident("backward")
        else:
            p.set_option("resident", resident)
        syn = p.forward(src)
        out.append([t.cpu().numpy() for t in (syn,) + tuple(p.adjoint(src, (syn * 1e-2).contiguous()))])
        p.close()
    for o in out[1:]:
        for a, b in zip(o, out[0]):
            np.testing.assert_array_equal(a, b)


@pytest.mark.gpu
def test_autotuner_leaves_a_plan_without_resident_loops():
    import torch
    w = workloads.small(seed=3, nx=150, nz=60, npml=20, nt=60, ns=3)
    p = _plan(w)
    p.set_model(torch.from_numpy(w.vp_init), torch.from_numpy(workloads.gardner(w.vp_init)))
    p.set_option("resident", 0)
    tuned = p.autotune(5)
    assert not p.resident("forward") and not p.resident("backward") and not p.resident("exact")
    assert tuned["fwd_us"] > 0 and tuned["bwd_us"] > 0
    p.set_option("resident", 1)
    p.autotune(5)                            # times both; either way the results are the same
    p.close()

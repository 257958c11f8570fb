"""Calls that took what memory there is still do where the larger workspaces and the resident loops'
arrays do not fit: they run with less."""
import numpy as np
import pytest

from helpers import integrated_sources
from swit_amd import workloads


@pytest.mark.gpu
def test_processing_with_room_for_the_smallest_workspace():
    """40000 traces: 657 MB to filter all at once, 269 MB for the least; 400 MB left."""
    import torch
    from swit_amd import engine
    from test_gpu_process import _optim
    rng = np.random.default_rng(5)
    d = torch.from_numpy(rng.standard_normal((1, 40000, 2000), dtype=np.float32)).cuda()
    o = _optim(fre_filter='bandpass', fre_low=4.0, fre_high=18.0)
    want = engine.process_gathers(o, d.clone(), 0.002)
    torch.cuda.synchronize()
    got = d.clone()
    del d
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 400 * 2**20) / total)
    try:
        engine.process_gathers(o, got, 0.002)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(got, want)


@pytest.mark.gpu
def test_plan_without_room_for_the_resident_arrays():
    """Half of the reverse loop's accumulators (0.8 GB) are left beside the rest of the plan: it is
    created, runs that loop by step kernels and gives the same results."""
    import torch
    from swit_amd.engine import Plan
    w = workloads.small(seed=6, nx=600, nz=180, npml=20, nt=24, ns=400)
    src = torch.from_numpy(integrated_sources(w)).cuda()
    vp, rho = torch.from_numpy(w.vp_init).cuda(), torch.from_numpy(workloads.gardner(w.vp_init)).cuda()

    def run():
        p = Plan(w.nx, w.nz, w.dx, w.dt, w.nt, w.npml, w.src_xz, w.rec_xz)
        p.set_model(vp, rho)
        syn = p.forward(src)
        res = [syn.cpu()] + [t.cpu() for t in p.adjoint(src, (syn * 1e-2).contiguous())]
        route, size = (p.resident("forward"), p.resident("backward")), p.scratch_bytes
        p.close()
        return res, route, size
    want, route, size = run()
    assert route == (True, True)
    acc = w.ns * (w.nx + 2 * w.npml) * 3 * 64 * 4 * 4          # four rows a lane
    assert acc > 0.7e9
    torch.cuda.empty_cache()
    # the seismograms, adjoint sources and gradients of run() come from torch: leave their room too
    room = size - acc // 2 + 4 * w.ns * w.rec_xz.shape[1] * w.nt * 4 + 64 * 2**20
    held = []
    try:
        for _ in range(3):                   # a large allocation sets a reserve free
            more = torch.cuda.mem_get_info()[0] - room
            if more > 0:
                held.append(torch.empty(more, dtype=torch.uint8, device="cuda"))
        got, route, small = run()
    finally:
        del held
        torch.cuda.empty_cache()
    assert route == (True, False) and small <= size - acc
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a.numpy(), b.numpy())

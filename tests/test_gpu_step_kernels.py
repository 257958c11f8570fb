"""The step kernels on plans whose loops would run resident (SWIT_OPT_RESIDENT 0, asserted): replayed
graphs and direct launches, two streams, both backward kernels, 16-bit strips, the exact adjoint's
fused and separate passes, the launch counters, and calls on a capturing stream.  Everything equals the
resident loops' bits, and these the oracle's.  Also resident loops on several streams at once,
of plans that do not fit the chip together."""
import numpy as np
import pytest

from helpers import integrated_sources, rel_l2
from swit_amd import workloads


def _plan(w, resident, **kw):
    import torch
    from swit_amd.engine import Plan
    p = Plan(w.nx, w.nz, w.dx, w.dt, w.nt, w.npml, w.src_xz, w.rec_xz, **kw)
    p.set_model(torch.from_numpy(w.vp_init), torch.from_numpy(workloads.gardner(w.vp_init)))
    p.set_option("resident", resident)
    assert p.resident("forward") == p.resident("backward") == bool(resident)
    return p


def _run(p, src):
    import torch
    s = torch.from_numpy(src)
    syn = p.forward(s, save_strips=True)
    return [t.cpu().numpy() for t in [syn, p.saved_strips()] + list(p.adjoint(s, (syn * 1e-2).contiguous()))]


def _same(a, b):
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [1, 0])
@pytest.mark.parametrize("streams,steps,strips,ns", [
    (1, 2, "f32", 3), (1, 1, "f16", 3), (2, 1, "f32", 2), (2, 2, "f32", 5), (2, 1, "f16", 3), (2, 2, "bf16", 4),
    (2, 2, "f32", 1)])
def test_step_kernels_against_resident(graph, streams, steps, strips, ns):
    w = workloads.small(seed=ns, nx=60, nz=40, npml=10, nt=200 + ns, ns=ns)
    src = integrated_sources(w)
    p = _plan(w, 1, strips=strips)
    want = _run(p, src)
    p.close()
    p = _plan(w, 0, strips=strips)
    for option, value in (("graph", graph), ("streams", streams), ("bwd_steps", steps)):
        p.set_option(option, value)
    _same(_run(p, src), want)
    _same(_run(p, src), want)                     # the captured graphs replayed
    p.set_option("fwd_group", ns)                 # drops them
    p.set_option("bwd_tile_x", 16)
    p.set_option("profile", 1)
    _same(_run(p, src), want)
    assert not p.resident("forward") and not p.resident("backward")
    assert p.kernel_time("forward")[1] == p.kernel_time("backward")[1] == w.nt - 1
    p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [1, 0])
def test_step_kernels_against_the_oracle(graph):
    from oracle import oracle as O
    w = workloads.small(seed=12, nx=56, nz=36, npml=10, nt=220, ns=3)
    src = integrated_sources(w)
    m = O.Model(w.vp_init, workloads.gardner(w.vp_init), w.dx, w.npml, "f32")
    f = O.forward(m, w.nt, w.dt, w.src_xz, w.rec_xz, src)
    a = O.adjoint(m, w.nt, w.dt, w.src_xz, w.rec_xz, src, (f["seis"] * np.float32(1e-2)).astype(np.float32), f)
    p = _plan(w, 0)
    p.set_option("graph", graph)
    syn, strips, g, fw, bk = _run(p, src)
    p.close()
    np.testing.assert_array_equal(syn, f["seis"])
    np.testing.assert_array_equal(strips, f["boundary"])
    for x, name in ((g, "grad"), (fw, "illum_forw"), (bk, "illum_back")):
        assert rel_l2(x, a[name]) <= 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [True, "checkpoint"])
@pytest.mark.parametrize("streams,graph,fused,ns", [(1, 1, 1, 3), (1, 0, 0, 2), (2, 1, 1, 5), (2, 0, 1, 4), (2, 1, 0, 3)])
def test_exact_step_kernels_against_resident(kind, streams, graph, fused, ns):
    import torch
    w = workloads.small(seed=ns + 20, nx=52, nz=36, npml=10, nt=150 + ns, ns=ns)
    src = torch.from_numpy(integrated_sources(w))
    out = []
    for resident in (1, 0):
        p = _plan(w, resident, exact=kind)
        if not resident:
            for option, value in (("streams", streams), ("graph", graph), ("exact_fused", fused)):
                p.set_option(option, value)
        assert p.resident("exact") == bool(resident)
        for _ in range(2):
            syn = p.forward_exact(src)
            out.append((syn.cpu().numpy(), p.adjoint_exact((syn * 1e-2).contiguous()).cpu().numpy()))
        p.close()
    for o in out[1:]:
        _same(o, out[0])


@pytest.mark.gpu
def test_group_graph_after_an_option_change():
    import torch
    from swit_amd.engine import PlanGroup
    ws = [workloads.small(seed=51, nx=50, nz=34, npml=10, nt=210, ns=3),
          workloads.small(seed=52, nx=64, nz=28, npml=8, nt=160, ns=2)]
    srcs = [torch.from_numpy(integrated_sources(w)).cuda() for w in ws]
    plans = [_plan(w, 1) for w in ws]
    want = []
    for p, s in zip(plans, srcs):
        syn = p.forward(s)
        want.append([t.cpu().numpy() for t in (syn,) + tuple(p.adjoint(s, (syn * 1e-2).contiguous()))])
    adj = [torch.from_numpy(o[0]).cuda() * 1e-2 for o in want]
    for p in plans:
        p.set_option("resident", 0)
    grp = PlanGroup(plans)
    for rep in range(3):
        if rep == 2:
            plans[1].set_option("bwd_steps", 1)       # captured arguments change: recapture
            plans[1].set_option("fwd_group", 1)
        assert grp.sets("forward") == grp.sets("backward") == 0
        seis = grp.forward(srcs)
        for o, s, g in zip(want, seis, grp.adjoint(srcs, adj)):
            _same([s.cpu().numpy()] + [t.cpu().numpy() for t in g], o)
    grp.close()
    for p in plans:
        p.close()


@pytest.mark.gpu
def test_captured_calls():
    """On a capturing stream a plan takes its step kernels; replays between resident jobs."""
    import torch
    w = workloads.small(seed=31, nx=58, nz=38, npml=10, nt=140, ns=2)
    src = torch.from_numpy(integrated_sources(w)).cuda()
    p = _plan(w, 1, strips="f16")
    p.set_option("graph", 0)                          # the caller's capture holds the launches
    syn = p.forward(src)
    adj = (syn * 1e-2).contiguous()
    want = [t.cpu().numpy() for t in (syn,) + tuple(p.adjoint(src, adj))]
    torch.cuda.synchronize()
    st, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(g, stream=st):
        out = (p.forward(src),) + tuple(p.adjoint(src, adj))
    for _ in range(3):
        for t in out:
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        _same([t.cpu().numpy() for t in out], want)
        _same([t.cpu().numpy() for t in (p.forward(src),) + tuple(p.adjoint(src, adj))], want)
    del out, g
    p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 4])
def test_resident_plans_on_streams_of_their_own(n):
    """Each plan's 40 shots take more than one round of the chip."""
    import torch
    w = workloads.small(seed=35, nx=300, nz=100, npml=20, nt=80, ns=40)
    src = torch.from_numpy(integrated_sources(w)).cuda()
    plans = [_plan(w, 1) for _ in range(n)]
    syn = plans[0].forward(src)
    adj = (syn * 1e-2).contiguous()
    want = [t.cpu().numpy() for t in (syn,) + tuple(plans[0].adjoint(src, adj))]
    streams = [torch.cuda.Stream() for _ in plans]
    torch.cuda.synchronize()
    for _ in range(3):
        outs = []
        for p, st in zip(plans, streams):
            with torch.cuda.stream(st):
                outs.append((p.forward(src),) + tuple(p.adjoint(src, adj)))
        torch.cuda.synchronize()
        for o in outs:
            _same([t.cpu().numpy() for t in o], want)
    for p in plans:
        p.close()

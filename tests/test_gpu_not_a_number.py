"""What becomes of a forward that is not a number (a time loop that gave up, an unstable
model): the misfits of its traces and the group gradient's are NaN, not those of a perfect model;
dead and ordinary traces keep the toolbox's rules; the drop-in solver reports a crash."""
import numpy as np
import pytest

from helpers import integrated_sources
from swit_amd import misfit as host
from swit_amd import workloads

KINDS = {"Waveform": (host.misfit_waveform, host.adjoint_source_waveform),
         "Globalcorrelation": (host.misfit_global_correlation, host.adjoint_source_global_correlation),
         "Envelope": (host.misfit_envelope, host.adjoint_source_envelope),
         "Traveltime": (host.misfit_traveltime, host.adjoint_source_traveltime)}


@pytest.mark.gpu
@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("ntr,nt", [(6, 2), (6, 300), (700, 1000), (6, 4400)])
def test_traces_that_are_no_number(kind, ntr, nt):
    """Trace 1: every sample; 2: the last one.  3: NaN in the observed one (dead by norm > 0); 4:
    NaN against an observed trace without energy (dead).  The others as without them."""
    import torch
    from swit_amd.engine import misfit
    rng = np.random.default_rng(nt)
    t = np.arange(nt) * 0.002
    obs = (np.sin(2 * np.pi * (3.0 + rng.random((ntr, 1))) * (t + 0.01)) + 0.1).astype(np.float32)
    syn = (np.roll(obs, 1, axis=1) * np.float32(1.2) + np.float32(0.01) * (t > 0.1)).astype(np.float32)
    clean = misfit(kind, torch.from_numpy(obs).cuda(), torch.from_numpy(syn).cuda(), 0.002)
    syn[1] = np.nan
    syn[2, -1] = np.nan
    obs[3, nt // 2] = np.nan
    obs[4] = 0.0
    syn[4] = np.nan
    J, adj, per = misfit(kind, torch.from_numpy(obs).cuda(), torch.from_numpy(syn).cuda(), 0.002)
    adj, per = adj.cpu().numpy(), per.cpu().numpy()
    assert np.isnan(adj[1:3]).all() and np.isnan(per[1:3]).all() and np.isnan(float(J))
    assert not adj[3:5].any() and not per[3:5].any()
    rest = [0] + list(range(5, ntr))
    np.testing.assert_array_equal(adj[rest], clean[1].cpu().numpy()[rest])
    np.testing.assert_array_equal(per[rest], clean[2].cpu().numpy()[rest])


def _plan(w):
    import torch
    from swit_amd.engine import Plan
    p = Plan(w.nx, w.nz, w.dx, w.dt, w.nt, w.npml, w.src_xz, w.rec_xz)
    p.set_model(torch.from_numpy(w.vp_init), torch.from_numpy(workloads.gardner(w.vp_init)))
    p.set_option("resident", 1)
    return p


@pytest.mark.gpu
@pytest.mark.parametrize("kind", list(KINDS))
def test_group_gradient_that_gives_up(kind):
    import torch
    from swit_amd.engine import PlanGroup
    w = workloads.small(seed=78, nx=150, nz=40, npml=10, nt=200, ns=2)
    src = torch.from_numpy(integrated_sources(w)).cuda()
    plans = [_plan(w), _plan(w)]
    obs = [(plans[0].forward(src) * 1.1).contiguous() for _ in plans]
    grp = PlanGroup(plans)
    ref = [float(J) for J in grp.gradient([src, src], obs, kind)[0]]
    plans[1].set_option("resident_wait", 0)
    Js, seis, outs = grp.gradient([src, src], obs, kind)
    assert float(Js[0]) == ref[0] and np.isnan(float(Js[1]))
    assert all(bool(t.isnan().all()) for t in outs[1]) and not any(bool(t.isnan().any()) for t in outs[0])
    grp.close()
    for p in plans:
        p.close()


@pytest.mark.gpu
def test_dropin_reports_a_crash(tmp_path):
    from test_gpu_dropin import _optim, _simu
    from swit_amd import preprocess, solver
    w = workloads.small(seed=22, nx=150, nz=36, npml=10, nt=200, ns=2)
    w.rec_xz = w.rec_xz[:, :w.nx]
    home = str(tmp_path) + "/"
    simu, optim = _simu(home, w, w.vp_init), _optim()
    solver.forward(_simu(home, w, w.vp_true), 'obs')
    solver.forward(simu, 'syn', savesnap=1)
    preprocess.process_workflow(simu, optim, 'obs')
    preprocess.process_workflow(simu, optim, 'syn')
    plan = solver._JOBS[simu.system.homepath].plan
    plan.set_option("resident", 1)
    plan.set_option("resident_wait", 0)
    with pytest.raises(ValueError, match="Adjoint solver crash"):
        solver.adjoint(simu, optim)
    with pytest.raises(ValueError, match="Forward solver crash"):
        solver.forward(simu, 'syn', savesnap=1)
    plan.set_option("resident_wait", 30000)
    solver.forward(simu, 'syn', savesnap=1)
    preprocess.process_workflow(simu, optim, 'syn')
    assert np.isfinite(solver.adjoint(simu, optim)).all()
    solver.release(simu.system.homepath)

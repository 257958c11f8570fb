"""The ways a plan group runs: plans side by side where their resident loops fit the chip together (at
most four), one after the other where each fills it, plans of step kernels by themselves, or all
as one graph of step kernels.  Each gives the bits of every plan run alone, in forward, adjoint and
whole gradient, call after call.  Few shots a line one after the other were slower than the graph:
three lines of one shot (220x259 and two smaller, 765 steps) 19.8 ms, the graph 12.5."""
import numpy as np
import pytest

from helpers import integrated_sources
from swit_amd import workloads


def _lines(*cases):
    return [workloads.small(seed=60 + i, **c) for i, c in enumerate(cases)]


ONE_SHOT = [dict(nx=200, nz=80, npml=20, nt=150, ns=1), dict(nx=190, nz=56, npml=20, nt=120, ns=1),
            dict(nx=120, nz=48, npml=20, nt=90, ns=1)]
MANY = [dict(nx=400, nz=170, npml=20, nt=40, ns=22), dict(nx=380, nz=121, npml=20, nt=32, ns=21),
        dict(nx=240, nz=102, npml=20, nt=24, ns=21)]
# one shot each: too tall for a resident loop; many shots
TALL = [dict(nx=60, nz=520, npml=20, nt=50, ns=1)] + MANY[1:]
# (lines, resident option by plan or None, sets forward, sets backward)
CASES = {"few shots side by side": (ONE_SHOT, None, 1, 1),
         "at most four": (ONE_SHOT + ONE_SHOT[1:], None, 2, 2),
         "many shots in turn": (MANY, None, 3, 3),
         "a plan of step kernels by itself": (TALL, None, 3, 3),
         "an option on one plan": (MANY, [1, 0, 1], 3, 3),
         "one graph": (ONE_SHOT, [0, 0, 0], 0, 0)}


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
def test_route(case):
    import torch
    from swit_amd.engine import Plan, PlanGroup, misfit
    cases, resident, sets_f, sets_b = CASES[case]
    plans, srcs, obs, ref = [], [], [], []
    for i, w in enumerate(_lines(*cases)):
        src = torch.from_numpy(integrated_sources(w)).cuda()
        p = Plan(w.nx, w.nz, w.dx, w.dt, w.nt, w.npml, w.src_xz, w.rec_xz, strips=["f32", "f16", "f32"][i % 3])
        p.set_model(torch.from_numpy(w.vp_init), torch.from_numpy(workloads.gardner(w.vp_init)))
        if resident:
            p.set_option("resident", resident[i])
        syn = p.forward(src, save_strips=True)
        o = (1.1 * torch.roll(syn, 1, 2)).contiguous()
        J, adj, _ = misfit("Waveform", o, syn, w.dt)
        g = p.adjoint(src, adj)
        ref.append((float(J), syn.cpu().numpy(), adj, [t.cpu().numpy() for t in g]))
        plans.append(p)
        srcs.append(src)
        obs.append(o)
    grp = PlanGroup(plans)
    assert grp.sets("forward") == sets_f and grp.sets("backward") == sets_b
    for _ in range(2):
        seis = grp.forward(srcs, save_strips=True)
        outs = grp.adjoint(srcs, [r[2] for r in ref])
        for (J0, s0, _, g0), s, g in zip(ref, seis, outs):
            np.testing.assert_array_equal(s.cpu().numpy(), s0)
            for a, b in zip(g, g0):
                np.testing.assert_array_equal(a.cpu().numpy(), b)
        Js, seis, outs = grp.gradient(srcs, obs, "Waveform")
        for (J0, s0, _, g0), J, s, g in zip(ref, Js, seis, outs):
            assert float(J) == J0
            np.testing.assert_array_equal(s.cpu().numpy(), s0)
            for a, b in zip(g, g0):
                np.testing.assert_array_equal(a.cpu().numpy(), b)
    grp.close()
    for p in plans:
        p.close()

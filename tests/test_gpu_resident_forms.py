"""Resident loops against the step kernels over drawn forms: sizes, layers, shot counts, record
lengths, sources at any depth, receivers on the surface, on several rows, on the last row, several
to a cell, at random cells, fewer on later shots, strip precisions, exact histories, either
surface condition.  Seismograms, strips, gradient, illuminations and the exact gradient are the same
bits, in two passes."""
import math
import random

import numpy as np
import pytest

from helpers import integrated_sources
from swit_amd import workloads


def _form(seed):
    rng, nrg = random.Random(seed), np.random.default_rng(seed)

    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))
    while True:
        nx, nz, npml, ns = log(8, 700), log(9, 400), rng.choice([3, 8, 10, 20, 30, 50]), log(1, 60)
        if (nx + 2 * npml) * (nz + 2 * npml) * ns < 6e6:
            break
    w = workloads.small(seed=seed, nx=nx, nz=nz, npml=npml, nt=rng.choice([2, 3, 20, 60, 130, 140]), ns=ns)
    kind = rng.choice(["surface", "rows", "ragged", "shared", "deep", "any"])
    surface = [(x, 0) for x in range(nx)]
    cells = {"rows": [(x, z) for z in rng.sample(range(nz), min(nz, rng.randint(2, 7)))
                      for x in range(0, nx, rng.choice([1, 2, 5]))],
             "deep": [(x, nz - 1) for x in range(nx)],
             "shared": [(x, 2) for x in range(nx)] + [(x, 2) for x in range(0, nx, 3)],
             "any": [(nrg.integers(0, nx), nrg.integers(0, nz)) for _ in range(60)]}.get(kind, surface)
    rec = np.asarray(cells, np.float32) * np.float32(w.dx)
    w.rec_xz = [rec[:max(1, len(rec) - (3 * i if kind == "ragged" else 0))] for i in range(ns)]
    w.src_xz = np.stack([nrg.integers(0, nx, ns), nrg.integers(0, max(1, nz - 1), ns)], 1).astype(np.float32) * w.dx
    return w, dict(strips=rng.choice(["f32", "f32", "f16", "bf16"]), exact=rng.choice([False, True, "checkpoint"]),
                   free_surface=rng.choice([1, 1, 0]))


@pytest.mark.gpu
@pytest.mark.parametrize("first", range(1140, 1340, 20))
def test_forms(first):
    import torch
    from swit_amd.engine import Plan
    for seed in range(first, first + 20):
        w, kw = _form(seed)
        p = Plan(w.nx, w.nz, w.dx, w.dt, w.nt, w.npml, w.src_xz, w.rec_xz, **kw)
        p.set_model(torch.from_numpy(w.vp_init), torch.from_numpy(workloads.gardner(w.vp_init)))
        src = torch.from_numpy(integrated_sources(w)).cuda()
        adj, want = None, None
        for resident in (0, 1, 1):
            p.set_option("resident", resident)
            syn = p.forward(src)
            if adj is None:
                adj = torch.randn(syn.shape, generator=torch.Generator("cuda").manual_seed(seed), device="cuda")
            out = [syn, p.saved_strips()] + list(p.adjoint(src, adj))
            if kw["exact"]:
                out += [p.forward_exact(src), p.adjoint_exact(adj)]
            if want is None:
                want = out
            for k, (a, b) in enumerate(zip(out, want)):
                assert torch.equal(a, b), (seed, w.nx, w.nz, w.npml, w.nt, w.ns, kw, "output %d" % k)
        p.close()

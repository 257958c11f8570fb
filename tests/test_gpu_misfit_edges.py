"""Waveform and global-correlation misfits at the edges of their layout: 256 samples a pass, 16 of
each trace per thread in registers (4096), longer records from memory, more traces than one pass
of the final sum; and norms outside the range of the division by a shared divisor."""
import numpy as np
import pytest

from swit_amd import misfit as host


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [2, 3, 255, 256, 257, 4095, 4096, 4097, 4400])
def test_lengths(nt):
    """The adjoint source is the FP64 value rounded to float32 (two units of the last place for
    sums in another order); the waveform's is exact."""
    import torch
    from swit_amd.engine import misfit
    rng = np.random.default_rng(nt)
    obs = rng.standard_normal((4100 if nt < 300 else 5, nt)).astype(np.float32)
    syn = (0.7 * obs + 0.5 * rng.standard_normal(obs.shape)).astype(np.float32)
    o, s = torch.from_numpy(obs).cuda(), torch.from_numpy(syn).cuda()
    J, adj, _ = misfit("Waveform", o, s, 0.002)
    np.testing.assert_array_equal(adj.cpu().numpy(), syn - obs)
    o64, s64 = obs.astype(np.float64), syn.astype(np.float64)
    dt = float(np.float32(0.002))
    r = (syn - obs).astype(np.float64)                   # the residual is a float32 array
    assert float(J) == pytest.approx(np.sum(np.sqrt(np.sum(r * r, axis=1) * dt)), rel=1e-12)
    J, adj, _ = misfit("Globalcorrelation", o, s, 0.002)
    want = host.adjoint_source_global_correlation(o64, s64, dt)
    np.testing.assert_allclose(adj.cpu().numpy(), want, rtol=0, atol=2.0 ** -22 * np.abs(want).max())
    assert float(J) == pytest.approx(host.misfit_global_correlation(o64, s64, dt), rel=1e-12, abs=1e-12 * len(obs))


@pytest.mark.gpu
def test_infinite_sample():
    """An infinite sample makes its own adjoint sample NaN and the finite ones 0 (x / inf), as the
    division does; the other traces are untouched."""
    import torch
    from swit_amd.engine import misfit
    rng = np.random.default_rng(1)
    obs = rng.standard_normal((3, 300)).astype(np.float32)
    syn = rng.standard_normal((3, 300)).astype(np.float32)
    clean = misfit("Globalcorrelation", torch.from_numpy(obs).cuda(), torch.from_numpy(syn).cuda(), 0.002)[1].cpu().numpy()
    syn[1, 7] = np.inf
    adj = misfit("Globalcorrelation", torch.from_numpy(obs).cuda(), torch.from_numpy(syn).cuda(), 0.002)[1].cpu().numpy()
    np.testing.assert_array_equal(adj[[0, 2]], clean[[0, 2]])
    assert np.isnan(adj[1, 7]) and np.all(np.delete(adj[1], 7) == 0)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["Envelope", "Traveltime"])
@pytest.mark.parametrize("nt", [2, 8, 200, 1000, 2000, 2048, 2003, 1001])
def test_fft_misfits_of_many_traces(nt, kind):
    """More than 512 traces (256 threads each where every stage is a register butterfly) against
    the same traces in calls of 100 (512 threads each): the transforms' operations are the same,
    the FP64 sums over a trace go in another order."""
    import torch
    from swit_amd.engine import misfit
    rng = np.random.default_rng(nt)
    t = np.arange(nt) * 0.002
    obs = (np.sin(2 * np.pi * (3.0 + rng.random((700, 1))) * t) + 0.1 * rng.standard_normal((700, nt))).astype(np.float32)
    syn = np.roll(obs, 3, axis=1) * np.float32(1.2)
    obs[5] = 0.0
    o, s = torch.from_numpy(obs).cuda(), torch.from_numpy(syn).cuda()
    J, adj, per = misfit(kind, o, s, 0.002)
    parts = [misfit(kind, o[a:a + 100].contiguous(), s[a:a + 100].contiguous(), 0.002) for a in range(0, 700, 100)]
    want = np.concatenate([p[1].cpu().numpy() for p in parts])
    np.testing.assert_allclose(adj.cpu().numpy(), want, rtol=0, atol=2e-7 * max(np.abs(want).max(), 1e-30))
    wper = np.concatenate([p[2].cpu().numpy() for p in parts])
    np.testing.assert_allclose(per.cpu().numpy(), wper, rtol=1e-12, atol=1e-300)
    assert float(J) == pytest.approx(wper.sum(), rel=1e-12)

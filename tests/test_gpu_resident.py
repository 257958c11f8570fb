"""Resident time loops (the wavefields of a shot in registers, many steps per launch) against
the step kernels: the same bits for seismograms, strips and everything computed from them.
Sizes lie at the edges of the layout: heights around a multiple of 64 rows (each number of
rows per lane), widths that leave one to a few columns to the last window or fit one window,
records of 2, 3 and a few steps, 16-bit strips whose record ends at, before and after a full
ring, many receivers on many rows (written directly) and a few rows (staged), several
receivers in a cell, sources next to window edges, more shots than run at once."""
import numpy as np
import pytest

from helpers import integrated_sources
from swit_amd import workloads


def _outputs(w, strips, resident, free_surface=1, sources=None):
    import torch
    from swit_amd.engine import Plan
    p = Plan(w.nx, w.nz, w.dx, w.dt, w.nt, w.npml, w.src_xz, w.rec_xz, strips=strips, free_surface=free_surface)
    p.set_model(torch.from_numpy(w.vp_init), torch.from_numpy(workloads.gardner(w.vp_init)))
    p.set_option("resident", resident)
    src = torch.from_numpy(integrated_sources(w) if sources is None else sources)
    out = []
    for _ in range(2):                       # a second job on the same plan
        syn = p.forward(src, save_strips=strips != "none")
        res = [syn]
        if strips != "none":
            res.append(p.saved_strips())
            res += list(p.adjoint(src, (syn * 1e-2).contiguous()))
        out.append([t.cpu().numpy() for t in res])
    p.close()
    return out


def _check(w, strips, free_surface=1):
    ref = _outputs(w, strips, 0, free_surface)
    got = _outputs(w, strips, 1, free_surface)
    assert np.abs(ref[0][0]).max() > 0
    for a, b in zip(ref, got):
        for name, x, y in zip(("seismograms", "strips", "gradient", "forward illumination",
                               "backward illumination"), a, b):
            np.testing.assert_array_equal(y, x, err_msg=name)


@pytest.mark.gpu
@pytest.mark.parametrize("nz,npml", [(117, 10), (118, 10), (181, 10), (182, 10), (246, 9), (309, 10), (310, 10),
                                     (373, 10), (438, 9), (501, 10)])
def test_rows_per_lane(nz, npml):
    """nz + npml + 1 rows: 128, 129, 192, 193, 256, 320, 321, 384, 448, 512."""
    w = workloads.small(seed=nz, nx=70, nz=nz, npml=npml, nt=60, ns=2)
    _check(w, "f32")


@pytest.mark.gpu
@pytest.mark.parametrize("nx", [8, 9, 34, 41, 49, 50, 51, 52, 53, 54, 55, 61, 118, 119, 120, 121, 122, 123, 240])
def test_widths(nx):
    w = workloads.small(seed=nx, nx=nx, nz=40, npml=10, nt=70, ns=2)
    _check(w, "f32", free_surface=nx % 2)


@pytest.mark.gpu
@pytest.mark.parametrize("strips", ["f16", "bf16"])
@pytest.mark.parametrize("nt", [2, 3, 127, 128, 129, 130, 256, 257])
def test_sixteen_bit_rings(nt, strips):
    w = workloads.small(seed=nt, nx=60, nz=30, npml=8, nt=nt, ns=3)
    ref, got = _outputs(w, strips, 0), _outputs(w, strips, 1)
    for a, b in zip(ref, got):
        for x, y in zip(a, b):
            np.testing.assert_array_equal(y, x)


@pytest.mark.gpu
@pytest.mark.parametrize("strips", ["none", "f32"])
def test_receivers_on_every_row_and_shared_cells(strips):
    w = workloads.small(seed=3, nx=90, nz=70, npml=12, nt=90, ns=3)
    rec = [[x * w.dx, 0.0] for x in range(w.nx)]
    rec += [[x * w.dx, z * w.dx] for x in (0, 17, 44, 89) for z in range(1, w.nz)]
    rec += [[17 * w.dx, 5 * w.dx], [17 * w.dx + 1.0, 5 * w.dx + 1.0], [3 * w.dx, 0.0], [3 * w.dx, 1.0 * w.dx]]
    w.rec_xz = np.broadcast_to(np.asarray(rec, np.float32), (w.ns, len(rec), 2)).copy()
    _check(w, strips)


@pytest.mark.gpu
def test_many_receivers_on_one_row_ragged():
    """More receivers than columns (several to a cell), fewer on the later shots."""
    w = workloads.small(seed=4, nx=110, nz=40, npml=10, nt=80, ns=4)
    rec = np.array([[x * w.dx * 0.25, 3.0 * w.dx] for x in range(4 * w.nx - 4)], np.float32)
    w.rec_xz = [rec[:len(rec) - 60 * i] for i in range(w.ns)]
    _check(w, "f32")


@pytest.mark.gpu
def test_sources_at_every_depth_and_more_shots_than_run_at_once():
    w = workloads.small(seed=6, nx=260, nz=180, npml=30, nt=40, ns=6)
    n = 90
    rng = np.random.default_rng(6)
    w.src_xz = np.stack([rng.integers(0, w.nx, n) * w.dx, rng.integers(0, w.nz - 1, n) * w.dx], 1).astype(np.float32)
    w.rec_xz = np.broadcast_to(w.rec_xz[0], (n,) + w.rec_xz[0].shape).copy()
    _check(w, "f32")


@pytest.mark.gpu
def test_seismograms_against_the_oracle():
    import torch
    from oracle import oracle as O
    from swit_amd.engine import Plan
    w = workloads.small(seed=8, nx=150, nz=60, npml=20, nt=300, ns=2)
    src = integrated_sources(w)
    m = O.Model(w.vp_init, workloads.gardner(w.vp_init), w.dx, w.npml, "f32")
    f = O.forward(m, w.nt, w.dt, w.src_xz, w.rec_xz, src)
    p = Plan(w.nx, w.nz, w.dx, w.dt, w.nt, w.npml, w.src_xz, w.rec_xz)
    p.set_model(torch.from_numpy(w.vp_init), torch.from_numpy(workloads.gardner(w.vp_init)))
    np.testing.assert_array_equal(p.forward(torch.from_numpy(src)).cpu().numpy(), f["seis"])
    p.close()


def _exact_outputs(w, kind, resident, free_surface=1):
    import torch
    from swit_amd.engine import Plan
    p = Plan(w.nx, w.nz, w.dx, w.dt, w.nt, w.npml, w.src_xz, w.rec_xz, strips="none", exact=kind,
             free_surface=free_surface)
    p.set_model(torch.from_numpy(w.vp_init), torch.from_numpy(workloads.gardner(w.vp_init)))
    p.set_option("resident", resident)
    src = torch.from_numpy(integrated_sources(w))
    out = []
    for _ in range(2):
        syn = p.forward_exact(src)
        g = torch.flip(syn, (2,)) + syn
        out.append([syn.cpu().numpy(), p.adjoint_exact(g.contiguous()).cpu().numpy()])
    p.close()
    return out


def _check_exact(w, kind, free_surface=1):
    """The reverse loop's operations and their order are the step kernels': equal but for the
    sign of zeros (cells outside an update region multiply by 0 there, here they are skipped)."""
    ref, got = (_exact_outputs(w, kind, r, free_surface) for r in (0, 1))
    assert np.abs(ref[0][0]).max() > 0
    for a, b in zip(ref, got):
        np.testing.assert_array_equal(b[0], a[0])
        np.testing.assert_array_equal(b[1], a[1])


@pytest.mark.gpu
@pytest.mark.parametrize("nz,npml", [(117, 10), (118, 10), (181, 10), (182, 10), (246, 9), (310, 10), (373, 10),
                                     (438, 9), (501, 10)])
def test_exact_rows_per_lane(nz, npml):
    w = workloads.small(seed=nz, nx=70, nz=nz, npml=npml, nt=90, ns=2)
    _check_exact(w, True)


@pytest.mark.gpu
@pytest.mark.parametrize("nx", [8, 9, 34, 49, 50, 51, 52, 53, 61, 121, 240])
def test_exact_widths(nx):
    w = workloads.small(seed=nx, nx=nx, nz=40, npml=10, nt=70, ns=2)
    _check_exact(w, "checkpoint" if nx % 3 else True, free_surface=nx % 2)


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [2, 3, 5, 49, 50, 101])
def test_exact_checkpoint_segments(nt):
    """Records of one segment, of a last segment of one step, of full segments."""
    w = workloads.small(seed=nt, nx=60, nz=30, npml=8, nt=nt, ns=3)
    _check_exact(w, "checkpoint")


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [True, "checkpoint"])
def test_exact_shared_cells_and_many_shots(kind):
    w = workloads.small(seed=6, nx=130, nz=50, npml=10, nt=80, ns=70)
    rec = [[x * w.dx, z * w.dx] for x in range(w.nx) for z in (1.0, 9.0)]
    rec += [[17 * w.dx, w.dx], [18 * w.dx, 9.0 * w.dx], [29 * w.dx, w.dx]]
    w.rec_xz = [np.asarray(rec[:len(rec) - i], np.float32) for i in range(w.ns)]
    _check_exact(w, kind)

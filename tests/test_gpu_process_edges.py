"""Trace lengths at the edges of the processing kernels' layout (blocks of 16 samples in the
filter, 16 samples of a trace per thread in registers: 4096, the rest from memory), and a
workspace that filters the traces in more than one launch.  Bit-exact against scipy's filtfilt
and the host restatement, as the tests of the ordinary lengths."""
import ctypes

import numpy as np
import pytest

from swit_amd import preprocess
from test_gpu_process import _device, _gathers, _host, _optim


@pytest.mark.gpu
@pytest.mark.parametrize("nt", [28, 31, 32, 33, 47, 48, 4095, 4096, 4097])
def test_filter_lengths(nt):
    from scipy.signal import filtfilt
    from swit_amd import engine
    d, off = _gathers(nt=nt)
    o = _optim(fre_filter='bandpass', fre_low=4.0, fre_high=18.0)
    p, win, taper = engine.process_params(o, *d.shape, 0.002)
    p.detrend_taper = 0
    b, a = preprocess.filter_design(o, 0.002)
    np.testing.assert_array_equal(_device(o, d, 0.002, off, params=(p, win, None)), filtfilt(b, a, d).astype(np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("window", [0.08, -0.08])
@pytest.mark.parametrize("nt", [255, 256, 4096, 4097, 4500])
def test_mute_and_maximum_lengths(nt, window):
    d, off = _gathers(nt=nt)
    o = _optim(mute_late_arrival=1, mute_late_window=window, normalize=['Max-Trace'])
    np.testing.assert_array_equal(_device(o, d, 0.002, off), _host(o, d, 0.002, off))


@pytest.mark.gpu
def test_filter_in_several_launches():
    import torch
    from swit_amd import _native, engine
    rng = np.random.default_rng(3)
    d = rng.standard_normal((1, 16384 + 70, 60)).astype(np.float32)
    o = _optim(fre_filter='lowpass', fre_low=15.0, fre_high=15.0)
    p, _, _ = engine.process_params(o, *d.shape, 0.002)
    p.detrend_taper = 0
    want = _device(o, d, 0.002, None, params=(p, None, None))
    lib = _native.load()
    nb = ctypes.c_size_t()
    _native.check(lib.swit_process_work(ctypes.byref(p), ctypes.byref(nb)))
    assert nb.value == 8 * (60 + 6 * p.filter_taps) * 16384
    x = torch.from_numpy(d).cuda()
    work = torch.empty(nb.value, dtype=torch.uint8, device="cuda")
    _native.check(lib.swit_process(ctypes.byref(p), None, None, None, None, ctypes.c_void_p(x.data_ptr()),
                                   ctypes.c_void_p(work.data_ptr()), nb.value,
                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    np.testing.assert_array_equal(x.cpu().numpy(), want)

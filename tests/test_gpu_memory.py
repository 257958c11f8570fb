"""Calls that took what memory there is still do where a larger workspace does not fit: they run
with less."""
import numpy as np
import pytest


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

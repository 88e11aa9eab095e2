"""-m gpu: host tensors that reach the device in one copy (models/flash_causal_lm.py)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1,), (0, 5, 1), (64, 7, 33, 1000)])
def test_to_device_together(gpu_device, sizes):
    from tgis_amd.models.flash_causal_lm import to_device_together

    dtypes = [torch.int64, torch.int32, torch.uint8]
    host = [torch.arange(n * (1 + i % 2)).to(dtypes[i % 3]).view(1 + i % 2, n) for i, n in enumerate(sizes)]
    there = to_device_together(host, gpu_device)
    for h, d in zip(host, there):
        assert d.is_cuda and d.dtype == h.dtype and d.is_contiguous() and d.data_ptr() % 64 == 0 and torch.equal(d.cpu(), h)
    kept = [h.clone() for h in host]
    for d in there:  # no part reaches into another one
        d.fill_(1)
        for h, o in zip(kept, there):
            assert o is d or torch.equal(o.cpu(), h)
        d.copy_(kept[[o is d for o in there].index(True)])

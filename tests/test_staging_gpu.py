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


def test_batch_of_prompts(gpu_device):
    """The indices of a new batch: prompts of one token and many, one behind a prefix, a second one without."""
    from tgis_amd.models.flash_causal_lm import FlashCausalLMBatch
    from tgis_amd.testing import SyntheticTokenizer, make_batch_pb

    tok = SyntheticTokenizer(1000)
    prefix = torch.full((3, 8), 5.0, device=gpu_device)
    cache = type("Cache", (), {"get": lambda self, name: prefix})()
    table = torch.arange(8000, dtype=torch.float32, device=gpu_device).view(1000, 8)
    for lens in ([1], [5], [40, 1, 7]):
        for prefixed in (False, True):
            pb = make_batch_pb(lens, max_new=4)
            if prefixed:
                pb.requests[0].prefix_id = "p"
            batch, errors = FlashCausalLMBatch.from_pb(pb, tok, torch.float16, gpu_device, lambda ids: table[ids], cache, True)
            assert not errors
            words = [t[-n:] for t, n in zip(tok([r.inputs for r in pb.requests], truncation=True, max_length=max(lens), return_token_type_ids=False)["input_ids"], lens)]
            words = [[tok.pad_token_id] * (3 if prefixed and i == 0 else 0) + list(w) for i, w in enumerate(words)]
            full = [len(w) for w in words]
            assert batch.input_lengths == full and batch.cu_seqlens.tolist() == [sum(full[:i]) for i in range(len(full) + 1)]
            assert batch.cu_seqlens.dtype == torch.int32 and batch.position_ids.dtype == torch.int64
            assert batch.position_ids.tolist() == [p for n in full for p in range(n)]
            for row, w in zip(batch.all_input_ids_tensor.tolist(), words):
                assert row == w + [tok.pad_token_id] * (len(row) - len(w)) and len(row) == max(full) + 4
            flat = torch.tensor([t for w in words for t in w])
            if prefixed:
                want = table.cpu()[flat]
                want[:3] = 5.0
                assert batch.input_ids is None and torch.equal(batch.inputs_embeds.cpu(), want)
            else:
                assert torch.equal(batch.input_ids.cpu(), flat) and batch.inputs_embeds is None

"""-m gpu: decode steps of a few rows of a dense Llama model on the launches that norm their operand (FlashLlamaModel.forward_rows), against the same
steps through `forward`: the logits and the pages written, from a captured graph and step by step; and the models and steps that go the other way."""
import pytest
import torch

from tests.test_llama_prompt_gpu import model

pytestmark = pytest.mark.gpu

STEPS = 4


def decode(lm, vocab, rows, graphs):
    """Prompts of different lengths and STEPS forced tokens behind them (one sequence takes a new page): every step's logits, the pages left."""
    from tgis_amd.testing import SyntheticTokenizer, make_batch_pb

    lm.use_graphs = graphs
    lens = ([30, 9, 47, 17, 5] + [3 + i % 20 for i in range(rows)])[:rows]
    forced = torch.randint(3, vocab, (STEPS, rows), generator=torch.Generator().manual_seed(rows)).cuda()
    taken, run = [], lm._process_new_tokens
    lm._process_new_tokens = lambda batch, out, *a, **k: taken.append(out.clone()) or run(batch, out, *a, **k)
    for i in range(lm.num_layers):
        for pool in (lm.kv_cache.k_pool(i), lm.kv_cache.v_pool(i)):
            pool.zero_()
    with lm.context_manager():
        batch, errors = lm.batch_type.from_pb(make_batch_pb(lens, max_new=STEPS + 2), SyntheticTokenizer(vocab), lm.dtype, lm.device, lm.word_embeddings,
                                              None, lm.use_position_ids)
        assert not errors
        lm.generate_token(batch, first=True)
        for tokens in forced:
            batch.input_ids = tokens
            lm.generate_token(batch)
        flat = torch.tensor([p for seq in batch.pages for p in seq]).cuda()
        pages = [pool.view(64, -1)[flat].clone() for i in range(lm.num_layers) for pool in (lm.kv_cache.k_pool(i), lm.kv_cache.v_pool(i))]
    batch.release()
    return taken, pages


@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_same_steps(gpu_device, monkeypatch, dtype, graphs, rows):
    from tgis_amd.models.custom_modeling.flash_llama_modeling import FlashLlamaForCausalLM, FlashLlamaModel

    calls, run = [], FlashLlamaModel.forward_rows
    monkeypatch.setattr(FlashLlamaModel, "forward_rows", lambda self, ids, *a: calls.append(ids.shape[0]) or run(self, ids, *a))
    # (three and four rows of bf16 are forward_rows16's, but for TGIS_DEFER_REDUCE=0)
    monkeypatch.setattr(FlashLlamaForCausalLM, "rows16_path", lambda self, n: False)
    lm, cfg = model(dtype)
    got, pages = decode(lm, cfg.vocab_size, rows, graphs)
    # a warm-up and a capture, or every step; with the rows of its bucket
    assert calls == [1 << (rows - 1).bit_length()] * (2 if graphs else STEPS)
    monkeypatch.setattr(FlashLlamaForCausalLM, "rows_path", lambda self, n: False)
    del calls[:]
    lm, _ = model(dtype)
    want, pages_want = decode(lm, cfg.vocab_size, rows, graphs)
    assert not calls and len(got) == len(want) == STEPS + 1 and torch.equal(got[0], want[0])
    # sums in another order: here and there a value rounds to the other side (a step of the dtype), which three layers carry on: below four steps
    # in the norm of all
    step = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for a, b in zip(got[1:] + pages, want[1:] + pages_want):
        a, b = a.double(), b.double()
        assert a.shape == b.shape and float((a - b).norm() / b.norm()) < 4 * step


def test_other_steps(gpu_device, monkeypatch):
    """Five rows in f16, int4 layers and ranks of a group are not forward_rows's."""
    from tgis_amd.models.custom_modeling.flash_llama_modeling import FlashLlamaModel

    monkeypatch.setattr(FlashLlamaModel, "forward_rows", lambda *a: pytest.fail("served"))
    lm, cfg = model(torch.float16)
    assert [lm.model.rows_path(n) for n in (1, 4, 5, 64)] == [True, True, False, False]
    decode(lm, cfg.vocab_size, 5, False)
    lm.model._rows_path.clear()
    lm.model.model.tp_world_size = 2
    assert not lm.model.rows_path(1)
    lm, cfg = model(torch.float16, quantize="gptq")
    assert not lm.model.rows_path(1)
    decode(lm, cfg.vocab_size, 2, False)

"""-m gpu: a dense Llama model's layers on prompts, launched in one call, against the same launches one by one: the same bits in the logits and in
the pages; and the models and steps that go on one by one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def checkpoint(dtype, quantize=None, **kw):
    from oracle.tiny_models import TinyLlamaConfig, tiny_llama_tensors

    cfg = TinyLlamaConfig(**{**dict(hidden_size=2048, intermediate_size=1024, num_attention_heads=32, num_key_value_heads=4, num_hidden_layers=3), **kw})
    return cfg, {k: v.to(dtype) if v.is_floating_point() else v for k, v in tiny_llama_tensors(cfg, seed=7, quantize=quantize, groupsize=64).items()}


def model(dtype, **kw):
    from tgis_amd.inference_engine.synthetic import InferenceEngine
    from tgis_amd.models.custom_modeling.flash_llama_modeling import LlamaConfig
    from tgis_amd.models.flash_causal_lm import FlashCausalLM
    from tgis_amd.testing import SyntheticTokenizer

    quantize = kw.get("quantize")
    cfg, tensors = checkpoint(dtype, **kw)
    config = LlamaConfig(**cfg.to_dict())
    eng = InferenceEngine(tensors, config, dtype, quantize, tokenizer=SyntheticTokenizer(config.vocab_size), gptq_groupsize=64)
    return FlashCausalLM("synthetic", None, "synthetic", dtype, quantize, engine=eng, kv_cache_pages=64), config


def steps(lm, vocab, lens):
    """Prompts whole; the logits of every token, of the ends alone, and the pages left."""
    g = torch.Generator().manual_seed(11)
    pages = [lm.kv_cache.alloc(n // 32 + 1) for n in lens]
    last = (torch.tensor(lens).cumsum(0) - 1).cuda()
    ids = torch.randint(3, vocab, (sum(lens),), generator=g).cuda()
    for i in range(lm.num_layers):
        for pool in (lm.kv_cache.k_pool(i), lm.kv_cache.v_pool(i)):
            pool.zero_()  # (what lies behind a sequence's last token is either left or cleared)
    with lm.context_manager():
        out = [lm.ragged_forward(ids, pages, [0] * len(lens), lens),
               lm.ragged_forward(ids, pages, [0] * len(lens), lens, lm_head_indices=last, ends_only=True)]
        flat = torch.tensor([p for seq in pages for p in seq])
        for i in range(lm.num_layers):
            out += [pool.view(64, -1)[flat.cuda()].clone() for pool in (lm.kv_cache.k_pool(i), lm.kv_cache.v_pool(i))]
    for p in pages:
        lm.kv_cache.free(p)
    return out


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_same_bits(gpu_device, monkeypatch, dtype):
    from tgis_amd import native
    from tgis_amd.models.custom_modeling.flash_llama_modeling import FlashLlamaModel

    lm, cfg = model(dtype)
    calls, run = [], native.llama_prompt
    monkeypatch.setattr(native, "llama_prompt", lambda layers, x, *a, **k: calls.append((len(layers), x.shape[0])) or run(layers, x, *a, **k))
    for lens in ([1], [2], [47], [13, 1, 50], [65], [40, 30], [37, 1, 70, 33], [200, 57]):
        del calls[:]
        got = steps(lm, cfg.vocab_size, lens)
        assert calls[0] == (3, sum(lens)) and calls[1] == (2 if sum(lens) >= 128 else 3, sum(lens)), calls
        with monkeypatch.context() as m:
            m.setattr(FlashLlamaModel, "plain_layers", lambda self, *a: [])
            want = steps(lm, cfg.vocab_size, lens)
        assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want)), lens


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_cache_writes_token_by_token(gpu_device, monkeypatch, dtype):
    """TGIS_PREFILL_KV=0: the same bits."""
    from tgis_amd import native
    from tgis_amd.models import flash_causal_lm
    from tgis_amd.models.custom_modeling.flash_llama_modeling import FlashLlamaModel

    lm, cfg = model(dtype)
    monkeypatch.setattr(flash_causal_lm, "FRESH_PREFILL_KV", False)
    monkeypatch.setattr(native, "rope_kv_write_prefill", lambda *a, **k: pytest.fail("page by page"))
    calls, run = [], native.llama_prompt
    monkeypatch.setattr(native, "llama_prompt", lambda layers, x, *a, **k: calls.append(x.shape[0]) or run(layers, x, *a, **k))
    for lens in ([47], [13, 2, 40], [65], [100, 2, 90], [200, 57]):
        del calls[:]
        got = steps(lm, cfg.vocab_size, lens)
        assert calls == [sum(lens)] * 2
        with monkeypatch.context() as m:
            m.setattr(FlashLlamaModel, "plain_layers", lambda self, *a: [])
            want = steps(lm, cfg.vocab_size, lens)
        assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want)), lens


@pytest.mark.parametrize("kw,lens", [(dict(quantize="gptq"), [20]), (dict(hidden_size=256, num_attention_heads=4), [70]),
                                     (dict(), [1500])])
def test_one_by_one(gpu_device, monkeypatch, kw, lens):
    """int4 layers, products too narrow for the prefill kernel, rows past its rule: the oracle's logits."""
    from oracle.llama_ref import LlamaRef
    from tgis_amd import native

    lm, cfg = model(torch.float16, **kw)
    monkeypatch.setattr(native, "llama_prompt", lambda *a, **k: pytest.fail("served"))
    ids = torch.randint(3, cfg.vocab_size, (sum(lens),), generator=torch.Generator().manual_seed(3))
    pages = [lm.kv_cache.alloc(n // 32 + 1) for n in lens]
    with lm.context_manager():
        logits = lm.ragged_forward(ids.cuda(), pages, [0] * len(lens), lens)
    want = LlamaRef(*checkpoint(torch.float16, **kw), quantize=kw.get("quantize"), groupsize=64).forward(ids, torch.arange(lens[0]), [0] * lens[0], [[None] * 3])
    # every layer rounds its activations, keys and values, and the tables of its rotation, to 2 ** -11 of their size, which three layers carry on
    assert logits.shape == want.shape and float((logits.cpu().double() - want).norm() / want.double().norm()) < 8 * 2.0 ** -11


def test_no_split_sums_where_they_are_off(gpu_device, monkeypatch):
    """TGIS_DEFER_REDUCE=0: prompts of up to 256 rows go layer by layer, and no product leaves its sum to a norm."""
    from tgis_amd import native
    from tgis_amd.models.custom_modeling import flash_llama_modeling
    from tgis_amd.utils import layers

    lm, cfg = model(torch.bfloat16)
    served, run = [], native.llama_prompt
    monkeypatch.setattr(native, "llama_prompt", lambda got, x, *a, **k: served.append(x.shape[0]) or run(got, x, *a, **k))
    prompts = ([47], [70], [200, 56], [257])
    want = [steps(lm, cfg.vocab_size, lens)[0] for lens in prompts]
    assert {47, 70, 256, 257} == set(served)
    del served[:]
    monkeypatch.setattr(flash_llama_modeling, "DEFER_REDUCE", False)
    monkeypatch.setattr(layers, "DEFER_REDUCE", False)
    for name in ("dense_tall_partial", "dense_gemm_partial"):
        monkeypatch.setattr(native, name, lambda *a, **k: pytest.fail("left its sum"))
    got = [steps(lm, cfg.vocab_size, lens)[0] for lens in prompts]
    assert set(served) == {257}
    # every product is rounded to the model dtype in front of the norm either way: what differs is the order of the fp32 sums, and with it here and
    # there a rounding (a step of 2 ** -8), which three layers carry on: below four steps in the norm of all logits
    for a, b in zip(got, want):
        assert float((a.double() - b.double()).norm() / b.double().norm()) < 4 * 2.0 ** -8


def test_rows_that_the_user_divides(gpu_device, monkeypatch):
    """TGIS_SKINNY_MAX_M: dense linears are the streaming kernel and the library alone, in whole prompts and in the steps of a few rows as well."""
    from tgis_amd import native
    from tgis_amd.models.custom_modeling import flash_llama_modeling
    from tgis_amd.utils import layers

    lm, cfg = model(torch.float16)
    for module in (flash_llama_modeling, layers):
        monkeypatch.setattr(module, "DENSE_TALL", False)
        monkeypatch.setattr(module, "SKINNY_MAX_M", 2)
    for name in ("llama_prompt", "dense_tall", "dense_tall_partial"):
        monkeypatch.setattr(native, name, lambda *a, **k: pytest.fail("served"))
    for lens in ([20], [70], [300]):
        assert bool(torch.isfinite(steps(lm, cfg.vocab_size, lens)[0]).all())
    assert [lm.model.rows_path(rows) for rows in (1, 2, 3, 4)] == [True, True, False, False]

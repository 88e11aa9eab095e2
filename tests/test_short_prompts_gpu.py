"""-m gpu: whole prompts of up to 64 rows of an int4 model, at the widths and rows where the rotary launch is fused into the qkv GEMM and at
those where it is not, against the fp32 oracle."""
import pytest
import torch

from oracle.llama_ref import LlamaRef
from oracle.tiny_models import TinyLlamaConfig, tiny_llama_tensors

pytestmark = pytest.mark.gpu


# kv heads: as many as query heads (qkv three times as wide as the model: fused up to 32 rows), a third of them (never for prompts)
@pytest.mark.parametrize("kv_heads,fused_rows", [(24, 32), (8, 0)])
@pytest.mark.parametrize("act_order", [False, True])
def test_int4_prompts(gpu_device, monkeypatch, kv_heads, fused_rows, act_order):
    from tgis_amd import native
    from tgis_amd.inference_engine.synthetic import InferenceEngine
    from tgis_amd.models.custom_modeling.flash_llama_modeling import LlamaConfig
    from tgis_amd.models.flash_causal_lm import FlashCausalLM
    from tgis_amd.testing import SyntheticTokenizer, make_batch_pb

    tcfg = TinyLlamaConfig(hidden_size=1536, intermediate_size=1024, num_hidden_layers=2, num_attention_heads=24, num_key_value_heads=kv_heads)
    cfg = LlamaConfig(**tcfg.to_dict())
    tensors = tiny_llama_tensors(tcfg, seed=11, quantize="gptq", groupsize=64, act_order=act_order)
    tok = SyntheticTokenizer(cfg.vocab_size)
    eng = InferenceEngine({k: v.clone() for k, v in tensors.items()}, cfg, torch.float16, "gptq", tokenizer=tok, gptq_groupsize=64)
    lm = FlashCausalLM("synthetic", None, "synthetic", torch.float16, "gptq", engine=eng, kv_cache_pages=64)
    ref = LlamaRef(tcfg, tensors, quantize="gptq", groupsize=64)
    row_major = []  # rows of the fused launches that took their operand as rows

    def spied(x, *args, **kw):
        if not isinstance(x, native.FragAct):
            row_major.append(x.shape[0])
        return fused(x, *args, **kw)

    fused = native.gptq_gemm_rope
    monkeypatch.setattr(native, "gptq_gemm_rope", spied)
    for i, lens in enumerate(([1], [16], [20, 12], [33], [47], [1, 30, 33])):
        row_major.clear()
        with lm.context_manager():
            batch, errs = lm.batch_type.from_pb(make_batch_pb(lens, max_new=3, batch_id=i, first_request_id=10 * i, logprobs=True), tok, lm.dtype,
                                                lm.device, lm.word_embeddings, None, True)
            assert not errs
            prompts = [batch.all_input_ids_tensor[j, :n].tolist() for j, n in enumerate(lens)]
            got = [lm.generate_token(batch, first=True)[0]]
            assert row_major == ([sum(lens)] * 2 if sum(lens) <= fused_rows else []), lens
            got.append(lm.generate_token(batch)[0])  # reads the pages that the prompt wrote
        want = ref.generate_greedy(prompts, 2, forced=[[t.token_id for t in step] for step in got])
        for g, w in zip(got, want):
            assert [t.token_id for t in g] == w["token_ids"].tolist(), lens
            # logits of tens in f16 (2 ** -11 of them per rounding), a handful of roundings behind each other
            assert torch.allclose(torch.tensor([t.logprob for t in g]), w["logprobs"], atol=5e-2, rtol=0), lens
        batch.release()


@pytest.mark.parametrize("act_order", [False, True])
def test_int4_prompts_in_fragments(gpu_device, monkeypatch, act_order):
    """Prompts of 1 - 64 rows whose norms write the operands of the fused qkv and of the SiLU * up launch in fragment order, against the fp32 oracle."""
    from tgis_amd import native
    from tgis_amd.inference_engine.synthetic import InferenceEngine
    from tgis_amd.models.custom_modeling.flash_llama_modeling import LlamaConfig
    from tgis_amd.models.flash_causal_lm import FlashCausalLM
    from tgis_amd.testing import SyntheticTokenizer, make_batch_pb

    tcfg = TinyLlamaConfig(hidden_size=2560, intermediate_size=4096, num_hidden_layers=2, num_attention_heads=40, num_key_value_heads=10)
    cfg = LlamaConfig(**tcfg.to_dict())
    tensors = tiny_llama_tensors(tcfg, seed=12, quantize="gptq", groupsize=64, act_order=act_order)
    tok = SyntheticTokenizer(cfg.vocab_size)
    eng = InferenceEngine({k: v.clone() for k, v in tensors.items()}, cfg, torch.float16, "gptq", tokenizer=tok, gptq_groupsize=64)
    lm = FlashCausalLM("synthetic", None, "synthetic", torch.float16, "gptq", engine=eng, kv_cache_pages=64)
    ref = LlamaRef(tcfg, tensors, quantize="gptq", groupsize=64)
    calls = []  # rows of the launches behind the norms that took fragments

    def spied(x, *args, _launch, **kw):
        if isinstance(x, native.FragAct) and kw.get("act", 2) == 2:
            calls.append(x.shape[0])
        return _launch(x, *args, **kw)

    for name in ("gptq_gemm_rope", "gptq_gemm"):
        launch = getattr(native, name)
        monkeypatch.setattr(native, name, lambda x, *args, _launch=launch, **kw: spied(x, *args, _launch=_launch, **kw))
    for i, lens in enumerate(([1], [16], [17], [33], [20, 28], [49], [1, 30, 33])):
        calls.clear()
        with lm.context_manager():
            batch, errs = lm.batch_type.from_pb(make_batch_pb(lens, max_new=3, batch_id=i, first_request_id=10 * i, logprobs=True), tok, lm.dtype,
                                                lm.device, lm.word_embeddings, None, True)
            assert not errs
            prompts = [batch.all_input_ids_tensor[j, :n].tolist() for j, n in enumerate(lens)]
            got = [lm.generate_token(batch, first=True)[0]]
            assert len(calls) >= 2 and set(calls) == {sum(lens)}, (lens, calls)
            got.append(lm.generate_token(batch)[0])  # reads the pages that the prompt wrote
        want = ref.generate_greedy(prompts, 2, forced=[[t.token_id for t in step] for step in got])
        for g, w in zip(got, want):
            assert [t.token_id for t in g] == w["token_ids"].tolist(), lens
            assert torch.allclose(torch.tensor([t.logprob for t in g]), w["logprobs"], atol=5e-2, rtol=0), lens
        batch.release()

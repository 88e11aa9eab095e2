"""-m gpu: a prefill of which only the last tokens' logits are wanted goes through its last layer with those rows alone; against the same
prefill whole: the logits, and the pages and states that it leaves."""
import pytest
import torch

pytestmark = pytest.mark.gpu

LENS = [37, 1, 70, 33]


def llama(quantize, act_order, layers=2):
    from oracle.tiny_models import TinyLlamaConfig, tiny_llama_tensors
    from tgis_amd.models.custom_modeling.flash_llama_modeling import LlamaConfig

    cfg = TinyLlamaConfig(num_hidden_layers=layers)
    return LlamaConfig(**cfg.to_dict()), tiny_llama_tensors(cfg, seed=5, quantize=quantize, groupsize=64, act_order=act_order), torch.float16, quantize


def bigcode():
    from oracle.tiny_models import TinyBigCodeConfig, tiny_bigcode_tensors

    cfg = TinyBigCodeConfig()
    cfg.quantize = None
    return cfg, tiny_bigcode_tensors(cfg, seed=5), torch.float16, None


def lenisun(last, dtype):
    from oracle import lenisun_tiny as tiny
    from tgis_amd.models.custom_modeling.flash_lenisun_modeling import LenisunConfig

    layers = [tiny.attention_layer(v_mix=True, mlp=tiny.dense_mlp()), tiny.wkv_layer(mlp=tiny.dense_mlp())]
    layers += [tiny.attention_layer(v_mix=True, mlp=tiny.moe_mlp())] if last == "attention" else [tiny.wkv_layer(mlp=None)]
    cfg = tiny.make_config(layers)
    return LenisunConfig(**cfg), {k: v.to(dtype) for k, v in tiny.make_tensors(cfg, seed=5).items()}, dtype, None


CASES = {
    "llama": lambda: llama(None, False), "llama_one_layer": lambda: llama(None, False, layers=1), "llama_int4": lambda: llama("gptq", False),
    "llama_act_order": lambda: llama("gptq", True), "bigcode": bigcode, "lenisun_f32": lambda: lenisun("attention", torch.float32),
    "lenisun_wkv_f32": lambda: lenisun("wkv", torch.float32), "lenisun_bf16": lambda: lenisun("attention", torch.bfloat16),
}
# float32 models: sums in another order.  Two-byte ones: roundings of one layer that fall the other way (2 ** -11, 2 ** -8 each), a handful of them
TOL = {torch.float32: 2e-5, torch.float16: 8 * 2.0 ** -11, torch.bfloat16: 8 * 2.0 ** -8}


@pytest.mark.parametrize("case", sorted(CASES))
def test_prefill_of_the_ends(gpu_device, monkeypatch, case):
    from tgis_amd.inference_engine.synthetic import InferenceEngine
    from tgis_amd.models.custom_modeling import flash_llama_modeling
    from tgis_amd.models.flash_causal_lm import FlashCausalLM
    from tgis_amd.testing import SyntheticTokenizer

    cfg, tensors, dtype, quantize = CASES[case]()
    eng = InferenceEngine(tensors, cfg, dtype, quantize, tokenizer=SyntheticTokenizer(cfg.vocab_size), gptq_groupsize=64)
    lm = FlashCausalLM("synthetic", None, "synthetic", dtype, quantize, engine=eng, kv_cache_pages=32, state_slots=8)
    monkeypatch.setattr(flash_llama_modeling, "ENDS_FROM_ROWS", 64)
    pages = [lm.kv_cache.alloc(n // 32 + 1) for n in LENS]
    slots = lm.state_cache.alloc(len(LENS)) if lm.state_cache is not None else None
    ids = torch.randint(3, cfg.vocab_size, (sum(LENS),), generator=torch.Generator().manual_seed(3)).to(gpu_device)
    last = (torch.tensor(LENS).cumsum(0) - 1).to(gpu_device)

    def prefill(ends_only):
        with lm.context_manager():
            logits = lm.ragged_forward(ids, pages, [0] * len(LENS), LENS, slots, None, last, ends_only=ends_only)
            left = []
            for i in range(lm.num_layers):
                for pool in (lm.kv_cache.k_pool(i), lm.kv_cache.v_pool(i)):
                    left.append(None if pool is None else pool.clone())
                if lm.state_cache is not None and lm.state_cache.state[i] is not None:
                    left.append(lm.state_cache.state[i].clone())
        return logits, left

    want, want_left = prefill(False)
    got, left = prefill(True)
    assert got.shape == want.shape == (len(LENS), cfg.vocab_size)
    size = want.double().square().mean(-1, keepdim=True).sqrt()
    assert ((got - want).abs() <= TOL[dtype] * size).all(), float(((got - want).abs() / size).max())
    assert all((a is None and b is None) or torch.equal(a, b) for a, b in zip(left, want_left))


@pytest.mark.parametrize("lens,recurrent,cut", [([128], False, True), ([127], False, False), ([128], True, True), ([16] * 8, True, False), ([16] * 8, False, True),
                                                ([24] * 8, True, True), ([2] * 64, False, True), ([1] * 192, True, False), ([32] * 4, True, True)])
def test_rows_that_are_cut(gpu_device, lens, recurrent, cut):
    from tgis_amd.models.custom_modeling.flash_llama_modeling import KVArgs

    kv = KVArgs(cache=None, block_tables=None, ctx_lens=None, slots=None, max_q_len=max(lens), max_ctx=max(lens), num_splits=1,
                ends=torch.tensor(lens, device=gpu_device).cumsum(0) - 1)
    assert kv.cuts_to_ends(sum(lens), recurrent) == cut
    kv.residual_trace = []
    assert not kv.cuts_to_ends(sum(lens), recurrent)

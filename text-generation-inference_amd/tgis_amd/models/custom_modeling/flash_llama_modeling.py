"""Llama (MHA / GQA) forward for prefill and batched decode on the gfx950 kernels of libtgis_hip.so.

Mirrors custom_modeling/flash_llama_modeling.py of the reference — `LlamaConfig` (:37-99), `LlamaRMSNorm`
(:102-152), `FlashLlamaAttention` (:183-297), `LlamaMLP` (:300-335), `FlashLlamaLayer` (:338-395),
`FlashLlamaModel` (:398-497), `FlashLlamaForCausalLM` (:500-540) — with these deliberate differences:
  * the KV cache is the paged pool of utils/kv_cache.py instead of a per-batch contiguous tensor, so
    `forward` takes a `KVArgs` (block tables, context lengths, slots) where the reference takes
    `past_key_values` / `pre_allocate_past_size`;
  * RoPE, the KV write and the q/k/v split are one kernel; SiLU*mul is fused into down_proj's operand
    staging; every residual-add is fused into the following RMSNorm (as in the reference);
  * logits are produced in fp32.
Tensor-parallel sharding follows the reference exactly (heads split across ranks, qkv / gate_up
column-parallel, o_proj / down_proj row-parallel + all-reduce, vocab-parallel embedding and head)."""
import os
from dataclasses import dataclass, replace
from typing import List, Optional

import torch

from tgis_amd import native
from tgis_amd.utils.layers import (
    DEFER_REDUCE,
    DENSE_TALL,
    SKINNY_MAX_M,
    Ex4bitLinearV2,
    FastLinear,
    PositionRotaryEmbedding,
    TensorParallelColumnLinear,
    TensorParallelEmbedding,
    TensorParallelHead,
    TensorParallelRowLinear,
    workspace,
)


class LlamaConfig:
    """The subset of the HF Llama config the forward needs (reference :37-99; eps default 1e-6 there)."""

    def __init__(self, vocab_size=32000, hidden_size=4096, intermediate_size=11008, num_hidden_layers=32,
                 num_attention_heads=32, num_key_value_heads=None, hidden_act="silu", max_position_embeddings=2048,
                 rms_norm_eps=1e-6, rope_scaling=None, rope_theta=10000.0, attention_bias=False, mlp_bias=False,
                 pad_token_id=None, bos_token_id=1, eos_token_id=2, tie_word_embeddings=False, quantize=None,
                 **kwargs):
        self.vocab_size = vocab_size
        self.hidden_size = hidden_size
        self.intermediate_size = intermediate_size
        self.num_hidden_layers = num_hidden_layers
        self.num_attention_heads = num_attention_heads
        self.num_key_value_heads = num_key_value_heads if num_key_value_heads is not None else num_attention_heads
        self.hidden_act = hidden_act
        self.max_position_embeddings = max_position_embeddings
        self.rms_norm_eps = rms_norm_eps
        self.rope_scaling = rope_scaling
        self.rope_theta = rope_theta
        self.attention_bias = attention_bias
        self.mlp_bias = mlp_bias
        self.pad_token_id = pad_token_id
        self.bos_token_id = bos_token_id
        self.eos_token_id = eos_token_id
        self.tie_word_embeddings = tie_word_embeddings
        self.quantize = quantize
        self.model_type = "llama"
        for k, v in kwargs.items():
            setattr(self, k, v)

    def to_dict(self):
        return dict(vars(self))


# rows of a prefill from which its last layer is cut to the last tokens: below, the layer waits for its weights either way, and the cut is three
# launches more.  One prompt, us, whole / cut: 8 hybrid layers 70 rows 1134 / 1152, 140 1305 / 1283, 4 x 1024 5130 / 4750; 8 layers of a 15B code
# model 140 4391 / 4096, 2 x 4093 42.8 / 38.4 ms; 22 layers of a 1.1B model 130 2151 / 2113; 32 int4 layers 130 5416 / 5352, 16 x 1008 198 / 194 ms
ENDS_FROM_ROWS = 128


@dataclass
class KVArgs:
    """Where this forward's keys/values live in the paged cache."""
    cache: "object"                    # utils.kv_cache.PagedKVCache
    block_tables: torch.Tensor         # [B, max_pages] int32 (device)
    ctx_lens: Optional[torch.Tensor]   # [B] int32, tokens per sequence incl. this forward's (prefill); decode: filled in
    slots: Optional[torch.Tensor]      # [T] int32 physical slot per token (prefill); decode: filled in
    max_q_len: int                     # longest q run in this forward (1 for decode)
    max_ctx: int                       # upper bound of ctx_lens (launch shaping only)
    num_splits: int = 1                # attention key splits (decode)
    fresh_prefill: bool = False        # every sequence starts at cache position 0: page-wise cache writes
    # models with recurrent layers (utils/state_cache.py): the slot of every sequence of the step
    state: "object" = None             # utils.state_cache.RecurrentStateCache
    state_slots: Optional[torch.Tensor] = None  # [B] int32 (device)
    cu_seqlens_q: Optional[torch.Tensor] = None  # [B + 1] int32, for mixers that get the step description from here
    turns: Optional[dict] = None       # rotation tables of this step's tokens, made by the first layer that asks (utils/mixers.py)
    residual_trace: Optional[list] = None  # debugging: models that support it append the residual stream after every layer
    # [B] int64: the row of every sequence's last token, where no other row's logits are wanted (a whole prompt's prefill)
    ends: Optional[torch.Tensor] = None

    def cuts_to_ends(self, rows: int, recurrent: bool = False) -> bool:
        """Whether the last layer of a step of `rows` rows goes on with the sequences' last tokens alone behind its keys and values (whose
        outputs nothing else reads).  recurrent: of a model with linear-recurrence layers, whose short steps wait for the host: with sequences of
        fewer than 32 rows the cut's launches cost there what it saves up to half as many rows again (whole / cut, 8 hybrid layers: 8 x 16 rows 1159 / 1168, 32
        x 4 1328 / 1348, 64 x 2 1580 / 1600, 48 x 3 1479 / 1494, 16 x 12 1254 / 1251, 48 x 4 1523 / 1519, 1 x 160 1181 / 1172)."""
        if self.ends is None or self.residual_trace is not None:
            return False
        B = self.ends.shape[0]
        least = ENDS_FROM_ROWS * 3 // 2 if recurrent and rows < 32 * B else ENDS_FROM_ROWS
        return rows >= least and rows >= 2 * B

    def at_ends(self, heads: int, kv_heads: int) -> "KVArgs":
        """The step that the last tokens make: one token per sequence, all others cached."""
        B = self.ends.shape[0]
        return replace(self, max_q_len=1, fresh_prefill=False, ends=None, num_splits=native.attn_num_splits(B, kv_heads, heads, 1, self.max_ctx),
                       cu_seqlens_q=torch.arange(B + 1, dtype=torch.int32, device=self.ends.device))


# (The persistent decode tail, the rope-in-attention launch and the norm-as-a-GEMM-phase launches were all
# measured slower than the launches they replace: experiments/README.md is their ledger.)


def frag_rows(linear, rows: int, act: int = 0, gathers: bool = False) -> bool:
    """Up to 64 rows in front of an int4 linear that takes its operand in fragment order (native.FragAct); gathers: the
    producer can write an act-order matrix's column order."""
    return rows <= 64 and hasattr(linear, "wants_fragments") and linear.wants_fragments(rows, act, gathers)


class LlamaRMSNorm:
    def __init__(self, prefix, weights, eps=1e-6):
        self.weight = weights.get_tensor(f"{prefix}.weight").contiguous()
        self.variance_epsilon = eps

    def forward(self, hidden_states, residual=None, frag: bool = False, perm=None):
        # returns (normed, res) like the reference; res is hidden_states itself when residual is None
        # frag: the normed activation leaves in fragment order (native.FragAct) for the int4 GEMM behind it; perm: its columns
        # leave in that (act-order) GEMM's order
        if perm is not None:
            return native.rmsnorm_residual(hidden_states, residual, self.weight, self.variance_epsilon, frag=frag, perm=perm)
        return native.rmsnorm_residual(hidden_states, residual, self.weight, self.variance_epsilon, frag=frag)

    __call__ = forward


def rope_settings(config):
    """(theta, linear scaling factor) from either config generation: `rope_theta` + `rope_scaling{type, factor}` (the
    reference's transformers 4.40, flash_llama_modeling.py:181-191) or `rope_parameters{rope_theta, rope_type, factor}`
    (transformers >= 5, which dropped the flat attributes)."""
    params = getattr(config, "rope_parameters", None) or {}
    theta = getattr(config, "rope_theta", None)
    if theta is None:
        theta = params.get("rope_theta", 10000.0)
    rs = getattr(config, "rope_scaling", None) or {}
    kind = rs.get("type") or rs.get("rope_type") or params.get("rope_type") or "default"
    if kind in ("default", None):
        return float(theta), 1.0
    if kind == "linear":
        return float(theta), float(rs.get("factor", params.get("factor", 1.0)))
    raise ValueError(f"rope_scaling of type {kind} is not supported")


class FlashLlamaAttention:
    def __init__(self, prefix: str, config, weights):
        self.num_heads = config.num_attention_heads
        self.hidden_size = config.hidden_size
        self.head_size = self.hidden_size // self.num_heads
        theta, scaling = rope_settings(config)
        self.rotary_emb = PositionRotaryEmbedding.static(dim=self.head_size, base=theta,
                                                         device=weights.device, scaling_factor=scaling)
        self.softmax_scale = self.head_size ** -0.5
        tp = weights.process_group.size()
        if self.num_heads % tp != 0:
            raise ValueError(f"`num_heads` must be divisible by `num_shards` (got `num_heads`: {self.num_heads} "
                             f"and `num_shards`: {tp}")
        assert config.num_key_value_heads % tp == 0, "num_key_value_heads must be divisible by the shard count"
        self.num_heads = self.num_heads // tp
        self.num_key_value_heads = config.num_key_value_heads // tp
        self.query_key_value = TensorParallelColumnLinear.load_multi(
            config, prefixes=[f"{prefix}.q_proj", f"{prefix}.k_proj", f"{prefix}.v_proj"], dim=0, weights=weights,
            bias=config.attention_bias)
        self.o_proj = TensorParallelRowLinear.load(config, prefix=f"{prefix}.o_proj", weights=weights,
                                                   bias=config.attention_bias)
        # steps of up to 64 rows (where native.rope_gemm_ok) rotate q / k and write the cache in the GEMM epilogue, prompts where that pays
        if hasattr(self.query_key_value.linear, "rope_heads"):
            self.query_key_value.linear.rope_heads = (self.num_heads, self.num_key_value_heads, self.head_size)
        self.out_places: Optional[torch.Tensor] = None  # an act-order o_proj's order of the attention's output columns (post_init)

    def project_qkv(self, hidden_states, cos, sin, position_ids, cu_seqlens_q, layer_id: int, kv: KVArgs, gathered: bool = False,
                    attended: bool = False):
        """qkv GEMM, rotation of q and k in place, k and v scattered to their page slots (reference :251-268,282): the qkv rows, and what `attend`
        is to rotate q by (None: it is rotated).
        gathered: hidden_states' columns are in the order of an act-order qkv weight.  attended: all rows' q go to `attend`, which may rotate it."""
        H, Hkv, D = self.num_heads, self.num_key_value_heads, self.head_size
        k_pool, v_pool = kv.cache.k_pool(layer_id), kv.cache.v_pool(layer_id)
        lin = self.query_key_value.linear
        rope_w = getattr(lin, "rope_handle", None)
        decode = kv.max_q_len == 1 and not kv.fresh_prefill
        if isinstance(hidden_states, native.FragAct) or (
                rope_w is not None and kv.slots is not None
                and (gathered or getattr(lin, "perm", None) is None) and hidden_states.shape[0] <= 64 and cos.shape[1] * 2 == D
                and native.rope_gemm_ok(hidden_states.shape[0], rope_w, D)
                and (decode or native.rope_gemm_pays_for_prompts(hidden_states.shape[0], rope_w))):
            # one launch: GEMM + rotary embedding + cache write (native.gptq_gemm_rope / native.dense_gemm_rope)
            fused = native.gptq_gemm_rope if isinstance(rope_w, native.GptqWeight) else native.dense_gemm_rope
            return fused(hidden_states, rope_w, lin.bias, cos, sin, position_ids, kv.slots, k_pool, v_pool, H, Hkv, D), None
        # [T, (H + 2 Hkv) D]; at decode sizes the split-K sum of the GPTQ GEMM is finished inside the rope kernel; whole prompts on the dense
        # prefill kernel take the finished sum, and with it the page-wise cache writes
        whole = kv.fresh_prefill and isinstance(lin, FastLinear) and lin.tall(hidden_states) >= 0
        qkv = self.query_key_value(hidden_states, partial=not whole, **({"gathered": True} if gathered else {}))
        if kv.fresh_prefill and not isinstance(qkv, native.Partial):
            pages = (qkv, cos, sin, position_ids, cu_seqlens_q, kv.block_tables, k_pool, v_pool, kv.max_q_len, H, Hkv, D, D)
            if attended and qkv.is_cuda and kv.num_splits == 1 and cos.shape[1] * 2 == D and native.attn_rotates_q(H, Hkv, D, kv.max_q_len):
                return native.rope_kv_write_prefill(*pages, rotate_q=False), (cos, sin, position_ids)
            return native.rope_kv_write_prefill(*pages), None
        return native.rope_kv_write(qkv, cos, sin, position_ids, kv.slots, k_pool, v_pool, H, Hkv, D, D), None

    def attend(self, qkv, cu_seqlens_q, layer_id: int, kv: KVArgs, rope=None, frag: bool = False):
        """Attention of q (rotated, or to be rotated by `rope`) over the layer's cache pages (reference :271-295): [T, H D], a native.FragAct where the
        o_proj GEMM reads that, or with `frag`: decode steps, and prompts of up to 64 rows, on the launches of csrc/dense_rows.hip."""
        H, Hkv, D = self.num_heads, self.num_key_value_heads, self.head_size
        k_pool, v_pool = kv.cache.k_pool(layer_id), kv.cache.v_pool(layer_id)
        T = qkv.shape[0]
        B = kv.block_tables.shape[0]
        # decode: the o_proj GEMM reads its operand in fragment order, an act-order one with its columns in its own
        places = {} if rope is None else {"rope": rope}
        decode = kv.max_q_len == 1 and not kv.fresh_prefill
        if decode and frag_rows(self.o_proj.linear, T, gathers=self.out_places is not None):
            if self.out_places is not None:
                places = {"out_cols": self.out_places}
            attn_output = native.FragAct.empty(T, H * D, qkv.device)
        elif frag:
            attn_output = native.FragAct.empty(T, H * D, qkv.device, qkv.dtype)
        else:
            attn_output = torch.empty((T, H * D), dtype=qkv.dtype, device=qkv.device)
        ws = None
        if kv.num_splits > 1:
            from tgis_amd.utils.layers import workspace
            ws = workspace(qkv.device)
            ws.ensure(native.attn_workspace_bytes(T, H, Hkv, D, kv.num_splits))
        native.attn_paged(qkv, qkv.stride(0), k_pool, v_pool, kv.block_tables, kv.ctx_lens, cu_seqlens_q,
                          attn_output, B, H, Hkv, D, kv.max_q_len, kv.max_ctx, self.softmax_scale, kv.num_splits, ws, **places)
        return attn_output

    def forward(self, hidden_states, cos, sin, position_ids, cu_seqlens_q, layer_id: int, kv: KVArgs, gathered: bool = False):
        qkv, rope = self.project_qkv(hidden_states, cos, sin, position_ids, cu_seqlens_q, layer_id, kv, gathered, attended=True)
        attn_output = self.attend(qkv, cu_seqlens_q, layer_id, kv, rope)
        # may be a native.Partial: the following fused add+RMSNorm finishes the split-K sum
        return self.o_proj(attn_output, partial=True)

    __call__ = forward


class LlamaMLP:
    def __init__(self, prefix, config, weights):
        if config.hidden_act != "silu":
            raise NotImplementedError(f"hidden_act {config.hidden_act}: only silu is wired into the fused kernel")
        self.gate_up_proj = TensorParallelColumnLinear.load_multi(
            config, prefixes=[f"{prefix}.gate_proj", f"{prefix}.up_proj"], weights=weights, dim=0,
            bias=config.mlp_bias)
        self.down_proj = TensorParallelRowLinear.load(config, prefix=f"{prefix}.down_proj", weights=weights,
                                                      bias=config.mlp_bias)
        self.intermediate_size = config.intermediate_size // weights.process_group.size()
        # GPTQ: SiLU(gate)*up runs in the gate_up GEMM epilogue (columns interleaved at prepare time);
        # dense: it runs while down_proj stages its operand.  Reference: eager ops at :332-335.
        self.fused_epilogue = hasattr(self.gate_up_proj.linear, "gate_up") and self.intermediate_size % 16 == 0
        if self.fused_epilogue:
            self.gate_up_proj.linear.gate_up = True

    def post_init(self):
        """An act-order down projection wants its operand's columns in its own order: the gate and up columns that produce
        them are re-ordered once, and nothing is gathered per step."""
        down, gate_up = self.down_proj.linear, self.gate_up_proj.linear
        if not self.fused_epilogue or not hasattr(down, "order_columns") or not hasattr(gate_up, "order_columns"):
            return
        if gate_up.q_handle is None and down.perm is not None and down.height == self.intermediate_size:
            order = down.perm
            if bool((order >= 0).all()):
                gate_up.order_columns(torch.cat([order, order + self.intermediate_size]))
                down.take_ordered_input()

    def forward(self, hidden_states, gathered: bool = False):
        kw = {"gathered": True} if gathered else {}
        if self.fused_epilogue:
            if isinstance(hidden_states, native.FragAct):  # SiLU * up leaves in the layout down_proj reads
                rows = hidden_states.shape[0]
                act = self.gate_up_proj(hidden_states, out_frag=self.down_proj.linear.wants_fragments(rows))
                return self.down_proj(act, partial=True)
            act = self.gate_up_proj(hidden_states, **kw)  # [T, I], already silu(gate) * up
            return self.down_proj(act, partial=True)
        gate_up_states = self.gate_up_proj(hidden_states, **kw)  # [T, 2, I]
        return self.down_proj(gate_up_states, act=1, partial=True)

    __call__ = forward


class FlashLlamaLayer:
    def __init__(self, layer_id, config, weights):
        prefix = f"model.layers.{layer_id}"
        self.layer_id = layer_id
        self.self_attn = FlashLlamaAttention(prefix=f"{prefix}.self_attn", config=config, weights=weights)
        self.mlp = LlamaMLP(prefix=f"{prefix}.mlp", config=config, weights=weights)
        self.input_layernorm = LlamaRMSNorm(prefix=f"{prefix}.input_layernorm", weights=weights,
                                            eps=config.rms_norm_eps)
        self.post_attention_layernorm = LlamaRMSNorm(prefix=f"{prefix}.post_attention_layernorm", weights=weights,
                                                     eps=config.rms_norm_eps)
        self.int4 = hasattr(self.self_attn.query_key_value.linear, "wants_fragments")

    def hands_fragments(self, rows: int, kv: KVArgs) -> bool:
        """Whether the norms may hand the int4 GEMMs of up to 64 rows their operands in fragment order (native.FragAct): decode steps, and prompts but
        for those whose row-major fused qkv launch pays.  us, rows / fragments: a 7B model's prompts of 40 rows 3000 / 2660, two of 32 3223 / 2866, 60 in
        act order 3130 / 2822, four 70B layers' of 12, 48 868 / 801, 1069 / 1001; but a 7B model's of 16, 30 rows, the host's time either way, 2647 / 2668,
        2652 / 2692."""
        if rows > 64 or not self.int4:
            return False
        return ((kv.max_q_len == 1 and not kv.fresh_prefill)
                or not native.rope_gemm_pays_for_prompts(rows, self.self_attn.query_key_value.linear.rope_handle))

    def forward(self, hidden_states, residual, cos, sin, position_ids, cu_seqlens_q, kv: KVArgs):
        rows = hidden_states.shape[0]
        att = self.self_attn
        # the qkv + rotary launch takes its operand in fragment order when it serves the rows, the MLP when the SiLU * up epilogue does; the norms
        # gather for act-order weights
        qkv_perm = getattr(att.query_key_value.linear, "perm", None)
        qkv_frag = (self.hands_fragments(rows, kv) and kv.slots is not None and cos.shape[1] * 2 == att.head_size
                    and frag_rows(att.query_key_value.linear, rows, act=3, gathers=True))
        normed_hidden_states, res = self.input_layernorm(hidden_states, residual, frag=qkv_frag, perm=qkv_perm)
        attn_output = att(normed_hidden_states, cos, sin, position_ids, cu_seqlens_q, self.layer_id, kv, qkv_perm is not None)
        return self.feed_forward(attn_output, res, kv)

    def feed_forward(self, attn_output, res, kv: KVArgs):
        rows = attn_output.shape[0]
        mlp_perm = getattr(self.mlp.gate_up_proj.linear, "perm", None)
        mlp_frag = (self.hands_fragments(rows, kv) and self.mlp.fused_epilogue
                    and frag_rows(self.mlp.gate_up_proj.linear, rows, act=2, gathers=True))
        normed_attn_res_output, attn_res = self.post_attention_layernorm(attn_output, res, frag=mlp_frag, perm=mlp_perm)
        mlp_output = self.mlp(normed_attn_res_output, mlp_perm is not None)
        return mlp_output, attn_res

    def forward_ends(self, hidden_states, residual, cos, sin, position_ids, cu_seqlens_q, kv: KVArgs):
        """`forward` of which only the rows `kv.ends` are wanted: keys and values of all tokens, the rest of the layer for those rows."""
        att = self.self_attn
        qkv_perm = getattr(att.query_key_value.linear, "perm", None)
        normed_hidden_states, res = self.input_layernorm(hidden_states, residual, perm=qkv_perm)
        qkv, _ = att.project_qkv(normed_hidden_states, cos, sin, position_ids, cu_seqlens_q, self.layer_id, kv, qkv_perm is not None)
        step = kv.at_ends(att.num_heads, att.num_key_value_heads)
        attn_output = att.o_proj(att.attend(qkv.index_select(0, kv.ends), step.cu_seqlens_q, self.layer_id, step), partial=True)
        return self.feed_forward(attn_output, res.index_select(0, kv.ends), step)

    __call__ = forward


class FlashLlamaModel:
    def __init__(self, config, weights):
        self.config = config
        process_group = weights.process_group
        self.tp_rank = process_group.rank()
        self.tp_world_size = process_group.size()
        self.embed_tokens = TensorParallelEmbedding(prefix="model.embed_tokens", weights=weights)
        self.layers = [FlashLlamaLayer(i, config, weights) for i in range(config.num_hidden_layers)]
        self.norm = LlamaRMSNorm(prefix="model.norm", weights=weights, eps=config.rms_norm_eps)
        self.head_size = self.layers[0].self_attn.head_size
        self.num_heads = self.layers[0].self_attn.num_heads
        self.num_key_value_heads = config.num_key_value_heads // process_group.size()
        self.max_positions = 0
        self._rows16 = {}  # rows -> serves_rows16
        self.int4_norms, self._int4_rows = None, {}  # prepare_int4_rows; rows -> serves_int4_rows

    def rope_tables(self, dtype, device, max_s: int):
        # Sized once for the model's whole position range, so the tables normally never move.  A longer request
        # still works: PositionRotaryEmbedding keeps the replaced tables allocated, because decode graphs captured
        # earlier hold their raw pointers (and only ever index positions inside the table they captured).
        if max_s > self.max_positions:
            declared = min(int(getattr(self.config, "max_position_embeddings", 0) or 0), 1 << 17)
            self.max_positions = max(max_s, 2 * self.max_positions, declared, 2048)
        return self.layers[0].self_attn.rotary_emb.tables(dtype, device, self.max_positions)

    def forward_rows(self, input_ids, position_ids, cu_seqlens_q, max_s, kv: KVArgs):
        """A decode step of a few rows on the launches of csrc/dense_rows.hip: the residual stream (fp32, [rows, hidden]) in front of the final
        norm.  Five launches a layer; the values are those of `forward` but for the order of the sums."""
        h = native.embedding_scaled_f32(input_ids, self.embed_tokens.weight, 1.0)
        cos, sin = self.rope_tables(self.embed_tokens.weight.dtype, h.device, max_s)
        for layer in self.layers:
            att, mlp = layer.self_attn, layer.mlp
            qkv = native.dense_rows_rope(h, layer.input_layernorm.weight, layer.input_layernorm.variance_epsilon,
                                         att.query_key_value.linear.rope_handle, att.query_key_value.linear.bias, cos, sin, position_ids, kv.slots,
                                         kv.cache.k_pool(layer.layer_id), kv.cache.v_pool(layer.layer_id), att.num_heads, att.num_key_value_heads,
                                         att.head_size)
            native.dense_rows_residual(att.attend(qkv, cu_seqlens_q, layer.layer_id, kv), att.o_proj.linear.prepared, h)
            act = native.dense_rows_silu(h, layer.post_attention_layernorm.weight, layer.post_attention_layernorm.variance_epsilon,
                                         mlp.gate_up_proj.linear.prepared)
            native.dense_rows_residual(act, mlp.down_proj.linear.prepared, h)
        return h

    def forward_rows16(self, input_ids, position_ids, cu_seqlens_q, max_s, kv: KVArgs):
        """The same for more rows, in bf16, on the launches there that take the matrix instruction: a native.RowsStream."""
        h = native.RowsStream.embed(input_ids, self.embed_tokens.weight, self.layers[0].input_layernorm.weight)
        cos, sin = self.rope_tables(self.embed_tokens.weight.dtype, h.device, max_s)
        down = self._rows16_layers(h, cos, sin, position_ids, cu_seqlens_q, kv)
        native.dense_rows16_residual(*down, h, self.norm.weight)
        return h

    def _rows16_layers(self, h, cos, sin, position_ids, cu_seqlens_q, kv: KVArgs):
        """All layers but for the last one's down projection, whose operands it returns."""
        for i, layer in enumerate(self.layers):
            att, mlp = layer.self_attn, layer.mlp
            if i > 0:
                native.dense_rows16_residual(*down, h, layer.input_layernorm.weight)
            qkv = native.dense_rows16_rope(h, layer.input_layernorm.variance_epsilon, att.query_key_value.linear.rope_handle,
                                           att.query_key_value.linear.bias, cos, sin, position_ids, kv.slots, kv.cache.k_pool(layer.layer_id),
                                           kv.cache.v_pool(layer.layer_id), att.num_heads, att.num_key_value_heads, att.head_size)
            native.dense_rows16_residual(att.attend(qkv, cu_seqlens_q, layer.layer_id, kv, frag=True), att.o_proj.linear.prepared, h,
                                         layer.post_attention_layernorm.weight)
            down = (native.dense_rows16_silu(h, layer.post_attention_layernorm.variance_epsilon, mlp.gate_up_proj.linear.prepared),
                    mlp.down_proj.linear.prepared)
        return down

    def forward_int4_rows(self, input_ids, position_ids, cu_seqlens_q, max_s, kv: KVArgs):
        """A decode step of up to 32 rows of an int4 model on the launches of csrc/gptq_rows.hip: the normed hidden states.  Five launches a layer, or one more for sums that are split; the values are
        those of `forward` but for the order of the sums and where the norm's 1 / rms is multiplied in."""
        qkv_norms, mlp_norms = self.int4_norms
        table = self.embed_tokens.weight
        h = native.Int4RowsStream.embed(input_ids, table, qkv_norms[0])
        cos, sin = self.rope_tables(table.dtype, h.device, max_s)

        def add(x, lin, h, norm):
            if native.gptq_rows_ok(h.M, lin.ordered, False):
                native.gptq_rows_residual(x, lin.ordered, h, norm)
            else:
                native.gptq_rows_sum(native.gptq_gemm_partial(x, lin.ordered), h, norm)

        for i, layer in enumerate(self.layers):
            att, mlp = layer.self_attn, layer.mlp
            if i > 0:
                add(act, down, h, qkv_norms[i])
            qkv = native.gptq_rows_rope(h, layer.input_layernorm.variance_epsilon, att.query_key_value.linear.rope_handle, att.query_key_value.linear.bias, cos, sin,
                                        position_ids, kv.slots, kv.cache.k_pool(layer.layer_id), kv.cache.v_pool(layer.layer_id), att.num_heads,
                                        att.num_key_value_heads, att.head_size)
            add(att.attend(qkv, cu_seqlens_q, layer.layer_id, kv), att.o_proj.linear, h, mlp_norms[i])
            act = native.gptq_rows_silu(h, layer.post_attention_layernorm.variance_epsilon, mlp.gate_up_proj.linear.ordered)
            down = mlp.down_proj.linear
        return self.norm(self.layers[-1].mlp.down_proj(act, partial=True), h.h)[0]

    def prepare_int4_rows(self):
        """Once the int4 matrices are prepared: the norms as `forward_int4_rows` takes them, if all layers are int4, of one rank, in f16 and without a bias but that of
        qkv, and the orders of act-order matrices are ones that their operands' producers write."""
        self.int4_norms, self._int4_rows = None, {}
        if self.tp_world_size != 1 or self.embed_tokens.weight.dtype != torch.float16:
            return
        norms = ([], [])
        for layer in self.layers:
            att, mlp = layer.self_attn, layer.mlp
            qkv, o, gate_up, down = lins = (att.query_key_value.linear, att.o_proj.linear, mlp.gate_up_proj.linear, mlp.down_proj.linear)
            if (not all(isinstance(lin, Ex4bitLinearV2) for lin in lins) or qkv.rope_handle is None or not gate_up.gate_up or down.perm is not None
                    or any(lin.bias is not None for lin in lins[1:]) or (o.perm is not None and att.out_places is None)):
                return
            for lin, norm, inputs in ((qkv, layer.input_layernorm, norms[0]), (gate_up, layer.post_attention_layernorm, norms[1])):
                inputs.append((norm.weight, lin.places()))
                if lin.perm is not None and inputs[-1][1] is None:
                    return
        self.int4_norms = tuple(native.Int4NormInput.several(inputs) for inputs in norms)

    def serves_int4_rows(self, rows: int) -> bool:
        """Widths between 4096 and 6144 are 257 - 383 residual units, a second round of the chip that is mostly empty, and one unit at a time in front of a norm.  Whole
        steps, us, the other launches / these (with a form for five double steps a wave, which is gone), at 1, 4, 11, 16 rows: 4608, inner 12288 541 / 546, 548 / 552, 593 / 609,
        616 / 631; 5120, 12288 530 / 558, 540 / 563, 587 / 625, 609 / 645; 5120, 13824 563 / 564, 573 / 572, 622 / 626, 644 / 646, with eight kv heads 527 / 522, 535 / 524, 553 /
        548, 554 / 550.  Served: 6144, 16384 537 / 536, 544 / 539, 558 / 563, 561 / 566; 6144, 12288 484 / 470, 489 / 471, 502 / 500, 505 / 501; 6656, 17920 671 / 620, 681 / 628,
        733 / 687, 763 / 719; 7168, 20480 484 / 441, 487 / 442, 498 / 458, 499 / 460 (4 - 8 layers)."""
        got = self._int4_rows.get(rows)
        if got is None:
            got = rows <= native.GPTQ_ROWS_MAX_M and self.int4_norms is not None and not 4096 < self.config.hidden_size < 6144
            for layer in self.layers if got else ():
                att, mlp = layer.self_attn, layer.mlp
                o = att.o_proj.linear
                got = (got and native.gptq_rows_ok(rows, att.query_key_value.linear.rope_handle, True) and native.gptq_rows_ok(rows, mlp.gate_up_proj.linear.ordered, True)
                       and o.wants_fragments(rows, gathers=att.out_places is not None) and mlp.down_proj.linear.wants_fragments(rows)
                       and mlp.intermediate_size % 64 == 0)
            self._int4_rows[rows] = got
        return got

    def prompt_rows16(self, x, cos, kv: KVArgs) -> bool:
        """Whether a step of x's rows is a prompt's that the launches of `forward_rows16` serve."""
        return (DEFER_REDUCE and native.DENSE_ROWS16_MIN_M <= x.shape[0] <= min(native.DENSE_ROWS16_MAX_M, SKINNY_MAX_M) and kv.num_splits == 1
                and not (kv.max_q_len == 1 and not kv.fresh_prefill) and kv.slots is not None and kv.residual_trace is None
                and cos.shape[1] * 2 == self.head_size and x.is_contiguous() and self.serves_rows16(x.shape[0]))

    def serves_rows16(self, rows: int) -> bool:
        got = self._rows16.get(rows)
        if got is None:
            got = self._rows16[rows] = self.embed_tokens.weight.dtype == torch.bfloat16 and self.serves_rows(rows, native.dense_rows16_ok)
        return got

    def serves_rows(self, rows: int, ok) -> bool:
        """Whether all layers are dense, of one rank, and of shapes that `ok` says are served."""
        plain = lambda lin: isinstance(lin, FastLinear) and lin.streams and lin.bias is None
        if self.tp_world_size != 1 or not ok(rows, self.config.hidden_size, True):
            return False
        for layer in self.layers:
            qkv, o = layer.self_attn.query_key_value.linear, layer.self_attn.o_proj.linear
            gate_up, down = layer.mlp.gate_up_proj.linear, layer.mlp.down_proj.linear
            if not (isinstance(qkv, FastLinear) and qkv.rope_handle is not None and plain(o) and plain(gate_up) and gate_up.gate_up and plain(down)
                    and ok(rows, o.in_features, False) and ok(rows, down.in_features, False)):
                return False
        return True

    def plain_layers(self, count: int, x, cos, kv: KVArgs) -> list:
        """The weights and cache pages of the first `count` layers, as native.llama_prompt takes them, if a step of x's rows is a prompt's and
        each of its products one that the launches there serve; else nothing."""
        rows, hidden = x.shape
        att, mlp = self.layers[0].self_attn, self.layers[0].mlp
        H, Hkv, D, inner = att.num_heads, att.num_key_value_heads, att.head_size, mlp.intermediate_size
        if ((kv.max_q_len == 1 and not kv.fresh_prefill) or kv.num_splits != 1 or kv.slots is None or kv.residual_trace is not None or not rows
                or self.tp_world_size != 1 or cos.shape[1] * 2 != D or not x.is_contiguous()):
            return []
        tall = rows >= native.DENSE_TALL_MIN_M
        shapes = {"qkv": ((H + 2 * Hkv) * D, hidden), "o": (hidden, H * D), "gate_up": (2 * inner, hidden), "down": (hidden, inner)}
        if tall and any(K % 64 or N < native.DENSE_TALL_MIN_N for N, K in shapes.values()):
            return []
        # past the rows whose products may be left in parts, by either kernel, all four are the prefill kernel's
        if tall and not all(native.dense_tall_serves(rows, K, N, 2 if name == "gate_up" else 0) for name, (N, K) in shapes.items()
                            if rows > native.PARTIAL_MAX_M or name == "gate_up"):
            return []
        if rows <= native.PARTIAL_MAX_M and not DEFER_REDUCE:  # (the launches of such steps leave split sums to the norms)
            return []
        if not DENSE_TALL if tall else rows > SKINNY_MAX_M:
            return []
        got = []
        for layer in self.layers[:count]:
            att, mlp = layer.self_attn, layer.mlp
            lin = {"qkv": att.query_key_value.linear, "o": att.o_proj.linear, "gate_up": mlp.gate_up_proj.linear, "down": mlp.down_proj.linear}
            for name, (N, K) in shapes.items():
                w = lin[name]
                if not (isinstance(w, FastLinear) and w.streams and (w.out_features, w.in_features) == (N, K) and w.weight.dtype == x.dtype
                        and w.gate_up == (name == "gate_up") and (w.bias is None or name == "qkv")):
                    return []
            qkv = lin["qkv"]
            if not tall and (qkv.rope_handle is None or not native.rope_gemm_ok(rows, qkv.rope_handle, D)):
                return []
            got.append((layer.input_layernorm.weight, qkv.prepared.image, None if qkv.rope_handle is None else qkv.rope_handle.image, qkv.bias,
                        lin["o"].prepared.image, layer.post_attention_layernorm.weight, lin["gate_up"].prepared.image, lin["down"].prepared.image,
                        kv.cache.k_pool(layer.layer_id), kv.cache.v_pool(layer.layer_id)))
        return got

    def forward(self, input_ids, position_ids, cu_seqlens_q, max_s, inputs_embeds, kv: KVArgs):
        if input_ids is not None and inputs_embeds is not None:
            raise ValueError("You cannot specify both input_ids and inputs_embeds at the same time")
        hidden_states = inputs_embeds if inputs_embeds is not None else self.embed_tokens(input_ids)
        cos, sin = self.rope_tables(hidden_states.dtype, hidden_states.device, max_s)
        residual = None
        whole = len(self.layers) - kv.cuts_to_ends(hidden_states.shape[0])
        plain = self.plain_layers(whole, hidden_states, cos, kv)
        rows16 = whole == len(self.layers) and self.prompt_rows16(hidden_states, cos, kv)
        if plain:
            att = self.layers[0].self_attn
            hidden_states, residual = native.llama_prompt(
                plain, hidden_states, workspace(hidden_states.device), position_ids, kv.slots, cu_seqlens_q, kv.block_tables, kv.ctx_lens, cos, sin,
                att.num_heads, att.num_key_value_heads, att.head_size, self.layers[0].mlp.intermediate_size, kv.max_q_len, kv.max_ctx,
                kv.fresh_prefill, self.layers[0].input_layernorm.variance_epsilon, att.softmax_scale, rows16)
        elif rows16:
            h = native.RowsStream.of_rows(hidden_states, self.layers[0].input_layernorm.weight)
            down = self._rows16_layers(h, cos, sin, position_ids, cu_seqlens_q, kv)
            hidden_states, residual = native.dense_rows16_leave(*down, h)
            plain = self.layers
        for layer in self.layers[len(plain):whole]:
            hidden_states, residual = layer(hidden_states, residual, cos, sin, position_ids, cu_seqlens_q, kv)
        for layer in self.layers[whole:]:
            hidden_states, residual = layer.forward_ends(hidden_states, residual, cos, sin, position_ids, cu_seqlens_q, kv)
        hidden_states, _ = self.norm(hidden_states, residual)
        return hidden_states

    __call__ = forward


class FlashLlamaForCausalLM:
    def __init__(self, config, weights):
        self.config = config
        self.model = FlashLlamaModel(config, weights)
        self.lm_head = TensorParallelHead.load(config, prefix="lm_head", weights=weights)
        self._rows_path, self._rows16_path = {}, {}
        self.gptq_linears: List = []
        for layer in self.model.layers:
            for lin in (layer.self_attn.query_key_value.linear, layer.self_attn.o_proj.linear,
                        layer.mlp.gate_up_proj.linear, layer.mlp.down_proj.linear):
                if hasattr(lin, "post_init"):
                    self.gptq_linears.append(lin)

    def post_init(self):
        """Repack every GPTQ linear for the kernels (the reference does this in serve(), server.py:334-358)."""
        for layer in self.model.layers:
            layer.mlp.post_init()
        for lin in self.gptq_linears:
            if lin.q_handle is None:
                lin.post_init()
        for layer in self.model.layers:
            o_proj = layer.self_attn.o_proj.linear
            if hasattr(o_proj, "places"):
                layer.self_attn.out_places = o_proj.places()
        self.model.prepare_int4_rows()

    def rows_path(self, rows: int) -> bool:
        """Whether a decode step of `rows` rows runs on the launches that norm their operand themselves (FlashLlamaModel.forward_rows)."""
        got = self._rows_path.get(rows)
        if got is None:
            got = self._rows_path[rows] = rows <= min(native.DENSE_ROWS_MAX_M, SKINNY_MAX_M) and self._serves_rows(rows)
        return got

    def rows16_path(self, rows: int) -> bool:
        """The same of the launches for more rows (FlashLlamaModel.forward_rows16), which may split their sums (TGIS_DEFER_REDUCE)."""
        got = self._rows16_path.get(rows)
        if got is None:
            got = self._rows16_path[rows] = (native.DENSE_ROWS16_MIN_M <= rows <= min(native.DENSE_ROWS16_MAX_M, SKINNY_MAX_M)
                                             and self._plain_head() and self.model.serves_rows16(rows))
        return got and DEFER_REDUCE

    def _serves_rows(self, rows: int) -> bool:
        return self._plain_head() and self.model.serves_rows(rows, native.dense_rows_ok)

    def _plain_head(self) -> bool:
        head = self.lm_head.linear
        return isinstance(head, FastLinear) and head.streams and head.bias is None

    def get_input_embeddings(self):
        return self.model.embed_tokens

    @property
    def num_layers(self):
        return len(self.model.layers)

    def forward(self, input_ids, position_ids, cu_seqlens_q, max_s, inputs_embeds=None, kv: KVArgs = None,
                lm_head_indices: Optional[torch.Tensor] = None):
        """position_ids int32 [T]; returns fp32 logits [T or len(lm_head_indices), vocab]."""
        if kv.max_q_len == 1 and not kv.fresh_prefill and inputs_embeds is None and lm_head_indices is None and kv.slots is not None:
            rows, norm, head = input_ids.shape[0], self.model.norm, self.lm_head.linear
            step = (input_ids, position_ids, cu_seqlens_q, max_s, kv)
            if self.rows16_path(rows):
                return native.dense_rows16_head(self.model.forward_rows16(*step), norm.variance_epsilon, head.prepared)
            if self.rows_path(rows):
                return native.dense_rows_head(self.model.forward_rows(*step), norm.weight, norm.variance_epsilon, head.prepared)
            if DEFER_REDUCE and self.model.serves_int4_rows(rows):
                return self.lm_head(self.model.forward_int4_rows(*step))
        hidden_states = self.model(input_ids, position_ids, cu_seqlens_q, max_s, inputs_embeds, kv)
        if lm_head_indices is not None and not kv.cuts_to_ends(position_ids.shape[0]):
            hidden_states = hidden_states.index_select(0, lm_head_indices)
        return self.lm_head(hidden_states)

    __call__ = forward

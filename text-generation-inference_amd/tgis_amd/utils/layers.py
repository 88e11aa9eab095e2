"""Linear / embedding / head building blocks on the HIP kernels, with Megatron-style tensor parallelism.

Mirrors utils/layers.py of the reference: `FastLinear` (:104-111), the `get_linear` quant registry
(:172-203), `TensorParallelHead` (:215-277), `TensorParallelColumnLinear` (:280-297),
`TensorParallelRowLinear` (all-reduce, :300-322), `TensorParallelEmbedding` (:325-357) and
`PositionRotaryEmbedding` (:406-490); `Ex4bitLinearV2` mirrors utils/gptq/exllamav2.py:100-144.
Every forward runs a kernel of libtgis_hip.so or, for prefill-sized M where that is faster, a library GEMM
on the same device; there is no CPU path."""
import copy
import math
from typing import List, Optional

import torch
import torch.distributed
from torch.nn import functional as F

from tgis_amd import native
from tgis_amd.utils.graph_segments import collective

import os

# rows up to which the dense weight-streaming MFMA kernel is used (one pass over the weights per 32 / 64 rows); above,
# hipBLASLt; from 65 rows on the prefill kernel on the same image where it is faster than either (native.dense_tall_bytes).
# GPTQ linears ask the library how far its fused kernels reach (GptqWeight.fused_rows: 64-row streaming passes
# to 256 rows, the tall kernel from 65 / 129 rows to 8192 where it is faster; else dequantise once + hipBLASLt, exllamav2.py:87).
SKINNY_MAX_M = int(os.getenv("TGIS_SKINNY_MAX_M", "256"))
DENSE_TALL = os.getenv("TGIS_SKINNY_MAX_M") is None  # with the variable set, dense linears are the streaming kernel and the library alone
# fuse the split-K reduce of decode-sized GPTQ GEMMs into the consumer kernel (rmsnorm / rope+KV write)
DEFER_REDUCE = os.getenv("TGIS_DEFER_REDUCE", "true").lower() not in ("0", "false")
# steps of up to 64 rows, prompts where that pays (native.rope_gemm_pays_for_prompts): rotary embedding + cache write in the epilogue of the qkv
# GEMM (one launch instead of GEMM + tgis_rope_kv_write, no split-K slabs).  Costs a second image of the qkv weights.
FUSED_ROPE_GEMM = os.getenv("TGIS_FUSED_ROPE_GEMM", "true").lower() not in ("0", "false")
# GELU applied by the dense decode GEMM that produces its operand (TGIS_FUSED_GELU_GEMM=false: a launch of its own)
FUSED_GELU_GEMM = os.getenv("TGIS_FUSED_GELU_GEMM", "true").lower() not in ("0", "false")

_WORKSPACES = {}


def workspace(device) -> native.Workspace:
    key = str(device)
    ws = _WORKSPACES.get(key)
    if ws is None:
        ws = _WORKSPACES[key] = native.Workspace(64 << 20, device)
    return ws


def tall_bytes(x: torch.Tensor, image: native.DenseWeight, act: int = 0) -> int:
    """The scratch of the prefill kernel on this image where it serves the step, and sooner than the weight-streaming kernel or the library GEMM
    would; else -1."""
    return native.dense_tall_bytes(x, image, act) if x.shape[0] >= native.DENSE_TALL_MIN_M and DENSE_TALL else -1


class FastLinear:
    def __init__(self, weight: torch.Tensor, bias: Optional[torch.Tensor]):
        self.weight = weight
        self.bias = bias
        # the weight-streaming MFMA kernel takes two-byte dtypes and K a multiple of 8; anything else (fp32 serving, odd
        # widths) runs the library GEMM at every M
        self.streams = weight.dtype in (torch.float16, torch.bfloat16) and weight.shape[1] % 8 == 0
        self.prepared = native.DenseWeight(weight) if self.streams else None
        self.out_features, self.in_features = weight.shape
        self._gate_up = False
        self._rope_heads = None
        self.rope_handle: Optional[native.DenseWeight] = None

    def rows(self, first: int, n: int) -> "FastLinear":
        """Output columns [first, first + n) as a projection of their own on the same weight and image (first a multiple of 32)."""
        assert self.bias is None and not self._gate_up and self._rope_heads is None
        part = copy.copy(self)
        part.weight, part.out_features = self.weight[first:first + n], n
        part.prepared = self.prepared.rows(first, n) if self.streams else None
        return part

    @property
    def gate_up(self) -> bool:
        return self._gate_up

    @gate_up.setter
    def gate_up(self, on: bool):
        """Set by LlamaMLP on the fused [gate | up] projection: SiLU(gate)*up then runs in the GEMM epilogue (the image
        is rebuilt with interleaved pairs; the checkpoint-layout weight stays for the large-M library path)."""
        if bool(on) != self._gate_up and self.streams:
            self._gate_up = bool(on)
            self.prepared = native.DenseWeight(self.weight, gate_up=self._gate_up)

    @property
    def rope_heads(self):
        return self._rope_heads

    @rope_heads.setter
    def rope_heads(self, heads):
        """Set by FlashLlamaAttention on the fused qkv projection: (H, Hkv, D) of this shard.  Builds the rope image (a
        second copy of the weight with rotation pairs inside each tile) for native.dense_gemm_rope."""
        self._rope_heads = heads
        self.rope_handle = None
        if heads is not None and FUSED_ROPE_GEMM and heads[2] % 32 == 0 and self.streams:
            H, Hkv, D = heads
            # the image is a second copy of the weight: only build it where the fused launch will serve some decode batch
            # (tgis_dense_rope_ok asks for >= TGIS_ROPE_MIN_BLOCKS workgroups in the unsplit plan — TinyLlama has 40, a
            # 70B shard at TP = 8 has 20), as Ex4bitLinearV2.post_init does for the int4 image
            if any(native.rope_gemm_ok(m, self.prepared, D) for m in (1, 32, 64)):
                self.rope_handle = native.DenseWeight(self.weight, rope=(D, H + Hkv))

    def tall(self, x: torch.Tensor, act: int = 0) -> int:
        return tall_bytes(x, self.prepared, act) if self.streams else -1

    def forward(self, x: torch.Tensor, act: int = 0, out_f32: bool = False, partial: bool = False,
                gelu: Optional[bool] = None, out: Optional[torch.Tensor] = None) -> torch.Tensor:
        """`gelu` (None / False: exact erf form / True: tanh approximation): the activation behind this projection
        (santacoder's `c_fc`, flash_santacoder_modeling.py:303-305) — applied where the decode GEMM finishes its output
        instead of by a launch of its own; same bits as the two steps."""
        if out is not None:
            # the caller's buffer (a [M, N] view with unit column stride): plain projections only
            assert not act and not out_f32 and not partial and gelu is None and not self._gate_up and self.bias is None
            tall = self.tall(x)
            if tall >= 0:
                return native.dense_tall(x, self.prepared, workspace(x.device), tall, out=out)
            if self.streams and x.shape[0] <= SKINNY_MAX_M:
                return native.dense_gemm(x, self.prepared, workspace(x.device), out=out)
            if out.is_contiguous():
                return torch.mm(x, self.weight.t(), out=out)
            out.copy_(F.linear(x, self.weight))
            return out
        if not self.streams:
            assert not self._gate_up and not act and not partial
            out = F.linear(x, self.weight, self.bias)
            if gelu is not None:
                out = native.gelu(out, gelu)
            return out.float() if out_f32 else out
        if gelu is not None:
            assert act == 0 and not out_f32 and not partial and not self._gate_up
            tall = self.tall(x, 5 if gelu else 4) if FUSED_GELU_GEMM else -1
            if tall >= 0:
                return native.dense_tall(x, self.prepared, workspace(x.device), tall, bias=self.bias, act=5 if gelu else 4)
            if x.shape[0] <= SKINNY_MAX_M and FUSED_GELU_GEMM:
                return native.dense_gemm(x, self.prepared, workspace(x.device), bias=self.bias, act=5 if gelu else 4)
            return native.gelu(self.forward(x), gelu)
        if self._gate_up:
            # output is the activated [M, I] tensor
            tall = self.tall(x, 2)
            if tall >= 0:
                return native.dense_tall(x, self.prepared, workspace(x.device), tall, bias=self.bias, act=2)
            if x.shape[0] <= SKINNY_MAX_M:
                return native.dense_gemm(x, self.prepared, workspace(x.device), bias=self.bias, act=2)
            return native.act_mul(F.linear(x, self.weight, self.bias), self.out_features // 2)
        defers = partial and x.shape[0] <= native.PARTIAL_MAX_M and DEFER_REDUCE and not out_f32
        if defers and not act and DENSE_TALL and native.dense_tall_partial_bytes(x, self.prepared) >= 0:
            return native.dense_tall_partial(x, self.prepared, bias=self.bias)
        tall = self.tall(x) if not act and not defers and (not out_f32 or x.shape[0] <= SKINNY_MAX_M) else -1
        if tall >= 0:
            return native.dense_tall(x, self.prepared, workspace(x.device), tall, bias=self.bias, out_f32=out_f32)
        if defers:
            # the split-K sum (and the bias) is finished by the consumer kernel (add+norm / rope): no reduce launch
            return native.dense_gemm_partial(x, self.prepared, bias=self.bias, act=act)
        if x.shape[0] <= SKINNY_MAX_M:
            return native.dense_gemm(x, self.prepared, workspace(x.device), bias=self.bias, out_f32=out_f32, act=act)
        if act:
            x = native.act_mul(x, self.in_features)
        out = F.linear(x, self.weight, self.bias)
        return out.float() if out_f32 else out

    __call__ = forward


class Ex4bitLinearV2:
    """4-bit GPTQ linear.  Construction keeps the checkpoint tensors; `post_init` repacks them for the
    kernels (the reference defers this the same way, server.py:347-354)."""
    _temp_dq = {}

    def __init__(self, qweight, qzeros, scales, g_idx, bias, bits, groupsize):
        assert bits == 4
        self.device = qweight.device
        self.qweight, self.qzeros, self.scales = qweight, qzeros, scales
        # ("perm", gather index, x columns): an explicit activation permutation (act-order row shards, utils/weights.py)
        self.g_idx = g_idx if isinstance(g_idx, tuple) else (g_idx.cpu() if g_idx is not None else None)
        self.bias = bias
        self.bits, self.groupsize = bits, groupsize
        self.height = qweight.shape[0] * 8
        self.width = qweight.shape[1]
        # (no device check here: native.GptqWeight refuses tensors that are not on the GPU — server.py:290-291)
        assert self.height % 32 == 0 and self.width % 32 == 0
        self.q_handle: Optional[native.GptqWeight] = None
        self.ordered: Optional[native.GptqWeight] = None  # the same image for operands in its own order: what the kernels run on
        # set by LlamaMLP on the fused [gate | up] projection: SiLU(gate)*up runs in the GEMM epilogue
        self.gate_up = False
        # set by FlashLlamaAttention on the fused qkv projection: (H, Hkv, D) of this shard -> post_init also builds the
        # rope image (a second copy of the int4 matrix with rotation pairs inside each tile, +K*N/2 bytes) for
        # native.gptq_gemm_rope, the decode launch that rotates q / k and writes the cache in its epilogue
        self.rope_heads = None
        self.rope_handle: Optional[native.GptqWeight] = None
        self._perm: Optional[torch.Tensor] = None  # see `perm`
        self._fused = {}  # act -> rows up to which the library's fused kernels are used
        self._whole = {}  # (rows, act) -> whether the library finishes the sums by itself

    def post_init(self):
        handle = native.GptqWeight(self.qweight, self.qzeros, self.scales, self.g_idx, self.bits, self.groupsize,
                                   gate_up=self.gate_up)
        # act-order: the operand is gathered once, in front of the GEMM, and every kernel takes the matrix as if it had no
        # act-order (7B, 11 rows: the four GEMMs of a layer and the rotary launch 163 us when the GEMMs gather while they stage their operand,
        # 48 us with one gather launch in front of o_proj and the norms gathering for qkv and gate_up)
        self._perm = handle.perm
        self.q_handle, self.ordered = handle, handle if self._perm is None else handle.in_order()
        if self.rope_heads is not None and FUSED_ROPE_GEMM:
            H, Hkv, D = self.rope_heads
            if any(native.gptq_rope_ok(m, self.ordered, D) for m in (1, 32, 64)):
                rope = native.GptqWeight(self.qweight, self.qzeros, self.scales, self.g_idx if self._perm is not None else None,
                                         self.bits, self.groupsize, rope=(D, H + Hkv))
                self.rope_handle = rope if rope.perm is None else rope.in_order()
        self.qweight = self.qzeros = self.scales = None  # the prepared image replaces them

    @property
    def perm(self) -> Optional[torch.Tensor]:
        """Columns of the activation in the order the image wants them (int32, -1 = a zero column), None = as they are.  A
        producer that can gather (native.rmsnorm_residual) passes `gathered=True` on to forward."""
        if self.q_handle is None:
            self.post_init()
        return self._perm

    def places(self) -> Optional[torch.Tensor]:
        """Where each column of the activation goes in the image's order (int32): for a producer that writes its columns one by one (decode
        attention).  None without act-order and where `perm` is no permutation of the columns."""
        if self.perm is None or self._perm.numel() != self.height:
            return None
        order, columns = self._perm.long(), torch.arange(self.height, device=self._perm.device)
        if not bool((order.sort().values == columns).all()):
            return None
        return torch.empty_like(order).scatter_(0, order, columns).to(torch.int32)

    def order_columns(self, order: torch.Tensor):
        """Before post_init: re-order the output columns, y[:, i] = old y[:, order[i]]."""
        assert self.q_handle is None
        order = order.to(self.device).long()
        self.qweight = self.qweight.index_select(1, order)
        self.scales = self.scales.index_select(1, order)
        shifts = 4 * torch.arange(8, dtype=torch.int32, device=self.device)
        zeros = ((self.qzeros[:, :, None] >> shifts) & 15).view(self.qzeros.shape[0], -1).index_select(1, order)
        self.qzeros = (zeros.view(self.qzeros.shape[0], -1, 8) << shifts).sum(-1, dtype=torch.int32)
        if self.bias is not None:
            self.bias = self.bias.index_select(0, order)

    def take_ordered_input(self):
        """From now on the activation arrives in the image's order (its producer's columns were re-ordered to match)."""
        self._perm = None

    def _fused_rows(self, act: int) -> int:
        got = self._fused.get(act)
        if got is None:
            got = self._fused[act] = self.ordered.fused_rows(act)
        return got

    def _whole_sums(self, rows: int, act: int) -> bool:
        if rows <= 64 or self._fused_rows(act) <= 256:
            return False
        got = self._whole.get((rows, act))  # (up to 256 rows: PARTIAL_MAX_M)
        if got is None:
            got = self._whole[(rows, act)] = self.ordered.whole_sums(rows, act)
        return got

    def _dequant_scratch(self) -> torch.Tensor:
        key = (str(self.device), self.height, self.width)
        buf = Ex4bitLinearV2._temp_dq.get(key)
        if buf is None:
            Ex4bitLinearV2._temp_dq.clear()  # one scratch at a time, like exllama's temp_dq
            buf = Ex4bitLinearV2._temp_dq[key] = torch.empty((self.width, self.height), dtype=torch.float16,
                                                             device=self.device)
        return buf

    def wants_fragments(self, rows: int, act: int = 0, gathers: bool = False) -> bool:
        """Should the producer of this linear's operand write it in fragment order (native.FragAct) for `rows` decode
        rows?  act: 0 plain / partial, 2 the SiLU * up image, 3 the rope image (the fused qkv + rotary launch).  An act-order
        matrix asks for it only of a producer that can gather the columns (`gathers`)."""
        if self.perm is not None and not gathers:
            return False
        if act == 2 and not self.gate_up:
            act = 0
        w = self.rope_handle if act == 3 else self.ordered
        return w is not None and rows <= 64 and native.gptq_fragments_ok(rows, w, act)

    def forward(self, x, act: int = 0, partial: bool = False, out_frag: bool = False, gathered: bool = False):
        """partial=True (decode-sized M only): return native.Partial — the consumer kernel finishes the split-K sum.
        x may be a native.FragAct (decode, <= 64 rows; see wants_fragments); out_frag: the SiLU * up output leaves as one.
        gathered: x is in the order of `perm` already (a FragAct always is)."""
        if self.perm is not None and not gathered and not isinstance(x, native.FragAct):
            if act:
                x, act = native.act_mul(x, self.height), 0
            rows = x.shape[0]
            x = native.gather_columns(x, self._perm, frag=1 <= rows <= 64 and native.gptq_fragments_ok(
                rows, self.ordered, 2 if self.gate_up else 0))
        if isinstance(x, native.FragAct):
            if self.gate_up:
                return native.gptq_gemm(x, self.ordered, workspace(x.device), bias=self.bias, act=2, out_frag=out_frag)
            assert act == 0
            if partial and DEFER_REDUCE:
                return native.gptq_gemm_partial(x, self.ordered, bias=self.bias)
            return native.gptq_gemm(x, self.ordered, workspace(x.device), bias=self.bias)
        if self.gate_up:
            # output is the activated [M, I] tensor
            if x.shape[0] <= self._fused_rows(2) and (x.shape[0] <= 256 or self.ordered.fused_pays(x.shape[0], 2)):
                return native.gptq_gemm(x, self.ordered, workspace(x.device), bias=self.bias, act=2)
            return native.act_mul(self._large_m(x), self.width // 2)
        # where the tall kernel finishes its own sums sooner than a consumer adds the slabs of 64-row passes, nothing is deferred
        if partial and x.shape[0] <= native.PARTIAL_MAX_M and DEFER_REDUCE and not self._whole_sums(x.shape[0], act):
            return native.gptq_gemm_partial(x, self.ordered, bias=self.bias, act=act)
        if x.shape[0] <= self._fused_rows(act) and (x.shape[0] <= 256 or self.ordered.fused_pays(x.shape[0], act)):
            return native.gptq_gemm(x, self.ordered, workspace(x.device), bias=self.bias, act=act)
        if act:
            x = native.act_mul(x, self.height)
        return self._large_m(x)

    def _large_m(self, x: torch.Tensor) -> torch.Tensor:
        """prefill-sized M: dequantise once into scratch, then a library GEMM (exllamav2.py:87 "M > 50"); x in image order."""
        out = torch.matmul(x, native.gptq_dequant_t(self.ordered, self._dequant_scratch()).t())
        if self.bias is not None:
            out.add_(self.bias)
        return out

    __call__ = forward


def get_linear(weight, bias, quantize):
    if quantize is None:
        return FastLinear(weight, bias)
    if quantize == "gptq":
        try:
            qweight, qzeros, scales, g_idx, bits, groupsize, _use = weight
        except Exception:
            raise NotImplementedError("The passed weight is not `gptq` compatible, loader needs to be updated.")
        return Ex4bitLinearV2(qweight, qzeros, scales, g_idx, bias, bits, groupsize)
    raise NotImplementedError(f"Quantization `{quantize}` is not implemented yet.")


class SuperLayer:
    def __init__(self, linear):
        self.linear = linear

    def forward(self, x, **kw):
        return self.linear.forward(x, **kw)

    __call__ = forward


class TensorParallelHead(SuperLayer):
    def __init__(self, linear, process_group, should_gather: bool):
        super().__init__(linear)
        self.process_group = process_group
        self.should_gather = should_gather

    @staticmethod
    def load(config, prefix: str, weights):
        if weights.process_group.size() > 1:
            try:
                weight = weights.get_sharded(f"{prefix}.weight", dim=0)
                should_gather = True
            except AssertionError:
                # vocab not divisible by the number of shards: every rank keeps the full head
                weight = weights.get_tensor(f"{prefix}.weight")
                should_gather = False
        else:
            weight = weights.get_tensor(f"{prefix}.weight")
            should_gather = False
        # GPTQ doesn't quantize heads (nor embeddings)
        return TensorParallelHead(get_linear(weight, bias=None, quantize=None), weights.process_group, should_gather)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        """fp32 logits [T, V]; vocab shards are gathered so every rank holds identical logits."""
        local = self.linear.forward(x, out_f32=True)
        if not self.should_gather:
            return local
        world = self.process_group.size()
        # Every rank contributes its [T, V/tp] block; the gathered [tp, T, V/tp] buffer is re-laid out ONCE into the
        # row-major [T, V] the fused argmax / warper kernels read.  (The reference gathers transposed [V/tp, T] blocks
        # and returns a transposed view, layers.py:244-269 — two transposing copies on this side of the gather.)
        local = local.contiguous()
        T, vp = local.shape
        gathered = torch.empty((world, T, vp), dtype=local.dtype, device=local.device)
        pg = self.process_group
        collective(lambda o=gathered, i=local: torch.distributed.all_gather_into_tensor(o.view(world * T, vp), i, group=pg))
        return gathered.permute(1, 0, 2).reshape(T, world * vp)

    __call__ = forward


class TensorParallelColumnLinear(SuperLayer):
    @classmethod
    def load(cls, config, prefix: str, weights, bias: bool):
        return cls.load_multi(config, [prefix], weights, bias, dim=0)

    @classmethod
    def load_multi(cls, config, prefixes: List[str], weights, bias: bool, dim: int):
        weight = weights.get_multi_weights_col(prefixes, quantize=config.quantize, dim=dim)
        if bias:
            b = [weights.get_sharded(f"{p}.bias", dim=0) for p in prefixes]
            bias = torch.cat(b, dim=dim)
        else:
            bias = None
        return cls(get_linear(weight, bias, config.quantize))


class TensorParallelRowLinear(SuperLayer):
    def __init__(self, linear, process_group):
        super().__init__(linear)
        self.process_group = process_group

    @classmethod
    def load(cls, config, prefix: str, weights, bias: bool):
        weight = weights.get_multi_weights_row(prefix, quantize=config.quantize)
        if bias and weights.process_group.rank() == 0:
            bias = weights.get_tensor(f"{prefix}.bias")  # bias only on the first rank
        else:
            bias = None
        return cls(get_linear(weight, bias, config.quantize), process_group=weights.process_group)

    def forward(self, x: torch.Tensor, **kw) -> torch.Tensor:
        if self.process_group.size() > 1:
            kw.pop("partial", None)  # the all-reduce needs the reduced f16 tensor
            out = self.linear.forward(x, **kw)
            pg = self.process_group
            collective(lambda t=out: torch.distributed.all_reduce(t, group=pg))
            return out
        return self.linear.forward(x, **kw)

    __call__ = forward


class TensorParallelEmbedding:
    def __init__(self, prefix: str, weights, reduce=True):
        self.weight = weights.get_partial_sharded(f"{prefix}.weight", dim=0).contiguous()
        num_embeddings = weights.get_shape(f"{prefix}.weight")[0]
        self.process_group = weights.process_group
        world_size = self.process_group.size()
        rank = self.process_group.rank()
        block_size = num_embeddings // world_size
        self.min_id = rank * block_size
        self.max_id = min(num_embeddings, (rank + 1) * block_size)
        self.reduce = reduce

    def forward(self, input_ids: torch.Tensor, positions=None, pos_table=None) -> torch.Tensor:
        # ids outside [min_id, max_id) read the null (zero) row, then shards are summed (layers.py:346-357)
        out = native.embedding(input_ids, self.weight, positions=positions, pos_table=pos_table,
                               id_offset=self.min_id)
        if self.reduce and self.process_group.size() > 1:
            pg = self.process_group
            collective(lambda t=out: torch.distributed.all_reduce(t, group=pg))
        return out

    __call__ = forward


class PositionRotaryEmbedding:
    """cos/sin caches: inv_freq and freqs in fp32, tables cast to the model dtype (layers.py:419-451)."""

    def __init__(self, inv_freq: torch.Tensor, scaling_factor: float = 1.0):
        self.inv_freq = inv_freq
        self.scaling_factor = scaling_factor
        self._seq_len_cached = 0
        self._cos_cached = None
        self._sin_cached = None
        # tables that were replaced by longer ones: captured decode graphs hold raw pointers into them, and every
        # position such a graph can see lies inside the table it captured, so they only have to stay allocated
        self._retired = []

    @classmethod
    def static(cls, dim, base, device, scaling_factor=1.0):
        inv_freq = 1.0 / (base ** (torch.arange(0, dim, 2, device=device, dtype=torch.float32) / dim))
        return cls(inv_freq, scaling_factor)

    def tables(self, dtype, device, seqlen: int):
        if seqlen > self._seq_len_cached or self._cos_cached.device != device or self._cos_cached.dtype != dtype:
            if self._cos_cached is not None:
                self._retired.append((self._cos_cached, self._sin_cached))
            self._seq_len_cached = seqlen
            t = torch.arange(seqlen, device=device, dtype=self.inv_freq.dtype)
            if self.scaling_factor != 1.0:
                t = t / self.scaling_factor
            freqs = torch.outer(t, self.inv_freq.to(device=t.device))
            self._cos_cached = torch.cos(freqs).to(dtype).contiguous()
            self._sin_cached = torch.sin(freqs).to(dtype).contiguous()
        return self._cos_cached, self._sin_cached

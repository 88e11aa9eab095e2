"""The work a server asks of this framework, as cases that can be timed and checked one by one.

A case is one call a shard servicer makes: a decode step of a running batch (`FlashCausalLM.generate_token`, the NextToken RPC), the
prefill of a new batch (`from_pb` + `generate_token(first=True)`, the Prefill RPC), or a short completion (a prefill and the decode
steps behind it).  Models have the layer shapes of the benchmark's configurations, some with fewer layers than the checkpoint they
stand for; weights and prompts are seeded noise.  The embedding of the vocabulary in the head is heavy-tailed, as trained heads are,
so that the best token is seldom a near tie.

Decode steps are teacher-forced: the step's input token is seeded and the batch is set back to the same position before every pass,
which is the state a batch is in after a `concatenate` or `prune` (its inputs are staged anew)."""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "text-generation-inference_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

F64 = torch.float64
GROUP = 128  # GPTQ group size
PAGE = 32    # tokens per cache page

# layer shapes of the benchmark's models; `layers` may be a slice of the whole depth
MODELS = {
    # Llama-2-7B, int4 GPTQ, at full depth
    "llama7b": dict(kind="llama", width=4096, ff=11008, heads=32, kv_heads=32, layers=32, vocab=32000, quant=True, dtype="float16"),
    # Llama-2-70B, int4 GPTQ: 4 of 80 layers
    "llama70b": dict(kind="llama", width=8192, ff=28672, heads=64, kv_heads=8, layers=4, vocab=32000, quant=True, dtype="float16"),
    # TinyLlama-1.1B, bf16, at full depth
    "tinyllama": dict(kind="llama", width=2048, ff=5632, heads=32, kv_heads=4, layers=22, vocab=32000, quant=False, dtype="bfloat16"),
    # Starcoder-15B, bf16, multi-query attention: 8 of 40 layers
    "starcoder": dict(kind="bigcode", width=6144, ff=24576, heads=48, kv_heads=1, layers=8, vocab=49152, quant=False,
                      dtype="bfloat16"),
    # Lenisun at the 1b size: recurrence and attention in turn, clamped gated units; 8 of 22 layers
    "lenisun": dict(kind="lenisun", width=2048, ff=5632, heads=32, kv_heads=4, layers=8, vocab=32000, quant=False, dtype="bfloat16"),
}


def _case(name, task, model, batch, length, ragged=False, sampled=False, act_order=False, new=1):
    return {"name": name, "task": task, "model": model, "batch": batch, "length": length, "ragged": ragged, "sampled": sampled,
            "act_order": act_order, "new": new}


def listed():
    return [
        # one interactive user of a small model: a step is all launches and latency
        _case("decode_one_user", "decode", "tinyllama", 1, 137),
        # a small model under ordinary load (the benchmark's TinyLlama configuration)
        _case("decode_small_model", "decode", "tinyllama", 16, 512),
        # the headline: a 7B int4 model, a full batch at a common context
        _case("decode_int4_full_batch", "decode", "llama7b", 32, 1024),
        # chat traffic on an act-order checkpoint: contexts of all lengths, every request with its own sampling parameters
        _case("decode_int4_sampled_ragged", "decode", "llama7b", 11, 700, ragged=True, sampled=True, act_order=True),
        # a large grouped-query model, two row tiles per step
        _case("decode_70b_int4", "decode", "llama70b", 64, 2048),
        # a code model with one kv head and long contexts
        _case("decode_code_long", "decode", "starcoder", 32, 4096),
        # time to first token of a short prompt
        _case("prefill_short", "prefill", "tinyllama", 1, 47),
        # a few arriving requests beside a running int4 batch
        _case("prefill_int4_few", "prefill", "llama7b", 3, 433, ragged=True),
        # a wave of prompts, the largest prefill a router would form
        _case("prefill_int4_many", "prefill", "llama7b", 16, 1008),
        # two long files for a code model: attention over thousands of keys
        _case("prefill_code_long", "prefill", "starcoder", 2, 4093),
        # prompts of a hybrid decoder: recurrent scans and normed attention
        _case("prefill_hybrid", "prefill", "lenisun", 4, 1024),
        # short completions of a hybrid decoder: prompts of a chat turn, eight tokens each
        _case("complete_hybrid", "complete", "lenisun", 24, 96, ragged=True, new=8),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    task = rng.choice(["decode", "decode", "prefill", "prefill", "complete"])
    if task == "complete":
        return _unnamed(_case("", task, "lenisun", log_int(1, 32), log_int(8, 300), ragged=rng.random() < 0.7, new=rng.randint(2, 12)))
    if task == "decode":
        model = rng.choice(["tinyllama", "llama7b", "llama7b", "llama70b", "starcoder"])
        batch = log_int(1, 64)
        length = log_int(20, min(4096, 65536 // batch))
        if model == "llama7b":
            length = min(length, 32768 // batch)
    else:
        model = rng.choice(["tinyllama", "llama7b", "llama70b", "starcoder", "lenisun"])
        tokens = log_int(16, 8192)
        batch = log_int(1, min(16, tokens // 8))
        length = min(4096, max(8, tokens // batch))
    return _unnamed(_case("", task, model, batch, length, ragged=rng.random() < 0.6, sampled=rng.random() < 0.25,
                          act_order=MODELS[model]["quant"] and rng.random() < 0.3))


def _unnamed(case):
    return {k: v for k, v in case.items() if k != "name"}


# ---- inputs ---------------------------------------------------------------------------------------------------------------


def _lengths(case):
    """Prompt lengths: all equal, or spread between a quarter of the nominal length and the length itself."""
    n, b = case["length"], case["batch"]
    if not case["ragged"]:
        return [n] * b
    return [max(1, int(n * (0.25 + 0.75 * ((i * 0.618034 + 0.5) % 1.0)))) for i in range(b)]


def _prompts(case, seed):
    """Token ids of every prompt and of the forced tokens behind it."""
    g = torch.Generator().manual_seed(seed * 1000003 + 17)
    vocab = MODELS[case["model"]]["vocab"]
    return [torch.randint(3, vocab, (n + case["new"],), generator=g) for n in _lengths(case)]


class _Recipe:
    """Seeded weights, made on `device` in the order they are asked for."""

    def __init__(self, seed, device, dtype):
        self.g = torch.Generator(device=device).manual_seed(seed)
        self.device, self.dtype, self.t = device, dtype, {}

    def normal(self, name, *shape, std=1.0, mean=0.0):
        self.t[name] = torch.empty(shape, device=self.device, dtype=self.dtype).normal_(mean, std, generator=self.g)

    def uniform(self, name, *shape, lo=0.0, hi=1.0):
        self.t[name] = torch.empty(shape, device=self.device, dtype=torch.float32).uniform_(lo, hi, generator=self.g).to(self.dtype)

    def linear(self, name, n, k, suffix=".weight", bias=False):
        self.normal(name + suffix, n, k, std=k ** -0.5)
        if bias:
            self.normal(name + ".bias", n, std=0.02)

    def head(self, name, n, k):
        self.normal(name, n, k, std=k ** -0.5)
        self.t[name] *= torch.empty((n, 1), device=self.device).normal_(0.0, 0.5, generator=self.g).exp().to(self.dtype)

    def gptq(self, name, n, k, g_idx):
        """Uniform nibbles, zero points 1..14, scales that give the matrix a standard deviation of k ** -0.5."""
        dev, G = self.device, k // GROUP
        bits = dict(device=dev, dtype=torch.int32, generator=self.g)
        self.t[f"{name}.qweight"] = torch.randint(-2**31, 2**31 - 1, (k // 8, n), **bits)
        zeros = torch.randint(0, 14, (G, n // 8, 8), **bits)
        self.t[f"{name}.qzeros"] = (zeros << (4 * torch.arange(8, device=dev, dtype=torch.int32))).sum(-1, dtype=torch.int32)
        scale = torch.empty((G, n), device=dev).uniform_(0.5, 1.5, generator=self.g)
        self.t[f"{name}.scales"] = (scale * (k ** -0.5 / 6.4)).to(torch.float16)
        self.t[f"{name}.g_idx"] = g_idx

    def group_index(self, k, shuffled):
        g_idx = torch.arange(k, device=self.device, dtype=torch.int32) // GROUP
        return g_idx[torch.randperm(k, device=self.device, generator=self.g)] if shuffled else g_idx


def _lenisun_layers(m):
    dim = m["width"] // m["heads"]
    attention = {"heads": m["heads"], "kv_heads": m["kv_heads"], "dim": dim, "vdim": dim, "scale": dim ** -0.5,
                 "q_temp": {"coef": 0.1, "every": 1024}, "v_mix": True}
    recurrence = {"heads": m["width"] // 64, "dim": 64}
    return [{"type": "attention" if i % 2 else "wkv", "mixer": attention if i % 2 else recurrence,
             "mlp": {"kind": "dense", "ff": m["ff"], "limit": 7.0}} for i in range(m["layers"])]


def _weights(case, seed, device):
    m = MODELS[case["model"]]
    W, ff, L, vocab = m["width"], m["ff"], m["layers"], m["vocab"]
    dim = W // m["heads"]
    kv = m["kv_heads"] * dim
    r = _Recipe(seed, device, getattr(torch, m["dtype"]))
    if m["kind"] == "llama":
        r.normal("model.embed_tokens.weight", vocab, W)
        for i in range(L):
            p = f"model.layers.{i}"
            groups = [r.group_index(k, case["act_order"]) for k in (W, W, W, ff)]
            for name, n, k, g in (("self_attn.q_proj", W, W, 0), ("self_attn.k_proj", kv, W, 0), ("self_attn.v_proj", kv, W, 0),
                                  ("self_attn.o_proj", W, W, 1), ("mlp.gate_proj", ff, W, 2), ("mlp.up_proj", ff, W, 2),
                                  ("mlp.down_proj", W, ff, 3)):
                if m["quant"]:
                    r.gptq(f"{p}.{name}", n, k, groups[g])
                else:
                    r.linear(f"{p}.{name}", n, k)
            for n in ("input_layernorm", "post_attention_layernorm"):
                r.normal(f"{p}.{n}.weight", W, mean=1.0, std=0.05)
        r.normal("model.norm.weight", W, mean=1.0, std=0.05)
        r.head("lm_head.weight", vocab, W)
    elif m["kind"] == "bigcode":
        r.head("transformer.wte.weight", vocab, W)
        r.normal("transformer.wpe.weight", 8192, W, std=0.02)
        for i in range(L):
            p = f"transformer.h.{i}"
            for name, n, k in (("attn.c_attn", W + 2 * dim, W), ("attn.c_proj", W, W), ("mlp.c_fc", ff, W), ("mlp.c_proj", W, ff)):
                r.linear(f"{p}.{name}", n, k, bias=True)
            for n in ("ln_1", "ln_2"):
                r.normal(f"{p}.{n}.weight", W, mean=1.0, std=0.05)
                r.normal(f"{p}.{n}.bias", W, std=0.05)
        r.normal("transformer.ln_f.weight", W, mean=1.0, std=0.05)
        r.normal("transformer.ln_f.bias", W, std=0.05)
    else:
        r.normal("embed", vocab, W)
        for i, lay in enumerate(_lenisun_layers(m)):
            p, x = f"l{i}.mix", lay["mixer"]
            for n in ("norm1", "norm1b", "norm2", "norm2b"):
                r.normal(f"l{i}.{n}", W, std=0.05)
            if lay["type"] == "attention":
                for n, rows in (("q", W), ("k", kv), ("v", kv), ("o", W)):
                    r.linear(f"{p}.{n}", rows, W, suffix="")
                r.normal(f"{p}.q.norm", dim, mean=1.0, std=0.05)
                r.normal(f"{p}.k.norm", dim, mean=1.0, std=0.05)
                r.uniform(f"{p}.vmix", lo=0.3, hi=0.7)
            else:
                for n in ("r", "k", "v", "g", "w"):
                    r.uniform(f"{p}.mu.{n}", W)
                for n in ("r", "k", "v", "g", "o"):
                    r.linear(f"{p}.{n}", W, W, suffix="")
                r.linear(f"{p}.w1", 64, W, suffix="")
                r.linear(f"{p}.w2", W, 64, suffix="")
                r.normal(f"{p}.w0", W, mean=-1.0)
                r.normal(f"{p}.u", x["heads"], x["dim"], std=0.3)
                r.normal(f"{p}.norm", W, mean=1.0, std=0.05)
            for n, rows, k in (("gate", ff, W), ("up", ff, W), ("down", W, ff)):
                r.linear(f"l{i}.mlp.{n}", rows, k, suffix="")
        r.normal("final.norm", W, std=0.05)
        r.head("head", vocab, W)
    return r.t


def _config(case):
    m = MODELS[case["model"]]
    if m["kind"] == "llama":
        from tgis_amd.models.custom_modeling.flash_llama_modeling import LlamaConfig

        return LlamaConfig(vocab_size=m["vocab"], hidden_size=m["width"], intermediate_size=m["ff"], num_hidden_layers=m["layers"],
                           num_attention_heads=m["heads"], num_key_value_heads=m["kv_heads"], rms_norm_eps=1e-5, pad_token_id=0,
                           max_position_embeddings=4096)
    if m["kind"] == "bigcode":
        from tgis_amd.inference_engine.synthetic import BigCodeConfig

        return BigCodeConfig(vocab_size=m["vocab"], hidden_size=m["width"], n_inner=m["ff"], num_hidden_layers=m["layers"],
                             num_attention_heads=m["heads"], n_positions=8192)
    from tgis_amd.models.custom_modeling.flash_lenisun_modeling import LenisunConfig

    return LenisunConfig(width=m["width"], vocab=m["vocab"], layers=_lenisun_layers(m), norm={"eps": 1e-5}, embedding={"scale": 1.0})


class _Prompts:
    """Stands for the checkpoint's tokenizer: the prompt texts are keys of prompts that are tokenized already."""
    pad_token_id, bos_token_id, eos_token_id = 0, 1, 2
    add_bos_token, padding_side, truncation_side = False, "left", "left"

    def __init__(self, ids):
        self.ids = ids

    def __call__(self, texts, truncation=True, max_length=None, return_token_type_ids=False):
        return {"input_ids": [self.ids[t] for t in texts]}


def _model(case, seed, tokenizer):
    from tgis_amd.inference_engine.synthetic import InferenceEngine
    from tgis_amd.models.flash_causal_lm import FlashCausalLM

    class Model(FlashCausalLM):
        """Keeps the last step's logits beside the tokens chosen from them."""

        def _process_new_tokens(self, batch, out, *args):
            self.last_logits = out
            return super()._process_new_tokens(batch, out, *args)

    m = MODELS[case["model"]]
    dtype, quantize = getattr(torch, m["dtype"]), "gptq" if m["quant"] else None
    engine = InferenceEngine(_weights(case, seed, torch.device("cuda")), _config(case), dtype, quantize, tokenizer=tokenizer,
                             gptq_groupsize=GROUP)
    pages = sum((n + case["new"]) // PAGE + 1 for n in _lengths(case)) + 64
    return Model("synthetic", None, "synthetic", dtype, quantize, engine=engine, kv_cache_pages=pages, state_slots=64)


def _request_batch(case, indices, lengths):
    from tgis_amd.pb import generate_pb2

    requests = []
    for i in indices:
        r = generate_pb2.Request(id=i, inputs=f"prompt {i}", input_length=lengths[i], truncate=True,
                                 max_output_length=case["new"] + 1)
        if case["sampled"]:
            p = r.parameters
            p.seed = 1000 + i
            p.temperature = 0.7 + 0.1 * (i % 5)
            if i % 3 == 0:
                p.top_k = 50
            if i % 2 == 0:
                p.top_p = 0.9
            p.repetition_penalty = 1.1 if i % 2 else 1.0
        else:
            r.details.logprobs = True
        requests.append(r)
    return generate_pb2.Batch(id=indices[0], requests=requests, total_tokens=sum(lengths[i] for i in indices))


def _prefill(lm, pb):
    batch, errors = lm.batch_type.from_pb(pb, lm.tokenizer, lm.dtype, lm.device, lm.word_embeddings, lm.prefix_cache,
                                          lm.use_position_ids)
    assert not errors
    return batch, lm.generate_token(batch, first=True)[0]


def prepare(case, seed):
    lengths, prompts = _lengths(case), _prompts(case, seed)
    lm = _model(case, seed, _Prompts({f"prompt {i}": p[:n].tolist() for i, (p, n) in enumerate(zip(prompts, lengths))}))
    forced = torch.stack([p[n:] for p, n in zip(prompts, lengths)], dim=1).to("cuda")  # [new, batch]
    state = {"case": case, "lm": lm, "lengths": lengths, "forced": list(forced),
             "request": _request_batch(case, list(range(len(lengths))), lengths)}
    if case["task"] == "decode":
        # a running batch: requests were prefilled in waves of up to 16k tokens and joined
        waves, tokens = [[]], 0
        for i, n in enumerate(lengths):
            if waves[-1] and tokens + n > 16384:
                waves.append([])
                tokens = 0
            waves[-1].append(i)
            tokens += n
        with lm.context_manager():
            batches = [_prefill(lm, _request_batch(case, w, lengths))[0] for w in waves]
            batch = batches[0] if len(batches) == 1 else lm.batch_type.concatenate(batches)
            batch.all_input_ids_tensor.scatter_(1, batch.position_ids[:, None], state["forced"][0][:, None])
        state.update(batch=batch, positions=batch.position_ids.clone(), input_lengths=list(batch.input_lengths),
                     max_seqlen=batch.max_seqlen)
    return state


def run(state):
    """Logits of the pass's last step, and the requests' token ids with the chosen ones written behind the prompts."""
    case, lm = state["case"], state["lm"]
    with lm.context_manager():
        if case["task"] == "decode":
            batch = state["batch"]
            batch.input_ids, batch.position_ids = state["forced"][0], state["positions"].clone()
            batch.input_lengths, batch.max_seqlen = list(state["input_lengths"]), state["max_seqlen"]
            lm.generate_token(batch)
            return {"logits": lm.last_logits, "ids": batch.all_input_ids_tensor}
        batch, _ = _prefill(lm, state["request"])
        if case["task"] == "complete":
            for forced in state["forced"]:
                batch.input_ids = forced
                lm.generate_token(batch)
        batch.release()
        return {"logits": lm.last_logits, "ids": batch.all_input_ids_tensor}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------


def work(case):
    m, lengths = MODELS[case["model"]], _lengths(case)
    W, ff, L, B = m["width"], m["ff"], m["layers"], case["batch"]
    dim = W // m["heads"]
    kv = m["kv_heads"] * dim
    attention = W * (W + 2 * kv) + W * W
    recurrence = 5 * W * W + 2 * 64 * W
    n_att = L // 2 if m["kind"] == "lenisun" else L
    params = n_att * attention + (L - n_att) * recurrence + L * (2 if m["kind"] == "bigcode" else 3) * W * ff
    head = W * m["vocab"]
    weight_bytes = params * (0.5 + 2.5 / GROUP if m["quant"] else 2.0) + head * 2
    state_bytes = (L - n_att) * W * 64 * 4  # matrix states of one sequence
    kv_token = n_att * 2 * kv * 2
    out_bytes = B * m["vocab"] * 4

    def step(new, cached):
        """(bytes, flops) of a forward that adds `new[i]` tokens to `cached[i]`."""
        tokens = sum(new)
        pairs = sum(n * c + n * (n + 1) // 2 for n, c in zip(new, cached))
        moved = weight_bytes + kv_token * (tokens + sum(c for c in cached)) + out_bytes + tokens * W * 2
        moved += state_bytes * sum(2 if c else 1 for c in cached)
        return moved, 2 * params * tokens + 2 * head * B + 4 * n_att * W * pairs + 6 * (L - n_att) * W * 64 * tokens

    ones = [1] * B
    if case["task"] == "decode":
        parts = [step(ones, lengths)]
    else:
        parts = [step(lengths, [0] * B)]
        if case["task"] == "complete":
            parts += [step(ones, [n + j for n in lengths]) for j in range(case["new"])]
    return {"bytes": int(sum(p[0] for p in parts)), "flops": int(sum(p[1] for p in parts))}


def tolerance(case):
    # four times what the path shows against `exact` (rounding of activations and cached keys and values to the model's two-byte type
    # in every layer): 2.5e-3, 0.95e-3, 1.65e-2, 6.6e-3 and 1.7e-2; among the ids, a chosen token may differ where two candidates are
    # within that error of each other
    rel = {"llama7b": 1e-2, "llama70b": 4e-3, "tinyllama": 6.5e-2, "starcoder": 2.6e-2, "lenisun": 6.5e-2}[case["model"]]
    chosen = case["batch"] * (case["new"] + 1)
    ids = case["batch"] * (max(_lengths(case)) + case["new"] + 1)
    return {"rel": rel, "differ": max(1.0, 0.08 * chosen) * 1.001 / ids}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------------


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _rotate(x, pos, base=10000.0):
    d = x.shape[-1]
    angle = pos.to(F64)[:, None] * base ** (-torch.arange(0, d, 2, device=x.device, dtype=F64) / d)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _attend(q, k, v, scale):
    """q [n, H, d] are the last n positions of k, v [t, G, d]: causal softmax attention, [n, H, d]."""
    n, H, _ = q.shape
    t, G, _ = k.shape
    out = torch.empty_like(q)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    keys = torch.arange(t, device=q.device)
    rows = max(1, int(2e8) // (H * t))
    for a in range(0, n, rows):
        part = q[a:a + rows]
        c = part.shape[0]
        s = torch.bmm(part.reshape(c, G, H // G, -1).permute(1, 0, 2, 3).reshape(G, c * (H // G), -1), kt) * scale
        s = s.view(G, c, H // G, t)
        limit = torch.arange(t - n + a, t - n + a + c, device=q.device)
        s.masked_fill_((keys[None, :] > limit[:, None])[None, :, None, :], float("-inf"))
        o = torch.bmm(torch.softmax(s, -1).view(G, -1, t), vt).view(G, c, H // G, -1)
        out[a:a + rows] = o.permute(1, 0, 2, 3).reshape(c, H, -1)
    return out


def _dequantize(t, name):
    qw, qz = t[f"{name}.qweight"], t[f"{name}.qzeros"]
    shifts = 4 * torch.arange(8, device=qw.device, dtype=torch.int32)
    q = ((qw[:, None, :] >> shifts[None, :, None]) & 15).reshape(-1, qw.shape[1])
    z = ((qz[:, :, None] >> shifts) & 15).reshape(qz.shape[0], -1) + 1
    g = t[f"{name}.g_idx"].long()
    return (q - z[g]).to(F64) * t[f"{name}.scales"].to(F64)[g]  # [in, out]


def exact(case, seed):
    m, lengths, prompts = MODELS[case["model"]], _lengths(case), _prompts(case, seed)
    dev = torch.device("cuda")
    t = _weights(case, seed, dev)
    new = 0 if case["task"] == "prefill" else case["new"]
    ids = torch.cat([p[:n + new] for p, n in zip(prompts, lengths)]).to(dev)
    runs, at = [], 0
    for n in lengths:
        runs.append((at, at + n + new))
        at += n + new
    pos = torch.cat([torch.arange(b - a, device=dev) for a, b in runs])
    last = torch.tensor([b - 1 for _, b in runs], device=dev)
    with torch.inference_mode():
        logits = _lenisun_exact(m, t, ids, pos, runs, last) if m["kind"] == "lenisun" else _decoder_exact(m, t, ids, pos, runs, last)
    return {"logits": logits, "ids": None}  # (a token may be settled by a near tie or a draw)


def _by_rows(x, f, rows=16384):
    return torch.cat([f(x[i:i + rows]) for i in range(0, x.shape[0], rows)])


def _decoder_exact(m, t, ids, pos, runs, last):
    """Llama or GPT-BigCode over whole sequences; logits of each one's last token."""
    W, H, G, ff = m["width"], m["heads"], m["kv_heads"], m["ff"]
    dim = W // H
    llama = m["kind"] == "llama"

    def product(x, name):
        if f"{name}.qweight" in t:
            return x @ _dequantize(t, name)
        y = x @ t[f"{name}.weight"].to(F64).t()
        return y + t[f"{name}.bias"].to(F64) if f"{name}.bias" in t else y

    def norm(x, name):
        w = t[f"{name}.weight"].to(F64)
        if llama:
            return _rms(x, 1e-5) * w
        return torch.nn.functional.layer_norm(x, (W,), w, t[f"{name}.bias"].to(F64), 1e-5)

    if llama:
        x = t["model.embed_tokens.weight"][ids].to(F64)
    else:
        x = t["transformer.wte.weight"][ids].to(F64) + t["transformer.wpe.weight"][pos].to(F64)
    for i in range(m["layers"]):
        p = f"model.layers.{i}" if llama else f"transformer.h.{i}"
        h = norm(x, f"{p}.input_layernorm" if llama else f"{p}.ln_1")
        if llama:
            q, k, v = (product(h, f"{p}.self_attn.{n}_proj").view(-1, heads, dim) for n, heads in (("q", H), ("k", G), ("v", G)))
            q, k = _rotate(q, pos), _rotate(k, pos)
        else:
            q, k, v = (y.reshape(-1, heads, dim) for y, heads in zip(product(h, f"{p}.attn.c_attn").split([W, dim, dim], -1), (H, 1, 1)))
        del h
        if i + 1 == m["layers"]:  # nothing reads the other tokens' last layer
            o = torch.cat([_attend(q[b - 1:b], k[a:b], v[a:b], dim ** -0.5) for a, b in runs])
            x = x[last]
        else:
            o = torch.cat([_attend(q[a:b], k[a:b], v[a:b], dim ** -0.5) for a, b in runs])
        del q, k, v
        x = x + product(o.reshape(-1, W), f"{p}.self_attn.o_proj" if llama else f"{p}.attn.c_proj")
        del o
        h = norm(x, f"{p}.post_attention_layernorm" if llama else f"{p}.ln_2")
        if llama:
            h = torch.nn.functional.silu(product(h, f"{p}.mlp.gate_proj")).mul_(product(h, f"{p}.mlp.up_proj"))
            x = x + product(h, f"{p}.mlp.down_proj")
        else:
            h = torch.nn.functional.gelu(product(h, f"{p}.mlp.c_fc"), approximate="tanh")
            x = x + product(h, f"{p}.mlp.c_proj")
        del h
    return norm(x, "model.norm" if llama else "transformer.ln_f") @ t["lm_head.weight" if llama else "transformer.wte.weight"].to(F64).t()


def _lenisun_exact(m, t, ids, pos, runs, last):
    """Lenisun over whole sequences; logits of each one's last token."""
    eps = 1e-5
    w = lambda name: t[name].to(F64)
    norm = lambda x, name: _rms(x, eps) * (1.0 + w(name))
    x = w("embed")[ids]
    v_first = None
    for i, lay in enumerate(_lenisun_layers(m)):
        p, c = f"l{i}.mix", lay["mixer"]
        H, d = c["heads"], c["dim"]
        h = norm(x, f"l{i}.norm1")
        if lay["type"] == "attention":
            q, k, v = (h @ w(f"{p}.{n}").t() for n in ("q", "k", "v"))
            q, k, v = q.view(-1, H, d), k.view(-1, c["kv_heads"], d), v.view(-1, c["kv_heads"], d)
            gain = 1.0 + c["q_temp"]["coef"] * torch.log((pos + 1).div(c["q_temp"]["every"], rounding_mode="floor").to(F64) + 1.0)
            q, k = _rms(q, eps) * w(f"{p}.q.norm") * gain[:, None, None], _rms(k, eps) * w(f"{p}.k.norm")
            if v_first is None:
                v_first = v
            else:
                v = (1.0 - w(f"{p}.vmix")) * v + w(f"{p}.vmix") * v_first
            y = torch.cat([_attend(q[a:b], k[a:b], v[a:b], c["scale"]) for a, b in runs]).reshape(-1, H * d)
        else:
            before = torch.cat([torch.cat([torch.zeros_like(h[:1]), h[a:b - 1]]) for a, b in runs])
            mix = lambda n: h + (before - h) * w(f"{p}.mu.{n}")
            r, k, v = ((mix(n) @ w(f"{p}.{n}").t()).view(-1, H, d) for n in ("r", "k", "v"))
            decay = torch.exp(-torch.exp(torch.tanh(mix("w") @ w(f"{p}.w1").t()) @ w(f"{p}.w2").t() + w(f"{p}.w0"))).view(-1, H, d)
            # all sequences side by side, padded to the longest
            n, B = max(b - a for a, b in runs), len(runs)
            wide = [torch.zeros((n, B, H, d), dtype=F64, device=x.device) for _ in range(4)]
            for j, (a, b) in enumerate(runs):
                for dst, src in zip(wide, (r, k, v, decay)):
                    dst[:b - a, j] = src[a:b]
            S, o, u = torch.zeros((B, H, d, d), dtype=F64, device=x.device), torch.empty_like(wide[0]), w(f"{p}.u")[None, :, :, None]
            for s in range(n):
                kv = wide[1][s][..., :, None] * wide[2][s][..., None, :]
                o[s] = (wide[0][s][..., None, :] @ (S + u * kv))[..., 0, :]
                S = S * wide[3][s][..., :, None] + kv
            o = torch.cat([o[:b - a, j] for j, (a, b) in enumerate(runs)])
            y = _rms(o, eps).reshape(-1, H * d) * w(f"{p}.norm") * torch.nn.functional.silu(mix("g") @ w(f"{p}.g").t())
        x = x + norm(y @ w(f"{p}.o").t(), f"l{i}.norm1b")
        h = norm(x, f"l{i}.norm2")
        g = torch.clamp(h @ w(f"l{i}.mlp.gate").t(), max=7.0)
        u = torch.clamp(h @ w(f"l{i}.mlp.up").t(), -7.0, 7.0)
        x = x + norm((g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(f"l{i}.mlp.down").t(), f"l{i}.norm2b")
    return norm(x[last], "final.norm") @ w("head").t()

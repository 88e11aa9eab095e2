"""-m gpu: the decode products of csrc/dense_rows.hip that take the matrix instruction, against float64, and decode steps on them against `forward`."""
import pytest
import torch

from tests.test_dense_rows_gpu import close, normed
from tests.test_dense_rows_model_gpu import STEPS, decode
from tests.test_llama_prompt_gpu import model

pytestmark = pytest.mark.gpu


def to_stream(h, nw, dev):
    """An fp32 stream [M, width] in front of the norm of weight nw; rows past M poisoned."""
    from tgis_amd import native

    (M, width), dtype = h.shape, torch.bfloat16
    stream = native.RowsStream(M, width, dev)
    full = torch.full((64, width), float("nan"))
    for act, value in ((stream.h, h), (stream.hw, h * nw.float())):
        full[:M] = value
        act.buf.copy_(native.FragAct.from_rows(full.to(dtype)).buf[:act.buf.numel()])
    full[:M] = h
    stream.sums.copy_((full * full).view(64, -1, 4, 8).sum(-1).transpose(0, 1).reshape(-1))
    return stream


# K: one step of 64, fewer steps than waves, one more than a round of them, more than are asked for at once
@pytest.mark.parametrize("M", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("K,N", [(64, 64), (1088, 192), (2112, 2048), (6208, 64), (12288, 64)])
def test_residual(gpu_device, M, K, N):
    from tgis_amd import native

    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(M + K)
    x, w = torch.randn(M, K, generator=g).to(dtype), (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype)
    h, nw = torch.randn(M, N, generator=g), (torch.rand(N, generator=g) + 0.5).to(dtype)
    stream = to_stream(h, nw, gpu_device)
    native.dense_rows16_residual(native.FragAct.from_rows(x.to(gpu_device)), native.DenseWeight(w.to(gpu_device)), stream, nw.to(gpu_device))
    rows = lambda act: native.FragAct(act.buf, act.buf.numel() // N, N).to_rows().cpu().double()
    sums = stream.sums.cpu().view(-1, 64, 4).transpose(0, 1).reshape(64, -1).double()
    y = x.double() @ w.double().t()
    want = y.to(dtype).double() + h.to(dtype).double()
    u = 2.0 ** -8
    # the product's rounding may fall the other way (a step of it), and then the stream's
    slack = 2 * u * y.abs() + 1e-5
    assert ((rows(stream.h)[:M] - want).abs() <= slack + u * want.abs()).all()
    assert ((rows(stream.hw)[:M] - want * nw.double()).abs() <= slack * nw.double() + u * (want * nw.double()).abs()).all()
    assert ((sums[:M] - (want * want).view(M, -1, 8).sum(-1)).abs() <= (2 * slack * want.abs() + slack * slack).view(M, -1, 8).sum(-1) + 1e-5).all()
    assert bool(rows(stream.h)[M:].isnan().all()) and bool(rows(stream.hw)[M:].isnan().all()) and bool(sums[M:].isnan().all())


# ff, vocab: one unit, an odd number of units a workgroup, tiles that end within four columns
@pytest.mark.parametrize("M", [5, 16, 17, 48, 64])
@pytest.mark.parametrize("K,ff,vocab", [(64, 64, 50), (1088, 4160, 8203), (2048, 5632, 40), (2560, 64, 40), (3072, 64, 40), (4096, 128, 72)])
def test_norm_silu_and_head(gpu_device, M, K, ff, vocab):
    from tgis_amd import native

    dtype = torch.bfloat16
    if not native.dense_rows16_ok(M, K, True):
        with pytest.raises(RuntimeError, match="up to 64 rows"):
            native.dense_rows16_head(native.RowsStream(M, K, gpu_device), 1e-5, native.DenseWeight(torch.zeros(64, K, dtype=dtype, device=gpu_device)))
        return
    g = torch.Generator().manual_seed(M + K)
    h, nw = torch.randn(M, K, generator=g) * 3, (torch.rand(K, generator=g) + 0.5).to(dtype)
    wg, wh = ((torch.randn(n, K, generator=g) * K ** -0.5).to(dtype) for n in (2 * ff, vocab))
    dev = lambda t: t.to(gpu_device)
    x = (h * nw.float()).to(dtype).double() / torch.sqrt((h.double() ** 2).mean(-1, keepdim=True) + 1e-5)  # (what the launches multiply by)
    gate, up = (x @ wg.double().t()).split(ff, -1)
    act = native.dense_rows16_silu(to_stream(h, nw, gpu_device), 1e-5, native.DenseWeight(dev(wg), gate_up=True)).to_rows().cpu()
    close(act, torch.nn.functional.silu(gate) * up, K, dtype, 4)
    logits = native.dense_rows16_head(to_stream(h, nw, gpu_device), 1e-5, native.DenseWeight(dev(wh))).cpu()
    close(logits, x @ wh.double().t(), K, dtype, 0)


@pytest.mark.parametrize("M", [5, 31, 47, 64])
@pytest.mark.parametrize("K,H,Hkv,D,bias", [(2048, 32, 4, 64, False), (448, 3, 1, 32, True), (1984, 32, 16, 128, True)])
def test_norm_rope(gpu_device, M, K, H, Hkv, D, bias):
    """The same launch as norm + dense_gemm_rope: q, and the pages that it wrote, element for element within roundings."""
    from tgis_amd import native

    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(M + K)
    N, pages = (H + 2 * Hkv) * D, 3
    h, nw = torch.randn(M, K, generator=g) * 2, (torch.rand(K, generator=g) + 0.5).to(dtype)
    w, b = (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype), torch.randn(N, generator=g).to(dtype) if bias else None
    angle = torch.outer(torch.arange(100), 10000.0 ** (-torch.arange(0, D, 2) / D))
    cos, sin = angle.cos().to(dtype), angle.sin().to(dtype)
    pos, slots = torch.randint(0, 100, (M,), generator=g).int(), torch.randperm(pages * 32, generator=g)[:M].int()
    dev = lambda t: None if t is None else t.to(gpu_device)
    image = native.DenseWeight(dev(w), rope=(D, H + Hkv))
    pools = [torch.full((pages, Hkv, 32 * D), 7.0, dtype=dtype, device=gpu_device) for _ in range(4)]
    q = native.dense_rows16_rope(to_stream(h, nw, gpu_device), 1e-5, image, dev(b), dev(cos), dev(sin), dev(pos), dev(slots), pools[0], pools[1], H, Hkv, D)
    x = normed(h, nw, 1e-5, dtype).to(dtype)
    want = native.dense_gemm_rope(dev(x), image, dev(b), dev(cos), dev(sin), dev(pos), dev(slots), pools[2], pools[3], H, Hkv, D)
    # roundings of the result, of a pair of size up to 4 in front of its rotation, and of the operands in front of and behind the norm: K terms of u
    # 2 ** 0.5 / 3 ** 0.5 times K ** -0.5 each, six times their deviation
    u = 2.0 ** -8
    for got, ref in ((q[:, :H * D], want[:, :H * D]), (pools[0], pools[2]), (pools[1], pools[3])):
        got, ref = got.cpu().double(), ref.cpu().double()
        assert ((got - ref).abs() <= 2 * u * ref.abs() + 8 * u + 5 * u).all()


# two to four blocks of sixteen rows; the last two split the down projection
@pytest.mark.parametrize("rows,inner", [(3, 1024), (5, 1024), (17, 1024), (40, 4096), (56, 4096)])
def test_same_steps(gpu_device, monkeypatch, rows, inner):
    from tgis_amd import native
    from tgis_amd.models.custom_modeling.flash_llama_modeling import FlashLlamaForCausalLM, FlashLlamaModel

    calls, run = [], FlashLlamaModel.forward_rows16
    monkeypatch.setattr(FlashLlamaModel, "forward_rows16", lambda self, ids, *a: calls.append(ids.shape[0]) or run(self, ids, *a))
    lm, cfg = model(torch.bfloat16, intermediate_size=inner)
    got, pages = decode(lm, cfg.vocab_size, rows, True)
    assert calls == [{3: 4, 5: 8, 17: 24, 40: 40, 56: 56}[rows]] * 2  # a warm-up and a capture, with the rows of the bucket
    assert (native.load_library().tgis_dense_rows16_slab_bytes(rows, inner, cfg.hidden_size, 0) > 0) == (rows >= 40)
    for path in ("rows_path", "rows16_path"):
        monkeypatch.setattr(FlashLlamaForCausalLM, path, lambda self, n: False)
    lm, _ = model(torch.bfloat16, intermediate_size=inner)
    want, pages_want = decode(lm, cfg.vocab_size, rows, True)
    assert len(calls) == 2 and len(got) == len(want) == STEPS + 1 and torch.equal(got[0], want[0])
    # (as with fewer rows: sums in another order, which three layers carry on)
    step = 2.0 ** -8
    for a, b in zip(got[1:] + pages, want[1:] + pages_want):
        a, b = a.double(), b.double()
        assert a.shape == b.shape and float((a - b).norm() / b.norm()) < 4 * step


# (query tokens, keys) of each sequence: prompts of few and of many query tokens, some behind a prefix, up to two blocks of rows; decode steps, whole and behind key splits
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("H,Hkv,D", [(32, 4, 64), (8, 8, 128), (16, 1, 128), (6, 2, 64)])
@pytest.mark.parametrize("runs", [[(3, 3), (1, 40), (2, 2)], [(20, 20), (7, 100), (1, 1), (36, 36)], [(64, 64)], [(1, 700)] * 3, [(1, 5 + 9 * i) for i in range(40)]])
def test_attention_in_fragment_order(gpu_device, dtype, H, Hkv, D, runs):
    """The attention of the launches around it: the bits that the same launch leaves as rows."""
    from tgis_amd import native

    g = torch.Generator().manual_seed(len(runs) + D)
    B, T, longest, ctx = len(runs), sum(n for n, _ in runs), max(n for n, _ in runs), max(k for _, k in runs)
    per = (ctx + 31) // 32
    pools = [(torch.randn(B * per + 1, Hkv, 32 * D, generator=g) * 0.5).to(dtype).to(gpu_device) for _ in range(2)]
    table = torch.randperm(B * per, generator=g).int().view(B, per).to(gpu_device)
    q = (torch.randn(T, (H + 2) * D, generator=g) * 0.5).to(dtype).to(gpu_device)
    lens = torch.tensor([k for _, k in runs], dtype=torch.int32, device=gpu_device)
    cu = torch.tensor([0] + [n for n, _ in runs], device=gpu_device).cumsum(0).int()
    for splits in sorted({1, native.attn_num_splits(B, Hkv, H, longest, ctx)}):
        ws = native.Workspace(native.attn_workspace_bytes(B, H, Hkv, D, splits), gpu_device) if splits > 1 else None
        rows, frag = torch.empty((T, H * D), dtype=dtype, device=gpu_device), native.FragAct.empty(T, H * D, gpu_device, dtype)
        for out in (rows, frag):
            native.attn_paged(q, q.stride(0), *pools, table, lens, cu, out, B, H, Hkv, D, longest, ctx, D ** -0.5, splits, ws)
        assert torch.equal(frag.to_rows(), rows), splits


@pytest.mark.parametrize("lens", [[3], [30, 1, 33], [47], [64]])
def test_prompts(gpu_device, monkeypatch, lens):
    """Prompts of up to 64 rows: every token's logits and the pages, against the launches of `forward`."""
    from tests.test_llama_prompt_gpu import steps
    from tgis_amd.models.custom_modeling.flash_llama_modeling import FlashLlamaModel

    lm, cfg = model(torch.bfloat16)
    got = steps(lm, cfg.vocab_size, lens)
    monkeypatch.setattr(FlashLlamaModel, "serves_rows16", lambda self, rows: False)
    want = steps(lm, cfg.vocab_size, lens)
    assert len(got) == len(want) and not torch.equal(got[0], want[0])
    for a, b in zip(got, want):  # (as above)
        assert float((a.double() - b.double()).norm() / b.double().norm()) < 4 * 2.0 ** -8

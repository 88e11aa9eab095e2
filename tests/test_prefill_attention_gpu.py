"""-m gpu: prefill attention (csrc/attention_prefill.hip) over both page layouts: ragged runs, tile and page edges, group widths."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _pages(k, v, lens, layout, order):
    """k, v: per sequence [ctx, G, D] -> pools of 32-token pages dealt in `order`, and the block table.  What is past a context, the page that
    no sequence owns and the table entries past a sequence's pages (which name it) hold large values of either sign: a previous owner's."""
    G, D = k[0].shape[1:]
    per = [(n + 31) // 32 for n in lens]
    dice = torch.Generator().manual_seed(len(order))
    stale = lambda *shape: (60000 * (2 * torch.randint(0, 2, shape, generator=dice) - 1)).to(k[0].dtype)
    kp, vp = stale(sum(per) + 1, G, 32 * D), stale(sum(per) + 1, G, 32 * D)
    table = torch.full((len(lens), max(per) + 2), sum(per), dtype=torch.int32)
    it = iter(order)
    for b, n in enumerate(lens):
        for p in range(per[b]):
            page = next(it)
            table[b, p] = page
            kb, vb = stale(32, G, D), stale(32, G, D)
            m = min(32, n - 32 * p)
            kb[:m], vb[:m] = k[b][32 * p:32 * p + m], v[b][32 * p:32 * p + m]
            kb, vb = kb.transpose(0, 1), vb.transpose(0, 1)  # [G, 32, D]
            if layout == "rows":
                kp[page], vp[page] = kb.reshape(G, -1), vb.transpose(1, 2).reshape(G, -1)
            else:
                kp[page] = kb.reshape(G, 2, 16, D // 8, 8).transpose(2, 3).reshape(G, -1)
                tok = torch.arange(32)
                col = (tok % 16 // 4) * 8 + tok // 16 * 4 + tok % 4
                cols = torch.empty(G, 32, D, dtype=kp.dtype)
                cols[:, col] = vb
                vp[page] = cols.reshape(G, 4, 8, D).transpose(2, 3).reshape(G, -1)
    return kp, vp, table


def _oracle(q, k, v, scale):
    """q [n, H, D] are the last n positions of k, v [ctx, G, D]; float64."""
    n, H, D = q.shape
    ctx, G = k.shape[:2]
    kk, vv = (t.double().repeat_interleave(H // G, dim=1) for t in (k, v))
    s = torch.matmul(q.double().transpose(0, 1), kk.permute(1, 2, 0)) * scale
    hidden = torch.arange(ctx)[None, :] > (ctx - n + torch.arange(n))[:, None]
    p = torch.softmax(s.masked_fill(hidden, -math.inf), dim=-1)
    return torch.matmul(p, vv.transpose(0, 1)).transpose(0, 1), torch.matmul(p, vv.abs().transpose(0, 1)).transpose(0, 1)


# heads per kv head: one, not a power of two, one chunk of 16, more than a chunk; eight kv heads: tiles dealt to the XCDs by group
@pytest.mark.parametrize("H,G,D,dtype", [(8, 8, 128, torch.float16), (6, 2, 64, torch.bfloat16), (8, 1, 64, torch.float16), (16, 1, 128, torch.bfloat16),
                                         (20, 1, 128, torch.float16), (16, 8, 64, torch.bfloat16)])
@pytest.mark.parametrize("layout", ["fragments", "rows"])
@pytest.mark.parametrize("groups_per_wave", ["1", "2"])
@pytest.mark.parametrize("runs", [((65, 65),), ((17, 20), (64, 64), (70, 96)), ((127, 127), (1, 40)), ((128, 128), (129, 129), (31, 32)), ((33, 97), (300, 300), (2, 2)), ((161, 500),)])
def test_against_float64(gpu_device, H, G, D, dtype, layout, groups_per_wave, runs, monkeypatch):
    from tgis_amd import native

    monkeypatch.setenv("TGIS_PREFILL_CG", groups_per_wave)
    g = torch.Generator().manual_seed(H * D + len(runs))
    q = [torch.randn(n, H, D, generator=g).to(dtype) for n, _ in runs]
    k = [(2 * torch.randn(c, G, D, generator=g)).to(dtype) for _, c in runs]
    v = [torch.randn(c, G, D, generator=g).to(dtype) for _, c in runs]
    lens = [c for _, c in runs]
    order = torch.randperm(sum((c + 31) // 32 for c in lens), generator=g).tolist()
    kp, vp, table = (t.to(gpu_device) for t in _pages(k, v, lens, layout, order))
    ctx = torch.tensor(lens, dtype=torch.int32, device=gpu_device)
    cu = torch.tensor([0] + [n for n, _ in runs]).cumsum(0).int().to(gpu_device)
    wide = torch.full((int(cu[-1]), H * D + 16), 3.0, dtype=dtype)  # rows with a stride of their own
    wide[:, :H * D] = torch.cat([t.reshape(len(t), -1) for t in q])
    qd = wide.to(gpu_device)
    most = max(n for n, _ in runs)
    u = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    for scale in (D ** -0.5, -0.3 * D ** -0.5, 0.0):
        if layout == "rows":
            out = native.attn_varlen(qd[:, :H * D], kp, vp, table, ctx, cu, H, G, D, D, scale, max_q_len=most, max_ctx=max(lens))
        else:
            out = torch.empty(len(qd), H * D, dtype=dtype, device=gpu_device)
            native.attn_paged(qd, qd.stride(0), kp, vp, table, ctx, cu, out, len(lens), H, G, D, most, max(lens), scale, 1, None)
        got = out.view(-1, H, D).double().cpu()
        for b in range(len(runs)):
            want, size = _oracle(q[b], k[b], v[b], scale)
            # each probability is rounded to the type (and their sum with them), then the result; fp32 scores of up to ~60
            tol = (2 * u + 64 * D * 2.0 ** -24) * size + u * want.abs() + 1e-6
            err = (got[int(cu[b]):int(cu[b + 1])] - want).abs()
            assert (err <= tol).all(), (scale, b, float((err - tol).max()))


@pytest.mark.parametrize("groups_per_wave", ["1", "2"])
def test_large_and_missing_scores(gpu_device, groups_per_wave, monkeypatch):
    """Scores of every size: a maximum that moves late, keys whose scores are -inf, a row that sees one key."""
    from tgis_amd import native

    monkeypatch.setenv("TGIS_PREFILL_CG", groups_per_wave)
    H = G = 8
    n, D = 200, 64
    g = torch.Generator().manual_seed(5)
    q, v = torch.randn(n, H, D, generator=g).half(), torch.randn(n, G, D, generator=g).half()
    k = torch.randn(n, G, D, generator=g).half()
    q[:, :, 0] = 8.0
    k[100:, :, 0] = 300.0       # the late maximum
    k[150, :, 0] = -math.inf    # a key that no query sees
    kp, vp, table = (t.to(gpu_device) for t in _pages([k], [v], [n], "fragments", list(range(7))))
    out = torch.empty(n, H * D, dtype=torch.float16, device=gpu_device)
    cu = torch.tensor([0, n], dtype=torch.int32, device=gpu_device)
    native.attn_paged(q.view(n, -1).to(gpu_device), H * D, kp, vp, table, cu[1:].contiguous(), cu, out, 1, H, G, D, n, n, D ** -0.5, 1, None)
    want, size = _oracle(q, k, v, D ** -0.5)
    # scores of ~300: an fp32 sum's error moves a probability by up to 300 * 64 * 2 ** -24 of it
    tol = (3 * 2.0 ** -11 + 2 * 300 * D * 2.0 ** -24) * size + 1e-6
    assert ((out.view(n, H, D).double().cpu() - want).abs() <= tol).all()


# both head sizes, group widths, tile widths; positions from anywhere in the table; a row stride of its own
@pytest.mark.parametrize("H,G,D,dtype", [(8, 8, 128, torch.float16), (6, 2, 64, torch.bfloat16), (16, 1, 128, torch.bfloat16), (20, 1, 64, torch.float16)])
@pytest.mark.parametrize("groups_per_wave", ["1", "2"])
@pytest.mark.parametrize("lens", [[65], [129, 1, 70], [300, 33]])
def test_q_rotated_as_it_is_read(gpu_device, H, G, D, dtype, groups_per_wave, lens, monkeypatch):
    """The bits of a q that is rotated in front of the attention; the same cache pages."""
    from tgis_amd import native

    monkeypatch.setenv("TGIS_PREFILL_CG", groups_per_wave)
    g = torch.Generator().manual_seed(H + D + len(lens))
    T, row = sum(lens), (H + 2 * G) * D
    qkv = torch.randn(T, row + 8, generator=g).to(dtype).to(gpu_device)
    angle = torch.rand(700, D // 2, generator=g) * 6.28
    cos, sin = angle.cos().to(dtype).to(gpu_device), angle.sin().to(dtype).to(gpu_device)
    pos = torch.randint(0, 700, (T,), generator=g, dtype=torch.int32).to(gpu_device)
    cu = torch.tensor([0] + lens).cumsum(0).int().to(gpu_device)
    ctx = torch.tensor(lens, dtype=torch.int32, device=gpu_device)
    per = [(n + 31) // 32 for n in lens]
    table = torch.full((len(lens), max(per)), sum(per), dtype=torch.int32)
    for b, n in enumerate(per):
        table[b, :n] = torch.arange(sum(per[:b]), sum(per[:b]) + n)
    table = table.to(gpu_device)
    assert native.attn_rotates_q(H, G, D, max(lens)) == (max(lens) * min(16, 1 << (H // G - 1).bit_length()) > 64)

    def run(later):
        x = qkv.clone()
        kp, vp = (torch.zeros(sum(per) + 1, G, 32 * D, dtype=dtype, device=gpu_device) for _ in range(2))
        native.rope_kv_write_prefill(x, cos, sin, pos, cu, table, kp, vp, max(lens), H, G, D, D, rotate_q=not later)
        assert torch.equal(x, qkv) == later
        out = torch.empty(T, H * D, dtype=dtype, device=gpu_device)
        native.attn_paged(x, x.stride(0), kp, vp, table, ctx, cu, out, len(lens), H, G, D, max(lens), max(lens), D ** -0.5, 1, None,
                          **({"rope": (cos, sin, pos)} if later else {}))
        return out, kp, vp

    for a, b in zip(run(False), run(True)):
        assert torch.equal(a, b)


def test_q_not_rotated_for_short_queries(gpu_device):
    from tgis_amd import native

    q = torch.zeros(4, 8 * 64, dtype=torch.float16, device=gpu_device)
    one = torch.ones(1, dtype=torch.int32, device=gpu_device)
    pool, table = torch.zeros(1, 8, 32 * 64, dtype=torch.float16, device=gpu_device), torch.zeros(1, 1, dtype=torch.int32, device=gpu_device)
    tables = torch.zeros(8, 32, dtype=torch.float16, device=gpu_device)
    assert not native.attn_rotates_q(8, 8, 64, 4) and not native.attn_rotates_q(8, 8, 96, 400)
    with pytest.raises(RuntimeError, match="not for these heads"):
        native.attn_paged(q, q.stride(0), pool, pool, table, 4 * one, torch.tensor([0, 4], dtype=torch.int32, device=gpu_device), torch.empty_like(q), 1, 8, 8, 64,
                          4, 4, 0.1, 1, None, rope=(tables, tables, torch.zeros(4, dtype=torch.int32, device=gpu_device)))

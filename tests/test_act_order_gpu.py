"""-m gpu: act-order int4 linears whose operand is gathered in front of the GEMM (column gather, norm with a gather, re-ordered gate and
up columns)."""
import pytest
import torch

from oracle import ops_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,cols,K,offset", [
    (1, 8, 8, 0), (3, 72, 64, 0), (64, 4096, 4096, 0), (11, 11008, 11008, 0), (65, 352, 384, 0), (2500, 136, 136, 0),
    (5, 100, 128, 3),     # rows that are not 16-byte aligned
    (7, 32768, 128, 0),   # the longest row that is staged
    (7, 33000, 192, 0),   # longer: gathered from memory
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_gather_columns(gpu_device, M, cols, K, offset, dtype):
    from tgis_amd import native

    g = torch.Generator().manual_seed(M + cols)
    wide = torch.randn(M, cols + offset, generator=g).to(dtype).to(gpu_device)
    x = wide[:, offset:]
    perm = torch.randint(-1, cols, (K,), generator=g, dtype=torch.int32)
    perm[0], perm[-1] = cols - 1, -1
    want = torch.where(perm.to(gpu_device) >= 0, x[:, perm.clamp(min=0).long().to(gpu_device)], torch.zeros((), dtype=dtype, device=gpu_device))
    assert torch.equal(native.gather_columns(x, perm.to(gpu_device)), want)
    if M <= 64 and K % 64 == 0 and dtype == torch.float16:
        assert torch.equal(native.gather_columns(x, perm.to(gpu_device), frag=True).to_rows(), want)


@pytest.mark.parametrize("rows,hidden", [(1, 64), (11, 4096), (64, 2048), (65, 4096), (3, 16384)])
@pytest.mark.parametrize("partial", [False, True])
def test_norm_gathers(gpu_device, rows, hidden, partial):
    from tgis_amd import native

    g = torch.Generator().manual_seed(rows + hidden)
    x = torch.randn(rows, hidden, generator=g).half().to(gpu_device)
    if partial:
        slabs = torch.randn((rows + 31) // 32, 3, 32, hidden, generator=g).to(gpu_device)
        x = native.Partial(slabs, 3, hidden, rows, hidden, x[0].clone())
    res, w = torch.randn(rows, hidden, generator=g).half().to(gpu_device), torch.randn(hidden, generator=g).half().to(gpu_device)
    perm = torch.randperm(hidden, generator=g).to(torch.int32).to(gpu_device)
    y, r = native.rmsnorm_residual(x, res, w, 1e-5)
    got, got_r = native.rmsnorm_residual(x, res, w, 1e-5, perm=perm)
    assert torch.equal(got, y[:, perm.long()]) and torch.equal(got_r, r)
    if rows <= 64:
        assert torch.equal(native.rmsnorm_residual(x, res, w, 1e-5, frag=True, perm=perm)[0].to_rows(), y[:, perm.long()])


@pytest.mark.parametrize("M", [1, 32, 64, 65, 300, 3200])
@pytest.mark.parametrize("groupsize", [128, 32])
def test_linear_gathers_its_operand(gpu_device, M, groupsize):
    """Every path behind the gather (fragment order, row-major streaming, tall, dequantise) against the fp32 restatement, plain,
    deferred and with the SiLU * up epilogue over re-ordered columns."""
    from tgis_amd import native
    from tgis_amd.utils.layers import Ex4bitLinearV2, workspace

    K, I = 512, 384
    g = torch.Generator().manual_seed(M)
    up_t = ops_ref.make_gptq_tensors(K, 2 * I, groupsize, seed=1, act_order=True)
    down_t = ops_ref.make_gptq_tensors(I, 256, groupsize, seed=2, act_order=True)
    dev = lambda t: [torch.from_numpy(a).to(gpu_device) for a in t[:3]] + [torch.from_numpy(t[3])]
    # (the library path adds the bias to a product that is rounded already: another rounding, so no bias there)
    bias = (torch.randn(2 * I, generator=g) * (0.1 if M <= (3072 if groupsize == 128 else 256) else 0.0)).half()
    x = torch.randn(M, K, generator=g).half()
    w_up, w_down = (ops_ref.gptq_dequant(*t, groupsize).half().double() for t in (up_t, down_t))  # weights are rounded to f16 once
    y = x.double() @ w_up + bias.double()
    gate, up_ = y.half()[:, :I], y.half()[:, I:]
    act = (torch.nn.functional.silu(gate.float()).half().float() * up_.float()).half()
    want = act.double() @ w_down
    # One f16 rounding of an fp32 sum: 2 ** -11 of it, and the sum's own order (1e-6 of terms that add up to a few times the result).
    # Before the activation that order may turn a rounding the other way (2 ** -10 of gate or up, so 3 * 2 ** -10 of their product);
    # that happens to one value in some thousands: two in a row of 768 at the most reach one output.
    ulp = 2.0 ** -10
    tol_act = 3 * ulp * (gate.double() * up_.double()).abs() + 1e-5
    tol_out = ulp * want.abs() + 2 * float(tol_act.max()) * float(w_down.abs().max()) + 1e-5

    def close(got, want, tol):
        err = (got.double().cpu() - want).abs()
        assert (err <= tol).all(), float((err - tol).max())

    plain = Ex4bitLinearV2(*dev(up_t), bias.to(gpu_device), 4, groupsize)
    close(plain(x.to(gpu_device)), y, ulp * y.abs() + 1e-5)
    for fold in (False, True):
        up, down = Ex4bitLinearV2(*dev(up_t), bias.to(gpu_device), 4, groupsize), Ex4bitLinearV2(*dev(down_t), None, 4, groupsize)
        up.gate_up = True
        if fold:
            up.order_columns(torch.cat([down.perm, down.perm + I]))
            order = down.perm.long().cpu()
            down.take_ordered_input()
        h = up(x.to(gpu_device))
        close(h, act[:, order].double() if fold else act.double(), tol_act[:, order] if fold else tol_act)
        close(down(h), want, tol_out)
        if M <= 256:
            part = down(h, partial=True)
            rows = part.slabs.view(-1)[:(M + 31) // 32 * part.S * 32 * part.ld].view(-1, part.S, 32, part.ld).sum(1).reshape(-1, part.ld)
            close(rows[:M, :256], want, tol_out)


# unsplit blocks of four and eight waves, splits merged in the launch, the combine launch of multi-chunk blocks; more than 32 rows
@pytest.mark.parametrize("B,H,Hkv,D,ctx", [(11, 32, 32, 128, 200), (3, 8, 2, 64, 70), (2, 32, 32, 128, 1500), (2, 48, 1, 128, 1500), (40, 16, 4, 128, 90)])
def test_decode_attention_writes_columns_at_their_places(gpu_device, B, H, Hkv, D, ctx):
    from tgis_amd import native

    g = torch.Generator().manual_seed(B + ctx)
    W = (ctx + 31) // 32
    ctx_lens = torch.randint(1, ctx + 1, (B,), generator=g).int()
    ctx_lens[0] = ctx
    k_pool, v_pool = (torch.randn(B * W, Hkv, 32 * D, generator=g).half().to(gpu_device) for _ in range(2))
    q = torch.randn(B, H * D, generator=g).half().to(gpu_device)
    tables = torch.randperm(B * W, generator=g).int().view(B, W).to(gpu_device)
    places = torch.randperm(H * D, generator=g).int().to(gpu_device)
    splits = native.attn_num_splits(B, Hkv, H, 1, ctx)
    ws = native.Workspace(max(native.attn_workspace_bytes(B, H, Hkv, D, splits), 256), gpu_device)
    cu = torch.arange(B + 1, dtype=torch.int32, device=gpu_device)
    plain, placed = native.FragAct.empty(B, H * D, gpu_device), native.FragAct.empty(B, H * D, gpu_device)
    for out, cols in ((plain, None), (placed, places)):
        native.attn_paged(q, H * D, k_pool, v_pool, tables, ctx_lens.to(gpu_device), cu, out, B, H, Hkv, D, 1, ctx, D ** -0.5, splits, ws, out_cols=cols)
    assert torch.equal(placed.to_rows()[:, places.long()], plain.to_rows())

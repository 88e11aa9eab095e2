"""-m gpu: the dense decode GEMM that asks for its whole operand at once (csrc/dense_wide_body.h), at the edges of its rules."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bound(x, w, eps):
    """An fp32 sum of |x||w| over K in any order (2 ** -24 per addition, doubled), then one rounding to the output type."""
    return lambda want: eps * want.abs() + 2 * x.shape[1] * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t()) + 1e-6


# K: fewer steps than waves, a ragged last round of steps, one phase exactly, several phases; N: one ragged tile, several, a head (512+)
@pytest.mark.parametrize("K,N,M", [(*shape, M) for shape in [(64, 40), (448, 96), (576, 128), (2048, 2048), (2048, 100), (4160, 4128), (6144, 4096), (320, 16400),
                                                             (4160, 16400)] for M in (1, 2, 5, 15, 16, 17, 31, 32, 33, 47, 64, 65)]
                         + [(*shape, M) for shape in [(1280, 16384), (4160, 16384)] for M in (1, 4, 5, 16, 17)])
def test_finished(gpu_device, K, N, M):
    from tgis_amd import native

    g = torch.Generator().manual_seed(K + N + M)
    dtype = torch.bfloat16 if M & 1 else torch.float16
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    x, wt = torch.randn(M, K, generator=g).to(dtype), (torch.randn(N, K, generator=g) * 0.05).to(dtype)
    bias = (torch.randn(N, generator=g) * 0.1).to(dtype)
    w = native.DenseWeight(wt.to(gpu_device))
    ws = native.Workspace(w.workspace_bytes(M), gpu_device)
    wide = torch.full((M, K + 16), float("nan"), dtype=dtype)  # rows with a stride of their own
    wide[:, :K] = x
    xd = wide.to(gpu_device)[:, :K]
    plain = x.double() @ wt.double().t()
    want = plain + bias.double()
    bound = _bound(x, wt, eps)
    for out_f32 in (False, True):
        out = torch.full((M, N + 3), 7.0, dtype=torch.float32 if out_f32 else dtype, device=gpu_device)
        native.dense_gemm(xd, w, ws, bias=bias.to(gpu_device), out_f32=out_f32, out=out[:, :N])
        # an unsplit sum is rounded to the type before the bias, whatever it is stored as
        err = (out[:, :N].double().cpu() - want).abs()
        assert (err <= bound(want) + eps * plain.abs()).all(), (out_f32, float((err - bound(want)).max()))
        assert (out[:, N:] == 7.0).all()
    y = native.dense_gemm(xd, w, ws, act=4)
    want = torch.nn.functional.gelu(plain, approximate="tanh")
    assert ((y.double().cpu() - want).abs() <= eps * want.abs() + 1.13 * bound(plain) + 1e-3 * eps).all()  # |gelu'| <= 1.13


# (and the sizes between which the form with the whole operand in flight runs: 256 to 512 tiles, the last ones ragged)
@pytest.mark.parametrize("K,I", [(64, 16), (576, 48), (2048, 208), (2112, 64), (1152, 4080), (1152, 4096), (2048, 8192)])
@pytest.mark.parametrize("M", [32, 33, 47, 64])
def test_gate_up(gpu_device, K, I, M):
    from tgis_amd import native

    g = torch.Generator().manual_seed(K + I + M)
    x, wt = torch.randn(M, K, generator=g).bfloat16(), (torch.randn(2 * I, K, generator=g) * 0.05).bfloat16()
    w = native.DenseWeight(wt.to(gpu_device), gate_up=True)
    ws = native.Workspace(w.workspace_bytes(M), gpu_device)
    out = torch.full((M, I + 5), 7.0, dtype=torch.bfloat16, device=gpu_device)
    native.dense_gemm(x.to(gpu_device), w, ws, act=2, out=out[:, :I])
    y = x.double() @ wt.double().t()
    tol = _bound(x, wt, 2.0 ** -8)(y)
    gate, up = y[:, :I], y[:, I:]
    silu = torch.nn.functional.silu(gate)
    # |silu'| <= 1.1; silu is rounded, then the product
    bound = 1.1 * tol[:, :I] * up.abs() + silu.abs() * tol[:, I:] + 2 * 2.0 ** -8 * (silu * up).abs() + 1e-4
    assert ((out[:, :I].double().cpu() - silu * up).abs() <= bound).all()
    assert (out[:, I:] == 7.0).all()


@pytest.mark.parametrize("K,H,Hkv,D,M", [(*shape, M) for shape in [(1088, 48, 8, 32), (2048, 32, 4, 64), (2112, 16, 4, 128), (4096, 16, 8, 64),
                                                                   (4160, 16, 8, 64)] for M in (1, 2, 15, 16, 17)]
                         + [(*shape, M) for shape in [(64, 48, 8, 32), (1088, 48, 8, 32), (2048, 32, 4, 64)] for M in (33, 47, 63, 64)]
                         + [(*shape, M) for shape in [(1024, 32, 8, 64), (3072, 24, 8, 128)] for M in (8, 9, 16)])
def test_rope(gpu_device, K, H, Hkv, D, M):
    """Against the plain image's GEMM followed by the rotary launch: the two differ by the order of their fp32 sums alone."""
    from tgis_amd import native

    g = torch.Generator().manual_seed(K + M)
    N = (H + 2 * Hkv) * D
    x, wt = torch.randn(M, K, generator=g).bfloat16().to(gpu_device), (torch.randn(N, K, generator=g) * 0.05).bfloat16().to(gpu_device)
    bias = (torch.randn(N, generator=g) * 0.1).bfloat16().to(gpu_device)
    w, wr = native.DenseWeight(wt), native.DenseWeight(wt, rope=(D, H + Hkv))
    assert native.rope_gemm_ok(M, wr, D)
    ws = native.Workspace(w.workspace_bytes(M), gpu_device)
    cos, sin = (torch.randn(80, D // 2, generator=g).clamp(-1, 1).bfloat16().to(gpu_device) for _ in range(2))
    pos = torch.randint(0, 80, (M,), generator=g).int().to(gpu_device)
    slots = torch.randperm(8 * 32, generator=g)[:M].int().to(gpu_device)
    pools = [torch.zeros((8, Hkv, 32 * D), dtype=torch.bfloat16, device=gpu_device) for _ in range(4)]
    q0 = native.rope_kv_write(native.dense_gemm(x, w, ws, bias=bias), cos, sin, pos, slots, pools[0], pools[1], H, Hkv, D, D)
    q1 = native.dense_gemm_rope(x, wr, bias, cos, sin, pos, slots, pools[2], pools[3], H, Hkv, D)
    # one flipped rounding of either half of a pair (2 ** -8), of each product and of the rotated sum
    scale = float((x.float().abs() @ wt.float().abs().t()).max()) * K * 2.0 ** -23 + 4 * 2.0 ** -8 * float((x.float() @ wt.float().t()).abs().max() + 0.5)
    for a, b in ((q0[:, :H * D], q1[:, :H * D]), (pools[0], pools[2]), (pools[1], pools[3])):
        diff = (a.float() - b.float()).abs()
        assert float(diff.max()) <= scale and float((diff > 0).float().mean()) < 0.05


# groups: one, and several with a last one that is whole / one ragged tile / several tiles; the last has more tiles than there are CUs, whose phases of x are shorter
@pytest.mark.parametrize("K,n_group,N,G", [(64, 32, 20, 1), (448, 96, 288, 3), (576, 64, 150, 3), (2048, 512, 2048 + 64, 5), (4160, 64, 4 * 64 + 33, 5), (2112, 2080, 4 * 2080 + 33, 5)])
@pytest.mark.parametrize("M", [1, 8, 15, 16, 17, 32, 33, 64])
def test_groups(gpu_device, K, n_group, N, G, M):
    from tgis_amd import native

    g = torch.Generator().manual_seed(K + N + M)
    dtype = torch.bfloat16 if M & 1 else torch.float16
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    x, wt = torch.randn(G, M, K, generator=g).to(dtype), (torch.randn(N, K, generator=g) * 0.05).to(dtype)
    w = native.DenseWeight(wt.to(gpu_device))
    out = torch.full((G, M, n_group + 8), 7.0, dtype=dtype, device=gpu_device)
    native.dense_gemm_groups(x.to(gpu_device), w, n_group, out)
    for i in range(G):
        rows = wt[i * n_group:(i + 1) * n_group]
        want = x[i].double() @ rows.double().t()
        assert ((out[i, :, :len(rows)].double().cpu() - want).abs() <= _bound(x[i], rows, eps)(want)).all(), i
        assert (out[i, :, len(rows):] == 7.0).all()
        # a group as a weight of its own
        part = w.rows(i * n_group, len(rows))
        y = native.dense_gemm(x[i].to(gpu_device), part, native.Workspace(part.workspace_bytes(M), gpu_device))
        assert ((y.double().cpu() - want).abs() <= _bound(x[i], rows, eps)(want)).all(), i


def test_groups_refuses(gpu_device):
    from tgis_amd import native

    w = native.DenseWeight(torch.zeros(96, 72, dtype=torch.float16, device=gpu_device))
    with pytest.raises(RuntimeError, match="multiple of 64"):
        native.dense_gemm_groups(torch.zeros(3, 4, 72, dtype=torch.float16, device=gpu_device), w, 32, torch.zeros(3, 4, 32, dtype=torch.float16, device=gpu_device))

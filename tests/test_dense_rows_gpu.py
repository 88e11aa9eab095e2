"""-m gpu: the decode products of a few rows that norm their operand and add to the residual stream (csrc/dense_rows.hip), against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def normed(h, w, eps, dtype):
    h = h.double()
    return (h / torch.sqrt((h * h).mean(-1, keepdim=True) + eps) * w.double()).to(dtype).double()


def close(got, want, K, dtype, roundings, turned=0.0):
    """fp32 sums of K terms of size K ** -0.5 (2e-6), `roundings` roundings of the result to the model dtype, and up to two elements of the normed
    operand (of size up to 4: a step of 4 u) that round the other way than float64's, each times a weight of up to four times K ** -0.5;
    turned: the size of a pair whose two halves may each round the other way before they are rotated into each other."""
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    err = (got.double() - want).abs()
    tol = roundings * u * want.abs() + 2 * 4 * u * 4 * K ** -0.5 + 2e-6 + 2 * u * turned
    assert (err <= tol).all(), float((err / tol).max())


def refused(dev, M, K, dtype, norm):
    """More rows than fit LDS, or than are served at this width: an error in front of any launch, and outputs as they were."""
    from tgis_amd import native

    N, stream = 64, torch.full((M, K if norm else 64), 3.0, device=dev)
    image, w = native.DenseWeight(torch.zeros(N, K, dtype=dtype, device=dev)), torch.ones(K, dtype=dtype, device=dev)
    with pytest.raises(RuntimeError, match="up to 4 rows"):
        if norm:
            native.dense_rows_head(stream, w, 1e-5, image)
        else:
            native.dense_rows_residual(torch.ones(M, K, dtype=dtype, device=dev), image, stream)
    if norm:
        with pytest.raises(RuntimeError, match="up to 4 rows"):
            native.dense_rows_silu(stream, w, 1e-5, native.DenseWeight(torch.zeros(N, K, dtype=dtype, device=dev), gate_up=True))
    assert bool((stream == 3.0).all())


# K: one step of 64, fewer steps than waves, every depth at its edge and past it; N: not a multiple of a tile, of a workgroup's columns
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("K,N", [(64, 40), (448, 72), (2048, 2048), (2112, 96), (4096, 32), (4160, 100), (5632, 256), (6208, 40), (12288, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_residual(gpu_device, M, K, N, dtype):
    from tgis_amd import native

    if not native.dense_rows_ok(M, K, False):
        return refused(gpu_device, M, K, dtype, norm=False)
    g = torch.Generator().manual_seed(M + K)
    x, w = torch.randn(M, K + 8, generator=g).to(dtype), (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype)
    h = torch.randn(M, N, generator=g)
    got = h.to(gpu_device)
    native.dense_rows_residual(x.to(gpu_device)[:, :K], native.DenseWeight(w.to(gpu_device)), got)
    y = x[:, :K].double() @ w.double().t()
    want = y.to(dtype).double() + h.to(dtype).double()
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    # the product's rounding may fall the other way; the sum itself is in fp32
    assert ((got.cpu().double() - want).abs() <= 2 * u * y.abs() + 1e-5).all()


@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("K,ff,vocab", [(64, 16, 50), (2048, 528, 1000), (2112, 64, 72), (3072, 16, 40), (3136, 48, 40), (4096, 48, 40)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_norm_silu_and_head(gpu_device, M, K, ff, vocab, dtype):
    from tgis_amd import native

    if not native.dense_rows_ok(M, K, True):
        return refused(gpu_device, M, K, dtype, norm=True)
    g = torch.Generator().manual_seed(M + K)
    h, nw = torch.randn(M, K, generator=g) * 3, (torch.rand(K, generator=g) + 0.5).to(dtype)
    wg, wh = ((torch.randn(n, K, generator=g) * K ** -0.5).to(dtype) for n in (2 * ff, vocab))
    dev = lambda t: t.to(gpu_device)
    x = normed(h, nw, 1e-5, dtype)
    gate, up = (x @ wg.double().t()).split(ff, -1)
    act = native.dense_rows_silu(dev(h), dev(nw), 1e-5, native.DenseWeight(dev(wg), gate_up=True)).cpu()
    close(act, torch.nn.functional.silu(gate) * up, K, dtype, 4)
    logits = native.dense_rows_head(dev(h), dev(nw), 1e-5, native.DenseWeight(dev(wh))).cpu()
    close(logits, x @ wh.double().t(), K, dtype, 0)


@pytest.mark.parametrize("M", [1, 2, 4])
@pytest.mark.parametrize("K,H,Hkv,D,bias", [(2048, 32, 4, 64, False), (448, 3, 1, 32, True), (2176, 4, 4, 128, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_norm_rope(gpu_device, M, K, H, Hkv, D, bias, dtype):
    """The same launch as norm + dense_gemm_rope: q, and the pages that it wrote, element for element within a rounding."""
    from tgis_amd import native

    if not native.dense_rows_ok(M, K, True):
        return refused(gpu_device, M, K, dtype, norm=True)
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
    q = native.dense_rows_rope(dev(h), dev(nw), 1e-5, image, dev(b), dev(cos), dev(sin), dev(pos), dev(slots), pools[0], pools[1], H, Hkv, D)
    x = normed(h, nw, 1e-5, dtype).to(dtype)
    want = native.dense_gemm_rope(dev(x), image, dev(b), dev(cos), dev(sin), dev(pos), dev(slots), pools[2], pools[3], H, Hkv, D)
    close(q[:, :H * D].cpu(), want[:, :H * D].cpu().double(), K, dtype, 2, 4.0)
    for got, ref in ((pools[0], pools[2]), (pools[1], pools[3])):
        close(got.cpu(), ref.cpu().double(), K, dtype, 2, 4.0)

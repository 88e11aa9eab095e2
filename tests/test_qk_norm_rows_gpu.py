"""-m gpu: the norm of q and k and the cache write of long steps (csrc/attn_varlen.hip, qk_norm_rows_kernel) against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# lanes per head 8, 16 and 32, full and part used; pad 8: a row stride that is longer than the row; pad 4: rows that are not 16-byte groups
@pytest.mark.parametrize("H,G,dk,dv,pad", [(4, 2, 64, 64, 0), (3, 1, 8, 16, 8), (6, 3, 72, 64, 0), (5, 5, 128, 128, 8), (2, 1, 200, 64, 0), (2, 2, 256, 256, 8),
                                           (4, 2, 64, 64, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_long_step(gpu_device, H, G, dk, dv, pad, dtype):
    from tgis_amd import native

    T, eps, PAGE = 517, 1e-5, 32
    g = torch.Generator().manual_seed(dk + pad)
    qkv = torch.randn(T, (H + G) * dk + G * dv + pad, generator=g).to(dtype)
    qw, kw = torch.rand(dk, generator=g) + 0.5, torch.rand(dk, generator=g) + 0.5
    pages = T // PAGE + 3
    slots, pos = torch.randperm(pages * PAGE, generator=g)[:T].int(), torch.randint(0, 5000, (T,), generator=g).int()
    dev = lambda t: t.to(gpu_device)
    buf = dev(qkv)
    rows = buf[:, :buf.shape[1] - pad] if pad else buf
    k_pool = torch.full((pages, G, PAGE, dk), 7.0, dtype=dtype, device=gpu_device)
    v_pool = torch.full((pages, G, dv, PAGE), 7.0, dtype=dtype, device=gpu_device)
    native.qk_norm_kv_write(rows, dev(pos), dev(slots), dev(qw), dev(kw), eps, 0.1, 1024, None, None, k_pool, v_pool, H, G, dk, dv)
    x = qkv[:, :(H + G) * dk].double().view(T, H + G, dk)
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    gain = 1 + 0.1 * torch.log((pos.double() + 1).div(1024, rounding_mode="floor") + 1)
    q, k = y[:, :H] * qw.double() * gain[:, None, None], y[:, H:] * kw.double()
    v = qkv[:, (H + G) * dk:(H + G) * dk + G * dv].view(T, G, dv)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11  # one rounding of the result; fp32 sums of up to 256 squares are 1e-6 at the most
    got = buf.cpu()
    # (+ half of float16's smallest step, 2 ** -24, which values below 2 ** -14 are rounded to)
    close = lambda a, b: bool(((a.double() - b).abs() <= (u + 2e-6) * b.abs() + 2.0 ** -25).all())
    assert close(got[:, :H * dk].view(T, H, dk), q)
    assert torch.equal(got[:, H * dk:], qkv[:, H * dk:])  # k and v stay in the projection's output as they were
    at = (slots.long() // PAGE, slots.long() % PAGE)
    assert close(k_pool.cpu()[at[0], :, at[1]], k) and torch.equal(v_pool.cpu()[at[0], :, :, at[1]], v)
    unused = torch.ones(pages * PAGE, dtype=torch.bool)
    unused[slots.long()] = False
    assert (k_pool.cpu().transpose(1, 2).reshape(pages * PAGE, -1)[unused] == 7).all()


# heads of one and two halves of a wave's channels; rows on both sides of a slab block; values of one block and more
@pytest.mark.parametrize("T,S,H,G,dk,dv", [(1, 1, 4, 2, 64, 64), (24, 4, 32, 4, 64, 64), (33, 3, 3, 1, 130, 18), (70, 8, 6, 3, 72, 512), (256, 2, 5, 5, 256, 40)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("blend", [False, True])
def test_of_partial_sums(gpu_device, T, S, H, G, dk, dv, dtype, blend):
    """The projection left as partial sums: the bits of their sum, added in order and rounded, and then normed and written."""
    from tgis_amd import native

    N, PAGE = (H + G) * dk + G * dv, 32
    g = torch.Generator().manual_seed(T + S)
    ld, blocks = -N // 32 * -32, -T // 32 * -1
    slabs = torch.randn(blocks, S, 32, ld, generator=g).to(gpu_device)
    part = native.Partial(slabs, S, ld, T, N, None)
    part.dtype = dtype
    total = slabs[:, 0]
    for s in range(1, S):
        total = total + slabs[:, s]
    whole = total.reshape(-1, ld)[:T, :N].to(dtype).contiguous()
    qw, kw = (torch.rand(dk, generator=g) + 0.5).to(gpu_device), (torch.rand(dk, generator=g) + 0.5).to(gpu_device)
    pages = T // PAGE + 3
    slots, pos = torch.randperm(pages * PAGE, generator=g)[:T].int().to(gpu_device), torch.randint(0, 5000, (T,), generator=g).int().to(gpu_device)
    first = torch.randn(T, G * dv, generator=g).to(dtype).to(gpu_device) if blend else None
    lam = torch.tensor([0.375], device=gpu_device) if blend else None

    def run(x):
        k_pool = torch.full((pages, G, PAGE, dk), 7.0, dtype=dtype, device=gpu_device)
        v_pool = torch.full((pages, G, dv, PAGE), 7.0, dtype=dtype, device=gpu_device)
        out = native.qk_norm_kv_write(x, pos, slots, qw, kw, 1e-5, 0.1, 1024, first, lam, k_pool, v_pool, H, G, dk, dv)
        return out, k_pool, v_pool

    assert all(torch.equal(a, b) for a, b in zip(run(part), run(whole)))

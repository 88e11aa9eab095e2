"""-m gpu: the int4 GEMM at prefill sizes (csrc/gptq_tall.hip): every tile shape, unsplit tiles, tiles split over k, ragged edges."""
import pytest
import torch

from oracle import ops_ref

pytestmark = pytest.mark.gpu


# K: one step, fewer and more steps than the ring of buffers, a whole number of rings; N: one tile, ragged and several column blocks; the last
# sizes have more tiles than the 256 of a whole round, so that a split plan launches whole tiles and split ones behind them: of the smallest tile, of each
@pytest.mark.parametrize("K,N,groupsize,M", [(*shape, M) for shape in [(64, 32, 64), (192, 288, 64), (320, 512, 64), (1024, 1120, 128), (1152, 96, 1152)]
                                             for M in (129, 161, 300)] + [(320, 4128, 64, 700), (320, 4128, 64, 2100)])
@pytest.mark.parametrize("act", [0, 2])
def test_every_plan(gpu_device, K, N, groupsize, M, act, monkeypatch):
    from tgis_amd import native

    qw, qz, sc, gi = ops_ref.make_gptq_tensors(K, N, groupsize, seed=K + N)
    w = native.GptqWeight(*(torch.from_numpy(t).to(gpu_device) for t in (qw, qz, sc)), torch.from_numpy(gi), 4, groupsize, gate_up=act == 2)
    g = torch.Generator().manual_seed(M)
    x, bias = torch.randn(M, K, generator=g).half(), (torch.randn(N, generator=g) * 0.1).half()
    ws = native.Workspace(64 << 20, gpu_device)
    y = x.double() @ ops_ref.gptq_dequant(qw, qz, sc, gi, groupsize).half().double() + bias.double()
    # a rounding of an fp32 sum to f16 (2 ** -11 of it) plus the sum's own order; before the activation that order may turn the
    # rounding of gate or up the other way (2 ** -10 of either, so 3 * 2 ** -10 of the product)
    ulp = 2.0 ** -10
    want, tol = y, ulp * y.abs() + 1e-5
    if act == 2:
        gate, up = y.half()[:, :N // 2], y.half()[:, N // 2:]
        want = (torch.nn.functional.silu(gate.float()).half().float() * up.float()).half().double()
        tol = 3 * ulp * (gate.double() * up.double()).abs() + 1e-5
    cols = want.shape[1]
    # (the last split needs a k64-step of its own)
    steps = K // 64
    plans = [None] + [f"{b},{t},{p}" for b in (2, 3, 4) for t in (1, 2) for p in (1, 2, 5) if (p - 1) * -(-steps // p) < steps]
    for plan in plans:
        if plan is None:
            monkeypatch.delenv("TGIS_TALL_PLAN", raising=False)
        else:
            monkeypatch.setenv("TGIS_TALL_PLAN", plan)
        for pad in (0, 3):  # rows of the output that take 16-byte stores, and rows that do not
            wide = torch.full((M, cols + pad), 7.0, dtype=torch.float16, device=gpu_device)
            native.gptq_gemm(x.to(gpu_device), w, ws, bias=bias.to(gpu_device), act=act, out=wide[:, :cols])
            err = (wide[:, :cols].double().cpu() - want).abs()
            assert (err <= tol).all(), (plan, pad, float((err - tol).max()))
            assert (wide[:, cols:] == 7.0).all()


# behind a whole turn of the ring of four buffers: one, two and three steps, and none; behind none, and in the parts of a split
# (the larger product has more than 256 tiles of each size, which take the other shape of the matrix instruction)
@pytest.mark.parametrize("steps,S", [(1, 1), (2, 1), (3, 1), (4, 1), (5, 1), (6, 1), (7, 1), (11, 1), (14, 2)])
@pytest.mark.parametrize("N,M", [(288, 290), (4128, 2100)])
def test_tails_of_the_ring(gpu_device, steps, S, N, M, monkeypatch):
    from tgis_amd import native

    K = 64 * steps
    qw, qz, sc, gi = ops_ref.make_gptq_tensors(K, N, 64, seed=steps)
    w = native.GptqWeight(*(torch.from_numpy(t).to(gpu_device) for t in (qw, qz, sc)), torch.from_numpy(gi), 4, 64)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(steps)).half()
    want = x.double() @ ops_ref.gptq_dequant(qw, qz, sc, gi, 64).half().double()
    ws = native.Workspace(64 << 20, gpu_device)
    for tile in ("2,1", "2,2", "3,1", "3,2", "4,1", "4,2"):
        monkeypatch.setenv("TGIS_TALL_PLAN", f"{tile},{S}")
        got = native.gptq_gemm(x.to(gpu_device), w, ws).double().cpu()
        assert ((got - want).abs() <= 2.0 ** -10 * want.abs() + 1e-5).all(), tile  # (as in test_every_plan)


def test_linear_takes_whole_sums_past_128_rows(gpu_device):
    """129 .. 256 rows: the linear returns a finished tensor where 64-row passes left slabs to the consumer."""
    from tgis_amd import native
    from tgis_amd.utils.layers import Ex4bitLinearV2

    qw, qz, sc, gi = ops_ref.make_gptq_tensors(256, 128, 128, seed=3)
    lin = Ex4bitLinearV2(*(torch.from_numpy(t).to(gpu_device) for t in (qw, qz, sc)), torch.from_numpy(gi), None, 4, 128)
    for M in (128, 129, 256):
        x = torch.randn(M, 256, generator=torch.Generator().manual_seed(M)).half()
        got = lin(x.to(gpu_device), partial=True)
        assert isinstance(got, native.Partial) == (M == 128)
        if M > 128:
            want = x.double() @ ops_ref.gptq_dequant(qw, qz, sc, gi, 128).half().double()
            assert ((got.double().cpu() - want).abs() <= 2.0 ** -10 * want.abs() + 1e-5).all()


def test_deferred_sums_at_any_row_count(gpu_device):
    """The C entry's slabs past the rows that the linears defer."""
    import ctypes

    from tgis_amd import native

    K, N, M = 512, 224, 300
    qw, qz, sc, gi = ops_ref.make_gptq_tensors(K, N, 128, seed=5)
    w = native.GptqWeight(*(torch.from_numpy(t).to(gpu_device) for t in (qw, qz, sc)), torch.from_numpy(gi), 4, 128)
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half().to(gpu_device)
    lib = native.load_library()
    slabs = torch.full((lib.tgis_gptq_gemm_partial_bytes(M, K, N) // 4,), float("nan"), device=gpu_device)
    S, ld = ctypes.c_int(), ctypes.c_int64()
    assert lib.tgis_gptq_gemm_f16_partial(x.data_ptr(), K, w.image.data_ptr(), None, M, K, N, w.groups, 0, slabs.data_ptr(), slabs.numel() * 4,
                                          ctypes.byref(S), ctypes.byref(ld), torch.cuda.current_stream().cuda_stream) == 0
    units = (M + 31) // 32
    got = slabs[:units * S.value * 32 * ld.value].view(units, S.value, 32, ld.value).sum(1).reshape(-1, ld.value)[:M, :N].double().cpu()
    want = x.double().cpu() @ ops_ref.gptq_dequant(qw, qz, sc, gi, 128).half().double()
    assert ((got - want).abs() <= 1e-5 * (1 + want.abs())).all()


# K: half a k64-step, whole ones, a ragged last; N: one tile, a block of eight and ragged ones; groups shorter than a step
# (and a matrix on each side of the 768 blocks of eight tiles)
@pytest.mark.parametrize("K,N,groupsize", [(32, 32, 32), (96, 288, 32), (256, 256, 128), (320, 544, 64), (160, 1024, 160), (512, 64, 128), (544, 96, 32), (2016, 6112, 32),
                                           (2048, 5888, 128)])
@pytest.mark.parametrize("image", ["plain", "gate_up", "rope"])
def test_dequant_bits(gpu_device, K, N, groupsize, image):
    """The image back to [K, N]: the bits of the reference formula, from each column order, into aligned and unaligned memory; and to [N, K]."""
    from tgis_amd import native

    qw, qz, sc, gi = ops_ref.make_gptq_tensors(K, N, groupsize, seed=K + N)
    kind = {"gate_up": {"gate_up": True}, "rope": {"rope": (32, max(1, N // 32 - 1))}}.get(image, {})
    w = native.GptqWeight(*(torch.from_numpy(t).to(gpu_device) for t in (qw, qz, sc)), torch.from_numpy(gi), 4, groupsize, **kind)
    want = ops_ref.gptq_dequant(qw, qz, sc, gi, groupsize).half()
    assert torch.equal(native.gptq_dequant(w).cpu(), want)
    buf = torch.full((K * N + 16,), 7.0, dtype=torch.float16, device=gpu_device)
    assert torch.equal(native.gptq_dequant_t(w, buf[8:-8].view(N, K)).t().cpu(), want) and (buf[:8] == 7.0).all() and (buf[-8:] == 7.0).all()
    buf = torch.full((K * N + 2,), 7.0, dtype=torch.float16, device=gpu_device)
    lib = native.load_library()
    assert lib.tgis_gptq_dequant_f16(w.image.data_ptr(), buf.data_ptr() + 2, K, N, w.groups, w.flags, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(buf[1:-1].view(K, N).cpu(), want) and buf[0] == 7.0 and buf[-1] == 7.0

"""-m gpu: the int4 SiLU * up GEMM of up to 64 rows whose blocks are pairs of waves on eight tiles (csrc/gptq_wide_body.h), against float64."""
import pytest
import torch

from oracle import ops_ref

pytestmark = pytest.mark.gpu
U = 2.0 ** -11


# N: a last block of four tiles (one group), and of five; K: fewer steps than k-parts, shares that differ
@pytest.mark.parametrize("M", [17, 33, 48, 64])
@pytest.mark.parametrize("K,N,frag", [(128, 32896, True), (448, 32928, False)])
def test_pairs(gpu_device, M, K, N, frag):
    from tgis_amd import native

    qw, qz, sc, gi = ops_ref.make_gptq_tensors(K, N, 64, seed=K, w_std=K ** -0.5)
    w = native.GptqWeight(*(torch.from_numpy(t).to(gpu_device) for t in (qw, qz, sc)), None, 4, 64, gate_up=True)
    g = torch.Generator().manual_seed(M)
    x, bias = torch.randn(M, K, generator=g).half(), (torch.randn(N, generator=g) * 0.1).half()
    y = x.double() @ ops_ref.gptq_dequant(qw, qz, sc, gi, 64).half().double() + bias.double()
    gate, up = y.split(N // 2, -1)
    s = torch.nn.functional.silu(gate)
    act = native.FragAct.from_rows(x.to(gpu_device))
    got = native.gptq_gemm(act, w, native.Workspace(64 << 20, gpu_device), bias=bias.to(gpu_device), act=2, out_frag=frag)
    got = (got.to_rows() if frag else got).cpu().double()
    # roundings of gate, SiLU(gate) (whose slope is below 1.1), up and the result, half a step each, and fp32 sums of K terms of size K ** -0.5
    assert ((got - s * up).abs() <= U * (4 * (s * up).abs() + 1.1 * (gate * up).abs()) + 1e-5 * (1 + up.abs() + s.abs())).all()

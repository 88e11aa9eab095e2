"""GELU in its tanh form: one function of the rounded value, wherever it is applied (csrc/common.h)."""
import pytest
import torch

from tgis_amd import native

pytestmark = pytest.mark.gpu


def _gelu_tanh(x):
    u = 0.7978845608028654 * (x + 0.044715 * x ** 3)
    return x / (1.0 + torch.exp(-2.0 * u))  # (1 + tanh u would lose the digits of its tail in 64 bits too)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_every_finite_value(gpu_device, dtype):
    x = torch.arange(-2 ** 15, 2 ** 15, dtype=torch.int32).to(torch.int16).view(dtype)
    x = x[torch.isfinite(x)].contiguous()
    got, want = native.gelu(x.to(gpu_device), True).cpu().double(), _gelu_tanh(x.double())
    unit, least = (2.0 ** -11, 2.0 ** -24) if dtype == torch.float16 else (2.0 ** -8, 2.0 ** -133)
    # one rounding of the type; in front of it the exponential of a = 2 u log2 e, whose own roundings weigh a times as much, and the reciprocal.  Past
    # a = 126 the denominator has no reciprocal among the normal numbers: up to |x| 2 ** -126, |x| about 10, may be lost.
    a = (2.302208198 * x.double() * (1 + 0.044715 * x.double() ** 2)).abs().clamp(max=128)
    bound = want.abs() * (unit + (8 + 4 * a) * 2.0 ** -24) + least / 2 + 11 * 2.0 ** -126
    assert bool(torch.isfinite(got).all())
    worst = (got - want).abs() - bound
    assert bool((worst <= 0).all()), (x[worst.argmax()], got[worst.argmax()], want[worst.argmax()])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N", [(1, 256, 72), (7, 512, 256), (32, 4096, 256), (33, 1024, 1160), (64, 2048, 2048), (200, 2048, 256)])
def test_gated_lookup_in_the_gemm_is_the_same_as_behind_it(gpu_device, dtype, M, K, N):
    """Unsplit plans and split ones, whose sums the reduce finishes; gates from far below zero to above; ids outside of the table."""
    g = torch.Generator().manual_seed(M + K + N)
    x = torch.randn(M, K, generator=g).to(dtype).to(gpu_device)
    w = native.DenseWeight((torch.randn(N, K, generator=g) * 3 * K ** -0.5).to(dtype).to(gpu_device))
    table = torch.randn(50, N + 24, generator=g).to(dtype).to(gpu_device)
    ids = torch.randint(-1, 51, (M,), generator=g).to(gpu_device)
    ws = native.Workspace(w.workspace_bytes(M), gpu_device)
    gate = native.dense_gemm(x, w, ws)
    one = native.dense_gemm_gelu_lookup(x, w, ws, ids, table, 16)
    assert torch.equal(one, native.gelu_gated_lookup(gate, ids, table, 16))
    assert float(gate.min()) < -3 and bool((one[(ids < 0) | (ids >= 50)] == 0).all())


def test_gated_lookup_in_32_bits(gpu_device):
    """Against 64 bits: the exponential's argument a carries a times its own roundings into a value that is 2 ** -a of the gate below zero."""
    x = torch.linspace(-8, 8, 1 << 16)[:, None].contiguous()
    table, ids = torch.ones(1, 1), torch.zeros(1 << 16, dtype=torch.int64)
    got = native.gelu_gated_lookup(x.to(gpu_device), ids.to(gpu_device), table.to(gpu_device), 0).cpu().double()
    want, f = _gelu_tanh(x.double()), x.double()
    a = (2.302208198 * f * (1 + 0.044715 * f ** 2)).abs()
    assert bool(((got - want).abs() <= want.abs() * (8 + 4 * a / (1 + torch.exp2(a * f.sign()))) * 2.0 ** -24).all())

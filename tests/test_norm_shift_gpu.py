"""-m gpu: the norm that leaves the token-shift mixes of a decode step as well (tgis_sandwich_norm_shift), against its two launches: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# E: a few columns of a block, each number of column groups of a thread, whole and not
@pytest.mark.parametrize("delta", ["none", "rows", "fp32", "slabs"])
@pytest.mark.parametrize("rows,E", [(1, 64), (24, 2048), (3, 2052), (40, 4096), (2, 5000), (5, 8192)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_same_bits(gpu_device, dtype, rows, E, delta):
    from tgis_amd import native

    g = torch.Generator().manual_seed(rows + E)
    rand = lambda *shape: torch.randn(shape, generator=g).to(gpu_device)
    x, post, pre, mu, state = rand(rows, E), rand(E), rand(E), rand(5, E), rand(rows + 3, E)
    slots = torch.randperm(rows + 3, generator=g)[:rows].int().to(gpu_device)
    positions = torch.arange(rows).int().to(gpu_device)  # (the first row is a sequence's first token)
    d = None
    if delta == "rows":
        d = rand(rows, E + 8).to(dtype)[:, :E]
    elif delta == "fp32":
        d = rand(rows, E)
    elif delta == "slabs":
        d = native.Partial(rand((rows + 31) // 32 * 3 * 32 * E), 3, E, rows, E, None)
    want_x, got_x = x.clone(), x.clone()
    want = native.sandwich_norm_f32(want_x, d, post if d is not None else None, pre, 1e-5, torch.float32)
    cu = torch.arange(rows + 1).int().to(gpu_device)
    want_mixes = native.token_shift_mix(want, state, slots, cu, positions, mu, dtype)
    got, mixes = native.sandwich_norm_shift(got_x, d, post if d is not None else None, pre, 1e-5, state, slots, positions, mu, dtype)
    assert torch.equal(got_x, want_x) and torch.equal(got, want) and torch.equal(mixes, want_mixes)


def test_refusals(gpu_device):
    from tgis_amd import native

    z = lambda *shape: torch.zeros(shape, device=gpu_device)
    i = torch.zeros(2, dtype=torch.int32, device=gpu_device)
    for E, mixes, dtype in ((2050, 5, torch.float16), (8200, 5, torch.float16), (64, 4, torch.float16), (64, 5, torch.float32)):
        with pytest.raises(RuntimeError):
            native.sandwich_norm_shift(z(2, E), None, None, z(E), 1e-5, z(2, E), i, i, z(mixes, E), dtype)

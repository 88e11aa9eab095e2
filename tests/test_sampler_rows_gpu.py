"""-m gpu: the chooser's row-in-registers form at the edges of its rows: ties, rows of one element to 32 per thread, masses at the cut."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rows(V, seed):
    g = torch.Generator().manual_seed(seed)
    few = torch.randint(-3, 4, (V,), generator=g).float() * 0.5                       # ties everywhere
    wide = torch.randn(V, generator=g) * torch.logspace(-20, 1, V)                    # keys of every exponent, both signs
    gone = torch.randn(V, generator=g).masked_fill(torch.rand(V, generator=g) < 0.5, float("-inf"))
    gone[0] = 0.0
    return torch.stack([few, wide, gone])


@pytest.mark.parametrize("V", [1, 63, 255, 1023, 1024, 1025, 32767, 32768])
@pytest.mark.parametrize("part", [0.0, 0.3, 0.999])
def test_top_k_keeps_the_ties_of_the_kth(gpu_device, V, part):
    from tgis_amd import native

    x = _rows(V, V)
    k = max(1, int(part * V))
    ids, _, _, got = native.warp_sample(x.to(gpu_device), top_k=torch.full((3,), k, dtype=torch.int32, device=gpu_device))
    kth = x.sort(dim=1, descending=True).values[:, k - 1:k]
    want = x.masked_fill(x < kth, float("-inf")) if k < V else x
    assert torch.equal(got.cpu(), want)
    assert torch.equal(ids.cpu(), x.argmax(dim=1)) or all(x[b, i] == x[b].max() for b, i in enumerate(ids.tolist()))


@pytest.mark.parametrize("V", [2, 1024, 1025, 32000, 32768])
@pytest.mark.parametrize("top_p", [0.05, 0.5, 0.9, 0.999])
def test_top_p_removes_all_that_fits_the_cut(gpu_device, V, top_p):
    from tgis_amd import native

    x = _rows(V, V + 1)
    cut = 1.0 - top_p
    _, _, _, got = native.warp_sample(x.to(gpu_device), top_p_cut=torch.full((3,), cut, device=gpu_device))
    got = got.cpu()
    kept = ~torch.isneginf(got)
    assert torch.equal(got[kept], x[kept])
    p = torch.softmax(x.double(), dim=1)
    slack = 4 * V ** 0.5 * 2.0 ** -24 + 1e-6  # fp32 sums of V terms in 1024 threads, the cut's own rounding
    for b in range(3):
        low = x[b][kept[b]].min()
        assert (kept[b] == (x[b] >= low)).all()  # a prefix of the order goes, ties together
        removed = p[b][x[b] < low].sum()
        assert removed <= cut + slack
        if low < x[b].max():
            assert removed + p[b][x[b] == low].sum() > cut - slack


@pytest.mark.parametrize("V", [255, 1025, 32768])
@pytest.mark.parametrize("k", [1, 4, 50, 254, 256, 257])
def test_top_p_behind_top_k(gpu_device, V, k):
    """One launch for both removes, to the bit, what a top-k and a top-p of its scores remove: rows with ties past the list and past a thread's four places among them."""
    from tgis_amd import native

    x = torch.cat([_rows(V, V + k), torch.randn(1, V, generator=torch.Generator().manual_seed(k))]).to(gpu_device)
    top_k, cut = torch.full((4,), k, dtype=torch.int32, device=gpu_device), torch.full((4,), 0.1, device=gpu_device)
    first = native.warp_sample(x, top_k=top_k)[3]
    ids, logprob, lse, want = native.warp_sample(first.clone(), top_p_cut=cut)
    got = native.warp_sample(x, top_k=top_k, top_p_cut=cut)
    assert torch.equal(got[3], want) and torch.equal(got[0], ids) and torch.equal(got[1], logprob) and torch.equal(got[2], lse)
    kept = torch.isfinite(want).sum(dim=1)
    assert int(kept.min()) >= 1 and (k >= V or int(kept[3]) <= k)

"""-m gpu: the recurrence of csrc/wkv.hip in chunks of 16 tokens and token by token, against its definition in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def definition(r, k, v, gate, logw, u, gain, S, eps):
    """One sequence: r, k, v, gate, logw [T, H, d], u [H, d], gain [H, d], S [H, d, d] -> (out [T, H, d], S)."""
    out = torch.empty_like(v)
    for t in range(r.shape[0]):
        kv = k[t][:, :, None] * v[t][:, None, :]
        o = torch.einsum("hi,hij->hj", r[t], S + u[:, :, None] * kv)
        S = logw[t].exp()[:, :, None] * S + kv
        out[t] = o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * gain * torch.nn.functional.silu(gate[t])
    return out, S


# dims: every template width, padded ones, one that is not a multiple of 4; pad: rows that are not aligned groups of four
@pytest.mark.parametrize("d,pad", [(64, 0), (64, 2), (32, 0), (8, 0), (48, 0), (128, 0), (100, 0), (18, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_scan_in_chunks(gpu_device, d, pad, dtype):
    from tgis_amd import native

    H, W, eps = 3, 40, 1e-4
    lens = [1, 4, 5, 16, 17, 31, 48, 50]  # both ways of walking, whole and ragged chunks
    fresh = [i % 3 == 0 for i in range(len(lens))]
    T, B = sum(lens), len(lens)
    g = torch.Generator().manual_seed(d)
    r, k, v, gate = ((torch.randn(T, H, d, generator=g) * s).to(dtype) for s in (0.5, 0.5, 1.0, 1.0))
    # decays near one, ordinary, and so strong that their products underflow
    logw = -torch.exp(torch.randn(T, H, d, generator=g) * 1.5 - 1.0)
    logw[torch.rand(T, H, d, generator=g) < 0.05] = -60.0
    u, gain = torch.randn(H, d, generator=g) * 0.3, torch.rand(H, d, generator=g) + 0.5
    state = torch.randn(B + 1, H, d, d, generator=g)
    h, shift = torch.randn(T, W, generator=g), torch.zeros(B + 1, W)
    slots = torch.randperm(B, generator=g).to(torch.int32)
    cu = torch.tensor([0] + lens).cumsum(0)
    pos = torch.cat([torch.arange(n) + (0 if f else 7) for n, f in zip(lens, fresh)]).to(torch.int32)
    dev = lambda t: t.to(gpu_device)
    rows = lambda t: torch.nn.functional.pad(t.reshape(T, H * d), (0, pad)).to(gpu_device)[:, :H * d]
    st, sh = dev(state).clone(), dev(shift)
    got = native.wkv_scan(rows(r), rows(k), rows(v), rows(gate), dev(logw.reshape(T, -1)), dev(u.reshape(-1)), dev(gain.reshape(-1)),
                          st, sh, dev(h), dev(slots), dev(cu.to(torch.int32)), dev(pos), H, d, eps).double().cpu().view(T, H, d)
    for b, (n, f) in enumerate(zip(lens, fresh)):
        a, e = int(cu[b]), int(cu[b + 1])
        S0 = torch.zeros(H, d, d, dtype=torch.float64) if f else state[int(slots[b])].double()
        want, S = definition(*(t[a:e].double() for t in (r, k, v, gate, logw)), u.double(), gain.double(), S0, eps)
        # fp32 sums of up to d + 16 terms of either sign and products of up to 16 decays: some tens of roundings (2e-7 each at the
        # most, relative to the row's size), and exp's own error; two-byte outputs add their rounding (2 ** -9 of the value)
        size = want.square().mean(-1, keepdim=True).sqrt()
        tol = 2e-5 * size + (0.0 if dtype == torch.float32 else 2.0 ** -8 * want.abs())
        assert ((got[a:e] - want).abs() <= tol).all(), (n, float(((got[a:e] - want).abs() / size).max()))
        got_S = st[int(slots[b])].double().cpu()
        assert (got_S - S).abs().max() <= 1e-5 * S.abs().max(), n
        assert torch.equal(sh[int(slots[b])].cpu(), h[e - 1])
    assert torch.equal(st[B].cpu(), state[B])


@pytest.mark.parametrize("W", [40, 1024, 1030])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_token_shift_and_decay(gpu_device, W, dtype):
    from tgis_amd import native

    g = torch.Generator().manual_seed(W)
    lens, T = [1, 1100], 1101
    h, shift, mu = torch.randn(T, W, generator=g), torch.randn(3, W, generator=g), torch.rand(5, W, generator=g)
    pos = torch.cat([torch.tensor([9]), torch.arange(1100)]).to(torch.int32)
    dev = lambda t: t.to(gpu_device)
    got = native.token_shift_mix(dev(h), dev(shift), dev(torch.tensor([2, 0], dtype=torch.int32)),
                                 dev(torch.tensor([0, 1, T], dtype=torch.int32)), dev(pos), dev(mu), dtype).cpu()
    before = torch.cat([shift[2:3], torch.zeros(1, W), h[1:-1]])
    want = h[None] + (before - h)[None] * mu[:, None]
    tol = 1e-6 if dtype == torch.float32 else 2.0 ** -10
    assert ((got.float() - want).abs() <= tol * (1 + want.abs())).all()
    for T2 in (3, 1024, 1101):  # single tokens, whole and ragged groups of tokens per workgroup
        a, w2t, w0 = torch.randn(T2, 24, generator=g).to(dtype), torch.randn(24, W, generator=g) * 0.2, torch.randn(W, generator=g)
        lw = native.wkv_decay(dev(a), dev(w2t), dev(w0)).cpu().double()
        z = w0.double() + torch.tanh(a.double()) @ w2t.double()
        assert ((lw + z.exp()).abs() <= 1e-5 * (1 + z.exp())).all()


# tokens, channels, rank: whole tiles of 64 x 256 and ragged ones, ranks of one and two blocks of 64 and past them
@pytest.mark.parametrize("T,W,rank", [(513, 2100, 64), (1000, 1100, 130), (2049, 1536, 67), (3200, 1030, 128)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_decay_in_tiles(gpu_device, T, W, rank, dtype):
    from tgis_amd import native

    g = torch.Generator().manual_seed(T)
    a = torch.randn(T, rank + 3, generator=g).to(dtype).to(gpu_device)[:, :rank]
    w2t, w0 = (torch.randn(rank, W, generator=g) * rank ** -0.5).to(gpu_device), torch.randn(W, generator=g).to(gpu_device)
    lw = native.wkv_decay(a, w2t, w0).double()
    z = w0.double() + torch.tanh(a.double()) @ w2t.double()
    # an fp32 sum of up to 130 terms of size rank ** -0.5 (some ten roundings of 6e-8 of a sum of up to 5), which exp turns into a relative error
    assert lw.shape == (T, W) and ((lw + z.exp()).abs() <= 1e-5 * z.exp()).all()


# ranks: one, fewer than a thread's first load, exactly those, more; lens: single tokens, none, and a few one after another
@pytest.mark.parametrize("d,rank", [(64, 64), (64, 5), (32, 1), (8, 70), (48, 200), (128, 32), (100, 129)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_step_with_its_decay(gpu_device, d, rank, dtype):
    from tgis_amd import native

    H, W, eps = 3, 300, 1e-4
    lens = [1, 0, 1, 3, 1, 1]
    fresh = [False, True, True, False, False, True]
    T, B = sum(lens), len(lens)
    g = torch.Generator().manual_seed(d + rank)
    r, k, v, gate = ((torch.randn(T, H, d, generator=g) * s).to(dtype) for s in (0.5, 0.5, 1.0, 1.0))
    low = torch.randn(T, rank, generator=g).to(dtype)
    w2t, w0 = torch.randn(rank, H * d, generator=g) * 0.3 * rank ** -0.5, torch.randn(H * d, generator=g) - 1.0
    logw = -torch.exp(w0.double() + torch.tanh(low.double()) @ w2t.double()).view(T, H, d)
    u, gain = torch.randn(H, d, generator=g) * 0.3, torch.rand(H, d, generator=g) + 0.5
    state = torch.randn(B + 1, H, d, d, generator=g)
    state[1::2, :, :, 0] = float("nan")  # what a fresh sequence's slot holds must not matter
    slots = torch.tensor([0, 3, 1, 2, 4, 5], dtype=torch.int32)
    fresh = [int(s) % 2 == 1 for s in slots]
    h, shift = torch.randn(T, W, generator=g), torch.zeros(B + 1, W)
    cu = torch.tensor([0] + lens).cumsum(0)
    pos = torch.cat([torch.arange(n) + (0 if f else 7) for n, f in zip(lens, fresh)]).to(torch.int32)
    dev = lambda t: t.to(gpu_device)
    rows = lambda t: torch.nn.functional.pad(t.reshape(T, H * d), (0, 4)).to(gpu_device)[:, :H * d]
    st, sh = dev(state).clone(), dev(shift)
    got = native.wkv_step(rows(r), rows(k), rows(v), rows(gate), torch.nn.functional.pad(dev(low), (0, 3))[:, :rank], dev(w2t), dev(w0),
                          dev(u.reshape(-1)), dev(gain.reshape(-1)), st, sh, dev(h), dev(slots), dev(cu.to(torch.int32)), dev(pos), H, d,
                          eps).double().cpu().view(T, H, d)
    for b, (n, f) in enumerate(zip(lens, fresh)):
        a, e, slot = int(cu[b]), int(cu[b + 1]), int(slots[b])
        if n == 0:
            assert torch.equal(st[slot].cpu().nan_to_num(), state[slot].nan_to_num()) and not sh[slot].any()
            continue
        S0 = torch.zeros(H, d, d, dtype=torch.float64) if f else state[slot].double()
        want, S = definition(*(t[a:e].double() for t in (r, k, v, gate, logw)), u.double(), gain.double(), S0, eps)
        size = want.square().mean(-1, keepdim=True).sqrt()
        # as above; the decay's exponent adds the fp32 sum of `rank` terms (2e-7 of its size per term at the most)
        tol = 4e-5 * size + (0.0 if dtype == torch.float32 else 2.0 ** -8 * want.abs())
        assert ((got[a:e] - want).abs() <= tol).all(), (b, float(((got[a:e] - want).abs() / size).max()))
        got_S = st[slot].double().cpu()
        assert (got_S - S).abs().max() <= 2e-5 * S.abs().max(), b
        assert torch.equal(sh[slot].cpu(), h[e - 1])
    assert torch.equal(st[B].cpu(), state[B])


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_values_that_are_not_finite_stay_with_later_tokens(gpu_device, dtype, bad):
    """Prompts of several chunks, one value channel of one token not finite: every token in front of it keeps its output, every one from
    it on loses its own, as when the tokens are walked one by one."""
    from tgis_amd import native

    H, d, W, eps = 2, 64, 40, 1e-4
    lens, at = [40, 33, 20], [25, 16, 18]  # inside a chunk, its first token, a ragged last chunk
    T, B = sum(lens), len(lens)
    g = torch.Generator().manual_seed(3)
    r, k, v, gate = (torch.randn(T, H, d, generator=g).to(dtype) for _ in range(4))
    logw = -torch.exp(torch.randn(T, H, d, generator=g) - 1.0)
    u, gain = torch.randn(H, d, generator=g) * 0.3, torch.rand(H, d, generator=g) + 0.5
    cu = torch.tensor([0] + lens).cumsum(0)
    pos = torch.cat([torch.arange(n) for n in lens]).to(torch.int32)
    dev = lambda t: t.to(gpu_device)
    rows = lambda t: dev(t.reshape(T, H * d))

    def scan(v):
        return native.wkv_scan(rows(r), rows(k), rows(v), rows(gate), rows(logw), dev(u.reshape(-1)), dev(gain.reshape(-1)),
                               torch.zeros(B, H, d, d, device=gpu_device), torch.zeros(B, W, device=gpu_device), torch.zeros(T, W, device=gpu_device),
                               dev(torch.arange(B, dtype=torch.int32)), dev(cu.int()), dev(pos), H, d, eps).float().cpu().view(T, H, d)

    clean = scan(v)
    for b, s in enumerate(at):
        v[int(cu[b]) + s, 0, 7] = bad
    got = scan(v)
    # (the sums of a token in a chunk with such a value are added in another order: fp32 roundings, then the output's)
    tol = 2e-5 + (0.0 if dtype == torch.float32 else 2.0 ** -7)
    for b, s in enumerate(at):
        a, e = int(cu[b]), int(cu[b + 1])
        assert ((got[a:a + s] - clean[a:a + s]).abs() <= tol * (1 + clean[a:a + s].abs())).all(), b
        assert not got[a + s:e, 0, 7].isfinite().any(), b
        assert torch.equal(got[a:e, 1], clean[a:e, 1]), b  # the other head


# heads and ranks on each side of what the step launch is for
@pytest.mark.parametrize("d,rank,stepped", [(64, 64, True), (64, 65, False), (32, 16, True), (68, 32, False), (128, 64, False)])
def test_single_tokens_of_a_mixer(gpu_device, monkeypatch, d, rank, stepped):
    """A decode step of the mixer takes the step launch where it pays, and the decay and the scan elsewhere, with the same result."""
    from types import SimpleNamespace

    from tgis_amd import native
    from tgis_amd.utils.mixers import WkvMixer

    H, B = 2, 3
    W = HD = H * d
    g = torch.Generator().manual_seed(d + rank)
    shapes = {**{f"m.mu.{s}": (W,) for s in WkvMixer.MIXES}, **{f"m.{s}": (HD, W) for s in "rkvgo"}, "m.w1": (rank, W), "m.w2": (HD, rank),
              "m.w0": (HD,), "m.u": (H, d), "m.norm": (HD,)}
    t = {n: (torch.randn(s, generator=g) * (W ** -0.5 if len(s) == 2 else 0.3)).bfloat16().to(gpu_device) for n, s in shapes.items()}
    weights = SimpleNamespace(get_tensor=lambda n, **kw: t[n], dtype=torch.bfloat16, device=gpu_device)
    m = WkvMixer(weights, "m", 0, H, d, 1e-5)
    state, shift = torch.randn(B, H, d, d, generator=g).to(gpu_device), torch.randn(B, W, generator=g).to(gpu_device)
    calls = []
    real = native.wkv_step
    monkeypatch.setattr(native, "wkv_step", lambda *a: calls.append(1) or real(*a))
    index = torch.arange(B + 1, dtype=torch.int32, device=gpu_device)
    h = torch.randn(B, W, generator=g).to(gpu_device)
    pos = torch.full((B,), 9, dtype=torch.int32, device=gpu_device)
    out = []
    for pays in (None, True, False):
        if pays is not None:
            monkeypatch.setattr(native, "wkv_step_pays", lambda *a: pays and d % 4 == 0)
        kept = SimpleNamespace(state=[state.clone()], shift=[shift.clone()])
        step = SimpleNamespace(state=kept, state_slots=index[:B], cu_seqlens_q=index, max_q_len=1)
        m.defer = False
        out.append(torch.cat([m.forward(h, pos, step, torch.bfloat16).float().flatten(), kept.state[0].flatten(), kept.shift[0].flatten()]))
        assert bool(calls) == (stepped if pays is None else pays)
        calls.clear()
    # fp32 sums in other orders, rounded to bf16 once before and once behind the output projection
    for a in out[1:]:
        assert ((a - out[0]).abs() <= 2.0 ** -6 * (out[0].abs() + out[0].square().mean().sqrt())).all()


# (heads, sequences, head width): more blocks than a CU holds of the chunk kernel, and not more; runs: the longest that is walked by token, one more
@pytest.mark.parametrize("H,B,d,by_token", [(8, 40, 64, True), (8, 32, 64, False), (6, 90, 32, True), (6, 40, 32, False), (3, 90, 68, False)])
@pytest.mark.parametrize("longest", [1, 10, 11, 16, 17, 18])
def test_scan_of_short_runs(gpu_device, H, B, d, by_token, longest):
    """Many short runs: the bits of the token-by-token walk where it is chosen (rows that are no groups of four take it always)."""
    from tgis_amd import native

    g = torch.Generator().manual_seed(H + B + longest)
    lens = torch.randint(0, longest + 1, (B,), generator=g)
    lens[B // 2] = longest
    T, W = int(lens.sum()), 8
    cu = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)]).int().to(gpu_device)
    rkvg = [torch.randn(T, H * d, generator=g).bfloat16().to(gpu_device) for _ in range(4)]
    logw = -torch.exp(torch.randn(T, H * d, generator=g) - 1.0).to(gpu_device)
    u, gain, state = (torch.randn(*s, generator=g).to(gpu_device) for s in ((H * d,), (H * d,), (B, H, d, d)))
    slots, pos = torch.randperm(B, generator=g).int().to(gpu_device), torch.randint(0, 2, (T,), generator=g).int().to(gpu_device)

    def scan(pad, hint):
        rows = [torch.nn.functional.pad(t, (0, pad))[:, :H * d] for t in rkvg]
        st = state.clone()
        out = native.wkv_scan(*rows, logw, u, gain, st, torch.zeros(B, W, device=gpu_device), torch.zeros(T, W, device=gpu_device), slots, cu, pos, H, d,
                              1e-5, max_q_len=hint)
        return out.float(), st

    walked, walked_st = scan(2, 0)
    got, got_st = scan(0, longest)
    if by_token and (longest <= 10 or longest == 17):
        assert torch.equal(got, walked) and torch.equal(got_st, walked_st)
    # fp32 sums in another order, one rounding to bf16
    assert ((got - walked).abs() <= 2.0 ** -7 * (walked.abs() + walked.square().mean().sqrt())).all()
    assert (got_st - walked_st).abs().max() <= 1e-5 * walked_st.abs().max()


# longest: fewer tokens than are cut, just enough, a last segment of one token and of whole sub-blocks, more segments than one launch takes
@pytest.mark.parametrize("d,longest", [(64, 127), (64, 128), (64, 449), (64, 2500), (32, 129), (48, 640), (128, 513), (100, 511)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_scan_in_segments(gpu_device, d, longest, dtype):
    """Long runs beside short ones, cut into segments, against the same step token by token (rows that are no groups of four, no hint)."""
    from tgis_amd import native

    H, W, eps = 2, 8, 1e-4
    lens = [longest, 1, min(129, longest), longest // 2, 64]
    fresh = [False, False, True, True, False]
    T, B = sum(lens), len(lens)
    g = torch.Generator().manual_seed(d + longest)
    r, k, v, gate = ((torch.randn(T, H * d, generator=g) * s).to(dtype) for s in (0.5, 0.5, 1.0, 1.0))
    # (r, k and u of one sign: r u k of a fresh run's first token is then no sum that cancels, which the unit norm would magnify)
    rkvg = [t.to(gpu_device) for t in (r.abs(), k.abs(), v, gate)]
    logw = -torch.exp(torch.randn(T, H * d, generator=g) * 1.5 - 4.0)  # decays that carry a state over hundreds of tokens, some that end it
    logw[torch.rand(T, H * d, generator=g) < 0.005] = -60.0
    u, gain = torch.rand(H * d, generator=g) * 0.5, torch.rand(H * d, generator=g) + 0.5
    state = torch.randn(B + 1, H, d, d, generator=g).to(gpu_device)
    state[4, :, :, 0] = float("nan")  # slot of the third sequence, which starts anew
    slots = torch.tensor([2, 0, 4, 1, 5], dtype=torch.int32)
    cu = torch.cat([torch.zeros(1, dtype=torch.int64), torch.tensor(lens).cumsum(0)])
    pos = torch.cat([torch.arange(n) + (0 if f else 7) for n, f in zip(lens, fresh)]).to(torch.int32)
    h = torch.randn(T, W, generator=g).to(gpu_device)
    dev = lambda t: t.to(gpu_device)

    def scan(pad, hint):
        rows = [torch.nn.functional.pad(t, (0, pad))[:, :H * d] for t in rkvg]
        st, sh = state.clone(), torch.zeros(B + 1, W, device=gpu_device)
        out = native.wkv_scan(*rows, dev(logw), dev(u), dev(gain), st, sh, h, dev(slots), dev(cu.to(torch.int32)), dev(pos), H, d, eps, max_q_len=hint)
        return out.double().view(T, H, d), st[slots.long()], sh, st[3]

    assert (native.load_library().tgis_wkv_scan_workspace(B, H, d, longest) > 0) == (longest >= (128 if d <= 64 else 512))
    want, want_st, want_sh, _ = scan(2, 0)
    got, got_st, got_sh, spare = scan(0, longest)
    # fp32 sums of either sign in another order and products of decays in another order (each a few roundings of 6e-8 per factor that
    # matters: a key is worth less than 1e-3 after some hundreds); two-byte outputs are rounded once on both sides
    size = want.square().mean(-1, keepdim=True).sqrt()
    tol = 4e-5 * size + (0.0 if dtype == torch.float32 else 2.0 ** -7 * want.abs())
    assert ((got - want).abs() <= tol).all(), float(((got - want).abs() / size).max())
    assert (got_st - want_st).abs().max() <= 2e-5 * want_st.abs().max()
    assert torch.equal(got_sh, want_sh) and torch.equal(spare, state[3])


def test_scan_entries_without_segments(gpu_device):
    """tgis_wkv_scan and tgis_wkv_scan_runs: the launches of a step that is not cut, with the hint 0 and with one, bit for bit."""
    from tgis_amd import native

    lib, H, W, d, eps = native.load_library(), 3, 8, 64, 1e-4
    lens = [5, 1, 33, 60]
    T, B = sum(lens), len(lens)
    g = torch.Generator().manual_seed(1)
    rkvg = [torch.randn(T, H * d, generator=g).to(torch.bfloat16).to(gpu_device) for _ in range(4)]
    logw, u, gain, state, h = (t.to(gpu_device) for t in (-torch.rand(T, H * d, generator=g), torch.rand(H * d, generator=g), torch.rand(H * d, generator=g),
                                                          torch.randn(B, H, d, d, generator=g), torch.randn(T, W, generator=g)))
    slots, pos = torch.arange(B).int().to(gpu_device), torch.cat([torch.arange(n) for n in lens]).int().to(gpu_device) + 3
    cu = torch.tensor([0] + lens).cumsum(0).int().to(gpu_device)
    ptr = lambda t: t.data_ptr()
    for name, hint in (("tgis_wkv_scan", 0), ("tgis_wkv_scan_runs", 60)):
        st, sh = state.clone(), torch.zeros(B, W, device=gpu_device)
        want = native.wkv_scan(*rkvg, logw, u, gain, st, sh, h, slots, cu, pos, H, d, eps, max_q_len=hint)
        st2, sh2, out = state.clone(), torch.zeros(B, W, device=gpu_device), torch.zeros_like(want)
        rest = (eps, hint, native.dtype_code3(out.dtype)) if hint else (eps, native.dtype_code3(out.dtype))
        assert lib.tgis_wkv_scan_workspace(B, H, d, hint) == 0
        assert getattr(lib, name)(*map(ptr, rkvg), H * d, ptr(logw), ptr(u), ptr(gain), ptr(st2), ptr(sh2), ptr(h), W, ptr(slots), ptr(cu), ptr(pos), ptr(out),
                                  H * d, B, H, d, *rest, torch.cuda.current_stream().cuda_stream) == 0
        assert torch.equal(out, want) and torch.equal(st2, st) and torch.equal(sh2, sh)

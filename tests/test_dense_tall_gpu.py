"""The dense GEMM of prefills on the prepared image (tgis_dense_tall) against the float64 product: every tile, whole and split over k, at the
edges of its rows and columns; and the projections that choose it, on both sides of the rule."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}  # half a step of the dtype, of a value's size


def _case(M, K, N, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(M, K, generator=g).to(dtype)
    w = (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype)
    bias = torch.randn(N, generator=g).to(dtype)
    z = x.double() @ w.double().t() + bias.double()
    # fp32 sums of K products in any order: K half-steps of 2^-24 of the sum of magnitudes
    acc = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + bias.double().abs())
    return x, w, bias, z, acc


def _expect(z, acc, dtype, act):
    """(value, bound): the sum may round to either neighbour (2 half-steps), the activation then moves by its slope (at most 1.13) times
    that, and every rounding behind it adds a half-step (a step where the intermediate is rounded too)."""
    u = ULP[dtype]
    r = z.to(dtype).double()
    dz = 2 * u * r.abs() + acc + 2.0 ** -24
    if act == 0:
        return r, dz
    if act in (4, 5):
        return torch.nn.functional.gelu(r, approximate="tanh" if act == 5 else "none"), 1.13 * dz + 2 * u * r.abs() + 2.0 ** -24
    h = z.shape[1] // 2
    gate, up, dg, du = r[:, :h], r[:, h:], dz[:, :h], dz[:, h:]
    if act == 2:
        s = gate * torch.sigmoid(gate)
        return s * up, 1.1 * dg * up.abs() + s.abs() * du + 4 * u * (s * up).abs() + 2.0 ** -24
    gc, uc = gate.clamp(max=3.0), up.clamp(-3.0, 3.0)
    s = gc * torch.sigmoid(1.7 * gc)
    return s * (uc + 1), 1.1 * dg * (uc + 1).abs() + s.abs() * du + 4 * u * (s * (uc + 1)).abs() + 2.0 ** -24


def _check(out, want):
    value, bound = want
    off = (out.double().cpu() - value).abs() - bound
    assert out.shape == value.shape and bool((off <= 0).all()), float(off.max())


def _run(M, K, N, dtype, act, plan, monkeypatch, ld_out=None):
    from tgis_amd import native

    if plan:
        monkeypatch.setenv("TGIS_DTALL_PLAN", plan)
    x, w, bias, z, acc = _case(M, K, N, dtype)
    clamped = act == 3
    image = native.DenseWeight(w.cuda(), gate_up=act in (2, 3))
    ws = native.Workspace(64 << 20, torch.device("cuda"))
    n_out = N // 2 if act in (2, 3) else N
    out = torch.full((M, ld_out or n_out), 7.0, dtype=dtype, device="cuda")
    native.dense_tall(x.cuda(), image, ws, 48 << 20, bias=bias.cuda(), act=2 if clamped else act, alpha=1.7, limit=3.0 if clamped else 0.0, out=out[:, :n_out])
    _check(out[:, :n_out], _expect(z, acc, dtype, act))
    assert bool((out[:, n_out:] == 7.0).all())


# tiles of 64 / 96 / 128 x 128 / 256, whole and in 2 and 3 parts; rows and columns one short of, at and past a tile; every remainder of the ring
@pytest.mark.parametrize("plan,M,K,N", [
    ("2,1,1", 65, 64, 128), ("2,1,2", 64, 320, 136), ("2,2,1", 129, 128, 257), ("2,2,3", 63, 1152, 520),
    ("3,1,1", 96, 192, 100), ("3,1,3", 97, 640, 129), ("3,2,2", 191, 448, 256), ("3,2,1", 290, 256, 31),
    ("4,1,1", 128, 384, 384), ("4,1,2", 127, 1088, 640), ("4,2,1", 257, 448, 300), ("4,2,3", 130, 896, 512),
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_plain(plan, M, K, N, dtype, monkeypatch):
    _run(M, K, N, dtype, 0, plan, monkeypatch, ld_out=N + 8 if M % 2 else None)


@pytest.mark.parametrize("plan,M", [("2,1,1", 97), ("2,2,3", 129), ("3,2,2", 190), ("4,2,1", 256), ("4,1,5", 65), (None, 108)])
def test_fp32_sums(plan, M, monkeypatch):
    """Without a rounding: the partial sums that a norm finishes, and a head's logits."""
    from tgis_amd import native
    from tgis_amd.utils.layers import FastLinear

    K, N = 576, 1100
    x, w, bias, z, acc = _case(M, K, N, torch.bfloat16, seed=5)
    lin = FastLinear(w.cuda(), bias.cuda())
    if plan:
        monkeypatch.setenv("TGIS_DTALL_PLAN", plan)
    part = lin(x.cuda(), partial=True)
    assert isinstance(part, native.Partial) and part.ld == 1120 and part.bias is lin.bias and (plan is None or part.S == int(plan[4]))
    sums = part.slabs.view(-1, part.S, 32, part.ld).sum(1, dtype=torch.float64).flatten(0, 1)
    _check(sums[:M, :N], (z - bias.double(), acc))
    _check(lin(x.cuda(), out_f32=True), (z, acc))


def test_parts_of_the_plan_that_ran(monkeypatch):
    """One projection whose plan is changed between two calls: the number of parts is that of the launch, not the first call's."""
    from tgis_amd.utils.layers import FastLinear

    x, w, bias, z, acc = _case(130, 576, 1100, torch.float16, seed=7)
    lin = FastLinear(w.cuda(), bias.cuda())
    for plan in ("2,1,3", "4,2,2", "3,1,1", "2,1,3"):
        monkeypatch.setenv("TGIS_DTALL_PLAN", plan)
        part = lin(x.cuda(), partial=True)
        assert part.S == int(plan[4])
        sums = part.slabs[:160 * part.S * part.ld].view(-1, part.S, 32, part.ld).sum(1, dtype=torch.float64).flatten(0, 1)
        _check(sums[:130, :1100], (z - bias.double(), acc))


@pytest.mark.parametrize("plan", ["2,1,1", "2,2,2", "3,1,3", "3,2,1", "4,1,2", "4,2,1"])
@pytest.mark.parametrize("act", [2, 3, 4, 5])
def test_activations(plan, act, monkeypatch):
    for dtype, M, K, N in ((torch.bfloat16, 131, 576, 352), (torch.float16, 98, 320, 544)):
        _run(M, K, N, dtype, act, plan, monkeypatch)


def test_chosen_plans(monkeypatch):
    # more than a round of 256 tiles with a split rest; several groups of row blocks; a narrow product
    for M, K, N, act in ((1100, 1024, 5632, 2), (2100, 256, 4224, 2), (700, 512, 64, 0), (300, 6144, 1024, 0)):
        _run(M, K, N, torch.bfloat16, act, None, monkeypatch)


@pytest.mark.parametrize("M,N", [(64, 1024), (65, 1024), (256, 1024), (257, 1024), (257, 992), (300, 2048), (501, 2048)])
def test_linear_on_both_sides(M, N):
    from tgis_amd.utils.layers import FastLinear

    K = 512
    x, w, bias, z, acc = _case(M, K, N, torch.float16, seed=3)
    lin = FastLinear(w.cuda(), bias.cuda())
    _check(lin(x.cuda()), _expect(z, acc, torch.float16, 0))
    _check(lin(x.cuda(), gelu=True), _expect(z, acc, torch.float16, 5))
    plain = FastLinear(w.cuda(), None)
    out = torch.empty(M, N, dtype=torch.float16, device="cuda")
    plain(x.cuda(), out=out)
    _check(out, _expect(z - bias.double(), acc, torch.float16, 0))
    lin.gate_up = True
    _check(lin(x.cuda()), _expect(z, acc, torch.float16, 2))


@pytest.mark.parametrize("pad,first", [(1, 0), (8, 1), (4, 0)])
def test_rows_it_cannot_read(pad, first):
    """Rows that are not 16-byte aligned go where they went: to the library."""
    from tgis_amd import native
    from tgis_amd.utils.layers import FastLinear

    x, w, bias, z, acc = _case(300, 512, 1024, torch.float16, seed=4)
    wide = torch.zeros(300, 512 + pad, dtype=torch.float16, device="cuda")
    view = wide[:, first:first + 512]
    view.copy_(x)
    lin = FastLinear(w.cuda(), bias.cuda())
    assert lin.tall(view) == -1 and lin.tall(x.cuda()) >= 0
    _check(lin(view), _expect(z, acc, torch.float16, 0))


# behind a whole turn of the ring of four buffers: one, two and three steps, and none; behind none, and in the parts of a split
@pytest.mark.parametrize("steps,S", [(1, 1), (2, 1), (3, 1), (4, 1), (5, 1), (6, 1), (7, 1), (11, 1), (14, 2)])
@pytest.mark.parametrize("tile", ["2,1", "2,2", "3,1", "3,2", "4,1", "4,2"])
def test_tails_of_the_ring(tile, steps, S, monkeypatch):
    _run(290, 64 * steps, 264, torch.bfloat16, 0, f"{tile},{S}", monkeypatch)


def test_rows_that_the_user_divides(monkeypatch):
    """TGIS_SKINNY_MAX_M: the streaming kernel up to that many rows, the library above, nothing else."""
    from tgis_amd import native
    from tgis_amd.utils import layers

    K, N = 512, 1024
    monkeypatch.setattr(layers, "DENSE_TALL", False)
    monkeypatch.setattr(layers, "SKINNY_MAX_M", 128)
    for name in ("dense_tall", "dense_tall_partial"):
        monkeypatch.setattr(native, name, lambda *a, **k: pytest.fail("the prefill kernel"))
    streamed, run = [], native.dense_gemm
    monkeypatch.setattr(native, "dense_gemm", lambda x, *a, **k: streamed.append(x.shape[0]) or run(x, *a, **k))
    for M in (65, 128, 129, 300):
        x, w, bias, z, acc = _case(M, K, N, torch.float16, seed=6)
        lin = layers.FastLinear(w.cuda(), bias.cuda())
        _check(lin(x.cuda()), _expect(z, acc, torch.float16, 0))
        _check(lin(x.cuda(), gelu=False), _expect(z, acc, torch.float16, 4))
        lin.gate_up = True
        _check(lin(x.cuda()), _expect(z, acc, torch.float16, 2))
    assert streamed == [65] * 3 + [128] * 3


# one launch of several products: one, several with a last one that is whole / part of a tile / a narrow one ahead of the others (past 5000 rows, or 6 M of their outputs)
@pytest.mark.parametrize("M,K,n_group,N,G,plans", [
    (65, 64, 32, 20, 1, "234"), (129, 448, 96, 288, 3, "234"), (97, 576, 64, 150, 3, "2"), (300, 2048, 512, 2048 + 64, 5, "234"), (257, 128, 160, 470, 3, "4"),
    (2049, 192, 256, 256 + 128, 2, "234"), (2050, 64, 288, 4 * 288 + 33, 5, "234"), (2049, 128, 256, 256 + 129, 2, "3"), (2111, 320, 32, 64, 2, "4"),
    (5001, 192, 256, 256 + 128, 2, "234"), (5002, 64, 288, 4 * 288 + 33, 5, "234"), (2100, 64, 2880, 2880 + 40, 2, "3"),
])
@pytest.mark.parametrize("width", [1, 2])
def test_groups(M, K, n_group, N, G, plans, width, monkeypatch):
    from tgis_amd import native

    dtype = torch.bfloat16 if M & 1 else torch.float16
    g = torch.Generator().manual_seed(K + N + M)
    x, wt = torch.randn(G, M, K, generator=g).to(dtype), (torch.randn(N, K, generator=g) * K ** -0.5).to(dtype)
    image, xd = native.DenseWeight(wt.cuda()), x.cuda()
    want = [_expect(x[i].double() @ wt[i * n_group:(i + 1) * n_group].double().t(),
                    K * 2.0 ** -24 * (x[i].double().abs() @ wt[i * n_group:(i + 1) * n_group].double().abs().t()), dtype, 0) for i in range(G)]
    for rows in [None, *plans]:
        if rows:
            monkeypatch.setenv("TGIS_DTALL_PLAN", f"{rows},{width},1")
        out = torch.full((G, M, n_group + (8 if M & 2 else 1)), 7.0, dtype=dtype, device="cuda")
        native.dense_tall_groups(xd, image, n_group, out)
        for i in range(G):
            cols = min(n_group, N - i * n_group)
            _check(out[i, :, :cols], want[i])
            assert bool((out[i, :, cols:] == 7.0).all())


def test_groups_rule():
    from tgis_amd import native

    pays = lambda *a: native.load_library().tgis_dense_tall_groups_pays(*a)
    assert pays(65, 2048, 2048, 4 * 2048 + 64, 5) and pays(4096, 2048, 2048, 4 * 2048 + 64, 5) and not pays(4097, 2048, 2048, 4 * 2048 + 64, 5)
    assert not pays(64, 2048, 2048, 4 * 2048 + 64, 5) and not pays(300, 96, 2048, 4 * 2048 + 64, 5) and not pays(300, 2048, 2048, 4 * 2048, 5)
    wide = native.DenseWeight(torch.zeros(96, 72, dtype=torch.float16, device="cuda"))
    with pytest.raises(RuntimeError, match="bad arguments"):
        native.dense_tall_groups(torch.zeros(3, 70, 72, dtype=torch.float16, device="cuda"), wide, 32, torch.zeros(3, 70, 32, dtype=torch.float16, device="cuda"))

"""The expert products over runs of up to 128 and 256 rows against float64: experts of one tile up to three runs that are
split evenly, contractions of one to five stages, column counts around the tiles of 128 and 256, tiles beyond the first
stretches of 64 of the table of runs, tiles in any order.  fp32 results carry the rounding of sums of K products of 16-bit
numbers only (1e-5 of the largest value); 16-bit results that of one store (2^-8)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
F = torch.float64
FORMS = [5, 6]


def rnd(shape, seed, std=1.0):
    return std * torch.randn(shape, generator=torch.Generator().manual_seed(seed))


def check(tiles_of, n, k, form, dtype, order=None):
    """Experts of so many row tiles; plain products in fp32, gated ones in 16 bits."""
    from vllm_legacy_amd import _seq_ops as ops
    experts = order if order is not None else [e for e, t in enumerate(tiles_of) for _ in range(t)]
    E = max(experts) + 1
    rows = 32 * len(experts)
    a, w = rnd((rows, k), 1).to(dtype), rnd((E, 2 * n, k), 2, k**-0.5).to(dtype)
    row_token = torch.randperm(rows, generator=torch.Generator().manual_seed(3)).to(torch.int32)
    row_token[::37] = -1
    scale = torch.rand(rows, generator=torch.Generator().manual_seed(4)) + 0.5
    src = torch.where((row_token < 0)[:, None], torch.zeros((), dtype=dtype), a[row_token.clamp(min=0).long()]).to(F)
    want = torch.full((rows, 2 * n), float("nan"), dtype=F)
    for e in range(E):
        mine = torch.tensor([x == e for x in experts]).repeat_interleave(32)
        want[mine] = src[mine] @ w[e].to(F).t() * scale[mine, None]
    used = torch.tensor([x >= 0 for x in experts]).repeat_interleave(32)
    tile_expert = torch.tensor(experts, dtype=torch.int32, device=DEV)
    args = (a.to(DEV), row_token.to(DEV), w.to(DEV), tile_expert)
    ops.set_grouped_linear_form(form)
    try:
        y = torch.full((rows, 2 * n), float("nan"), device=DEV)
        ops.grouped_linear(y, *args, "none", scale.to(DEV))
        y16 = torch.full((rows, 2 * n), float("nan"), dtype=dtype, device=DEV)
        ops.grouped_linear(y16, *args, "none", scale.to(DEV))
        z = torch.full((rows, n), float("nan"), dtype=dtype, device=DEV)
        ops.grouped_glu(z, *args, "silu", scale.to(DEV))
    finally:
        ops.set_grouped_linear_form(0)
    y, y16, z = y.cpu(), y16.cpu(), z.cpu()
    top = float(want[used].abs().max())
    assert float((y - want)[used].abs().max()) <= 1e-5 * top
    assert float((y16 - want)[used].abs().max()) <= 2.0**-8 * top
    glu = want[:, :n] * torch.sigmoid(want[:, :n]) * want[:, n:]
    assert float((z - glu)[used].abs().max()) <= 2.0**-8 * float(glu[used].abs().max())
    for t in (y, y16, z):
        assert bool(t[~used].isnan().all())                # tiles without an expert are left alone
        assert float(t[used & (row_token < 0)].abs().max()) == 0.0


@pytest.mark.parametrize("tiles_of", [[1], [4, 5], [2, 3, 7, 8, 9], [0, 6, 0, 17], [12, 24, 1]])
@pytest.mark.parametrize("n,k", [(64, 64), (128, 128), (129, 192), (36, 256), (250, 320)])
@pytest.mark.parametrize("form", FORMS)
def test_runs(tiles_of, n, k, form):
    check(tiles_of, n, k, form, torch.bfloat16)


@pytest.mark.parametrize("form", FORMS)
def test_float16(form):
    check([3, 8, 11], 136, 192, form, torch.float16)


@pytest.mark.parametrize("form", FORMS)
def test_more_tiles_than_a_stretch(form):
    check([63, 1, 2, 61, 1, 130, 9, 300], 40, 64, form, torch.bfloat16)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("order", [[0, 1] * 70, [-1] * 66 + [2] * 70 + [-1, 0, 0, -1, 1], [1] * 9 + [0] + [1] * 12])
def test_any_order(order, form):
    """More runs than a plan's order could leave: the workgroups walk them."""
    check(None, 72, 128, form, torch.bfloat16, order)


def test_values_at_the_ends_of_the_range():
    """silu of sums whose exponential overflows or vanishes, infinities and NaN."""
    from vllm_legacy_amd import _seq_ops as ops
    g = torch.tensor([0.0, -1e-30, 88.0, -88.0, -87.0, 126.0, -126.0, 1e4, -1e4, 3e38, -3e38, float("inf"), -float("inf"),
                      float("nan")])
    rows, n, k = 32 * 5, 16, 64
    a = torch.zeros(rows, k)
    a[:len(g), 0], a[:, 1] = g, 1.0
    w = torch.zeros(1, 2 * n, k)
    w[0, :n, 0], w[0, n:, 1] = 1.0, 1.0                    # gate = the value, up = 1
    a = a.to(torch.bfloat16)
    out = torch.empty(rows, n, dtype=torch.bfloat16, device=DEV)
    for form in FORMS:
        ops.set_grouped_linear_form(form)
        try:
            ops.grouped_glu(out, a.to(DEV), None, w.to(torch.bfloat16).to(DEV),
                            torch.zeros(5, dtype=torch.int32, device=DEV), "silu")
        finally:
            ops.set_grouped_linear_form(0)
        x = a[:len(g), 0].float()
        # 0 * inf in the products of a row that holds an infinity makes its ups NaN as well
        want = torch.where(x.isfinite(), x * torch.sigmoid(x), torch.full_like(x, float("nan")))
        got = out[:len(g), 0].float().cpu()
        assert bool((got.isnan() == want.isnan()).all())
        ok = ~want.isnan()
        assert bool(((got - want).abs()[ok] <= 2.0**-8 * want.abs()[ok] + 1e-37).all())

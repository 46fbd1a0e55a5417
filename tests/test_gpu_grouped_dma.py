"""The expert products on LDS-DMA, op by op against float64: runs of one to five row tiles per expert, experts
nobody chose, column counts around the tiles of 32, 64 and 128, contractions of one to six steps, gathered
and plain rows, scales, every activation and the clamped form.  fp32 results carry the rounding of sums of
K products of 16-bit numbers only (1e-5 of the largest value); 16-bit results that of one store (2^-8)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
F = torch.float64


def rnd(shape, seed, std=1.0):
    return std * torch.randn(shape, generator=torch.Generator().manual_seed(seed))


def act_of(z, act):
    return {"none": lambda: z, "relu2": lambda: torch.relu(z)**2, "silu": lambda: z * torch.sigmoid(z),
            "gelu_tanh": lambda: torch.nn.functional.gelu(z, approximate="tanh")}[act]()


def plan_of(counts, top=1):
    """Experts of the pairs so that expert e is chosen counts[e] times, in mixed order."""
    from vllm_legacy_amd import _seq_ops as ops
    pairs = torch.tensor([e for e, n in enumerate(counts) for _ in range(n)])
    pairs = pairs[torch.randperm(len(pairs), generator=torch.Generator().manual_seed(1))]
    experts = pairs.view(-1, top).to(torch.int32).to(DEV)
    return pairs, ops.moe_plan(experts, len(counts))


COUNTS = [[1], [0, 130, 0, 31, 33], [5, 4, 3, 2, 1, 0, 7, 64], [129, 257, 1, 128], [2] * 70]


@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("n,k", [(64, 64), (40, 128), (200, 192), (136, 384), (6, 64)])
@pytest.mark.parametrize("form", [0, 3, 4])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_plain_products(counts, n, k, form, dtype):
    from vllm_legacy_amd import _seq_ops as ops
    pairs, (pair_row, row_token, tile_expert) = plan_of(counts)
    E, P = len(counts), len(pairs)
    a, w = rnd((P, k), 2).to(dtype), rnd((E, n, k), 3, k**-0.5).to(dtype)
    scale = torch.rand((row_token.numel(), ), generator=torch.Generator().manual_seed(4)) + 0.5
    rows = pair_row.view(-1).cpu()
    want = torch.stack([w[pairs[i]].to(F) @ a[i].to(F) for i in range(P)])
    ops.set_grouped_linear_form(form)
    try:
        y = torch.full((row_token.numel(), n), float("nan"), device=DEV)
        ops.grouped_linear(y, a.to(DEV), row_token, w.to(DEV), tile_expert)
        assert float((y.cpu()[rows] - want).abs().max()) <= 1e-5 * float(want.abs().max())
        used = (tile_expert.cpu() >= 0).repeat_interleave(32)
        pad = used & (row_token.cpu() < 0)
        assert not pad.any() or float(y.cpu()[pad].abs().max()) == 0.0
        z = torch.empty((row_token.numel(), n), dtype=dtype, device=DEV)
        ops.grouped_linear(z, a.to(DEV), row_token, w.to(DEV), tile_expert, "silu", scale.to(DEV))
        w2 = act_of(want * scale[rows][:, None], "silu")
        assert float((z.cpu()[rows] - w2).abs().max()) <= 2.0**-8 * float(w2.abs().max())
        # rows that lie where the plan put them
        placed = torch.zeros((row_token.numel(), k), dtype=dtype)
        placed[rows] = a
        ops.grouped_linear(y, placed.to(DEV), None, w.to(DEV), tile_expert)
        assert float((y.cpu()[rows] - want).abs().max()) <= 1e-5 * float(want.abs().max())
    finally:
        ops.set_grouped_linear_form(0)


@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("ff,k", [(64, 64), (24, 128), (100, 192), (33, 320)])
@pytest.mark.parametrize("form", [0, 3, 4])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh", "clamped_glu"])
def test_gated_products(counts, ff, k, form, act):
    from vllm_legacy_amd import _seq_ops as ops
    dtype = torch.bfloat16
    pairs, (pair_row, row_token, tile_expert) = plan_of(counts)
    E, P = len(counts), len(pairs)
    a, w = rnd((P, k), 2).to(dtype), rnd((E, 2 * ff, k), 3, 2 * k**-0.5).to(dtype)
    scale = torch.rand((row_token.numel(), ), generator=torch.Generator().manual_seed(4)) + 0.5
    rows = pair_row.view(-1).cpu()
    both = torch.stack([w[pairs[i]].to(F) @ a[i].to(F) for i in range(P)]) * scale[rows][:, None]
    g, u = both[:, :ff], both[:, ff:]
    if act == "clamped_glu":
        gc, uc = g.clamp(max=1.2), u.clamp(-1.2, 1.2)
        want = gc * torch.sigmoid(1.7 * gc) * (uc + 1.0)
    else:
        want = act_of(g, act) * u
    ops.set_grouped_linear_form(form)
    try:
        out = torch.empty((row_token.numel(), ff), dtype=dtype, device=DEV)
        assert ops.grouped_glu_supported(a.to(DEV), w.to(DEV))
        ops.grouped_glu(out, a.to(DEV), row_token, w.to(DEV), tile_expert, act, scale.to(DEV), 1.2, 1.7, 1.0)
    finally:
        ops.set_grouped_linear_form(0)
    assert float((out.cpu()[rows] - want).abs().max()) <= 2.0**-8 * float(want.abs().max())


@pytest.mark.parametrize("experts", [[0, 1] * 20, [2, -1, 0, 0, -1, 1, 2, 2, 2, 2, 2, 0], [1] * 9 + [0] + [1] * 4])
@pytest.mark.parametrize("form", [0, 3, 4])
def test_tiles_in_any_order(experts, form):
    """Tiles that no plan put in order: an expert's tiles apart from each other, unused ones between them."""
    from vllm_legacy_amd import _seq_ops as ops
    n, k, E, dtype = 72, 128, 3, torch.bfloat16
    rows = 32 * len(experts)
    a, w = rnd((rows, k), 2).to(dtype), rnd((E, 2 * n, k), 3, k**-0.5).to(dtype)
    want = torch.stack([w[max(e, 0)].to(F) @ a[32 * i:32 * i + 32].to(F).t() for i, e in enumerate(experts)]).transpose(1, 2)
    used = torch.tensor(experts) >= 0
    tile_expert = torch.tensor(experts, dtype=torch.int32, device=DEV)
    ops.set_grouped_linear_form(form)
    try:
        y = torch.full((rows, 2 * n), float("nan"), device=DEV)
        ops.grouped_linear(y, a.to(DEV), None, w.to(DEV), tile_expert)
        z = torch.full((rows, n), float("nan"), dtype=dtype, device=DEV)
        ops.grouped_glu(z, a.to(DEV), None, w.to(DEV), tile_expert, "silu")
    finally:
        ops.set_grouped_linear_form(0)
    y, z = y.cpu().view(-1, 32, 2 * n), z.cpu().view(-1, 32, n)
    assert float((y - want)[used].abs().max()) <= 1e-5 * float(want.abs().max())
    glu = act_of(want[..., :n], "silu") * want[..., n:]
    assert float((z - glu)[used].abs().max()) <= 2.0**-8 * float(glu.abs().max())
    assert bool(y[~used].isnan().all() and z[~used].isnan().all())          # unused tiles are left alone


def test_gated_products_refuse_rows_whose_values_lie_apart():
    from vllm_legacy_amd import _seq_ops as ops
    k, ff = 64, 32
    w, tile_expert = torch.zeros((1, 2 * ff, k), dtype=torch.bfloat16, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV)
    a, out = torch.zeros((k, 32), dtype=torch.bfloat16, device=DEV).t(), torch.empty((32, ff), dtype=torch.bfloat16, device=DEV)
    with pytest.raises(AssertionError):
        ops.grouped_glu(out, a, None, w, tile_expert, "silu")

"""The router over 16 tokens a workgroup and the sum four columns at a time (csrc/seq_moe_kernels.hip) against float64, at
the edges of their tiles.  Logits are fp32 sums of `width` products: a score may be off by 1e-5 of itself."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
F = torch.float64


def rnd(shape, seed, std=1.0):
    return std * torch.randn(shape, generator=torch.Generator().manual_seed(seed))


@pytest.mark.parametrize("tokens,width", [(1, 32), (15, 64), (16, 288), (17, 2048), (300, 96)])
@pytest.mark.parametrize("routed,gated", [(2, False), (15, True), (16, True), (32, False), (33, True), (48, False), (63, True), (64, False)])
@pytest.mark.parametrize("score,dtype", [("softmax", torch.bfloat16), ("sigmoid", torch.float16), ("softmax", torch.float32)])
def test_route(tokens, width, routed, gated, score, dtype):
    from vllm_legacy_amd import _seq_ops as ops
    top = min(3, routed)
    h, r = rnd((tokens, width), 1).to(dtype), rnd((routed, width), 2, width**-0.5)
    bias, corr, sg = rnd((routed, ), 3), rnd((routed, ), 4, 0.1), rnd((width, ), 5, width**-0.5)
    groups, keep = (4, 2) if routed % 4 == 0 and top <= routed // 2 else (1, 1)
    hd = torch.zeros(tokens, width + 8, dtype=dtype, device=DEV)
    hd[:, :width] = h.to(DEV)
    hd = hd[:, :width]
    assert ops.moe_route_forms_logits(hd, r.to(DEV), sg.to(DEV) if gated else None) == (routed + gated <= 64)
    e, w, g = ops.moe_route(hd, r.to(DEV), corr.to(DEV), sg.to(DEV) if gated else None, top, None, bias.to(DEV), score, True,
                            groups, keep, 1.5)
    z = h.to(F) @ r.to(F).t() + bias.to(F)
    s = torch.softmax(z, 1) if score == "softmax" else torch.sigmoid(z)
    pick = s + corr.to(F)
    if groups > 1:
        best = pick.view(tokens, groups, -1).amax(2)
        keep_at = best.topk(keep, 1).indices
        shut = torch.ones(tokens, groups, dtype=torch.bool).scatter_(1, keep_at, False)
        pick = pick.masked_fill(shut.repeat_interleave(routed // groups, 1), -float("inf"))
    e = e.cpu().long()
    got = pick.gather(1, e)
    assert float((got - pick.topk(top, 1).values).abs().max()) <= 2e-5           # the best ones, but for ties
    assert all(len(set(row.tolist())) == top for row in e)
    want = s.gather(1, e)
    want = want / want.sum(1, keepdim=True) * 1.5
    assert float(((w.cpu() - want) / want).abs().max()) <= 4e-5
    if gated:
        want = torch.sigmoid(h.to(F) @ sg.to(F))
        assert float(((g.cpu() - want) / want).abs().max()) <= 2e-5


@pytest.mark.parametrize("width", [4, 36, 1020, 1024, 1028, 2052])
@pytest.mark.parametrize("top,shared", [(1, False), (2, True), (7, True)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_combine(width, top, shared, dtype):
    from vllm_legacy_amd import _seq_ops as ops
    T = 9
    y, h, sy = rnd((T * top, width), 1), rnd((T, width), 2).to(dtype), rnd((T, width), 3)
    w, sg = torch.rand(T, top), torch.rand(T)
    pair_row = torch.randperm(T * top, generator=torch.Generator().manual_seed(4)).view(T, top).to(torch.int32)
    pair_row[::4, 0] = -1
    rows = torch.where((pair_row < 0)[..., None], h.to(F)[:, None], y.to(F)[pair_row.clamp(min=0).long()])
    want = (rows * w.to(F)[..., None]).sum(1) + (sg.to(F)[:, None] * sy.to(F) if shared else 0.0)
    out = torch.empty(T, width, device=DEV)
    ops.moe_combine(out, y.to(DEV), pair_row.to(DEV), w.to(DEV), h.to(DEV), sy.to(DEV) if shared else None,
                    sg.to(DEV) if shared else None)
    assert float((out.cpu() - want).abs().max()) <= 2.0**-22 * (top + 2) * float(want.abs().max())

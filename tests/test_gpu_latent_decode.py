"""Latent attention of single rows (csrc/seq_latent_decode.hip) against float64, at the edges of its tiles of 16 keys,
the rows looked up ahead (1024) and the ranges that all sequences' keys are shared out in."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F = "cuda:0", torch.float64


def case(lens, heads, rank, rot, block, dtype, window=0, seed=0, slack=0):
    """A step whose rows see `lens` keys (no window): tensors on the GPU."""
    g = torch.Generator().manual_seed(seed)
    B = len(lens)
    need = [(n + slack + block - 1) // block for n in lens]
    ids = torch.randperm(sum(need) + 2, generator=g).tolist()
    tables, at = torch.zeros(B, max(need), dtype=torch.int32), 0
    for b, n in enumerate(need):
        tables[b, :n] = torch.tensor(ids[at:at + n], dtype=torch.int32)
        at += n

    def rnd(*shape, std=1.0):
        return (std * torch.randn(*shape, generator=g)).to(dtype).to(DEV)

    return dict(cache=rnd(sum(need) + 2, block, rank + rot), tables=tables.to(DEV), scale=0.06,
                q_lat=rnd(B, heads, rank), q_rot=rnd(B, heads, rot), starts=torch.arange(B + 1, dtype=torch.int32, device=DEV),
                ctx=torch.tensor([n - 1 for n in lens], dtype=torch.int32, device=DEV), window=window)


def run(c, gate=None, sinks=None, out=None, max_keys=None):
    from vllm_legacy_amd import _seq_ops as ops
    out = torch.empty_like(c["q_lat"]) if out is None else out
    assert ops.latent_decode_supported(out, c["q_lat"], c["q_rot"], c["cache"])
    ops.latent_decode(out, c["q_lat"], c["q_rot"], c["cache"], c["tables"], c["starts"], c["ctx"],
                      max_keys or int(c["ctx"].max()) + 1, c["scale"], c["window"], gate, sinks)
    return out


def reference(c, gate=None, sinks=None):
    out = []
    for b, n in enumerate((c["ctx"] + 1).tolist()):
        rows = c["cache"].to(F)[c["tables"][b].long()].flatten(0, 1)[max(0, n - c["window"]) if c["window"] else 0:n]
        q = torch.cat([c["q_lat"][b], c["q_rot"][b]], 1).to(F)
        s = (q @ rows.t()) * c["scale"]
        if sinks is not None:
            s = torch.cat([s, sinks.to(F)[:, None]], 1)
        p = torch.softmax(s, -1)[:, :rows.shape[0]]
        o = p @ rows[:, :c["q_lat"].shape[2]]
        out.append(o if gate is None else o * torch.sigmoid(gate[b].to(F))[:, None])
    return torch.stack(out)


def check(got, want, dtype):
    # a result is rounded to 16 bits (up to 2^-8 or 2^-11 of it; weights enter as two numbers); measured, per sequence, 0.002
    # and 0.0003
    rel = ((got.to(F) - want).flatten(1).norm(dim=1) / want.flatten(1).norm(dim=1)).max()
    assert float(rel) <= (0.008 if dtype == torch.bfloat16 else 0.001), float(rel)
    assert not torch.isnan(got).any()


LENS = [[1], [15], [16], [17], [31, 32, 33], [63, 1, 64, 65], [1023, 1024, 1025], [3000], [2048, 1, 2, 700, 96],
        [1 + 13 * i % 190 for i in range(130)], [40] * 600]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lens", LENS, ids=lambda x: f"{len(x)}x{max(x)}")
@pytest.mark.parametrize("rank,rot", [(512, 64), (256, 0)])
def test_lengths(rank, rot, lens, dtype):
    c = case(lens, 16, rank, rot, 16, dtype)
    check(run(c), reference(c), dtype)


@pytest.mark.parametrize("rank,rot", [(512, 0), (256, 64)])
@pytest.mark.parametrize("heads,block,window", [(1, 4, 0), (5, 7, 33), (17, 16, 100), (32, 1, 64), (40, 16, 1)])
def test_heads_pages_windows_gates_and_sinks(rank, rot, heads, block, window):
    lens = [200, 5, 33, 64, 129]
    c = case(lens, heads, rank, rot, block, torch.bfloat16, window)
    gate = torch.randn(len(lens), heads + 3, device=DEV).to(torch.bfloat16)[:, :heads]
    sinks = torch.randn(heads, device=DEV)
    flat = torch.empty(heads, len(lens), rank, dtype=torch.bfloat16, device=DEV).transpose(0, 1)
    check(run(c, gate, sinks, flat), reference(c, gate, sinks), torch.bfloat16)


@pytest.mark.parametrize("ranges_for", [1, 64, 100000])
def test_any_number_of_ranges(ranges_for):
    """How many workgroups share the keys is the host's guess; the result does not depend on it."""
    c = case([500, 31, 1200, 64], 16, 512, 64, 16, torch.bfloat16)
    check(run(c, max_keys=ranges_for), reference(c), torch.bfloat16)


def test_what_lies_behind_the_last_key_does_not_enter():
    lens = [20, 50, 1000]
    c = case(lens, 16, 512, 64, 16, torch.bfloat16)
    want = run(c).clone()
    for b, n in enumerate(lens):
        if n % 16:
            c["cache"][int(c["tables"][b, n // 16]), n % 16:] = math.inf
    assert torch.equal(run(c), want)


@pytest.mark.parametrize("rows", [(0, 16), (16, 32), (0, 64), (640, 768), (5, 6), (0, 33)])
@pytest.mark.parametrize("lens", [[100, 33, 190], [100, 3000, 190, 33]], ids=["whole", "shared"])
def test_scores_that_are_not_numbers(lens, rows):
    """NaN in the rotated part only (no value has it) of some keys, whole tiles and whole ranges among them: every output of
    the sequences that see one is NaN, all others are as they were."""
    c = case(lens, 16, 512, 64, 16, torch.bfloat16)
    want = run(c).clone()
    for b, n in enumerate(lens):
        for j in range(rows[0], min(rows[1], n)) if b else ():
            c["cache"][int(c["tables"][b, j // 16]), j % 16, 512 + j % 64] = math.nan
    got = run(c)
    for b, n in enumerate(lens):
        if b and n > rows[0]:
            assert bool(got[b].isnan().all()), b
        else:
            assert torch.equal(got[b], want[b])


def test_replayed_with_other_lengths():
    c = case([700, 90, 333], 16, 512, 64, 16, torch.bfloat16, slack=2200)
    out = torch.empty_like(c["q_lat"])
    run(c, out=out, max_keys=701)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(c, out=out, max_keys=701)
    for lens in ([700, 90, 333], [1, 2900, 16], [2222, 2223, 2224], [32, 64, 1]):
        c["ctx"].copy_(torch.tensor([n - 1 for n in lens], dtype=torch.int32))
        graph.replay()
        torch.cuda.synchronize()
        check(out, reference(c), torch.bfloat16)


@pytest.mark.parametrize("lens", [[400] * 300, [500] + [1 + 37 * i % 499 for i in range(270)]], ids=["even", "uneven"])
def test_many_sequences_stay_whole(lens):
    from vllm_legacy_amd import _lib
    assert _lib.seq_lib().vla_seq_latent_decode_ranges(len(lens), max(lens), 5) == 0
    c = case(lens, 5, 256, 64, 16, torch.bfloat16)
    check(run(c), reference(c), torch.bfloat16)


def test_no_further_off_than_the_kernel_for_all_steps():
    from vllm_legacy_amd import _seq_ops as ops
    c = case([300, 40, 7, 1100], 16, 512, 64, 16, torch.bfloat16)
    tiles = torch.empty_like(c["q_lat"])
    ops.latent_attention_tiles(tiles, c["q_lat"], c["q_rot"], c["cache"], c["tables"], c["starts"], c["ctx"], 1, c["scale"], 4)
    want, got = reference(c), run(c)
    error = [float((t.to(F) - want).norm() / want.norm()) for t in (tiles, got)]
    assert error[1] <= 1.1 * error[0], error


@pytest.mark.parametrize("heads,rank,rot,vdim,window,extras,takes_up", [
    (16, 512, 64, 128, 0, False, True), (5, 256, 0, 64, 700, True, True), (32, 512, 64, 96, 0, True, False),
    (3, 512, 64, 32, 40, True, None)])
@pytest.mark.parametrize("lens", [[300, 40, 7, 1100, 1], [90, 33, 190]], ids=["shared", "whole"])
def test_layers_take_it(monkeypatch, lens, heads, rank, rot, vdim, window, extras, takes_up):
    """A decode step of a layer goes this way, with its window, gate and sinks, and with its up-projection where the
    kernel takes it (None: weights at an odd address, which it does not)."""
    from vllm_legacy_amd import _seq_ops as ops
    from vllm_legacy_amd.attention.backends.latent_kv import LatentKVAttention
    from vllm_legacy_amd.attention.batch import SequenceBatch
    D, B, g = 48, len(lens), torch.Generator().manual_seed(7)

    def rnd(*shape, std=1.0, dtype=torch.bfloat16):
        return (std * torch.randn(*shape, generator=g)).to(dtype).to(DEV)

    layer = LatentKVAttention(heads, D, rot, vdim, rank, 0.06, rot, 1e4, None, 1e-5, torch.bfloat16, DEV, window=window or None,
                              sinks=extras)
    layer.set_weights(rnd(heads * D, rank, std=rank**-0.5), rnd(heads * vdim, rank, std=rank**-0.5), torch.ones(rank),
                      rnd(heads, dtype=torch.float32) if extras else None)
    if takes_up is None:
        odd = torch.empty(layer.w_uv_t.numel() + 1, dtype=torch.bfloat16, device=DEV)[1:].view(layer.w_uv_t.shape)
        layer.w_uv_t.data = odd.copy_(layer.w_uv_t.data)
    need = [(n + 15) // 16 for n in lens]
    ids, tables = torch.randperm(sum(need), generator=g).tolist(), []
    for n in need:
        tables.append([ids.pop() for _ in range(n)])
    batch = SequenceBatch.build([1] * B, [n - 1 for n in lens], tables, list(range(B)), 16, DEV)
    cache, q, kv = rnd(sum(need), 16, rank + rot), rnd(B, heads * (D + rot)), rnd(B, rank + rot)
    gate = rnd(B, heads) if extras else None
    calls, real = [], ops.latent_decode
    monkeypatch.setattr(ops, "latent_decode", lambda *a: calls.append(a) or real(*a))
    out = layer(q, kv, cache, batch, gate)
    assert len(calls) == 1 and (calls[0][12] is not None) == bool(takes_up)
    q3 = q.to(F).view(B, heads, D + rot)                   # rotated in place; the step's rows are in the cache
    for b, n in enumerate(lens):
        rows = cache.to(F)[torch.tensor(tables[b], device=DEV)].flatten(0, 1)[max(0, n - window) if window else 0:n]
        keys = torch.cat([torch.matmul(layer.w_uk.to(F), rows[:, :rank].t()),
                          rows[:, rank:].t()[None].expand(heads, -1, -1)], 1)             # [heads, D + rot, keys]
        s = torch.matmul(q3[b][:, None], keys.contiguous())[:, 0] * 0.06
        if extras:
            s = torch.cat([s, layer.sinks.to(F)[:, None]], 1)
        o = torch.matmul(torch.softmax(s, 1)[:, :rows.shape[0]], rows[:, :rank])
        if extras:
            o = o * torch.sigmoid(gate[b].to(F))[:, None]
        want = torch.matmul(o[:, None], layer.w_uv_t.to(F))[:, 0].reshape(-1)
        # three roundings to 16 bits: the query's product with W_uk (2^-9 of scores of a few units), the sums, the output
        assert float((out[b].to(F) - want).norm() / want.norm()) <= 0.015, b


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank,vdim,heads", [(512, 128, 16), (256, 32, 3), (512, 256, 2), (256, 64, 17)])
@pytest.mark.parametrize("lens", [[1], [5000], [15, 1, 700], [3000] + [1 + 13 * i % 190 for i in range(15)], [40] * 17, [900] * 33],
                         ids=lambda x: f"{len(x)}x{max(x)}")
def test_up_projection(lens, rank, vdim, heads, dtype):
    """The heads' up-projection in the merge: of the rounded sums, rounded once more."""
    from vllm_legacy_amd import _seq_ops as ops
    c = case(lens, heads, rank, 64, 16, dtype)
    gate = torch.randn(len(lens), heads, device=DEV).to(dtype)
    w = (torch.randn(heads, rank, vdim, device=DEV) * rank**-0.5).to(dtype)
    up = torch.full((len(lens), heads * vdim), float("nan"), dtype=dtype, device=DEV)
    out = torch.empty_like(c["q_lat"])
    assert ops.latent_decode_up_supported(w)
    ops.latent_decode(out, c["q_lat"], c["q_rot"], c["cache"], c["tables"], c["starts"], c["ctx"], max(lens), c["scale"], 0,
                      gate, None, up, w)
    o = reference(c, gate)
    want = torch.matmul(o.transpose(0, 1), w.to(F)).transpose(0, 1).reshape(len(lens), -1)
    check(up, want, dtype)
    alone = run(c, gate, max_keys=max(lens)).to(F)         # and of what the merge leaves
    near = torch.matmul(alone.transpose(0, 1), w.to(F)).transpose(0, 1).reshape(len(lens), -1)
    bound = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    assert float((up.to(F) - near).abs().max()) <= bound * float(near.abs().max()) + 1e-5


@pytest.mark.parametrize("rank,vdim,heads", [(512, 128, 16), (256, 64, 17)])
@pytest.mark.parametrize("lens", [[400] * 137, [9000] + [1 + 29 * i % 411 for i in range(128)]], ids=["even", "uneven"])
def test_up_projection_of_many_sequences(lens, rank, vdim, heads):
    """Sixteen sequences to a workgroup, where eight would be more workgroups than CUs: two to five parts of each, and seventy of one."""
    assert (len(lens) + 7) // 8 * heads > 256
    test_up_projection(lens, rank, vdim, heads, torch.bfloat16)


@pytest.mark.parametrize("rank,vdim,heads,lens", [(512, 256, 17, [400] * 70), (512, 256, 2, [500] * 65), (512, 256, 9, [90] * 70),
                                                  (256, 256, 5, [90] * 20), (256, 128, 5, [90] * 20), (512, 64, 3, [90] * 40)])
def test_up_projection_on_both_sides_of_the_rule(rank, vdim, heads, lens):
    """Sixteen and eight sequences to a workgroup by the columns, the latent dims and whether there are parts."""
    test_up_projection(lens, rank, vdim, heads, torch.bfloat16)


@pytest.mark.parametrize("window,sinks", [(0, True), (100, False), (70, True)])
@pytest.mark.parametrize("lens", [[33, 190, 64, 5], [3000, 33, 700, 64, 5]], ids=["whole", "shared"])
def test_up_projection_with_windows_sinks_and_sequences_without_a_row(lens, window, sinks):
    from vllm_legacy_amd import _seq_ops as ops
    heads, rank, vdim = 6, 512, 64
    c = case(lens, heads, rank, 64, 16, torch.bfloat16, window)
    sink = torch.randn(heads, device=DEV) if sinks else None
    w = (torch.randn(heads, rank, vdim, device=DEV) * rank**-0.5).to(torch.bfloat16)
    want = torch.matmul(reference(c, None, sink).transpose(0, 1), w.to(F)).transpose(0, 1).reshape(len(lens), -1)
    rows = [b for b in range(len(lens)) if b != 1]         # the second sequence has no row in this step
    c["q_lat"], c["q_rot"] = c["q_lat"][rows], c["q_rot"][rows]
    c["starts"] = torch.tensor([0, 1] + list(range(1, len(lens))), dtype=torch.int32, device=DEV)
    up = torch.full((len(rows), heads * vdim), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.latent_decode(torch.empty_like(c["q_lat"]), c["q_lat"], c["q_rot"], c["cache"], c["tables"], c["starts"], c["ctx"],
                      max(lens), c["scale"], window, None, sink, up, w)
    check(up, want[rows], torch.bfloat16)

"""Key / value and latent prompts of sequences of many lengths behind contexts of many lengths, in every way that a step is shared out:
one group of waves to a workgroup and two, tiles of rows found by their rank among one to four registers of sequences,
by the grid, and in the order of the rows -- which one is asserted.  Against the same attention in float64, 1 % of the largest value
in bfloat16 as in the single rows' test; every row is written, and none but those."""
import random

import pytest
import torch

from tests.test_gpu_kv_decode import DEV, rnd

pytestmark = pytest.mark.gpu
ONE, TWO, RANKED, IN_ORDER = 1, 2, 4, 8


def ragged(count, longest, context, seed=0):
    r = random.Random(seed)
    return [(r.randint(1, longest), r.randint(0, context)) for _ in range(count)]


@pytest.mark.parametrize("heads,kv_heads,runs,window,form", [
    (4, 1, [(300, 0)], 0, TWO + RANKED), (4, 1, [(300, 17)], 40, TWO),
    (8, 8, ragged(60, 150, 0), 0, ONE + RANKED), (8, 8, ragged(130, 150, 50, 1), 0, ONE + RANKED),
    (4, 2, ragged(70, 70, 300, 2), 33, TWO + RANKED), (4, 1, ragged(64, 300, 40, 3) + [(1, 900)] * 9, 0, TWO + RANKED),
    (4, 1, [(700, 5)] + ragged(190, 30, 600, 4), 0, TWO + RANKED), (4, 1, ragged(256, 60, 600, 5), 0, TWO + RANKED),
    (16, 4, ragged(250, 40, 90, 6), 0, ONE + RANKED), (16, 4, [(1300, 0), (129, 40), (700, 0), (2100, 0), (64, 8)], 0, ONE + RANKED),
    (8, 8, ragged(300, 130, 90, 7), 0, ONE), (4, 1, ragged(260, 32, 700, 8), 0, TWO),
    (16, 4, ragged(100, 32, 60, 9), 0, ONE), (16, 4, [(64, 0)] * 40, 0, ONE), (16, 4, [(32, 40), (32, 0), (32, 96)], 0, TWO),
    (2, 2, [(64, c % 60) for c in range(270)], 0, ONE), (64, 16, [(64, 0)] * 40, 0, ONE + IN_ORDER),
    (64, 16, [(32, 40), (32, 0), (32, 96)], 0, TWO + IN_ORDER), (64, 16, [(32, c % 60) for c in range(270)], 0, ONE + IN_ORDER)])
def test_all_rows(heads, kv_heads, runs, window, form):
    from vllm_legacy_amd import _lib
    from vllm_legacy_amd import _seq_ops as ops
    D, bs, longest = 32, 16, max(n for n, _ in runs)
    T, need = sum(n for n, _ in runs), [-(-(n + c) // bs) for n, c in runs]
    ids = torch.randperm(sum(need), generator=torch.Generator().manual_seed(3)).split(need)
    kc, vc = (rnd((sum(need), bs, kv_heads, D), s).to(torch.bfloat16) for s in (1, 2))
    tables = torch.zeros((len(runs), max(need)), dtype=torch.int32)
    for b, own in enumerate(ids):
        tables[b, :len(own)] = own
    q = rnd((T, heads * D), 4).to(torch.bfloat16)
    starts = torch.tensor([0] + [n for n, _ in runs]).cumsum(0)
    assert _lib.seq_lib().vla_seq_kv_attention_tiles_form(len(runs), longest, T, heads, kv_heads, D, max(need), bs, window, 0, 0) == form
    out = torch.full((T + 1, heads * D), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.kv_attention_tiles(out[:T], q.to(DEV), None, kc.to(DEV), vc.to(DEV), tables.to(DEV), starts.int().to(DEV),
                           torch.tensor([c for _, c in runs], dtype=torch.int32, device=DEV), longest, None, False, heads, window, D**-0.5)
    got, want = out[:T].double().cpu().view(T, heads, D), torch.empty((T, heads, D), dtype=torch.float64)
    for b, (n, c) in enumerate(runs):
        k, v = (t[ids[b]].reshape(-1, kv_heads, D)[:n + c].double().repeat_interleave(heads // kv_heads, 1).transpose(0, 1).contiguous()
                for t in (kc, vc))
        qs = q[starts[b]:starts[b + 1]].view(n, heads, D).double().transpose(0, 1)
        behind = (torch.arange(n) + c)[:, None] - torch.arange(n + c)[None, :]
        scores = (qs @ k.transpose(1, 2).contiguous()) * D**-0.5
        scores.masked_fill_((behind < 0) | ((behind >= window) & (window > 0)), float("-inf"))
        want[starts[b]:starts[b + 1]] = (torch.softmax(scores, 2) @ v).transpose(0, 1)
    assert float((got - want).abs().max()) <= 0.01 * float(want.abs().max())
    assert bool((out[T:] == 7.0).all())


@pytest.mark.parametrize("sizes,runs,window,form", [
    ((2, 128, 64, 128, 64), [(700, 0)], 0, TWO + RANKED), ((2, 128, 64, 128, 64), ragged(9, 300, 2000, 1), 700, TWO + RANKED),
    ((4, 64, 32, 64, 32), ragged(30, 128, 200, 2), 0, TWO), ((4, 64, 32, 64, 32), ragged(30, 200, 700, 2), 0, TWO + RANKED), ((1, 32, 16, 40, 32), ragged(200, 60, 500, 3), 0, TWO + RANKED),
    ((1, 32, 16, 40, 32), [(1030, 40)] + ragged(260, 30, 20, 4), 0, TWO), ((2, 136, 56, 128, 32), [(1030, 40)] + ragged(20, 200, 30, 5), 0, TWO + RANKED),
    ((2, 128, 64, 128, 64), [(130, 0), (100, 20)], 0, ONE + RANKED), ((8, 128, 64, 72, 64), ragged(80, 250, 500, 6), 300, ONE + RANKED),
    ((3, 64, 0, 64, 32), ragged(256, 120, 60, 7), 0, ONE), ((3, 64, 0, 64, 32), ragged(240, 200, 500, 8), 0, ONE + RANKED),
    ((8, 64, 16, 128, 32), ragged(300, 150, 90, 9), 70, ONE)])
def test_latent_prompts(sizes, runs, window, form):
    """Keys in two parts and values as given."""
    from vllm_legacy_amd import _lib
    from vllm_legacy_amd import _seq_ops as ops
    H, D, R, V, C = sizes
    seen = [n + c - (max(0, c - window + 1) if window else 0) for n, c in runs]
    T, N, longest, bf = sum(n for n, _ in runs), sum(seen), max(n for n, _ in runs), torch.bfloat16
    assert _lib.seq_lib().vla_seq_latent_prompt_form(N, len(runs), longest, H, D, R, V, 0) == form
    q, keys, values, rows = (rnd(s, i).to(bf) for i, s in enumerate([(T, H * (D + R)), (N, H * D), (N, H * V), (N, C + R)]))
    rest = rnd((N, H * D), 9, 2.0**-9).to(bf)
    starts = torch.tensor([0] + [n for n, _ in runs]).cumsum(0)
    out = torch.full((T + 1, H * V), 7.0, dtype=bf, device=DEV)
    scale = (D + R)**-0.5
    ops.latent_prompt(out[:T], *(t.to(DEV) for t in (q, keys, rest, values, rows)), starts.int().to(DEV),
                      torch.tensor([c for _, c in runs], dtype=torch.int32, device=DEV), longest, H, D, R, V, scale, window)
    got, want, at = out[:T].double().cpu().view(T, H, V), torch.empty((T, H, V), dtype=torch.float64), 0
    for b, ((n, c), m) in enumerate(zip(runs, seen)):
        k = (keys[at:at + m].double() + rest[at:at + m].double()).view(m, H, D)
        k = torch.cat([k, rows[at:at + m, C:].double()[:, None].expand(m, H, R)], 2).permute(1, 2, 0).contiguous()
        qs = q[starts[b]:starts[b + 1]].view(n, H, D + R).double().transpose(0, 1).contiguous()
        behind = (torch.arange(n) + c)[:, None] - (torch.arange(m) + c + n - m)[None, :]
        scores = (qs @ k * scale).masked_fill((behind < 0) | ((behind >= window) & (window > 0)), float("-inf"))
        v = values[at:at + m].double().view(m, H, V).transpose(0, 1).contiguous()
        want[starts[b]:starts[b + 1]] = (torch.softmax(scores, 2) @ v).transpose(0, 1)
        at += m
    assert float((got - want).abs().max()) <= 0.01 * float(want.abs().max())
    assert bool((out[T:] == 7.0).all())


def test_the_entry_without_the_number_of_rows():
    """It takes every sequence for as long as the longest: the same bits where that is so."""
    from vllm_legacy_amd import _lib
    from vllm_legacy_amd import _seq_ops as ops
    B, n, H, G, D, bs = 5, 70, 4, 2, 64, 16
    q, kc, vc = (rnd(s, i).to(torch.bfloat16).to(DEV) for i, s in enumerate([(B * n, H * D), (25, bs, G, D), (25, bs, G, D)]))
    tables = torch.randperm(25, generator=torch.Generator().manual_seed(1)).int().view(5, 5).to(DEV)
    starts, ctx = torch.arange(0, B * n + 1, n, dtype=torch.int32, device=DEV), torch.tensor([0, 3, 5, 10, 1], dtype=torch.int32, device=DEV)
    got, want = torch.empty_like(q), torch.empty_like(q)
    ops.kv_attention_tiles(want, q, None, kc, vc, tables, starts, ctx, n, None, False, H, 0, 0.125)
    assert _lib.seq_lib().vla_seq_kv_attention_tiles(
        got.data_ptr(), H * D, q.data_ptr(), H * D, None, 0, kc.data_ptr(), vc.data_ptr(), tables.data_ptr(), 5, starts.data_ptr(),
        ctx.data_ptr(), None, 0, B, n, H, G, D, D, bs, 25, 0, 0.125, _lib.BF16, 0, 0.0, 0, None,
        torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(got, want) and bool(want.isfinite().all())

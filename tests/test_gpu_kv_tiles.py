"""Runs of query rows on the LDS-DMA tile kernel: every key and value size class it exchanges differently, groups of
1 to 4 heads, pages of 1, 4 and 16 tokens, runs around its tiles of 32 rows and 64 keys, windows, chunks, kept
first tokens, caps, sinks, gates, values that turn back, scales of either sign, outputs at odd addresses, one to 1200
sequences of nearly equal lengths (uneven ones in every way that a step is shared out: test_gpu_uneven_prompts.py) -- against the same attention in
float64 and the bound of the single rows' test: 1 % of the largest value in bfloat16, an eighth in float16."""
import pytest
import torch

from tests.test_gpu_kv_decode import DEV, reference, rnd

pytestmark = pytest.mark.gpu

CASES = [
    # heads, kv heads, dim, vdim, page, [(rows, context)], options
    (4, 1, 128, 128, 16, [(65, 0), (1, 64), (33, 95)], {}),
    (4, 2, 64, 64, 4, [(31, 40), (70, 0)], dict(window=50)),
    (2, 2, 96, 32, 1, [(130, 3)], dict(window=40, keep=3, softcap=20.0)),
    (3, 1, 32, 96, 16, [(5, 0), (64, 64)], dict(chunk=48, sink=1.5)),
    (5, 1, 128, 64, 16, [(20, 300)], dict(gate=True, scale=-0.1)),
    (4, 1, 64, 128, 4, [(40, 150)], dict(turn="pairs", gate=True, odd=True)),
    (2, 1, 96, 96, 16, [(35, 129)], dict(turn="halves", window=100, keep=70)),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("copies", [1, 60, 600])
def test_runs_of_rows(case, dtype, copies):
    from vllm_legacy_amd import _seq_ops as ops
    H, G, D, V, bs, runs, opt = case
    window, keep, chunk = opt.get("window", 0), opt.get("keep", 0), opt.get("chunk", 0)
    need = [(n + c + bs - 1) // bs for n, c in runs]
    ids = torch.randperm(sum(need) + 2, generator=torch.Generator().manual_seed(3)).tolist()
    kc, vc = rnd((sum(need) + 2, bs, G, D), 1).to(dtype), rnd((sum(need) + 2, bs, G, V), 2).to(dtype)
    tables = torch.zeros((len(runs), max(need)), dtype=torch.int32)
    keys, values, positions, at = [], [], [], 0
    for i, (n, c) in enumerate(runs):
        own = torch.tensor(ids[at:at + need[i]])
        tables[i, :need[i]] = own
        at += need[i]
        keys += [kc[own].reshape(-1, G, D).double()] * n
        values += [vc[own].reshape(-1, G, V).double()] * n
        positions += list(range(c, c + n))
        if (n + c) % bs:
            kc[own[-1], (n + c) % bs:], vc[own[-1], (n + c) % bs:] = float("nan"), float("nan")
    T = len(positions)
    q, gate = rnd((T, H, D), 4).to(dtype), rnd((T, H + 1), 5).to(dtype) if opt.get("gate") else None
    inv = torch.rand(V // 2, generator=torch.Generator().manual_seed(6)) * 0.1 if opt.get("turn") else None
    inter, scale = opt.get("turn") == "pairs", opt.get("scale", D**-0.5)
    sinks = torch.full((H, ), opt["sink"], device=DEV) if "sink" in opt else None
    lens = torch.tensor([0] + [n for n, c in runs] * copies)
    odd = 1 if opt.get("odd") else 0
    out = torch.full((T * copies, H * V + 4), 7.0, dtype=dtype, device=DEV)
    assert ops.kv_attention_tiles_supported(q.to(DEV), D, V, inv is not None)
    ops.kv_attention_tiles(out[:, odd:odd + H * V], q.reshape(T, -1).repeat(copies, 1).to(DEV),
                           None if gate is None else gate.repeat(copies, 1).to(DEV)[:, :H], kc.to(DEV), vc.to(DEV),
                           tables.repeat(copies, 1).to(DEV), lens.cumsum(0).int().to(DEV),
                           torch.tensor([c for n, c in runs] * copies, dtype=torch.int32, device=DEV),
                           max(n for n, c in runs), None if inv is None else inv.to(DEV), inter, H, window, scale, keep,
                           opt.get("softcap", 0.0), chunk, sinks)

    def lo_of(p):
        return max(p - window + 1 if window else 0, p - p % chunk if chunk else 0)

    want = reference(q.double(), keys, values, None if gate is None else gate.double(), scale, lo_of,
                     keep if window or chunk else 0, opt.get("softcap", 0.0), opt.get("sink"), inv, inter, positions)
    got = out[:, odd:odd + H * V].double().cpu().view(copies, T, H, V)
    tol = (0.01 if dtype == torch.bfloat16 else 0.01 / 8) * float(want.abs().max())
    assert float((got - want).abs().max()) <= tol
    assert bool((out[:, :odd] == 7).all()) and bool((out[:, odd + H * V:] == 7).all())


def test_more_groups_of_heads_than_a_launch_takes():
    """65535 sequences of one row with 257 KV heads: a row that sees one key is that key's value."""
    from vllm_legacy_amd import _seq_ops as ops
    B, H, D = 65535, 257, 32
    q = torch.zeros((B, H * D), dtype=torch.bfloat16, device=DEV)
    kc, vc = (rnd((4, 1, H, D), s).to(torch.bfloat16).to(DEV) for s in (1, 2))
    table = (torch.arange(B, dtype=torch.int32, device=DEV) % 4).view(B, 1)
    out = torch.empty_like(q)
    ops.kv_attention_tiles(out, q, None, kc, vc, table, torch.arange(B + 1, dtype=torch.int32, device=DEV),
                           torch.zeros(B, dtype=torch.int32, device=DEV), 1, None, True, H, 0, 0.1)
    assert torch.equal(out.view(B, H, D), vc[table[:, 0].long(), 0])

"""Latent attention with keys and values formed per head: runs around the tiles of 128 rows and 64 keys, head
sizes around the padding of the two kernels (128 and 192 numbers a key, 64 and 128 a value), windows, gates,
steps that mix long runs with single rows, and what must keep taking the latent kernel.  Oracle and bound
(6 % of the largest value where operands and weights are rounded to bfloat16, an eighth of that in float16) are
those of the other latent tests; against the latent kernel itself the bound is half of that, since both round alike."""
import pytest
import torch

from tests.test_gpu_tekezen import DEV, latent_layer_of, latent_reference, rnd, run_latent

pytestmark = pytest.mark.gpu

SIZES = [(2, 128, 64, 128, 64), (3, 32, 16, 40, 32), (4, 64, 64, 72, 128), (2, 96, 0, 128, 512), (1, 136, 56, 8, 32),
         (2, 8, 8, 64, 32), (1, 136, 48, 8, 32), (2, 8, 16, 64, 64)]


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("cuts,window", [([127, 1, 129], 0), ([257], 70), ([64, 65, 2, 130], 129), ([300], 1), ([128, 128], 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_runs_around_a_tile(sizes, cuts, window, dtype):
    attn, uk, uv, nw = latent_layer_of(sizes, dtype, None, window)
    H, D, Rr, V, C = sizes
    n = sum(cuts)
    q, kv, gate = (t.to(dtype).float() for t in (rnd((n, H * (D + Rr)), 5, 1.5), rnd((n, C + Rr), 6, 1.5), rnd((n, H), 7, 2.0)))
    want, _ = latent_reference(sizes, q, kv, gate, uk, uv, nw, None, window)
    assert attn.formed_min_rows() <= 127
    attn.FORMED_MIN_WORK = 0
    got = run_latent(attn, sizes, q, kv, gate, cuts, dtype)
    bar = 0.06 if dtype == torch.bfloat16 else 0.06 / 8     # three bits more
    assert float((got - want).abs().max()) <= bar * float(want.abs().max())


def step(lens, contexts, block_size=16):
    from vllm_legacy_amd.attention.batch import SequenceBatch
    need = [-(-(n + c) // block_size) for n, c in zip(lens, contexts)]
    ids = torch.randperm(sum(need), generator=torch.Generator().manual_seed(1)).tolist()
    tables = [ids[sum(need[:i]):sum(need[:i + 1])] for i in range(len(need))]
    return SequenceBatch.build(lens, contexts, tables, list(range(len(lens))), block_size, DEV), sum(need)


@pytest.mark.parametrize("lens,contexts", [([1, 1, 200, 130, 1], [50, 3, 0, 77, 400]), ([150], [333]),
                                           ([140, 2, 150, 2, 160, 2], [0, 9, 10, 300, 5, 1]), ([31, 63, 300], [64, 0, 1])])
@pytest.mark.parametrize("window,sinks", [(0, True), (100, False)])
def test_stretches_of_a_step_agree_with_the_latent_kernel(lens, contexts, window, sinks):
    from dataclasses import replace
    from vllm_legacy_amd.attention.backends.latent_kv import LatentKVAttention
    H, D, Rr, V, C = 4, 128, 64, 128, 128
    batch, blocks = step(lens, contexts)
    attn = LatentKVAttention(H, D, Rr, V, C, (D + Rr)**-0.5, Rr, 1e4, None, 1e-5, torch.bfloat16, DEV, window=window or None,
                             sinks=sinks)
    attn.set_weights(rnd((H * D, C), 1, C**-0.5), rnd((H * V, C), 2, C**-0.5), 1 + 0.1 * rnd((C, ), 3),
                     rnd((H, ), 4) if sinks else None)
    attn.FORMED_MIN_WORK = 0
    T = sum(lens)
    q, kv, gate = (rnd((T, w), s).to(torch.bfloat16).to(DEV) for w, s in ((H * (D + Rr), 5), (C + Rr, 6), (H + 3, 7)))
    cache = rnd((blocks, 16, C + Rr), 8).to(torch.bfloat16).to(DEV)
    stretches = attn._stretches(batch)
    assert (stretches is None) == (len(lens) == 6)          # a step that alternates too often stays whole
    got = attn(q.clone(), kv, cache.clone(), batch, gate[:, 1:H + 1])
    want = attn(q.clone(), kv, cache.clone(), replace(batch, host_query_lens=None), gate[:, 1:H + 1])
    assert float((got - want).abs().max()) <= 0.03 * float(want.abs().max())
    assert torch.equal(got, want) == (stretches is None)


def test_what_keeps_the_latent_kernel():
    from vllm_legacy_amd.attention.backends.latent_kv import LatentKVAttention
    batch, _ = step([200], [0])
    for scale, rank, dtype, formed in ((0.1, 64, torch.bfloat16, True), (-0.1, 64, torch.bfloat16, False),
                                       (0.0, 64, torch.bfloat16, False)):
        attn = LatentKVAttention(2, 32, 0, 32, rank, scale, 0, 1e4, None, 1e-5, dtype, DEV)
        assert attn._stretches(batch) is None           # too little work for the launches
        attn.FORMED_MIN_WORK = 0
        assert (attn._stretches(batch) is not None) == formed


@pytest.mark.parametrize("common", [0.0, 3.0])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_no_further_from_64_bits_than_the_latent_kernel(common, dtype):
    """Latents with and without a part that all tokens share, values that do not see it, scores four times as large
    as usual: where a key's own rounding would show, since a query's is the same for all keys of a row.  (With keys
    rounded to 16 bits the errors' ratio is 1.03 without a common part.)"""
    from dataclasses import replace
    from vllm_legacy_amd.attention.backends.latent_kv import LatentKVAttention
    n, H, D, Rr, V, C, F = 512, 4, 128, 64, 128, 512, torch.float64
    batch, blocks = step([n], [0])
    attn = LatentKVAttention(H, D, Rr, V, C, 4 * (D + Rr)**-0.5, 0, 1e4, None, 1e-5, dtype, DEV)
    shared, uv = rnd((1, C), 9), rnd((H * V, C), 2, C**-0.5)
    uv = uv - (uv @ shared.t()) @ shared / (shared @ shared.t())
    attn.set_weights(rnd((H * D, C), 1, C**-0.5), uv, torch.ones(C))
    attn.FORMED_MIN_WORK = 0
    q = rnd((n, H * (D + Rr)), 5).to(dtype).to(DEV)
    kv = torch.cat([rnd((n, C), 6) + common * shared, rnd((n, Rr), 7)], 1).to(dtype).to(DEV)
    cache = torch.zeros((blocks, 16, C + Rr), dtype=dtype, device=DEV)
    formed = attn(q.clone(), kv, cache, batch)
    latent = attn(q.clone(), kv, cache, replace(batch, host_query_lens=None))
    rows = cache[batch.block_tables[0].long()].view(-1, C + Rr)[:n].to(F)
    unseen = torch.ones((n, n), dtype=torch.bool, device=DEV).triu(1)
    want = []
    for h in range(H):
        qh = q.view(n, H, D + Rr)[:, h].to(F)
        s = (qh[:, :D] @ (rows[:, :C] @ attn.w_uk.data[h].to(F).t()).t() + qh[:, D:] @ rows[:, C:].t()) * attn.scale
        want.append(torch.softmax(s.masked_fill(unseen, float("-inf")), 1) @ (rows[:, :C] @ attn.w_uv_t.data[h].to(F)))
    want = torch.stack(want, 1)
    errors = [float((x.view(n, H, V).to(F) - want).norm() / want.norm()) for x in (formed, latent)]
    assert errors[0] <= errors[1], errors


def layer_and_step(lens, contexts, sizes, window=0, sinks=False, dtype=torch.bfloat16):
    from vllm_legacy_amd.attention.backends.latent_kv import LatentKVAttention
    H, D, Rr, V, C = sizes
    batch, blocks = step(lens, contexts)
    attn = LatentKVAttention(H, D, Rr, V, C, (D + Rr)**-0.5, Rr, 1e4, None, 1e-5, dtype, DEV, window=window or None, sinks=sinks)
    attn.set_weights(rnd((H * D, C), 1, C**-0.5), rnd((H * V, C), 2, C**-0.5), 1 + 0.1 * rnd((C, ), 3),
                     rnd((H, ), 4) if sinks else None)
    attn.FORMED_MIN_WORK, attn.FORMED_MIN_ROWS = 0, 32
    T = sum(lens)
    q, kv, gate = (rnd((T, w), s).to(dtype).to(DEV) for w, s in ((H * (D + Rr), 5), (C + Rr, 6), (H, 7)))
    return attn, batch, q, kv, gate, rnd((blocks, 16, C + Rr), 8).to(dtype).to(DEV)


@pytest.mark.parametrize("sizes", [(4, 128, 64, 128, 128), (3, 40, 16, 56, 64), (2, 136, 56, 72, 32), (2, 136, 48, 72, 32)])
@pytest.mark.parametrize("lens,contexts", [([70, 64, 200], [500, 64, 0]), ([300], [1000]), ([50, 60], [1500, 3])])
@pytest.mark.parametrize("window,sinks", [(0, True), (150, False), (700, True)])
def test_a_workspace_of_few_keys(sizes, lens, contexts, window, sinks):
    """Sequences and ranges of a sequence's keys one after the other: as with all keys at once (the products over
    fewer rows may sum in another order: one rounding of a key), in no more memory than the workspace."""
    attn, batch, q, kv, gate, cache = layer_and_step(lens, contexts, sizes, window, sinks)
    want = attn(q.clone(), kv, cache.clone(), batch, gate)
    H, D, Rr, V, C = sizes
    each = 2 * (C + Rr + H * (2 * D + V))
    for keys in (64, 192, 640):
        attn.FORMED_WORKSPACE = keys * each
        assert attn.formed_keys(2) == keys
        q2, cache2 = q.clone(), cache.clone()
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        held = torch.cuda.memory_allocated()
        got = attn(q2, kv, cache2, batch, gate)
        assert float((got - want).abs().max()) <= 0.008 * float(want.abs().max())
        rows_own = sum(lens) * H * (4 * 132 + 2 * V) + 2 * H * C * V
        assert torch.cuda.max_memory_allocated() - held <= keys * each + rows_own + (1 << 20)


@pytest.mark.parametrize("sizes,formed", [((2, 64, 8, 64, 64), False), ((2, 64, 0, 64, 40), False), ((2, 128, 64, 128, 48), False),
                                          ((2, 64, 16, 64, 64), True)])
def test_sizes_whose_weights_have_32_bits(sizes, formed):
    """Ranks and rotated parts that the matrix-core latent kernel does not take go to the kernel that keeps a weight in
    32 bits, whatever the run's length."""
    from dataclasses import replace
    attn, batch, q, kv, gate, cache = layer_and_step([200, 3], [40, 9], sizes)
    assert attn._stretches(batch) is not None
    got = attn(q.clone(), kv, cache.clone(), batch, gate)
    want = attn(q.clone(), kv, cache.clone(), replace(batch, host_query_lens=None), gate)
    assert torch.equal(got, want) != formed


@pytest.mark.parametrize("which,size", [("uk", 1.0), ("uk", 3e4), ("uv", 3e3), ("uv", 3e4)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_values_that_leave_the_range(which, size, dtype):
    """Weights with which a key or a value can be more than float16 holds, where the sums on the latents' side are not:
    those stay there."""
    from vllm_legacy_amd.attention.backends.latent_kv import LatentKVAttention
    H, D, Rr, V, C, n = 2, 32, 16, 32, 64, 150
    batch, blocks = step([n], [0])
    attn = LatentKVAttention(H, D, Rr, V, C, 1e-4, 0, 1e4, None, 1e-5, dtype, DEV)
    w = {"uk": rnd((H * D, C), 1, C**-0.5), "uv": rnd((H * V, C), 2, C**-0.5)}
    w[which] = w[which] * size
    attn.set_weights(w["uk"], w["uv"], torch.ones(C))
    attn.FORMED_MIN_WORK = 0
    fits = dtype == torch.bfloat16 or size < 1e4
    assert (attn._stretches(batch) is not None) == fits
    q, kv = (rnd((n, x), s, 1.0 if s == 6 else 0.25).to(dtype).to(DEV) for x, s in ((H * (D + Rr), 5), (C + Rr, 6)))
    cache = torch.zeros((blocks, 16, C + Rr), dtype=dtype, device=DEV)
    got = attn(q, kv, cache, batch).view(n, H, V).double()
    rows = cache[batch.block_tables[0].long()].view(-1, C + Rr)[:n].double()
    unseen = torch.ones((n, n), dtype=torch.bool, device=DEV).triu(1)
    for h in range(H):
        qh, u = q.view(n, H, D + Rr)[:, h].double(), attn.w_uk.data[h].double()
        s = (qh[:, :D] @ (rows[:, :C] @ u.t()).t() + qh[:, D:] @ rows[:, C:].t()) * attn.scale
        want = torch.softmax(s.masked_fill(unseen, float("-inf")), 1) @ (rows[:, :C] @ attn.w_uv_t.data[h].double())
        live = want.abs().amax(1) < 6e4         # outputs that float16 holds
        bar = 0.06 if dtype == torch.bfloat16 else 0.06 / 8
        assert bool(live[20:].all()) and float((got[live, h] - want[live]).abs().max()) <= bar * float(want[live].abs().max())


@pytest.mark.parametrize("lens,contexts,most", [([48], [1 << 17], 19968), ([100, 3000, 64, 64], [0, 50000, 9, 900], 4096),
                                                ([64] * 40, [1000] * 40, 2048), ([64, 64], [0, 0], 64)])
@pytest.mark.parametrize("window", [0, 1024])
def test_parts_of_a_step(lens, contexts, most, window):
    """Every visible key of every sequence once, in order, at most so many at a time."""
    from vllm_legacy_amd.attention.backends.latent_kv import LatentKVAttention
    attn = LatentKVAttention(2, 32, 0, 32, 64, 0.1, 0, 1e4, None, 1e-5, torch.bfloat16, DEV, window=window or None)
    parts = attn._formed_parts(lens, contexts, most)
    counts = [c + n - (max(0, c - window + 1) if window else 0) for n, c in zip(lens, contexts)]
    at = key = 0
    for b0, b1, k0, count, total in parts:
        assert 0 < count <= most and (b0, k0) == (at, key)
        if b1 > b0 + 1 or count == total:
            assert k0 == 0 and count == total == sum(counts[b0:b1])
            at = b1
        else:
            assert total == counts[b0] and (count % 64 == 0 or k0 + count == total)
            at, key = (b1, 0) if k0 + count == total else (b0, k0 + count)
    assert (at, key) == (len(lens), 0)


@pytest.mark.parametrize("row", [0, 1, 31, 40, 63, 64, 127, 200])
@pytest.mark.parametrize("window", [0, 70])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_rows_that_do_not_see_one_that_is_not_finite(row, window, value):
    """Bit for bit what they are without it."""
    attn, batch, q, kv, gate, cache = layer_and_step([230, 66], [30, 0], (4, 128, 64, 128, 128), window)
    clean = attn(q.clone(), kv, cache.clone(), batch, gate)
    assert bool(clean.isfinite().all())
    kv[row, 5] = value
    got = attn(q.clone(), kv, cache.clone(), batch, gate)
    sees = torch.zeros(len(got), dtype=torch.bool, device=DEV)
    sees[row:min(230, row + window) if window else 230] = True
    assert torch.equal(got[~sees], clean[~sees]) and not got[sees].isfinite().any()


@pytest.mark.parametrize("seqs", [1, 40, 65, 130, 256, 257, 300])
@pytest.mark.parametrize("window", [0, 600])
def test_one_group_of_waves_and_two(seqs, window):
    """Many workgroups have one group of waves and find their tiles by their rank (up to 256 sequences) or by the grid;
    a small workspace makes few of them, which share a tile's keys out to two groups: one rounding of an output."""
    from vllm_legacy_amd import _lib
    lens, contexts = [129 + 11 * (i % 13) for i in range(seqs)], [420 + 7 * (i % 9) for i in range(seqs)]
    sizes = (4, 128, 64, 128, 128)
    attn, batch, q, kv, gate, cache = layer_and_step(lens, contexts, sizes, window)
    form = lambda n, c: _lib.seq_lib().vla_seq_latent_prompt_form(sum(n) + sum(c), len(n), max(n), 4, 128, 64, 128, 0)
    assert form(lens, contexts) == (1 if seqs > 256 else 5 if seqs > 30 else 6) and form(lens[:3], contexts[:3]) == 6
    want = attn(q.clone(), kv, cache.clone(), batch, gate)
    attn.FORMED_WORKSPACE = 2048 * 2 * (128 + 64 + 4 * 384)
    got = attn(q.clone(), kv, cache.clone(), batch, gate)
    assert float((got - want).abs().max()) <= 0.008 * float(want.abs().max())
    assert float(want.abs().max()) > 0.1 and bool(want.isfinite().all())
    assert torch.equal(got, want) == (seqs == 1)


def test_lengths_that_are_not_the_hosts():
    """Rows of a sequence that grew on the device are NaN, not what memory held; a captured step takes the latent
    kernel, which follows the device."""
    from dataclasses import replace
    attn, batch, q, kv, gate, cache = layer_and_step([100, 80], [200, 40], (2, 64, 0, 64, 64))
    good = attn(q.clone(), kv, cache.clone(), batch, gate)
    got = attn(q.clone(), kv, cache.clone(), replace(batch, host_context_lens=[136, 40]), gate)
    assert bool(got[100:].isnan().all()) and torch.equal(got[:100], good[:100])
    attn.FORMED_WORKSPACE = 0
    got = attn(q.clone(), kv, cache.clone(), replace(batch, host_context_lens=[136, 40]), gate)
    assert bool(got[:100].isnan().all())
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    assert attn._stretches(batch) is not None
    with torch.cuda.stream(stream):
        graph.capture_begin()
        inside = attn._stretches(batch)
        graph.capture_end()
    assert inside is None


@pytest.mark.parametrize("seqs,fit", [(4, 2), (4, 0), (70, 66), (200, 130), (300, 290)])
@pytest.mark.parametrize("window", [0, 400])
def test_sequences_that_rows_were_not_gathered_for(seqs, fit, window):
    """From the first sequence on that grew on the device all rows are NaN, those ahead of it what they are without; there
    are more tiles of rows than the host's lengths have."""
    from dataclasses import replace
    lens, contexts = [40 + 37 * (i % 4) for i in range(seqs)], [90 + 11 * (i % 5) for i in range(seqs)]
    grown = contexts[:fit] + [c + 200 for c in contexts[fit:]]
    attn, batch, q, kv, gate, cache = layer_and_step(lens, grown, (2, 64, 0, 64, 64), window)
    want = attn(q.clone(), kv, cache.clone(), batch, gate)
    got = attn(q.clone(), kv, cache.clone(), replace(batch, host_context_lens=contexts), gate)
    # (the first one may still find room among the rows of those behind it)
    ends = [sum(n + c for n, c in zip(lens[:b + 1], grown)) for b in range(seqs)]
    held = sum(1 for e in ends if e <= sum(lens) + sum(contexts))
    rows = sum(lens[:held])
    assert fit <= held < seqs and bool(want.isfinite().all())
    assert torch.equal(got[:rows], want[:rows]) and bool(got[rows:].isnan().all())


@pytest.mark.parametrize("workspace", [1 << 28, 1 << 22])
def test_a_portion_of_a_long_context(workspace):
    """A hundred thousand cached tokens, all at once and in ranges, beside the latent kernel."""
    from dataclasses import replace
    attn, batch, q, kv, gate, cache = layer_and_step([70, 50], [100000, 33], (2, 64, 32, 64, 64))
    attn.FORMED_WORKSPACE = workspace
    assert (attn.formed_keys(2) > 100200) == (workspace == 1 << 28)
    got = attn(q.clone(), kv, cache.clone(), batch, gate)
    want = attn(q.clone(), kv, cache.clone(), replace(batch, host_query_lens=None), gate)
    for rows in (slice(0, 70), slice(70, 120)):
        assert float((got[rows] - want[rows]).abs().max()) <= 0.03 * float(want[rows].abs().max())


@pytest.mark.parametrize("rows", [1, 255, 257, 600])
@pytest.mark.parametrize("sizes", [(1, 8, 16, 8, 32), (3, 40, 0, 72, 64), (2, 128, 64, 128, 96), (5, 136, 16, 120, 128), (16, 128, 64, 64, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_formed_keys_and_values(rows, sizes, dtype):
    """Around tiles of 256 rows and 128 columns, one to sixteen stages of the rank, heads that share a tile or part of one,
    weights at odd addresses: a key and what it lost together to 2 roundings of 16 bits and the sum's own (2^-24 of the
    terms' sum, by their number), a key or value alone to one."""
    from vllm_legacy_amd import _seq_ops as ops
    H, D, Rr, V, C = sizes
    x = rnd((rows, C + Rr), 1).to(dtype).to(DEV)
    w_uk, w_uv = (rnd((H * D * C + 1, ), 2, C**-0.5).to(dtype).to(DEV), rnd((H * C * V + 1, ), 3, C**-0.5).to(dtype).to(DEV))
    eps = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    tiny = 2.0**-24 if dtype == torch.float16 else 0.0      # what a remainder below the least normal number keeps
    for off in (0, 1):
        uk, uv = w_uk[off:off + H * D * C].view(H, D, C), w_uv[off:off + H * C * V].view(H, C, V)
        keys, rest, values = ops.latent_form(x, uk, uv)
        lat = x[:, :C].double().cpu()
        for got, left, w in ((keys, rest, uk.double().cpu().reshape(H * D, C).t()),
                             (values, None, uv.double().cpu().transpose(0, 1).reshape(C, H * V))):
            want, terms = lat @ w, lat.abs() @ w.abs()
            got = got.double().cpu()
            bar = eps * want.abs() + C * 2.0**-24 * terms + tiny
            assert bool(((got - want).abs() <= bar).all())
            if left is not None:
                assert bool(((got + left.double().cpu() - want).abs() <= 2 * eps * eps * want.abs() + C * 2.0**-24 * terms + tiny).all())


def test_which_steps_are_formed():
    """Short runs where few keys are ahead of them, heads are many and the rank is large, and steps of both kinds only where
    there is enough for two ways."""
    from vllm_legacy_amd.attention.backends.latent_kv import LatentKVAttention
    for H, C, lens, contexts, want in ((16, 512, [33], [0], [True]), (16, 512, [31], [0], None), (16, 512, [33], [300], [True]),
                                       (16, 512, [48], [300], [True]), (16, 512, [60], [2000], None), (16, 512, [64], [2000], None),
                                       (16, 512, [33] * 30, [1000] * 30, None), (16, 512, [64] * 30, [300] * 30, [True]),
                                       (16, 512, [54] * 3, [1240] * 3, [True]), (16, 512, [96], [4000], [True]), (16, 512, [48] * 4, [2000] * 4, [True]),
                                       (16, 512, [64, 20], [0, 0], None), (16, 512, [64, 60], [0, 2000], None),
                                       (16, 512, [1000, 20], [0, 0], [True, False]), (16, 512, [1000, 40], [0, 40], [True]),
                                       (16, 512, [1000, 33], [0, 4000], [True, False]), (16, 64, [96], [1500], None),
                                       (16, 64, [1024], [0], [True]), (1, 512, [128], [1500], None), (4, 512, [128], [2500], None), (1, 512, [512], [0], None)):
        attn = LatentKVAttention(H, 128, 64, 128, C, 192**-0.5, 64, 1e4, None, 1e-5, torch.bfloat16, DEV)
        got = attn._stretches(step(lens, contexts)[0])
        assert (got and [s[4] for s in got]) == want, (H, C, lens, contexts)

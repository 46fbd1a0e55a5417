"""The gated linear recurrence in chunks of 64 rows: runs around one and two chunks and blocks of 16 beside
single rows and continued sequences, every head size it takes, ranks 1 to 32, decays that underflow beside
decays of one, 16-bit rows -- against the float64 oracle of the recurrence's other tests and their bound for
fp32 rows (sums of a few hundred terms: 3e-5 of the largest value; 16-bit results: one rounding, 2^-8)."""
import pytest
import torch

from tests import lusadra_oracle as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def close(got, want, tol):
    assert float((got.double().cpu() - want).abs().max()) <= tol * float(want.abs().max())


def run(H, D, V, rank, lens, ctx, dtype, bias_of=None, offset=0):
    from vllm_legacy_amd.attention.batch import SequenceBatch
    from vllm_legacy_amd.attention.recurrent import GatedLinearRecurrence
    tau, eps, T = 5.0, 1e-5, sum(lens)
    layer = GatedLinearRecurrence(H, D, V, tau, eps)
    layer.CHUNK_ALONE_ROWS = 0              # however little there is to do
    g = torch.Generator().manual_seed(D + V + T)
    slots = list(range(len(lens)))[::-1]
    state = torch.randn(GatedLinearRecurrence.get_state_shape(len(lens), H, D, V), generator=g).to(DEV)
    before = state.cpu().double()
    w2 = (torch.randn(H * D, rank, generator=g) * 0.5).to(dtype)
    bias = torch.randn(H * D, generator=g) + 2 if bias_of is None else bias_of(H * D)
    norm_w = torch.randn(V, generator=g)
    widths = [H * D, H * D, H * V, H * V, rank]
    wide = torch.randn(T, sum(widths) + 8, generator=g).to(dtype)
    q, k, v, gate, y = wide[:, offset:offset + sum(widths)].split(widths, 1)
    q, k, v, gate, y = wide.to(DEV)[:, offset:offset + sum(widths)].split(widths, 1)
    b = SequenceBatch.build(lens, ctx, [[0] * 64] * len(lens), slots, 16, DEV)
    out = torch.empty(T, H * V, device=DEV, dtype=dtype)
    layer(out, q, k, v, gate, y, w2.to(DEV), bias.to(DEV), norm_w.to(DEV), state, b, 0.8)
    F, at, bar = R.F, 0, 3e-5 if dtype == torch.float32 else 2.0**-8
    q, k, v, gate, y = (t.cpu().to(F) for t in (q, k, v, gate, y))
    for i, (n, c) in enumerate(zip(lens, ctx)):
        rows = slice(at, at + n)
        ln_a = R.log_decay(y[rows], w2.to(F), bias.to(F), tau)
        S = before[slots[i]] if c else torch.zeros(H, D, V, dtype=F)
        a, o = torch.exp(ln_a).view(n, H, D), torch.empty(n, H, V, dtype=F)
        for t in range(n):
            S = a[t][:, :, None] * S + k[rows][t].view(H, D, 1) * v[rows][t].view(H, 1, V)
            o[t] = (S * (q[rows][t] * D**-0.5).view(H, D, 1)).sum(1)
        want = R.gated_head_norm(o, norm_w.to(F), gate[rows], eps, 0.8).reshape(n, H * V)
        close(out[rows], want, bar)
        close(state[slots[i]], S, 3e-5)
        at += n
    return layer


@pytest.mark.parametrize("shape", [(2, 16, 16, 1), (3, 32, 48, 5), (2, 64, 128, 16), (1, 128, 128, 32), (2, 128, 112, 7)])
@pytest.mark.parametrize("lens,ctx", [([64], [0]), ([63, 1, 65], [0, 7, 3]), ([130, 17, 2, 128], [5, 0, 1, 0]), ([1, 200], [0, 0])])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_runs_around_a_chunk(shape, lens, ctx, dtype):
    run(*shape, lens, ctx, dtype)


@pytest.mark.parametrize("shape", [(2, 64, 48, 8), (3, 32, 80, 16), (1, 128, 112, 8), (2, 16, 64, 24)])
@pytest.mark.parametrize("lens,ctx", [([64, 65], [0, 3]), ([127, 130, 2], [5, 0, 1])])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_results_eight_columns_at_a_time(shape, lens, ctx, dtype):
    """Rows of gates and results in 16-byte pieces, value sizes that fill the halves of 64 columns or leave part of one."""
    run(*shape, lens, ctx, dtype)


@pytest.mark.parametrize("lens,ctx", [([128, 129], [1, 0]), ([320, 321], [0, 2]), ([512, 513], [0, 0]), ([640, 641, 1], [3, 0, 0]),
                                      ([960, 64, 1000], [0, 1, 1])])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_runs_of_as_many_chunks_as_are_on_their_way(lens, ctx, dtype):
    """2, 5, 8 and 10 chunks and one more, whole groups of eight and the rest of one."""
    run(1, 32, 48, 5, lens, ctx, dtype)


def test_decays_are_as_exact_as_with_the_library(monkeypatch):
    """ln sigmoid(z) of one chunk (where the kernels leave it for each other) against float64: an error, root mean square,
    of no more than that of fp32 exp and log1p (3.3e-8), but for 5 % for the sample."""
    from vllm_legacy_amd import _seq_ops as ops
    H, D, V, n = 16, 128, 16, 64
    g = torch.Generator().manual_seed(5)
    y, w2 = torch.linspace(-3.0, 6.0, n)[:, None], torch.rand(H * D, 1, generator=g) * 0.5 + 0.5
    row = torch.zeros(n, H * D, device=DEV)
    small = torch.zeros(n, H * V, device=DEV)
    i32 = dict(dtype=torch.int32, device=DEV)
    need = ops.gla_chunks_scratch(row, row, small, H, D, V, 1, 1)
    kept, real = [], torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, **k: kept.append(real(*a, **k)) or kept[-1])
    ops.gla_chunks(torch.empty_like(small), row, row, small, small, y.to(DEV), w2.to(DEV), None, torch.ones(V, device=DEV),
                   torch.zeros(1, H, D, V, device=DEV), torch.tensor([0, n], **i32), torch.tensor([0], **i32),
                   torch.tensor([0], **i32), 1.0, 1.0, 1e-5, 1.0, need)
    monkeypatch.undo()
    scratch = next(t for t in kept if t.numel() == need).cpu()
    per = n * D + D + D * V
    got = torch.stack([scratch[h * per:h * per + n * D].view(n, D) for h in range(H)], 1).reshape(n, H * D)
    z = y * w2.t()                              # one rounding, as the kernel's
    want = torch.nn.functional.logsigmoid(z.double())
    plain = -((-z).clamp(min=0) + torch.log1p(torch.exp(-z.abs())))

    def error(t):
        return float(((t.double() - want) / want).square().mean().sqrt())

    assert error(got) <= 1.05 * error(plain), (error(got), error(plain))


def test_decays_of_nothing_and_of_one():
    def bias_of(n):
        b = torch.full((n, ), 60.0)         # 1
        b[::3] = -500.0                     # 0
        b[1::3] = -8.0
        return b

    run(2, 64, 128, 4, [150, 70], [3, 0], torch.float32, bias_of)


@pytest.mark.parametrize("offset", [0, 1, 4])
def test_rows_at_odd_addresses_go_the_other_way(offset):
    from vllm_legacy_amd import _seq_ops as ops
    run(2, 32, 32, 3, [100], [0], torch.bfloat16, offset=offset)
    rows = torch.empty((100, 200), dtype=torch.bfloat16, device=DEV)[:, offset:offset + 64]
    assert (ops.gla_chunks_scratch(rows, rows, rows, 2, 32, 32, 3, 1) > 0) == (offset % 4 == 0)
    rows = torch.empty((100, 200), dtype=torch.bfloat16, device=DEV)[:, :64]
    assert ops.gla_chunks_scratch(rows, rows, rows, 2, 24, 32, 3, 1) == 0
    assert ops.gla_chunks_scratch(rows, rows, rows, 2, 32, 32, 33, 1) == 0


@pytest.mark.parametrize("what,value", [("v", float("inf")), ("v", float("nan")), ("k", float("-inf")), ("y", float("nan")),
                                        ("q", float("inf"))])
@pytest.mark.parametrize("row", [0, 5, 15, 16, 63, 64, 100, 129])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rows_ahead_of_one_that_is_not_finite(what, value, row, dtype):
    """Bit for bit what they are without it, as token by token; it and the rows behind it are not finite exactly
    where a walk in float64 says so; other heads and sequences know nothing of it."""
    from vllm_legacy_amd.attention.batch import SequenceBatch
    from vllm_legacy_amd.attention.recurrent import GatedLinearRecurrence
    H, D, V, rank, lens = 2, 32, 48, 3, [130, 70]
    T, g = sum(lens), torch.Generator().manual_seed(row)
    layer = GatedLinearRecurrence(H, D, V, 5.0, 1e-5)
    rows = {"q": H * D, "k": H * D, "v": H * V, "gate": H * V, "y": rank}
    rows = {name: torch.randn(T, n, generator=g).to(dtype) for name, n in rows.items()}
    w2, bias, norm_w = torch.randn(H * D, rank, generator=g).to(dtype), torch.randn(H * D, generator=g) + 2, torch.ones(V)
    b = SequenceBatch.build(lens, [0, 0], [[0] * 64] * 2, [0, 1], 16, DEV)

    def go(r):
        state = torch.zeros(GatedLinearRecurrence.get_state_shape(2, H, D, V), device=DEV)
        out = torch.empty(T, H * V, device=DEV, dtype=dtype)
        layer(out, *(r[name].to(DEV) for name in ("q", "k", "v", "gate", "y")), w2.to(DEV), bias.to(DEV), norm_w.to(DEV), state, b,
              1.0)
        return out.float().cpu().view(T, H, V), state.cpu()

    clean, clean_state = go(rows)
    rows[what] = rows[what].clone()
    rows[what][row, 1] = value                  # head 0 (a decay's row: both heads)
    got, state = go(rows)
    assert torch.equal(got[:row], clean[:row]) and torch.equal(got[lens[0]:], clean[lens[0]:])
    assert torch.equal(state[1], clean_state[1])
    if what != "y":
        assert torch.equal(got[:, 1], clean[:, 1]) and torch.equal(state[0, 1], clean_state[0, 1])
    q, k, v, y = (rows[name].to(R.F)[:lens[0]] for name in ("q", "k", "v", "y"))
    a = torch.exp(R.log_decay(y, w2.to(R.F), bias.to(R.F), 5.0)).view(-1, H, D)
    S, o = torch.zeros(H, D, V, dtype=R.F), torch.empty(lens[0], H, V, dtype=R.F)
    for t in range(lens[0]):
        S = a[t][:, :, None] * S + k[t].view(H, D, 1) * v[t].view(H, 1, V)
        o[t] = (S * q[t].view(H, D, 1)).sum(1)
    want = R.gated_head_norm(o, norm_w.to(R.F), rows["gate"].to(R.F)[:lens[0]], 1e-5, 1.0).reshape(-1, H, V)
    assert torch.equal(got[:lens[0]].isfinite(), want.isfinite())
    assert torch.equal(state[0].isfinite(), S.isfinite())


@pytest.mark.parametrize("row", [0, 15, 16, 63, 64, 100, 129])
@pytest.mark.parametrize("D,V", [(16, 16), (32, 48), (64, 128), (128, 112)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_states_of_infinite_values(dtype, D, V, row):
    """A state that a walk in float64 leaves infinite is so, with its sign, not NaN; keys of 0 and values of both signs are
    NaN there and here; the other columns are, bit for bit, what they are without such values."""
    from vllm_legacy_amd.attention.batch import SequenceBatch
    from vllm_legacy_amd.attention.recurrent import GatedLinearRecurrence
    H, rank, n, g = 2, 3, 130, torch.Generator().manual_seed(row + D)
    layer = GatedLinearRecurrence(H, D, V, 5.0, 1e-5)
    layer.CHUNK_ALONE_ROWS = 0
    q, k, v, gate, y, w2 = (torch.randn(*shape, generator=g).to(dtype) for shape in [(n, H * D)] * 2 + [(n, H * V)] * 2 + [
        (n, rank), (H * D, rank)])
    bias = torch.randn(H * D, generator=g) + 2
    k[row, 2] = 0.0
    b = SequenceBatch.build([n], [0], [[0] * 64], [0], 16, DEV)

    def go(v):
        state = torch.zeros(1, H, D, V, device=DEV)
        layer(torch.empty(n, H * V, device=DEV, dtype=dtype), q.to(DEV), k.to(DEV), v.to(DEV), gate.to(DEV), y.to(DEV), w2.to(DEV),
              bias.to(DEV), torch.ones(V, device=DEV), state, b)
        return state[0].cpu().double()

    clean = go(v)
    v[row, 1], v[row, 5], v[row, 7] = float("inf"), float("-inf"), float("nan")
    v[row, 9], v[(row + 70) % n, 9] = float("inf"), float("-inf")
    got = go(v)
    a = torch.exp(R.log_decay(y.to(R.F), w2.to(R.F), bias.to(R.F), 5.0)).view(-1, H, D)
    S = torch.zeros(H, D, V, dtype=R.F)
    for t in range(n):
        S = a[t][:, :, None] * S + k[t].to(R.F).view(H, D, 1) * v[t].to(R.F).view(H, 1, V)
    assert int(S.isinf().sum()) > 2 * (D - 1) and int(S.isnan().sum()) > D
    assert torch.equal(got.isnan(), S.isnan())
    assert torch.equal(got[S.isinf()], S[S.isinf()])
    assert torch.equal(got[S.isfinite()], clean[S.isfinite()])


@pytest.mark.parametrize("H,lens,chunks", [(2, [99], False), (2, [100], True), (2, [100] + [1] * 6, False), (70, [64, 35], False),
                                           (70, [64, 36], True), (70, [63, 63], False)])
def test_steps_that_go_in_chunks(H, lens, chunks, monkeypatch):
    from vllm_legacy_amd import _seq_ops as ops
    from vllm_legacy_amd.attention.batch import SequenceBatch
    from vllm_legacy_amd.attention.recurrent import GatedLinearRecurrence
    D, V, rank, T, went = 16, 16, 1, sum(lens), []
    layer, taken = GatedLinearRecurrence(H, D, V, 5.0, 1e-5), ops.gla_chunks
    monkeypatch.setattr(ops, "gla_chunks", lambda *a: (went.append(1), taken(*a)))
    b = SequenceBatch.build(lens, [0] * len(lens), [[0] * 64] * len(lens), list(range(len(lens))), 16, DEV)
    q, k, v, gate, y, w2 = (torch.randn(*shape, generator=torch.Generator().manual_seed(i)).to(DEV) for i, shape in enumerate(
        [(T, H * D), (T, H * D), (T, H * V), (T, H * V), (T, rank), (H * D, rank)]))
    outs = []
    for alone in (None, 1 << 30):
        if alone:
            layer.CHUNK_ALONE_ROWS = layer.CHUNK_HEAD_ROWS = alone
        state = torch.zeros(GatedLinearRecurrence.get_state_shape(len(lens), H, D, V), device=DEV)
        out = torch.empty(T, H * V, device=DEV)
        layer(out, q, k, v, gate, y, w2, torch.ones(H * D, device=DEV), torch.ones(V, device=DEV), state, b, 1.0)
        outs.append(out)
    assert len(went) == int(chunks)
    assert float((outs[0] - outs[1]).abs().max()) <= 6e-5 * float(outs[1].abs().max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gates_of_any_size(dtype):
    """Gates at and beyond where exp(-gate) leaves fp32, in whole 16-byte pieces of a row: a result is its gate's silu times what
    the same row gives with a gate that silu leaves as it is (40), to one rounding of each."""
    from vllm_legacy_amd.attention.batch import SequenceBatch
    from vllm_legacy_amd.attention.recurrent import GatedLinearRecurrence
    H, D, V, rank, n = 2, 64, 128, 16, 100
    layer = GatedLinearRecurrence(H, D, V, 5.0, 1e-5)
    layer.CHUNK_ALONE_ROWS = 0
    g = torch.Generator().manual_seed(7)
    wide = torch.randn(n, 2 * H * D + H * V + rank, generator=g).to(dtype).to(DEV)
    q, k, v, y = wide.split([H * D, H * D, H * V, rank], 1)
    w2, bias, norm = torch.randn(H * D, rank, generator=g).to(dtype).to(DEV), torch.ones(H * D, device=DEV), torch.ones(V, device=DEV)
    b = SequenceBatch.build([n], [0], [[0] * 64], [0], 16, DEV)
    values = torch.tensor([-120.0, -95.0, -88.5, -87.5, -86.5, -20.0, -0.5, 0.0, 0.5, 20.0, 88.5, 300.0, float("inf")])

    def out(gate):
        got = torch.empty(n, H * V, device=DEV, dtype=dtype)
        layer(got, q, k, v, gate, y, w2, bias, norm, torch.zeros(1, H, D, V, device=DEV), b)
        return got.double().cpu()

    gate = values[torch.arange(n * H * V) % len(values)].view(n, H * V).to(dtype)
    plain = out(torch.full_like(gate, 40.0).to(DEV)) / 40
    gd = gate.double()
    want = plain * torch.where(gd.isinf(), gd, gd / (1 + torch.exp(-gd)))
    got, finite = out(gate.to(DEV)), want.isfinite() & (want.abs() < torch.finfo(dtype).max / 2)
    small = torch.finfo(dtype).tiny * 2          # below, a result may be rounded to a coarser step or to nothing
    eps = 2.0**-7 if dtype == torch.bfloat16 else 2.0**-10
    assert bool(((got - want).abs() <= eps * want.abs() + small)[finite].all())
    assert bool((got == want)[want.isinf()].all())


@pytest.mark.parametrize("lens,ctx", [([1000], [0]), ([300, 64, 200], [9, 0, 1])])
@pytest.mark.parametrize("dim", [64, 128])
def test_states_of_bfloat16_rows_are_as_exact_as_with_fp32_products(lens, ctx, dim):
    """Keys and A as three bfloat16 numbers each, values as they are: exact products, fewer roundings of the sums than fp32
    instructions make (states' relative errors 0.9e-7 where those left 1.3 to 1.4e-7)."""
    from vllm_legacy_amd.attention.batch import SequenceBatch
    from vllm_legacy_amd.attention.recurrent import GatedLinearRecurrence
    H, D, V, rank, T = 2, dim, 128, 16, sum(lens)
    layer = GatedLinearRecurrence(H, D, V, 8.0, 1e-5)
    layer.CHUNK_ALONE_ROWS = 0
    g = torch.Generator().manual_seed(T + dim)
    wide = torch.randn(T, 2 * H * D + 2 * H * V + rank, generator=g).to(torch.bfloat16)
    parts = [H * D, H * D, H * V, H * V, rank]
    w2, bias = (torch.randn(H * D, rank, generator=g) * 0.25).to(torch.bfloat16), torch.randn(H * D, generator=g) + 2
    state = torch.randn(len(lens), H, D, V, generator=g) * 0.1
    got = state.to(DEV)
    q, k, v, gate, y = wide.to(DEV).split(parts, 1)
    layer(torch.empty(T, H * V, device=DEV, dtype=torch.bfloat16), q, k, v, gate, y, w2.to(DEV), bias.to(DEV), torch.ones(V, device=DEV), got,
          SequenceBatch.build(lens, ctx, [[0] * 64] * len(lens), list(range(len(lens))), 16, DEV))
    q, k, v, gate, y = (t.double() for t in wide.split(parts, 1))
    decay = torch.exp(torch.nn.functional.logsigmoid(y @ w2.double().t() + bias.double()) / 8.0)
    at = 0
    for i, (n, c) in enumerate(zip(lens, ctx)):
        S = state[i].double() if c else torch.zeros(H, D, V, dtype=torch.float64)
        for t in range(at, at + n):
            S = decay[t].view(H, D, 1) * S + k[t].view(H, D, 1) * v[t].view(H, 1, V)
        at += n
        assert float((got[i].double().cpu() - S).norm() / S.norm()) <= 1.1e-7

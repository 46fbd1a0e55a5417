"""The delta rule's 32-row blocks at their edges: runs around one and two blocks, mixed with runs that go
token by token, head sizes around the padding of 64 rows and 16 columns, decays that underflow beside
decays of one, rows at odd addresses.  Oracle and bound (fp32 sums of a few hundred terms: 3e-5 of the
largest value) are those of the recurrence's other tests."""
import pytest
import torch

from tests.test_gpu_lamosun import DEV, close, make_batch, rnd, run_delta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(2, 1, 128, 128), (1, 1, 256, 24), (3, 3, 40, 20), (2, 2, 192, 130), (4, 2, 64, 16)])
@pytest.mark.parametrize("cuts", [[33], [63, 1, 34], [64, 64], [96, 4, 5, 65]])
def test_runs_around_a_block(shape, cuts):
    got, want = run_delta(*shape, sum(cuts), cuts, seed=11)
    close(got, want, 3e-5, (shape, cuts))


def test_decays_of_nothing_and_of_one():
    def craft(q, k, v, beta, dt):
        dt[::3] = 60.0          # exp(-rate * 60): underflows
        dt[1::3] = -40.0        # one
        dt[40:60] = -40.0
        beta[5::7] = -30.0      # writes nothing
        beta[6::7] = 30.0       # overwrites

    got, want = run_delta(2, 1, 128, 128, 130, [70, 60], seed=3, craft=craft)
    close(got, want, 3e-5)


@pytest.mark.parametrize("offset", [0, 1, 2])
def test_rows_at_odd_addresses_give_the_same_result(offset):
    from vllm_legacy_amd import _seq_ops as ops
    H, G, D, V, n = 2, 2, 128, 36, 75
    parts = [G * D, G * D, H * V, H * V, H, H]
    rows = rnd((n, sum(parts)), 5).to(DEV)
    batch = make_batch([n], [0], slots=[0])
    a_log, bias, w = rnd((H, ), 1, 0.5).to(DEV), rnd((H, ), 2, 0.5).to(DEV), torch.ones(V, device=DEV)

    def go(off):
        wide = torch.empty((n, sum(parts) + 3 + off), device=DEV)
        wide[:, off:off + sum(parts)] = rows
        q, k, v, gate, beta, dt = wide[:, off:off + sum(parts)].split(parts, 1)
        out, state = torch.empty((n, H * V), device=DEV), torch.zeros((1, H, V, D), device=DEV)
        ops.delta_rule_scan(out, q, k, v, gate, beta, dt, a_log, bias, w, state, batch.query_start_loc,
                            batch.context_lens, batch.state_slots, G, 1e-5, n)
        return out, state

    for x, y in zip(go(offset), go(0)):
        assert float((x - y).abs().max()) <= 1e-6 * float(y.abs().max())


@pytest.mark.parametrize("common,outputs,states", [(0.0, 1.0, 1.0), (1.0, 1.0, 1.0), (3.0, 1.0, 1.1)])
def test_as_close_to_64_bits_as_token_by_token(common, outputs, states):
    """Slow decays, where errors add up; keys that are independent and keys that share a part (an error in their
    products is then in every u behind them).  The bounds are those on the ratio of two errors of a few 1e-7 that
    average over 524288 outputs and 65536 numbers of state: 0.82 / 0.80, 0.84 / 0.87 and 0.90 / 1.01 with all that
    goes into U, and what a block adds to the state, in 64 bits; in 32 bits 1.27 / 1.26 without a common part and
    1.78 / 1.94 with the largest, with the key products alone in 64 bits 1.0 / 1.0 and 1.2 / 1.6."""
    from vllm_legacy_amd import _seq_ops as ops
    n, H, D, V = 1024, 4, 128, 128
    F = torch.float64
    q, k, v = rnd((n, H * D), 1), rnd((n, H * D), 2) + common * rnd((1, H * D), 3), rnd((n, H * V), 4)
    q = q + common * rnd((1, H * D), 8)
    beta, dt, gate = rnd((n, H), 5) + 2.0, rnd((n, H), 6, 0.5) - 4.0, torch.full((n, H * V), 40.0)
    batch = make_batch([n], [0], slots=[0])
    zero, one = torch.zeros(H, device=DEV), torch.ones(V, device=DEV)
    unit = [x.to(F).to(DEV).view(n, H, -1) for x in (q, k)]
    qn, kn = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in unit)
    b, a = torch.sigmoid(beta.to(F)).to(DEV), torch.exp(-torch.nn.functional.softplus(dt.to(F))).to(DEV)
    S, o, vv = torch.zeros((H, D, V), dtype=F, device=DEV), [], v.to(F).to(DEV).view(n, H, V)
    for t in range(n):
        S = S * a[t][:, None, None]
        u = b[t][:, None] * (vv[t] - (S * kn[t][:, :, None]).sum(1))
        S = S + kn[t][:, :, None] * u[:, None]
        o.append((S * qn[t][:, :, None]).sum(1) * D**-0.5)
    o = torch.stack(o)
    o = o / torch.sqrt((o * o).mean(-1, keepdim=True) + 1e-5) * 40.0
    errors = []
    for kernel in (2, 0):
        ops.set_delta_kernel(kernel)
        try:
            out, state = torch.empty((n, H * V), device=DEV), torch.zeros((1, H, V, D), device=DEV)
            ops.delta_rule_scan(out, *(x.to(DEV) for x in (q, k, v, gate, beta, dt)), zero, zero, one, state,
                                batch.query_start_loc, batch.context_lens, batch.state_slots, H, 1e-5, n)
        finally:
            ops.set_delta_kernel(0)
        errors.append([float((x.to(F) - want).norm() / want.norm())
                       for x, want in ((out.view(n, H, V), o), (state[0].transpose(1, 2), S))])
    assert errors[1][0] <= outputs * errors[0][0] and errors[1][1] <= states * errors[0][1], errors


@pytest.mark.parametrize("what,value", [("v", float("inf")), ("v", float("nan")), ("k", float("-inf")), ("k", float("nan")),
                                        ("beta", float("nan")), ("dt", float("nan")), ("q", float("inf"))])
@pytest.mark.parametrize("row", [0, 3, 15, 16, 22, 31, 32, 60, 65])
@pytest.mark.parametrize("V", [128, 40])
def test_rows_ahead_of_one_that_is_not_finite(what, value, row, V):
    """Bit for bit what they are without it, as token by token; the rows behind it are not finite exactly where
    the walk says so, and it itself nowhere (an infinity among a row's outputs leaves zeros beside it in the walk);
    other heads, columns and sequences know nothing of it."""
    from vllm_legacy_amd import _seq_ops as ops
    H, D, lens = 2, 64, [66, 40]
    n = sum(lens)
    rows = {"q": H * D, "k": H * D, "v": H * V, "gate": H * V, "beta": H, "dt": H}
    rows = {name: rnd((n, w), i) for i, (name, w) in enumerate(rows.items())}
    batch = make_batch(lens, [0, 0], slots=[0, 1])
    zero, one = torch.zeros(H, device=DEV), torch.ones(V, device=DEV)

    def go(kernel=0):
        out, state = torch.empty((n, H * V), device=DEV), torch.zeros((2, H, V, D), device=DEV)
        ops.set_delta_kernel(kernel)
        try:
            ops.delta_rule_scan(out, *(rows[x].to(DEV) for x in ("q", "k", "v", "gate", "beta", "dt")), zero, zero, one, state,
                                batch.query_start_loc, batch.context_lens, batch.state_slots, H, 1e-5, max(lens))
        finally:
            ops.set_delta_kernel(0)
        return out.cpu().view(n, H, V), state.cpu()

    clean, clean_state = go()
    rows[what] = rows[what].clone()
    rows[what][row, 0 if what in ("beta", "dt") else 1] = value                 # head 0
    got, state = go()
    want, want_state = go(2)
    assert torch.equal(got[:row], clean[:row]) and torch.equal(got[lens[0]:], clean[lens[0]:])
    assert torch.equal(got[:, 1], clean[:, 1]) and torch.equal(state[0, 1], clean_state[0, 1])
    assert torch.equal(state[1], clean_state[1])
    got, want = got.isfinite(), want.isfinite()
    assert not got[row, 0].any() and not want[row, 0].all()
    got[row, 0] = want[row, 0]
    assert torch.equal(got, want) and torch.equal(state.isfinite(), want_state.isfinite())


@pytest.mark.parametrize("rows", [1, 4, 5, 33])
@pytest.mark.parametrize("hint", [0, 33, 500])
def test_a_lone_run_shorter_than_the_hint(rows, hint):
    """max_query_len bounds the rows of a run; how many there are is read on the device."""
    from vllm_legacy_amd import _seq_ops as ops
    H, D, V = 2, 64, 48
    x = {name: rnd((rows, w), i).to(DEV) for i, (name, w) in enumerate(
        {"q": H * D, "k": H * D, "v": H * V, "gate": H * V, "beta": H, "dt": H}.items())}
    batch, zero, one = make_batch([rows], [0], slots=[0]), torch.zeros(H, device=DEV), torch.ones(V, device=DEV)

    def go(most):
        out, state = torch.full((rows, H * V), 7.0, device=DEV), torch.full((1, H, V, D), 7.0, device=DEV)
        ops.delta_rule_scan(out, *x.values(), zero, zero, one, state, batch.query_start_loc, batch.context_lens,
                            batch.state_slots, H, 1e-5, most)
        return out, state

    for got, want in zip(go(hint), go(min(rows, 32))):
        assert float((got - want).abs().max()) <= 3e-5 * float(want.abs().max())


@pytest.mark.parametrize("H,lens,blocks", [(2, [87], False), (2, [88], True), (2, [32] * 3, False), (128, [33, 30], False),
                                           (128, [33, 31], True), (128, [32, 32], False)])
def test_steps_that_go_in_blocks(H, lens, blocks):
    """The layer's choice, and both kernels' results."""
    from vllm_legacy_amd import _seq_ops as ops
    from vllm_legacy_amd.attention.recurrent import GatedDeltaRule
    D, V, n = 16, 64, sum(lens)
    layer = GatedDeltaRule(H, H, D, V, 1e-5, DEV)
    x = {name: rnd((n, w), i).to(DEV) for i, (name, w) in enumerate(
        {"q": H * D, "k": H * D, "v": H * V, "gate": H * V, "beta": H, "dt": H}.items())}
    batch = make_batch(lens, [0] * len(lens), slots=list(range(len(lens))))

    def go(which):
        out, state = torch.empty((n, H * V), device=DEV), torch.zeros((len(lens), H, V, D), device=DEV)
        if which is None:
            layer(out, *x.values(), state, batch)
        else:
            ops.delta_rule_scan(out, *x.values(), layer.a_log.data, layer.dt_bias.data, layer.norm_weight.data, state,
                                batch.query_start_loc, batch.context_lens, batch.state_slots, H, 1e-5, max(lens), which)
        return out, state

    got, walk, block = go(None), go(False), go(True)
    assert torch.equal(got[1], (block if blocks else walk)[1])
    assert not torch.equal(walk[1], block[1]) or max(lens) < 33
    for a, b in zip(walk, block):
        assert float((a - b).abs().max()) <= 3e-5 * float(b.abs().max())

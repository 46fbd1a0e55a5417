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

"""Entry points of the C interface that the package itself reaches only in their longer forms: each bit for bit what
the longer form gives where neither has a choice of its own, and against it where they choose kernels apart."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rnd(shape, seed, std=1.0):
    return (std * torch.randn(shape, generator=torch.Generator().manual_seed(seed))).to(DEV)


def at(t):
    return None if t is None else t.data_ptr()


def stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("n,k,tiles", [(40, 64, 3), (1200, 128, 130), (40, 72, 5)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_grouped_linear(n, k, tiles, dtype):
    """Few and many tiles by the rule that knows no number of experts, and sizes of the general kernels."""
    from vllm_legacy_amd import _lib, _seq_ops as ops
    E, rows = 3, 32 * tiles
    a, w = rnd((rows, k), 1).to(dtype), rnd((E, n, k), 2, k**-0.5).to(dtype)
    expert = (torch.arange(tiles, dtype=torch.int32) * E // tiles).to(DEV)
    got, want = (torch.empty((rows, n), device=DEV) for _ in range(2))
    ops.grouped_linear(want, a, None, w, expert, "silu")
    ops.seq_check(_lib.seq_lib().vla_seq_grouped_linear(
        at(got), n, _lib.F32, at(a), k, None, at(w), at(expert), tiles, n, k, ops.ACT["silu"], None, ops._dt(dtype),
        stream()), "grouped_linear")
    assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max())


def test_kv_attention():
    from vllm_legacy_amd import _lib, _seq_ops as ops
    T, H, G, D, keys, dtype = 2, 8, 2, 128, 3000, torch.bfloat16
    blocks = -(-keys // 16)
    kc, vc = (rnd((T * blocks, 16, G, D), s).to(dtype) for s in (1, 2))
    table = torch.arange(T * blocks, dtype=torch.int32, device=DEV).view(T, blocks)
    q = rnd((T, H * D), 3).to(dtype)
    seq, pos = torch.arange(T, dtype=torch.int32, device=DEV), torch.tensor([keys - 1, 70], device=DEV)
    got, whole, shared = (torch.empty_like(q) for _ in range(3))
    for out, most in ((whole, 0), (shared, keys)):
        ops.kv_attention(out, q, None, kc, vc, table, seq, pos, None, True, H, 0, D**-0.5, max_keys=most)
    ops.seq_check(_lib.seq_lib().vla_seq_kv_attention(
        at(got), H * D, at(q), H * D, None, 0, at(kc), at(vc), at(table), blocks, at(seq), at(pos), None, 1, T, H, G, D, D,
        16, T * blocks, 0, D**-0.5, ops._dt(dtype), 0, 0.0, 0, None, stream()), "kv_attention")
    assert torch.equal(got, whole)
    assert float((got - shared).abs().max()) <= 2.0**-7 * float(got.abs().max())


@pytest.mark.parametrize("rows", [3, 70])
def test_delta_rule_scan(rows):
    """Without scratch for blocks every run is walked token by token."""
    from tests.test_gpu_lamosun import make_batch
    from vllm_legacy_amd import _lib, _seq_ops as ops
    H, D, V = 2, 64, 48
    L = _lib.seq_lib()
    x = {name: rnd((rows, w), i) for i, (name, w) in enumerate(
        {"q": H * D, "k": H * D, "v": H * V, "gate": H * V, "beta": H, "dt": H}.items())}
    batch, zero, one = make_batch([rows], [0], slots=[0]), torch.zeros(H, device=DEV), torch.ones(V, device=DEV)
    want, want_state = torch.empty((rows, H * V), device=DEV), torch.zeros((1, H, V, D), device=DEV)
    ops.delta_rule_scan(want, *x.values(), zero, zero, one, want_state, batch.query_start_loc, batch.context_lens,
                        batch.state_slots, H, 1e-5, rows)
    got, state = torch.empty_like(want), torch.zeros_like(want_state)
    scratch = torch.empty(L.vla_seq_delta_rule_scratch_floats(rows, H, V), device=DEV)
    args = [y for t in x.values() for y in (at(t), t.shape[1])]
    ops.seq_check(L.vla_seq_delta_rule_scan(
        at(got), H * V, _lib.F32, *args, _lib.F32, at(zero), at(zero), at(one), at(state), at(batch.query_start_loc),
        at(batch.context_lens), at(batch.state_slots), rows, 1, rows, 1, H, H, D, V, 1e-5, at(scratch), stream()),
        "delta_rule_scan")
    for a, b in ((got, want), (state, want_state)):
        assert float((a - b).abs().max()) <= 3e-5 * float(b.abs().max())

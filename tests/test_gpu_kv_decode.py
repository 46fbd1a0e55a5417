"""Single rows on the LDS-DMA decode kernel: every head and value size it takes, groups of 1 to 16, pages of
1, 4 and 16 tokens, contexts around its tiles of 32 keys and its shares, windows, chunks, kept first tokens,
caps, sinks, gates and values that turn back -- against the same attention in float64.  The weights enter as
two 16-bit parts and the result is rounded once to 16 bits: 1 % of the largest value in bfloat16 (2^-8 and
the rounding of the operands' products), an eighth of that in float16."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rnd(shape, seed, std=1.0):
    return std * torch.randn(shape, generator=torch.Generator().manual_seed(seed))


def reference(q, keys, values, gate, scale, lo_of, keep, softcap, sink, inv_freq, interleaved, positions):
    T, H, D = q.shape
    out = torch.empty((T, H, values[0].shape[2]), dtype=torch.float64)
    for t in range(T):
        p = int(positions[t])
        lo = lo_of(p)
        seen = torch.tensor([j for j in range(p + 1) if j >= lo or j < keep])
        for h in range(H):
            g = h // (H // keys[t].shape[1])
            s = keys[t][seen, g] @ q[t, h] * scale
            s = softcap * torch.tanh(s / softcap) if softcap else s
            e = torch.exp(s - s.max())
            total = e.sum() + (torch.exp(torch.tensor(sink, dtype=torch.float64) - s.max()) if sink is not None else 0.0)
            o = (e / total) @ values[t][seen, g]
            if inv_freq is not None:
                half = o.shape[0] // 2
                a, b = (o[0::2], o[1::2]) if interleaved else (o[:half], o[half:])
                ang = (torch.tensor(float(p)) * inv_freq).double()
                x, y = a * ang.cos() + b * ang.sin(), b * ang.cos() - a * ang.sin()
                o = torch.stack([x, y], 1).reshape(-1) if interleaved else torch.cat([x, y])
            out[t, h] = o * (torch.sigmoid(gate[t, h]) if gate is not None else 1.0)
    return out


CASES = [
    # heads, kv heads, dim, vdim, page, positions, options
    (4, 1, 128, 128, 16, [0, 31, 32, 127, 128, 700], {}),
    (16, 1, 64, 128, 4, [5, 300], dict(window=100)),
    (3, 3, 128, 64, 1, [64, 33], dict(window=40, keep=3, softcap=20.0)),
    (10, 2, 64, 64, 16, [500, 17], dict(chunk=48, sink=1.5)),
    (8, 2, 128, 128, 16, [2047], dict(gate=True)),
    (8, 2, 128, 128, 4, [1500, 3], dict(turn="pairs", gate=True)),
    (4, 2, 64, 64, 16, [900], dict(turn="halves", window=600, keep=70)),
    (2, 1, 128, 128, 8, [4095], dict(sink=-2.0, softcap=30.0)),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("most", [0, 4096, 1 << 22])
def test_single_rows(case, dtype, most):
    """most: the bound on a row's keys that the launch is told: unknown, keys shared out, and (more than 256 MiB
    of keys and values by it) read past the last-level cache."""
    from vllm_legacy_amd import _seq_ops as ops
    H, G, D, V, bs, positions, opt = case
    T, window, keep, chunk = len(positions), opt.get("window", 0), opt.get("keep", 0), opt.get("chunk", 0)
    need = [p // bs + 1 for p in positions]
    ids = torch.randperm(sum(need) + 2, generator=torch.Generator().manual_seed(3)).tolist()
    kc, vc = rnd((sum(need) + 2, bs, G, D), 1).to(dtype), rnd((sum(need) + 2, bs, G, V), 2).to(dtype)
    tables = torch.zeros((T, max(need)), dtype=torch.int32)
    keys, values, at = [], [], 0
    for t, n in enumerate(need):
        own = torch.tensor(ids[at:at + n])
        tables[t, :n] = own
        keys.append(kc[own].reshape(-1, G, D).double())
        values.append(vc[own].reshape(-1, G, V).double())
        at += n
        kc[own[-1], positions[t] % bs + 1:], vc[own[-1], positions[t] % bs + 1:] = float("nan"), float("nan")
    q, gate = rnd((T, H, D), 4).to(dtype), rnd((T, H + 1), 5).to(dtype) if opt.get("gate") else None
    inv = torch.rand(V // 2, generator=torch.Generator().manual_seed(6)) * 0.1 if opt.get("turn") else None
    inter = opt.get("turn") == "pairs"
    pos = torch.tensor(positions)

    def lo_of(p):
        return max(0, p - window + 1 if window else 0, p - p % chunk if chunk else 0)

    want = reference(q.double(), keys, values, None if gate is None else gate[:, :H].double(), D**-0.5, lo_of,
                     keep if window or chunk else 0, opt.get("softcap", 0.0), opt.get("sink"), inv, inter, positions)
    out = torch.empty((T, H * V), dtype=dtype, device=DEV)
    sinks = None if opt.get("sink") is None else torch.full((H, ), opt["sink"], device=DEV)
    ops.kv_attention(out, q.view(T, H * D).to(DEV), None if gate is None else gate.to(DEV)[:, :H], kc.to(DEV), vc.to(DEV),
                     tables.to(DEV), torch.arange(T, dtype=torch.int32, device=DEV), pos.to(DEV),
                     None if inv is None else inv.to(DEV), inter, H, window, D**-0.5, keep, opt.get("softcap", 0.0), chunk,
                     sinks, most)
    got = out.cpu().double().view(T, H, V)
    bar = 0.01 if dtype == torch.bfloat16 else 0.00125
    assert float((got - want).abs().max()) <= bar * float(want.abs().max())

"""Rotary and latent rows written 16 bytes at a time against the kernel that takes any address: the same rows one element further on
go there.  Both form the same products and round once, so results are the same bits (float16: the compiler has a sum
rounded at once in one kernel and by way of 32 bits in the other, one unit in the last place where it lies half way): pairs side by side and in halves,
heads that turn in part, more pieces than a wave fetches ahead, rows that no cache takes, and tokens around the
sizes of a workgroup.  Which kernel takes the rows is asserted, and both are compared with a rotation in float64 by the same
fp32 angles: one rounding to 16 bits (2^-8 or 2^-11 of the result) and 2^-20 of the pair for sines and products."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def shifted(t, by):
    """The same rows in a wider tensor, `by` elements behind its start."""
    wide = torch.zeros(t.shape[0], t.shape[1] + 16, dtype=t.dtype, device=DEV)
    wide[:, by:by + t.shape[1]] = t
    return wide[:, by:by + t.shape[1]]


def turned(x, positions, freq, interleaved, magnitude=1.0):
    """[T, heads, 2 * len(freq)] by positions * freq -> the same in float64, and the size of every pair"""
    angle = (positions.float()[:, None] * freq).double()[:, None]
    sin, cos = angle.sin() * magnitude, angle.cos() * magnitude
    half, x = x.shape[2] // 2, x.double()
    a, b = (x[..., 0::2], x[..., 1::2]) if interleaved else (x[..., :half], x[..., half:])
    out = (a * cos - b * sin, b * cos + a * sin), (a.abs() + b.abs(), ) * 2
    return [torch.stack(t, 3).flatten(2) if interleaved else torch.cat(t, 2) for t in out]


def close(got, want, size):
    unit = 2.0**-8 if got.dtype == torch.bfloat16 else 2.0**-11
    return bool(((got.double() - want).abs() <= unit * want.abs() + 2.0**-20 * size + 2.0**-25).all())


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("T,heads,kv_heads,dim,vdim,rot", [
    (1, 1, 1, 16, 8, 16), (5, 16, 4, 128, 128, 128), (1023, 16, 4, 128, 128, 64), (1024, 4, 4, 64, 128, 64),
    (1029, 32, 8, 128, 128, 128), (7, 72, 24, 128, 72, 96), (6, 6, 3, 48, 40, 48), (3, 8, 8, 256, 256, 256),
    (3, 5, 1, 264, 24, 16), (70, 3, 3, 8 + 16, 8, 16), (2, 256, 16, 128, 64, 128), (2, 260, 4, 128, 64, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_same_bits_as_rows_anywhere(interleaved, T, heads, kv_heads, dim, vdim, rot, dtype):
    from vllm_legacy_amd import _lib
    from vllm_legacy_amd import _seq_ops as ops
    g = torch.Generator(device=DEV).manual_seed(T + heads)
    q, k, v = (torch.randn(T, n, generator=g, device=DEV).to(dtype) for n in (heads * dim, kv_heads * dim, kv_heads * vdim))
    blocks, size = T // 16 + 2, 16
    slots = torch.randperm(blocks * size, generator=g, device=DEV)[:T].contiguous()
    slots[T // 2] = -1 if T > 1 else slots[0]
    if T > 2:
        slots[T // 3] = blocks * size
    positions = torch.randint(0, 40000, (T, ), generator=g, device=DEV)
    freq = 10000.0**(-torch.arange(0, rot, 2, device=DEV, dtype=torch.float32) / rot)
    got = []
    for by in (8, 1):
        mine = [shifted(t, by) for t in (q, k, v)]
        caches = [torch.full((blocks, size, kv_heads, n), 7.0, dtype=dtype, device=DEV) for n in (dim, vdim)]
        rows = [x for t in mine for x in (t.data_ptr(), t.stride(0))]
        assert _lib.seq_lib().vla_seq_rotary_kv_write_form(*rows, caches[0].data_ptr(), caches[1].data_ptr(), heads, kv_heads, dim,
                                                           vdim, rot, _lib.BF16 if dtype == torch.bfloat16 else _lib.F16) == \
            (by == 8 and heads * rot // 16 <= 2048)
        ops.rotary_kv_write(*mine, *caches, positions, slots, freq, None, heads, rot, interleaved)
        got.append([mine[0].clone()] + caches)
        assert torch.equal(mine[1], k) and torch.equal(mine[2], v)
        x = mine[0].reshape(T, heads, dim)
        assert close(x[..., :rot], *turned(q.view(T, heads, dim)[..., :rot], positions, freq, interleaved))
        assert torch.equal(x[..., rot:], q.view(T, heads, dim)[..., rot:])
        held = (slots >= 0) & (slots < blocks * size)
        x = caches[0].view(-1, kv_heads, dim)[slots[held]]
        assert close(x[..., :rot], *turned(k.view(T, kv_heads, dim)[held][..., :rot], positions[held], freq, interleaved))
        assert torch.equal(x[..., rot:], k.view(T, kv_heads, dim)[held][..., rot:])
        assert torch.equal(caches[1].view(-1, kv_heads * vdim)[slots[held]], v[held])
    for a, b in zip(*got):
        if dtype == torch.bfloat16:
            assert torch.equal(a, b)
        else:       # a unit: 2^-10 of the value, 2^-24 below 2^-14
            a, b = a.double(), b.double()
            assert bool(((a - b).abs() <= 2.0**-10 * b.abs() + 2.0**-24).all()) and float((a != b).double().mean()) < 1e-3
    assert not torch.equal(got[0][0], q) and bool((got[0][1] == 7.0).any())


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("T,heads,rank,rot,rot_dims,head,first", [
    (1, 1, 8, 16, 16, 16, 0), (5, 16, 512, 64, 64, 192, 128), (1025, 16, 256, 64, 32, 128, 64), (7, 3, 520, 0, 0, 64, 8),
    (6, 40, 1024, 128, 128, 128, 0), (3, 5, 72, 272, 256, 280, 8), (1024, 4, 512, 64, 64, 64, 0), (9, 2, 504, 24, 16, 40, 8),
    # few pieces: on the general kernel up to 1024 tokens or 40960 pieces
    (1027, 1, 8, 16, 16, 16, 0), (1024, 1, 8, 16, 16, 16, 0), (640, 8, 256, 64, 64, 64, 0), (641, 8, 256, 64, 64, 64, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_latent_rows_as_rows_anywhere(interleaved, T, heads, rank, rot, rot_dims, head, first, dtype):
    """The latent's norm adds its squares in another order: relative differences of some 2^-22 ahead of one rounding."""
    from vllm_legacy_amd import _lib
    from vllm_legacy_amd import _seq_ops as ops
    pieces = heads * rot_dims // 16 + rank // 8
    whole = pieces > 64 or T > 1024 or T * pieces > 40960
    g = torch.Generator(device=DEV).manual_seed(T + heads)
    q, kv = (torch.randn(T, n, generator=g, device=DEV).to(dtype) for n in (heads * head, rank + rot))
    weight = torch.rand(rank, generator=g, device=DEV) + 0.5
    blocks, size = T // 16 + 2, 16
    slots = torch.randperm(blocks * size, generator=g, device=DEV)[:T].contiguous()
    if T > 2:
        slots[T // 2], slots[T // 3] = -1, blocks * size
    positions = torch.randint(0, 40000, (T, ), generator=g, device=DEV)
    freq = 10000.0**(-torch.arange(0, rot_dims, 2, device=DEV, dtype=torch.float32) / max(rot_dims, 1)) if rot_dims else None
    got = []
    for by in (8, 1):
        rows, lat = shifted(q, by), shifted(kv, by)
        cache = torch.full((blocks, size, rank + rot), 7.0, dtype=dtype, device=DEV)
        assert _lib.seq_lib().vla_seq_latent_rotary_write_form(
            rows.data_ptr(), rows.stride(0), head, first, lat.data_ptr(), lat.stride(0), weight.data_ptr(), cache.data_ptr(), T, heads,
            rank, rot, rot_dims, _lib.BF16 if dtype == torch.bfloat16 else _lib.F16) == (by == 8 and whole)
        ops.latent_rotary_write(rows, head, first, heads, lat, weight, 1e-5, cache, positions, slots, freq, 0.9, rot_dims,
                                interleaved)
        assert torch.equal(lat, kv)
        held = (slots >= 0) & (slots < blocks * size)
        row, c = cache.view(-1, rank + rot)[slots[held]], kv[held][:, :rank].double()
        normed = c / (c.square().mean(1, keepdim=True) + 1e-5).sqrt() * weight.double()
        assert close(row[:, :rank], normed, normed.abs())
        assert torch.equal(row[:, rank + rot_dims:], kv[held][:, rank + rot_dims:])
        x, y = (t.reshape(T, heads, head)[..., first:first + rot_dims] for t in (rows, q))
        if rot_dims:
            assert close(x, *turned(y, positions, freq, interleaved, 0.9))
            x, y = (t[:, rank:rank + rot_dims].reshape(-1, 1, rot_dims) for t in (row, kv[held]))
            assert close(x, *turned(y, positions[held], freq, interleaved, 0.9))
        got.append((rows.clone().double(), cache.double()))
    unit = 2.0**-7 if dtype == torch.bfloat16 else 2.0**-10
    for a, b in zip(*got):
        assert bool(((a - b).abs() <= unit * b.abs() + 2.0**-24).all()) and float((a != b).double().mean()) < 2e-3
    assert rot_dims == 0 or not torch.equal(got[0][0], q.double())
    assert bool((got[0][1] == 7.0).any()) and not bool((got[0][1] == 7.0).all())

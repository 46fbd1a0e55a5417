"""Attention sinks at the ends of float32's range, in the kernels for runs of rows: minus infinity, and the lowest number,
which overflows when it is scaled to base 2, count for nothing -- the same bits as without sinks, also for rows that see no
key of the first tiles they meet --, an infinite one leaves no number, as in a softmax, and a number between them counts."""
import math

import pytest
import torch

from tests.test_gpu_kv_decode import DEV, rnd
from tests.test_gpu_latent_prompt import layer_and_step

pytestmark = pytest.mark.gpu
SINKS = [-math.inf, torch.finfo(torch.float32).min, math.inf, 0.3]


def check(with_sinks, without):
    assert without.isfinite().all() and torch.equal(with_sinks[:, :2], without[:, :2])
    assert with_sinks[:, 2].isnan().all()
    assert with_sinks[:, 3].isfinite().all() and not torch.equal(with_sinks[:, 3], without[:, 3])


@pytest.mark.parametrize("opt", [dict(window=40), dict(window=40, scale=-0.1), dict(window=70, keep_first=3), dict(chunk=48),
                                 dict(window=0, softcap=20.0)])
@pytest.mark.parametrize("copies", [1, 150, 300])
def test_runs_of_rows(opt, copies):
    from vllm_legacy_amd import _seq_ops as ops
    runs, H, D, bs = [(65, 0), (33, 95)] * copies, 4, 64, 16
    T, opt = sum(n for n, _ in runs), dict(opt)
    kc, vc, q = (rnd(s, i).to(torch.bfloat16).to(DEV) for i, s in enumerate([(9, bs, 1, D), (9, bs, 1, D), (T, H * D)]))
    tables = torch.arange(len(runs) * 8, dtype=torch.int32, device=DEV).view(-1, 8) % 9
    lens = torch.tensor([0] + [n for n, _ in runs]).cumsum(0).int().to(DEV)
    ctx = torch.tensor([c for _, c in runs], dtype=torch.int32, device=DEV)
    window, scale = opt.pop("window", 0), opt.pop("scale", D**-0.5)
    got = []
    for sinks in (torch.tensor(SINKS, device=DEV), None):
        out = torch.empty_like(q)
        ops.kv_attention_tiles(out, q, None, kc, vc, tables, lens, ctx, 65, None, False, H, window, scale, sinks=sinks, **opt)
        got.append(out.view(T, H, D))
    check(*got)


@pytest.mark.parametrize("window", [0, 50, 90])
@pytest.mark.parametrize("seqs", [1, 70])
def test_latent_prompts(window, seqs):
    sizes = (4, 128, 64, 128, 128)
    got = []
    for sinks in (True, False):
        attn, batch, q, kv, gate, cache = layer_and_step([200, 129][:seqs] * seqs, [30, 170][:seqs] * seqs, sizes, window, sinks)
        if sinks:
            attn.sinks.data = torch.tensor(SINKS, device=DEV)
        got.append(attn(q, kv, cache, batch, gate).view(-1, 4, 128))
    check(*got)

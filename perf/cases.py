"""What a step of the framework is made of, at the sizes that serving meets, for measurement.

Five kinds of case, each through the layer that a model's forward calls, with the caches, weights and
step metadata that a serving loop keeps:

  llama    a decoder layer of the Llama-3-8B shape with AWQ int4 weights over the paged cache (16 bit or
           fp8), the final norm and a small head: decode steps of 1 to 256 sequences replayed from a
           graph, as the decode benchmark does, and prompts (also continued ones) run eagerly
  latent   attention over a cached latent (rank 512, with or without a rotated part, window, gate, sinks):
           prompts, portions of prompts and decode steps
  kv       rotary attention over paged keys and values with grouped queries (with or without window,
           capped scores, gate): prompts, portions and decode steps
  recur    the matrix-state recurrences: gated linear attention with a decay per key channel ("linear")
           and the gated delta rule ("delta"), over prompts, portions and single tokens
  experts  the routed feed-forward (gated silu experts, or squared ReLU with a shared expert), from a
           few tokens to a prompt

The sizes are those of the architecture benchmarks (2048 wide, 16 heads, 4 KV heads of 128, experts of
1408; the 4096-wide ones in some drawn cases) and of the decode benchmark.  16-bit models are measured in
the type they are served in: float16 for int4 weights, bfloat16 for the rest; recurrent rows of the
delta rule and every state are fp32.
"""
import math

import torch

from vllm_legacy_amd.attention.backends.gfx950_paged import Gfx950PagedAttentionMetadata
from vllm_legacy_amd.attention.backends.latent_kv import LatentKVAttention
from vllm_legacy_amd.attention.backends.rotary_kv import RotaryKVAttention
from vllm_legacy_amd.attention.batch import SequenceBatch
from vllm_legacy_amd.attention.recurrent import GatedDeltaRule, GatedLinearRecurrence
from vllm_legacy_amd.model.llama_decode import LlamaConfig, LlamaDecodeModel
from vllm_legacy_amd.routed_experts import RoutedExperts

F64 = torch.float64
EPS = 1e-5
BLOCK = 16          # tokens of a cache block


def _llama(name, seqs, context, new, ragged, kv):
    return dict(name=name, kind="llama", seqs=seqs, context=context, new=new, ragged=ragged, kv=kv)


def _latent(name, seqs, context, new, ragged, heads=16, rot=64, window=0, gate=False, sinks=False):
    return dict(name=name, kind="latent", seqs=seqs, context=context, new=new, ragged=ragged, heads=heads, dim=128,
                rot=rot, vdim=128, rank=512, window=window, gate=gate, sinks=sinks)


def _kv(name, seqs, context, new, ragged, heads=16, kv_heads=4, dim=128, rot_dims=128, interleaved=True, window=0,
        softcap=0.0, gate=False):
    return dict(name=name, kind="kv", seqs=seqs, context=context, new=new, ragged=ragged, heads=heads,
                kv_heads=kv_heads, dim=dim, rot_dims=rot_dims, interleaved=interleaved, window=window,
                softcap=softcap, gate=gate)


def _recur(name, rule, seqs, context, new, ragged, heads=16):
    dim, kv_heads = (64, heads) if rule == "linear" else (128, heads // 2)
    return dict(name=name, kind="recur", rule=rule, seqs=seqs, context=context, new=new, ragged=ragged, heads=heads,
                kv_heads=kv_heads, dim=dim, vdim=128)


def _experts(name, tokens, width=2048, experts=16, top=2, ff=1408, gated=True, shared=0):
    return dict(name=name, kind="experts", tokens=tokens, width=width, experts=experts, top=top, ff=ff, gated=gated,
                shared=shared)


def listed():
    return [
        # one user's chat: the next token of one sequence
        _llama("llama-decode-1", 1, 129, 1, False, "auto"),
        # a full server: the decode benchmark's batch at its context, fp8 cache
        _llama("llama-decode-256", 256, 4095, 1, False, "fp8"),
        # prompts of different lengths admitted in one step
        _llama("llama-prompt", 3, 0, 1501, True, "auto"),
        # a long prompt of a latent-attention model, from its first token
        _latent("latent-prompt", 1, 0, 4096, False),
        # a decode step of 64 requests at different points of their contexts
        _latent("latent-decode", 64, 4000, 1, True),
        # four prompts of different lengths, full causal attention
        _kv("kv-prompt", 4, 0, 2047, True),
        # decode of 64 requests at equal contexts
        _kv("kv-decode", 64, 4095, 1, False),
        # recurrent layers: one long prompt, two uneven prompts, a decode step
        _recur("linear-prompt", "linear", 1, 0, 4096, False),
        _recur("delta-prompt", "delta", 2, 0, 2999, True),
        _recur("delta-decode", "delta", 64, 1000, 1, False),
        # experts: a prompt's rows, and a decode step where every expert's weights are read for a few rows
        _experts("experts-prompt", 4096),
        _experts("experts-decode", 64),
    ]


def _spread(rng, low, high):
    """A whole number between low and high, even over its logarithm, odd as often as not."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))))


def draw(rng):
    kind = rng.choice(["llama", "latent", "kv", "recur", "experts"])
    if kind == "experts":
        wide = rng.random() < 0.25
        gated = rng.random() < 0.7
        c = _experts(None, _spread(rng, 1, 2048 if wide else 4096), *((4096, 32, 4) if wide else (2048, 16, 2)),
                     gated=gated, shared=0 if gated else 1408)
    else:
        form = rng.choice(["prompt", "portion", "decode", "decode"])
        ragged = rng.random() < 0.6
        if form == "decode":
            seqs, new = _spread(rng, 1, 256 if kind in ("llama", "recur") else 64), 1
            context = _spread(rng, 16, 4095)
        else:
            seqs = _spread(rng, 1, 6)
            new = _spread(rng, 33, 4096 // seqs)
            context = 0 if form == "prompt" else _spread(rng, 16, 2048)
        if kind == "llama":
            c = _llama(None, seqs, context, new, ragged, rng.choice(["auto", "fp8"]))
        elif kind == "latent":
            plain = rng.random() < 0.5
            c = _latent(None, seqs, context, new, ragged, rng.choice([16, 16, 32]) if form == "decode" else 16,
                        64 if plain else 0, 0 if plain else rng.choice([0, 1024]), not plain and rng.random() < 0.5,
                        not plain and rng.random() < 0.5)
        elif kind == "kv":
            heads, kv_heads = rng.choice([(16, 4), (16, 4), (32, 8)])
            dim = rng.choice([128, 128, 64])
            c = _kv(None, seqs, context, new, ragged, heads, kv_heads, dim, rng.choice([dim, dim // 2]),
                    rng.random() < 0.5, rng.choice([0, 0, 1024]), rng.choice([0.0, 0.0, 30.0]), rng.random() < 0.3)
        else:
            c = _recur(None, rng.choice(["linear", "delta"]), seqs, context, new, ragged, rng.choice([16, 16, 32]))
    del c["name"]
    return c


# ------------------------------------------------------------------------------- steps
def _lengths(case):
    """(new rows, cached tokens) of each sequence: the first sequence has the most of both; in a ragged step the
    others lie between one and that, spread evenly and in no order."""
    def spread(most, i, turn):
        if most <= 1 or not case["ragged"] or i == 0:
            return most
        return 1 + int((most - 1) * ((i * turn) % 1.0))
    return ([spread(case["new"], i, 0.6180339887) for i in range(case["seqs"])],
            [spread(case["context"], i, 0.7548776662) for i in range(case["seqs"])])


def _generator(seed, dev="cuda"):
    return torch.Generator(device=dev).manual_seed(int(seed))


def _tables(new, context, g):
    """Blocks of every sequence, scattered over the pool as an allocator leaves them, and the pool's size."""
    need = [(n + c + BLOCK - 1) // BLOCK for n, c in zip(new, context)]
    ids = torch.randperm(sum(need) + 3, device="cuda", generator=g).tolist()
    out, at = [], 0
    for n in need:
        out.append(ids[at:at + n])
        at += n
    return out, sum(need) + 3


def _randn(g, *shape, dtype=torch.bfloat16, std=1.0):
    """Normal values, filled in parts so that no temporary is larger than a gigabyte."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    for i in range(0, flat.numel(), 1 << 28):
        part = torch.randn(min(1 << 28, flat.numel() - i), device="cuda", generator=g)
        flat[i:i + part.numel()] = part.mul_(std).to(dtype)
    return out


def _batch(case, g):
    new, context = _lengths(case)
    tables, blocks = _tables(new, context, g)
    batch = SequenceBatch.build(new, context, tables, list(range(case["seqs"])), BLOCK, "cuda")
    return batch, tables, blocks, sum(new)


# ------------------------------------------------------------------------------- llama
def _llama_config():
    cfg = LlamaConfig.llama3_8b()
    cfg.num_hidden_layers, cfg.vocab_size = 1, 1024
    return cfg


def _llama_inputs(case, seed):
    g = _generator(seed)
    new, context = _lengths(case)
    tables, blocks = _tables(new, context, g)
    model = LlamaDecodeModel(_llama_config(), "awq", case["kv"], "cuda", seed=seed, dtype=torch.float16)
    model.layers[0].qkv_proj.scales.data.mul_(0.25)     # queries and keys of the size of the cached keys
    shape = model.kv_cache_shape(blocks, BLOCK)
    if case["kv"] == "fp8":
        cache = torch.empty(shape, dtype=torch.uint8, device="cuda")
        for half in cache:
            for part in half.split(8192):
                part.copy_(torch.randn(part.shape, device="cuda", generator=g).to(torch.float8_e4m3fn).view(torch.uint8))
    else:
        cache = torch.empty(shape, dtype=torch.float16, device="cuda")
        for half in cache:
            for part in half.split(8192):
                part.copy_(torch.randn(part.shape, device="cuda", generator=g))
    most = max(len(t) for t in tables)
    positions = [p for n, c in zip(new, context) for p in range(c, c + n)]
    slots = [t[p // BLOCK] * BLOCK + p % BLOCK for n, c, t in zip(new, context, tables) for p in range(c, c + n)]
    starts = [0]
    for n in new:
        starts.append(starts[-1] + n)
    i32 = dict(dtype=torch.int32, device="cuda")
    decode, lens = case["new"] == 1, [n + c for n, c in zip(new, context)]
    total = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    meta = Gfx950PagedAttentionMetadata(
        num_prefills=0 if decode else len(new), num_prefill_tokens=0 if decode else sum(new),
        num_decode_tokens=sum(new) if decode else 0, slot_mapping=torch.tensor(slots, device="cuda"), seq_lens=lens,
        seq_lens_tensor=torch.tensor(lens, **i32), max_query_len=max(new), max_prefill_seq_len=0 if decode else max(lens),
        max_decode_seq_len=max(lens) if decode else 0, query_start_loc=torch.tensor(starts, **i32), seq_start_loc=total,
        use_cuda_graph=decode, context_lens_tensor=torch.tensor(context, **i32),
        block_tables=torch.tensor([t + [0] * (most - len(t)) for t in tables], **i32))
    return dict(kind="llama", model=model, cache=cache, meta=meta, positions=torch.tensor(positions, device="cuda"),
                ids=torch.randint(0, 1024, (sum(new), ), device="cuda", generator=g),
                last=torch.tensor(starts[1:], device="cuda") - 1, graph=None)


def _llama_hidden(s):
    return s["model"](s["ids"], s["positions"], [s["cache"]], s["meta"])


def _llama_prepare(case, seed):
    """Weights are laid out on a first pass (as the reference does); a decode step is captured, as serving does."""
    s = _llama_inputs(case, seed)
    with torch.inference_mode():
        s["hidden"] = _llama_hidden(s)
        if case["new"] == 1:
            torch.cuda.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                s["hidden"] = _llama_hidden(s)
    return s


@torch.inference_mode()
def _llama_run(s):
    if s["graph"] is not None:
        s["graph"].replay()
        hidden = s["hidden"]
        logits = s["model"].compute_logits(hidden)
    else:
        hidden = _llama_hidden(s)
        logits = s["model"].compute_logits(hidden[s["last"]])
    return dict(hidden=hidden, logits=logits, key_cache=s["cache"][0], value_cache=s["cache"][1])


def _awq_columns(words):
    """int32 [rows, n] -> values 0 .. 15 [rows, 8 n], in the column order of the AWQ checkpoint format."""
    nibble = torch.tensor([0, 4, 1, 5, 2, 6, 3, 7], device=words.device) * 4
    return ((words[:, :, None] >> nibble) & 15).reshape(words.shape[0], -1)


def _awq_weight(lin):
    rows = lambda t: t.repeat_interleave(128, 0)  # noqa: E731
    return (_awq_columns(lin.qweight) - rows(_awq_columns(lin.qzeros))).to(F64) * rows(lin.scales.to(F64))


def _rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _softmax_core(q, k, v, scale, visible, softcap=0.0, sinks=None):
    """q [H, n, D], k [H, m, D], v [H, m, V], visible [n, m] -> [H, n, V], all float64."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
    if softcap:
        s = softcap * torch.tanh(s / softcap)
    s = s.masked_fill(~visible, -math.inf)
    top = s.amax(-1, keepdim=True)
    if sinks is not None:
        top = torch.maximum(top, sinks.to(F64)[:, None, None])
    e = torch.exp(s - top)
    total = e.sum(-1, keepdim=True)
    if sinks is not None:
        total = total + torch.exp(sinks.to(F64)[:, None, None] - top)
    return torch.matmul(e, v) / total


def _visible(c, n, window=0):
    i, j = torch.arange(c, c + n, device="cuda")[:, None], torch.arange(c + n, device="cuda")[None]
    return (j <= i) & (i - j < window) if window else j <= i


def _llama_exact(case, seed):
    s = _llama_inputs(case, seed)
    model, cfg = s["model"], s["model"].cfg
    layer, fp8 = model.layers[0], case["kv"] == "fp8"
    H, G, D = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    new, context = _lengths(case)
    x = model.embed_tokens[s["ids"]].to(F64)
    q, k, v = (_rms(x) @ _awq_weight(layer.qkv_proj)).split([H * D, G * D, G * D], 1)
    # rotary angles: the table is kept in the model's type
    ang = s["positions"][:, None] * (cfg.rope_theta**(-torch.arange(0, D, 2, device="cuda", dtype=torch.float32) / D))[None]
    cos, sin = ang.cos().half().to(F64)[:, None], ang.sin().half().to(F64)[:, None]

    def turned(t, heads):
        a, b = t.view(-1, heads, D).split(D // 2, 2)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], 2)

    q, k, v = turned(q, H), turned(k, G), v.reshape(-1, G, D)
    if fp8:         # what the cache holds of a row
        def held(t):
            return t.clamp(-448, 448).float().to(torch.float8_e4m3fn).to(F64)
    else:
        def held(t):
            return t
    per = 16 if fp8 else 8
    keys = s["cache"][0].view(-1, G, D // per, BLOCK, per)
    values = s["cache"][1].view(-1, G, D, BLOCK)

    def wide(t):
        return (t.view(torch.float8_e4m3fn) if fp8 else t).to(F64)

    out, at = torch.empty_like(q), 0
    for b, (n, c) in enumerate(zip(new, context)):
        table = s["meta"].block_tables[b, :(n + c + BLOCK - 1) // BLOCK].long()
        kb = wide(keys[table]).permute(1, 0, 3, 2, 4).reshape(G, -1, D)[:, :c]
        vb = wide(values[table]).permute(1, 0, 3, 2).reshape(G, -1, D)[:, :c]
        # a decode step reads its own row from the cache, a prompt its rows as they are
        kn, vn = (held(k[at:at + n]), held(v[at:at + n])) if case["new"] == 1 else (k[at:at + n], v[at:at + n])
        kb, vb = torch.cat([kb, kn.transpose(0, 1)], 1), torch.cat([vb, vn.transpose(0, 1)], 1)
        seen = _visible(c, n)
        for h in range(G):
            q_h = q[at:at + n, h * (H // G):(h + 1) * (H // G)].transpose(0, 1)
            out[at:at + n, h * (H // G):(h + 1) * (H // G)] = _softmax_core(
                q_h, kb[h:h + 1].expand(H // G, -1, -1), vb[h:h + 1].expand(H // G, -1, -1), D**-0.5,
                seen).transpose(0, 1)
        at += n
    x = x + out.reshape(-1, H * D) @ _awq_weight(layer.o_proj)
    gate, up = (_rms(x) @ _awq_weight(layer.gate_up_proj)).chunk(2, 1)
    x = x + (torch.nn.functional.silu(gate) * up) @ _awq_weight(layer.down_proj)
    hidden = _rms(x)
    logits = hidden[s["last"]] @ model.lm_head.to(F64).t()
    return dict(hidden=hidden, logits=logits, key_cache=None, value_cache=None)


# ------------------------------------------------------------------------------- latent
def _latent_prepare(case, seed):
    g = _generator(seed)
    batch, tables, blocks, T = _batch(case, g)
    H, D, R, V, C = case["heads"], case["dim"], case["rot"], case["vdim"], case["rank"]
    layer = LatentKVAttention(H, D, R, V, C, (D + R)**-0.5, R, 10000.0, None, EPS, torch.bfloat16, "cuda",
                              window=case["window"] or None, sinks=case["sinks"])
    layer.set_weights(_randn(g, H * D, C, std=C**-0.5), _randn(g, H * V, C, std=C**-0.5),
                      1.0 + 0.1 * torch.randn(C, device="cuda", generator=g),
                      torch.randn(H, device="cuda", generator=g) if case["sinks"] else None)
    return dict(kind="latent", layer=layer, batch=batch, tables=tables,
                cache=_randn(g, *LatentKVAttention.get_cache_shape(blocks, BLOCK, C, R)),
                q=_randn(g, T, H * (D + R)), kv=_randn(g, T, C + R), gate=_randn(g, T, H) if case["gate"] else None)


@torch.inference_mode()
def _latent_run(s):
    q = s["q"].clone()      # a projection's result: new rows in every step, turned in place by the layer
    return dict(out=s["layer"](q, s["kv"], s["cache"], s["batch"], s["gate"]), cache=s["cache"])


def _turn(t, positions, dims, base, interleaved):
    """The first `dims` elements of every head of t [T, heads, D] turned by their position."""
    f = (float(base)**(-torch.arange(0, dims, 2, dtype=F64, device="cuda") / dims)).float()
    ang = (positions.float()[:, None] * f[None]).to(F64)[:, None]
    a, b = (t[..., 0:dims:2], t[..., 1:dims:2]) if interleaved else (t[..., :dims // 2], t[..., dims // 2:dims])
    x, y = a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()
    head = torch.stack([x, y], -1).flatten(-2) if interleaved else torch.cat([x, y], -1)
    return torch.cat([head, t[..., dims:]], -1)


def _latent_exact(case, seed):
    s = _latent_prepare(case, seed)
    layer, batch = s["layer"], s["batch"]
    H, D, R, V, C = case["heads"], case["dim"], case["rot"], case["vdim"], case["rank"]
    q, kv = s["q"].to(F64).view(-1, H, D + R), s["kv"].to(F64)
    c, rot = _rms(kv[:, :C]) * layer.latent_norm.to(F64), kv[:, None, C:]
    if R:
        q = torch.cat([q[..., :D], _turn(q[..., D:], batch.positions, R, 1e4, True)], -1)
        rot = _turn(rot, batch.positions, R, 1e4, True)
    row = torch.cat([c, rot[:, 0]], 1)
    cache = s["cache"].to(F64)
    cache.view(-1, C + R)[batch.slot_mapping] = row
    out, at = torch.empty(q.shape[0], H, V, dtype=F64, device="cuda"), 0
    for (n, past), table in zip(zip(*_lengths(case)), s["tables"]):
        rows = cache[torch.tensor(table, device="cuda")].reshape(-1, C + R)[:n + past]
        seen = _visible(past, n, case["window"])
        for h in range(H):
            k = torch.cat([rows[:, :C] @ layer.w_uk[h].to(F64).t(), rows[:, C:]], 1)
            out[at:at + n, h] = _softmax_core(q[None, at:at + n, h], k[None], (rows[:, :C] @ layer.w_uv_t[h].to(F64))[None],
                                              (D + R)**-0.5, seen, 0.0, layer.sinks[h:h + 1] if case["sinks"] else None)[0]
        at += n
    if s["gate"] is not None:
        out = out * torch.sigmoid(s["gate"].to(F64))[..., None]
    return dict(out=out.reshape(-1, H * V), cache=cache)


# ------------------------------------------------------------------------------- kv
def _kv_prepare(case, seed):
    g = _generator(seed)
    batch, tables, blocks, T = _batch(case, g)
    H, G, D = case["heads"], case["kv_heads"], case["dim"]
    layer = RotaryKVAttention(H, G, D, D, D**-0.5, case["rot_dims"], 10000.0, case["interleaved"],
                              window=case["window"] or None, device="cuda", softcap=case["softcap"])
    ks, vs = RotaryKVAttention.get_cache_shapes(blocks, BLOCK, G, D, D)
    # q, k and v are parts of one projection's rows
    return dict(kind="kv", layer=layer, batch=batch, tables=tables, keys=_randn(g, *ks), values=_randn(g, *vs),
                proj=_randn(g, T, (H + 2 * G) * D), parts=[H * D, G * D, G * D],
                gate=_randn(g, T, H) if case["gate"] else None)


@torch.inference_mode()
def _kv_run(s):
    q, k, v = s["proj"].clone().split(s["parts"], 1)    # a projection's result, turned in place by the layer
    out = torch.empty((q.shape[0], s["parts"][0]), dtype=q.dtype, device=q.device)
    s["layer"](out, q, k, v, s["gate"], s["keys"], s["values"], s["batch"])
    return dict(out=out, keys=s["keys"], values=s["values"])


def _kv_exact(case, seed):
    s = _kv_prepare(case, seed)
    batch = s["batch"]
    H, G, D = case["heads"], case["kv_heads"], case["dim"]
    q, k, v = s["proj"].to(F64).split(s["parts"], 1)
    q = _turn(q.view(-1, H, D), batch.positions, case["rot_dims"], 1e4, case["interleaved"])
    k = _turn(k.view(-1, G, D), batch.positions, case["rot_dims"], 1e4, case["interleaved"])
    keys, values = s["keys"].to(F64), s["values"].to(F64)
    keys.view(-1, G, D)[batch.slot_mapping] = k
    values.view(-1, G, D)[batch.slot_mapping] = v.reshape(-1, G, D)
    out, at = torch.empty_like(q), 0
    for (n, past), table in zip(zip(*_lengths(case)), s["tables"]):
        table = torch.tensor(table, device="cuda")
        kb, vb = (t[table].reshape(-1, G, D)[:n + past] for t in (keys, values))
        seen = _visible(past, n, case["window"])
        for h in range(H):
            j = h // (H // G)
            out[at:at + n, h] = _softmax_core(q[None, at:at + n, h], kb[None, :, j], vb[None, :, j], D**-0.5, seen,
                                              case["softcap"])[0]
        at += n
    if s["gate"] is not None:
        out = out * torch.sigmoid(s["gate"].to(F64))[..., None]
    return dict(out=out.reshape(-1, H * D), keys=keys, values=values)


# ------------------------------------------------------------------------------- recur
def _recur_prepare(case, seed):
    g = _generator(seed)
    batch, _, _, T = _batch(case, g)
    H, G, D, V = case["heads"], case["kv_heads"], case["dim"], case["vdim"]

    def vec(n, mean, std):
        return mean + std * torch.randn(n, device="cuda", generator=g)

    s = dict(kind="recur", rule=case["rule"], batch=batch, norm=vec(V, 1.0, 0.1))
    if case["rule"] == "linear":
        s["layer"] = GatedLinearRecurrence(H, D, V, 8.0, EPS)
        shape = GatedLinearRecurrence.get_state_shape(case["seqs"], H, D, V)
        s["proj"], s["parts"] = _randn(g, T, 2 * H * D + 2 * H * V + 16), [H * D, H * D, H * V, H * V, 16]
        s["w2"], s["bias"] = _randn(g, H * D, 16, std=0.25), vec(H * D, 2.0, 1.0)
    else:
        s["layer"] = layer = GatedDeltaRule(H, G, D, V, EPS, "cuda")
        layer.a_log.data, layer.dt_bias.data, layer.norm_weight.data = vec(H, 0.0, 0.3), vec(H, -3.0, 1.0), s["norm"]
        shape = GatedDeltaRule.get_state_shape(case["seqs"], H, D, V)
        s["proj"], s["parts"] = _randn(g, T, 2 * G * D + 2 * H * V + 2 * H, dtype=torch.float32), \
            [G * D, G * D, H * V, H * V, H, H]
    s["state"] = _randn(g, *shape, dtype=torch.float32, std=0.1)
    s["seqs"] = case["seqs"]
    return s


@torch.inference_mode()
def _recur_run(s):
    parts = s["proj"].split(s["parts"], 1)
    out = torch.empty((s["proj"].shape[0], s["parts"][3]), dtype=torch.bfloat16, device="cuda")
    if s["rule"] == "linear":
        q, k, v, gate, y = parts
        s["layer"](out, q, k, v, gate, y, s["w2"], s["bias"], s["norm"], s["state"], s["batch"])
    else:
        q, k, v, gate, beta, dt = parts
        s["layer"](out, q, k, v, gate, beta, dt, s["state"], s["batch"])
    return dict(out=out, state=s["state"][:s["seqs"]])


def _recur_exact(case, seed):
    s = _recur_prepare(case, seed)
    H, G, D, V = case["heads"], case["kv_heads"], case["dim"], case["vdim"]
    parts = [t.to(F64) for t in s["proj"].split(s["parts"], 1)]
    q, k, v, gate = parts[0].view(-1, G, D), parts[1].view(-1, G, D), parts[2].view(-1, H, V), parts[3].view(-1, H, V)
    linear = case["rule"] == "linear"
    if linear:
        z = parts[4] @ s["w2"].to(F64).t() + s["bias"].to(F64)
        decay = torch.exp(torch.nn.functional.logsigmoid(z) / 8.0).view(-1, H, D)
        q = q * D**-0.5
    else:
        q = q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * D**-0.5
        k = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        q, k = q.repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1)
        layer = s["layer"]
        beta = torch.sigmoid(parts[4])
        decay = torch.exp(-torch.exp(layer.a_log.to(F64)) *
                          torch.nn.functional.softplus(parts[5] + layer.dt_bias.to(F64)))[..., None]
    new, context = _lengths(case)
    start = torch.tensor([sum(new[:b]) for b in range(len(new))], device="cuda")
    lens = torch.tensor(new, device="cuda")
    slots = s["state"][:case["seqs"]].to(F64)
    S = (slots if linear else slots.transpose(2, 3)) * torch.tensor(context, device="cuda").gt(0)[:, None, None, None]
    out = torch.empty(v.shape, dtype=F64, device="cuda")
    for t in range(max(new)):       # token by token, all sequences that still have one
        live = torch.tensor([b for b in range(len(new)) if new[b] > t], device="cuda")
        row = start[live] + t
        assert bool((lens[live] > t).all())
        Sl = S[live] * decay[row][..., None]
        u = v[row] if linear else beta[row][..., None] * (v[row] - (Sl * k[row][..., None]).sum(2))
        Sl = Sl + k[row][..., None] * u[:, :, None]
        S[live] = Sl
        out[row] = (Sl * q[row][..., None]).sum(2)
    out = _rms(out) * s["norm"].to(F64) * torch.nn.functional.silu(gate)
    return dict(out=out.reshape(-1, H * V), state=S if linear else S.transpose(2, 3))


# ------------------------------------------------------------------------------- experts
def _experts_prepare(case, seed):
    g = _generator(seed)
    W, E, F = case["width"], case["experts"], case["ff"]
    layer = RoutedExperts(W, E, 0, case["top"], F, case["shared"], act="silu" if case["gated"] else "relu2",
                          dtype=torch.bfloat16, device="cuda", gated=case["gated"])
    t = dict(router=_randn(g, E, W, dtype=torch.float32, std=W**-0.5))
    for e in range(E):
        for name in ("gate", "up") if case["gated"] else ("up", ):
            t[f"e{e}.{name}"] = _randn(g, F, W, std=W**-0.5)
        t[f"e{e}.down"] = _randn(g, W, F, std=F**-0.5)
    if case["shared"]:
        t["shared.up"], t["shared.down"] = _randn(g, case["shared"], W, std=W**-0.5), _randn(g, W, case["shared"], std=F**-0.5)
        t["shared.sg"] = _randn(g, W, dtype=torch.float32, std=W**-0.5)
    layer.set_weights(t)
    return dict(kind="experts", layer=layer, h=_randn(g, case["tokens"], W), weights=t)


@torch.inference_mode()
def _experts_run(s):
    return s["layer"](s["h"])


def _experts_exact(case, seed):
    s = _experts_prepare(case, seed)
    t, h, F = {k: v.to(F64) for k, v in s["weights"].items()}, s["h"].to(F64), torch.nn.functional
    top, chosen = torch.softmax(h @ t["router"].t(), -1).topk(case["top"], -1)
    top = top / top.sum(-1, keepdim=True)
    act = F.silu if case["gated"] else (lambda x: F.relu(x)**2)
    out = torch.zeros_like(h)
    for e in range(case["experts"]):
        row, place = (chosen == e).nonzero(as_tuple=True)
        x, up = h[row], h[row] @ t[f"e{e}.up"].t()
        y = (act(x @ t[f"e{e}.gate"].t()) * up if case["gated"] else act(up)) @ t[f"e{e}.down"].t()
        out.index_add_(0, row, y * top[row, place, None])
    if case["shared"]:
        out = out + torch.sigmoid(h @ t["shared.sg"])[:, None] * (act(h @ t["shared.up"].t()) @ t["shared.down"].t())
    return out


# ------------------------------------------------------------------------------- the file's functions
def prepare(case, seed):
    return {"llama": _llama_prepare, "latent": _latent_prepare, "kv": _kv_prepare, "recur": _recur_prepare,
            "experts": _experts_prepare}[case["kind"]](case, seed)


def run(state):
    return {"llama": _llama_run, "latent": _latent_run, "kv": _kv_run, "recur": _recur_run,
            "experts": _experts_run}[state["kind"]](state)


def exact(case, seed):
    with torch.inference_mode():
        return {"llama": _llama_exact, "latent": _latent_exact, "kv": _kv_exact, "recur": _recur_exact,
                "experts": _experts_exact}[case["kind"]](case, seed)


def _pairs(case, window=0):
    """(query, key) pairs that causality and the window let be seen, over all sequences."""
    total = 0
    for n, c in zip(*_lengths(case)):
        if window:
            total += sum(min(i + 1, window) for i in range(c, c + n))
        else:
            total += n * c + n * (n + 1) // 2
    return total


def work(case):
    kind = case["kind"]
    if kind == "experts":
        T, W, E, k, F = case["tokens"], case["width"], case["experts"], case["top"], case["ff"]
        mats, used = 3 if case["gated"] else 2, E * (1 - (1 - k / E)**T)       # experts that some token chooses
        return dict(bytes=2.0 * mats * used * F * W + 6.0 * T * W + 4.0 * E * W + 4.0 * case["shared"] * W,
                    flops=2.0 * mats * T * k * F * W + 2.0 * T * E * W + 4.0 * T * case["shared"] * W)
    new, context = _lengths(case)
    T, window = sum(new), case.get("window", 0)
    past = sum(min(c, window) if window else c for c in context)    # cached rows that some query sees
    if kind == "llama":
        h, ff, q, kv, size = 4096, 14336, 4096, 1024, 1 if case["kv"] == "fp8" else 2
        params = h * (q + 2 * kv) + q * h + 3 * h * ff
        rows = T if case["new"] == 1 else len(new)
        return dict(bytes=params * (0.5 + 2.5 / 128) + 2 * kv * size * (past + T) + 2.0 * 1024 * h + 4.0 * T * h + 2.0 * rows * 1024,
                    flops=2.0 * T * params + 4.0 * q * _pairs(case) + 2.0 * rows * 1024 * h)
    if kind == "latent":
        H, D, R, V, C = case["heads"], case["dim"], case["rot"], case["vdim"], case["rank"]
        pairs = _pairs(case, window)
        # the cheaper of scoring the latent itself and of forming every head's keys and values from it
        direct = 2.0 * pairs * H * (2 * C + R) + 2.0 * T * H * C * (D + V)
        formed = 2.0 * pairs * H * (D + R + V) + 2.0 * (past + T) * H * C * (D + V)
        return dict(bytes=2.0 * ((past + 2 * T) * (C + R) + T * H * (D + R + V) + H * C * (D + V)), flops=min(direct, formed))
    if kind == "kv":
        H, G, D = case["heads"], case["kv_heads"], case["dim"]
        return dict(bytes=2.0 * (2 * G * D * (past + 2 * T) + 2 * H * D * T), flops=4.0 * _pairs(case, window) * H * D)
    H, G, D, V = case["heads"], case["kv_heads"], case["dim"], case["vdim"]
    size, starts = 2 if case["rule"] == "linear" else 4, sum(c > 0 for c in context)
    extra = 16 if case["rule"] == "linear" else 2 * H
    return dict(bytes=float(T * (size * (2 * G * D + 2 * H * V + extra) + 2 * H * V) + 4 * (starts + len(new)) * H * D * V),
                flops=(4.0 if case["rule"] == "linear" else 6.0) * T * H * D * V)


def tolerance(case):
    """Results are rounded to 16 bits, and so are the operands between kernels: relative errors against 64 bits of
    0.0017 (recurrences, which are fp32 inside), 0.0024 to 0.0035 (attention, experts) and up to 0.0012 (a whole
    decoder layer in float16), and another order of sums moves each by as much; four times that."""
    rel = dict(recur=0.007, latent=0.014, kv=0.012, experts=0.012, llama=0.006)[case["kind"]]
    return dict(rel=rel, max=12 * rel, differ=0.01)

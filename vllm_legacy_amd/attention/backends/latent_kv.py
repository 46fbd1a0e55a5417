"""Causal softmax attention whose keys and values are up-projections of one cached latent.

Per token the layer caches one row [c | k_rot]: the RMS-normed latent c (`rank` numbers) and a
rotated key part (`rot` numbers) that all heads share -- cache [num_blocks, block_size, rank + rot].
Head h scores a query (q_plain [dim], q_rot [rot]) against key j as
(q_plain . W_uk,h c_j + q_rot . k_rot_j) * scale and sums values W_uv,h c_j.  For single rows and
short runs both up-projections are moved to the query's side, where they cost one batched matrix product per step each:
q_lat,h = W_uk,h^T q_plain,h scores the cached latent directly, and the head's output is
W_uv,h (sum_j p_j c_j).  Rotation: pairs (2i, 2i + 1) when `interleaved`, (i, i + rot_dims / 2)
otherwise, of the first `rot_dims` elements of the rotated parts turn by position * f_i, sine and
cosine times `magnitude` (a frequency table and a magnitude as YaRN scaling gives them, or plain
ones).  `scale` multiplies the scores as it is.  An optional `window` keeps 0 <= i - j < window;
an optional gate [T, heads] multiplies each head's output by its sigmoid (applied to the latent
sums, ahead of the linear up-projection).  `sinks` gives every head a learned number whose
exponential joins its softmax denominator (a key without a value, not scaled).  With
`own_latent=False` the layer forms no latents: it reads the cache another layer fills (same rank, no
rotated part), with queries and up-projections of its own.  In prompts, portions of prompts
and decode steps alike the step's rows are written to the cache, then every query row reads from there
(csrc/seq_latent_attention.hip: a matrix-core kernel for 16-bit models whose rank is a multiple of 32 and whose rotated part is a multiple of 16,
and an fp32 kernel for any dtype and size).  Runs of many rows with enough work, of sizes that the matrix-core
kernel takes, form every head's keys and values from the cached latents instead, in a workspace of fixed size, and
score those (csrc/seq_latent_prompt.hip).
"""
import math
from typing import Dict, Optional, Tuple

import torch
import torch.nn as nn

from vllm_legacy_amd import _seq_ops as ops
from vllm_legacy_amd.attention.batch import SequenceBatch


def yarn_frequencies(dims: int, base: float, scaling: Optional[Dict] = None,
                     device=None) -> Tuple[torch.Tensor, float]:
    """(f_i fp32 [dims / 2], magnitude).  Without scaling f_i = base^(-2i / dims) and the magnitude
    is 1.  With scaling {factor, original, fast, slow}: a pair that makes `t` turns over `original`
    positions sits at d(t) = dims ln(original / (2 pi t)) / (2 ln base); pairs below
    lo = floor(d(fast)) keep their frequency, pairs above hi = ceil(d(slow)) get f_i / factor, a
    linear ramp joins them, and sine and cosine are multiplied by 0.1 ln(factor) + 1.  Formed in
    float64, rounded once to fp32."""
    i = torch.arange(dims // 2, dtype=torch.float64)
    f = torch.pow(torch.tensor(float(base), dtype=torch.float64), -2.0 * i / float(dims))
    magnitude = 1.0
    if scaling:
        factor, original = float(scaling["factor"]), float(scaling["original"])

        def place(turns: float) -> float:
            return dims * math.log(original / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

        lo = max(math.floor(place(float(scaling["fast"]))), 0)
        hi = min(math.ceil(place(float(scaling["slow"]))), dims - 1)
        ramp = torch.clamp((i - lo) / max(hi - lo, 0.001), 0.0, 1.0)
        f = f / factor * ramp + f * (1.0 - ramp)
        magnitude = 0.1 * math.log(factor) + 1.0
    return f.to(torch.float32).to(device), magnitude


class LatentKVAttention(nn.Module):

    def __init__(self, num_heads: int, head_dim: int, rot_dim: int, value_dim: int, rank: int, scale: float,
                 rot_dims: int, rot_base: float, rot_scaling: Optional[Dict], eps: float, dtype=torch.bfloat16,
                 device=None, interleaved: bool = True, window: Optional[int] = None, sinks: bool = False,
                 own_latent: bool = True) -> None:
        super().__init__()
        if not own_latent and rot_dim:
            raise ValueError("a layer that reads another layer's latents has no rotated key part")
        self.own_latent = bool(own_latent)
        self.sinks = nn.Parameter(torch.zeros(num_heads, dtype=torch.float32, device=device),
                                  requires_grad=False) if sinks else None
        assert 0 <= rot_dims <= rot_dim and rot_dims % 2 == 0
        self.interleaved, self.window = bool(interleaved), int(window) if window else 0
        self.num_heads, self.head_dim, self.rot_dim, self.value_dim, self.rank = num_heads, head_dim, rot_dim, value_dim, rank
        self.scale, self.rot_dims, self.eps, self.dtype = float(scale), int(rot_dims), float(eps), dtype
        inv_freq, self.magnitude = yarn_frequencies(rot_dims, rot_base, rot_scaling, device) if rot_dims else (None, 1.0)
        self.register_buffer("inv_freq", inv_freq, persistent=False)
        self.latent_norm = nn.Parameter(torch.ones(rank, dtype=torch.float32, device=device),
                                        requires_grad=False) if own_latent else None
        # W_uk as [heads, dim, rank] (q_lat = q_plain W_uk,h) and W_uv^T as [heads, rank, vdim]
        self.w_uk = nn.Parameter(torch.zeros((num_heads, head_dim, rank), dtype=dtype, device=device),
                                 requires_grad=False)
        self.w_uv_t = nn.Parameter(torch.zeros((num_heads, rank, value_dim), dtype=dtype, device=device),
                                   requires_grad=False)
        self.formed_fits = True
        gain = 5 * (2 * rank + rot_dim) - 2 * (head_dim + rot_dim + value_dim)      # (formed_min_rows)
        self.least_rows = -(-rank * (head_dim + value_dim) // gain) if gain > 0 else 1 << 30
        self.few_rows = max(self.FORMED_FEW_ROWS, self.least_rows) if num_heads > 2 else 1 << 30
        self.tile_rows, self.tile_sets = 32 // min(num_heads, 32), -(-num_heads // min(num_heads, 32))
        # (formed_is_faster: us a (query, key) pair and a key of a CU's walk on the latent kernel; the keys of a part; us a key of
        # the longest walk, a pair and a key of them all, formed)
        self.costs = (2.1e-9 * num_heads * (2 * rank + rot_dim), 0.0155 + 0.0912 / 512 * rank, self.formed_keys(2),
                      0.0158 + 0.0046 / 128 * head_dim, 1.75e-9 * num_heads * (2 * head_dim + rot_dim + value_dim),
                      2.44e-9 * num_heads * (head_dim + value_dim) * (rank + 128) + 1.17e-6 * (rank + rot_dim))
        # keys behind which runs of FORMED_MIN_ROWS go formed (one or four of them): nothing more is asked of most steps
        self.near_keys, rows = self.FORMED_NEAR_KEYS, max(self.FORMED_MIN_ROWS, self.least_rows)
        while self.near_keys < 2400 and rows < 1024 and all(
                self.formed_is_faster([rows] * n, [2 * self.near_keys] * n) for n in (1, 4)):
            self.near_keys *= 2

    def set_weights(self, uk: torch.Tensor, uv: torch.Tensor, latent_norm: Optional[torch.Tensor] = None,
                    sinks: Optional[torch.Tensor] = None) -> None:
        """uk [heads * dim, rank], uv [heads * vdim, rank] (rows head by head), latent_norm [rank] (own
        latents), sinks [heads] (where the layer has them)."""
        dev = self.w_uk.device
        H, D, V, C = self.num_heads, self.head_dim, self.value_dim, self.rank
        self.w_uk.data = uk.to(self.dtype).view(H, D, C).to(dev).contiguous()
        self.w_uv_t.data = uv.to(self.dtype).view(H, V, C).transpose(1, 2).to(dev).contiguous()
        if self.own_latent:
            self.latent_norm.data = latent_norm.float().to(dev).contiguous()
        if self.sinks is not None:
            self.sinks.data = sinks.float().to(dev).contiguous()
        # No formed key or value may leave the dtype's range, where sums of latents stay in it.  A normed latent's
        # length is at most sqrt(rank) times the norm's largest weight (another layer's: taken as 8 at most).
        length = math.sqrt(C) * (float(latent_norm.abs().max()) if self.own_latent else 8.0)
        self.formed_fits = max(float(w.float().norm(dim=1).max()) for w in (uk, uv)) * length < torch.finfo(self.dtype).max

    # workgroups a launch should have before the keys of a row tile stay with one workgroup
    SPLIT_BELOW_WORKGROUPS = 512
    KEYS_PER_SPLIT = 256

    def key_splits(self, batch: SequenceBatch) -> int:
        """Steps of few rows over long contexts (decode steps) share every row tile's keys out to
        several workgroups: enough of them to fill the part, none with fewer than KEYS_PER_SPLIT
        keys."""
        return self._key_splits(batch.max_query_len, batch.num_seqs, batch.max_seq_len)

    def _key_splits(self, max_query_len: int, num_seqs: int, keys: int) -> int:
        tiles = -(-max_query_len // self.tile_rows) * self.tile_sets * num_seqs
        if tiles >= self.SPLIT_BELOW_WORKGROUPS:
            return 1
        if self.window:
            keys = min(keys, self.window + max_query_len)
        return max(1, min(-(-self.SPLIT_BELOW_WORKGROUPS // tiles), keys // self.KEYS_PER_SPLIT, 32))

    # the longest stretches of sequences a step is cut into; one that alternates more often stays whole
    MAX_STRETCHES = 4

    # Multiply-adds of a step's long runs on the latent kernel from which those runs go formed whatever else is in the step.
    FORMED_MIN_WORK = 6e9
    # Their rows at least: forming a key's numbers costs as much for few rows as for many.
    FORMED_MIN_ROWS = 96
    # Runs of so many rows go formed too, all of a step's, where that is the faster way: behind so few keys it always is (of 382
    # measured steps), behind more formed_is_faster says so.
    FORMED_FEW_ROWS = 32
    FORMED_NEAR_KEYS = 300

    def formed_min_rows(self) -> int:
        """Rows from which a run's keys and values are worth forming.  A (query, key) pair of a head costs the
        latent kernel 2 rank + rot multiply-adds at a fifth of a matrix product's rate (less where the rank is small),
        the formed one dim + rot + vdim at about half of it; forming costs rank (dim + vdim) per key at the full rate."""
        return max(self.FORMED_MIN_ROWS, self.least_rows)

    def formed_is_faster(self, lens, contexts) -> bool:
        """Both ways' time on the GPU for sequences of `lens` rows behind `contexts` keys, in us, as measured over 4 to 128
        heads of 32 to 128, ranks of 64 to 512, 1 to 30 sequences of 33 to 512 rows behind 0 to 8000 keys (750 steps;
        rms errors of 12 and 9 %).  Latent: launches, a merge where keys are shared out, the products, and the keys that
        a CU's workgroups walk (between the most that one may have and its share).  Formed: launches, the walk of the longest
        sequence's keys by one workgroup per 128 rows and head, forming, products and the gathered rows; one part of the
        workspace after the other.  Of those steps four are slower than on the latent kernel, by 2 to 10 %, of 439 of uneven lengths none; the
        host's part is less (65 us of Python and launches, 90).  Latent / formed, 16 heads of 128 + 64, rank 512: 33 rows
        x 300 keys 67 / 40, x 1000 68 / 57, x 2000 77 / 80, thirty of x 300 127 / 112 and x 1000 334 / 350; 48 x 1500 73 / 71;
        64 x 1000 69 / 59, x 2000 74 / 88; 96 x 500 72 / 48, x 2500 109 / 105; three of 54 x 1240 117 / 79, four of 48 x 2000
        177 / 121.  Rank 64, 96 x 1500 48 / 63, 1024 x 0 90 / 55.  One or two heads, whose few workgroups the sums are furthest
        off for, stay (one head, 128 x 1500 63 / 71, x 5000 66 / 152)."""
        w, rows_of_tile, tile_sets = self.window, self.tile_rows, self.tile_sets
        pairs = total = walked = longest = most_rows = 0
        for n, c in zip(lens, contexts):
            k = (min(c, w) if w else c) + n
            pairs += n * (k - n) + (n * (n + 1) // 2 if not w else n * min(n, w))
            total += k
            walked += -(-n // rows_of_tile) * k
            if k > longest:
                longest = k
            if n > most_rows:
                most_rows = n
        splits = self._key_splits(most_rows, len(lens), longest)
        share, walked = -(-longest // splits), walked * tile_sets
        most = -(-sum(-(-n // rows_of_tile) * -(-((min(c, w) if w else c) + n) // share) for n, c in zip(lens, contexts)) *
                 tile_sets // 256) * share
        of_pair, of_key, room, of_walk, of_formed_pair, of_formed_key = self.costs
        latent = 33.4 + 5.5 * (splits > 1) + of_pair * pairs + (most + max(share, walked / 256)) / 2 * of_key
        parts, walk = 1, longest
        if total > room:
            held = self._formed_parts(lens, contexts, room)
            parts, walk = len(held), sum(count if b1 == b0 + 1 else max((min(c, w) if w else c) + n for n, c in zip(
                lens[b0:b1], contexts[b0:b1])) for b0, b1, _, count, _ in held)
        return 26.5 * parts + walk * of_walk + of_formed_pair * pairs + total * of_formed_key < latent

    def _stretches(self, batch: SequenceBatch):
        """[[first sequence, one behind the last, first row, one behind the last, formed]]: neighbours that go
        the same way; None when the whole step takes the latent kernel."""
        q, ctx = batch.host_query_lens, batch.host_context_lens
        if q is None or ctx is None or not self.scale > 0 or not self.formed_fits or torch.cuda.is_current_stream_capturing():
            return None                 # a captured step is replayed with other lengths than the host's
        short = min(q)
        whole = short >= self.few_rows
        if whole and max(ctx) <= (self.near_keys if short >= self.formed_min_rows() else self.FORMED_NEAR_KEYS):
            return [[0, len(q), 0, batch.num_tokens, True]]
        each = self.num_heads * (2 * self.rank + self.rot_dim)          # multiply-adds of a (query, key) pair
        if batch.num_tokens * batch.max_seq_len * each >= self.FORMED_MIN_WORK and batch.max_query_len >= self.FORMED_MIN_ROWS:
            least = self.formed_min_rows()
            out, row, pairs = [], 0, 0
            for b, (n, c) in enumerate(zip(q, ctx)):
                if n >= least:
                    pairs += n * min(c, self.window or c) + (n * (n + 1) // 2 if not self.window else n * min(n, self.window))
                if out and out[-1][4] == (n >= least):
                    out[-1][1], out[-1][3] = b + 1, row + n
                else:
                    out.append([b, b + 1, row, row + n, n >= least])
                row += n
            if pairs * each >= self.FORMED_MIN_WORK:
                if len(out) > 1 and whole:
                    few = [(n, c) for n, c in zip(q, ctx) if n < least]
                    if self.formed_is_faster([n for n, _ in few], [c for _, c in few]):
                        return [[0, len(q), 0, row, True]]
                return out if len(out) <= self.MAX_STRETCHES else None
        if whole and self.formed_is_faster(q, ctx):
            return [[0, len(q), 0, batch.num_tokens, True]]
        return None

    # bytes of gathered rows and formed keys and values at a time: 20 thousand keys of 16 heads of 128 + 128
    FORMED_WORKSPACE = 1 << 28

    def formed_keys(self, size: int) -> int:
        """Keys that FORMED_WORKSPACE holds (whole tiles of 64, at least one): their cache rows, keys in two parts
        and values, `size` bytes a number."""
        each = size * (self.rank + self.rot_dim + self.num_heads * (2 * self.head_dim + self.value_dim))
        return max(64, self.FORMED_WORKSPACE // each // 64 * 64)

    def _formed_parts(self, lens, contexts, most: int):
        """[(first sequence, one behind the last, first key, keys, all keys)]: neighbours whose visible keys are at
        most `most` together, and ranges of the keys of one that has more by itself."""
        parts, first, held = [], 0, 0
        for b, (n, c) in enumerate(zip(lens, contexts)):
            count = c + n - (max(0, c - self.window + 1) if self.window else 0)
            if held and held + count > most:
                parts.append((first, b, 0, held, held))
                held = 0
            if count > most:
                parts += [(b, b + 1, k, min(most, count - k), count) for k in range(0, count, most)]
                first = b + 1
            else:
                first = first if held else b
                held += count
        if held:
            parts.append((first, len(lens), 0, held, held))
        return parts

    def _attend_formed(self, out, q, cache, batch: SequenceBatch, s0, s1, r0, r1, gate) -> None:
        """Sequences s0 .. s1 - 1 (rows r0 .. r1 - 1) with keys and values formed per head."""
        H, D, Rr, V, C = self.num_heads, self.head_dim, self.rot_dim, self.value_dim, self.rank
        ql, cl = batch.host_query_lens[s0:s1], batch.host_context_lens[s0:s1]
        sinks = None if self.sinks is None else self.sinks.data
        carry = None
        for b0, b1, k0, count, total in self._formed_parts(ql, cl, self.formed_keys(q.element_size())):
            if k0 == 0:
                t0 = r0 + sum(ql[:b0])
                t1 = t0 + sum(ql[b0:b1])
                tables, ctx = batch.block_tables[s0 + b0:s0 + b1], batch.context_lens[s0 + b0:s0 + b1]
                starts = batch.query_start_loc[s0 + b0:s0 + b1 + 1]
                if t0:
                    starts = starts - t0
                carry = ops.latent_prompt_carry(q[t0:t1], H, V) if count < total else None
            rows = torch.empty((count, C + Rr), dtype=q.dtype, device=q.device)
            longest = count if b1 == b0 + 1 else max(c + n for n, c in zip(ql[b0:b1], cl[b0:b1]))
            ops.latent_gather(rows, cache, tables, starts, ctx, longest, self.window, k0)
            # A key's rounding is its own, where that of a query on the latents' side is the same for all keys and
            # mostly cancels in the softmax: the keys keep what they lose.
            keys, keys_rest, values = ops.latent_form(rows, self.w_uk.data, self.w_uv_t.data)
            ops.latent_prompt(out[t0:t1], q[t0:t1], keys, keys_rest, values, rows, starts, ctx, max(ql[b0:b1]), H, D, Rr, V,
                              self.scale, self.window, None if gate is None else gate[t0:t1], sinks, k0,
                              total if carry is not None else 0, carry)
            del rows, keys, keys_rest, values          # the next part's take their place

    def _attend_latent(self, q, cache, batch: SequenceBatch, gate, part=None) -> torch.Tensor:
        """The step, or of part (s0, s1, r0, r1) sequences s0 .. s1 - 1 (rows r0 .. r1 - 1), on the cached latents ->
        [rows, heads * vdim]."""
        H, D, Rr, C = self.num_heads, self.head_dim, self.rot_dim, self.rank
        sinks = None if self.sinks is None else self.sinks.data
        if part is not None:
            s0, s1, r0, r1 = part
            q, gate = q[r0:r1], None if gate is None else gate[r0:r1]
        T = q.shape[0]
        q3 = q.view(T, H, D + Rr)
        q_lat = torch.bmm(q3.narrow(2, 0, D).transpose(0, 1), self.w_uk.data)       # [H, T, C]
        o_lat = torch.empty((H, T, C), dtype=q.dtype, device=q.device)
        q_lat, q_rot, o_rows = q_lat.transpose(0, 1), q3.narrow(2, D, Rr), o_lat.transpose(0, 1)
        if ops.latent_attention_tiles_supported(q_lat, q_rot, cache):
            # 16-bit models whose sizes fit: (token, head) rows in tiles of 32 on the matrix cores
            if part is None and batch.max_query_len == 1 and ops.latent_decode_supported(o_rows, q_lat, q_rot, cache):
                keys = min(batch.max_seq_len, self.window or batch.max_seq_len)
                w_uv = self.w_uv_t.data
                out = torch.empty((T, H * self.value_dim), dtype=q.dtype, device=q.device) \
                    if ops.latent_decode_up_supported(w_uv) else None
                ops.latent_decode(o_rows, q_lat, q_rot, cache, batch.block_tables, batch.query_start_loc,
                                  batch.context_lens, keys, self.scale, self.window, gate, sinks, out, w_uv)
                if out is not None:
                    return out
            elif part is None:
                ops.latent_attention_tiles(o_rows, q_lat, q_rot, cache, batch.block_tables, batch.query_start_loc,
                                           batch.context_lens, batch.max_query_len, self.scale, self.key_splits(batch),
                                           self.window, gate, sinks)
            else:
                ql, cl = batch.host_query_lens[s0:s1], batch.host_context_lens[s0:s1]
                longest = max(ql)
                splits = self._key_splits(longest, s1 - s0, max(c + n for n, c in zip(ql, cl)))
                ops.latent_attention_tiles(o_rows, q_lat, q_rot, cache, batch.block_tables[s0:s1],
                                           batch.query_start_loc[s0:s1 + 1] - r0, batch.context_lens[s0:s1], longest,
                                           self.scale, splits, self.window, gate, sinks)
        else:
            rows = slice(None) if part is None else slice(r0, r1)
            ops.latent_attention(o_rows, q_lat, q_rot, cache, batch.block_tables, batch.token_seq[rows],
                                 batch.positions[rows], self.scale, self.window, gate, sinks)
        o = torch.bmm(o_lat, self.w_uv_t.data)                                      # [H, T, V]
        return o.transpose(0, 1).reshape(T, H * self.value_dim)

    @staticmethod
    def get_cache_shape(num_blocks: int, block_size: int, rank: int, rot_dim: int) -> Tuple[int, ...]:
        return (num_blocks, block_size, rank + rot_dim)

    def forward(self, q: torch.Tensor, kv: Optional[torch.Tensor], cache: torch.Tensor, batch: SequenceBatch,
                gate: Optional[torch.Tensor] = None) -> torch.Tensor:
        """q [T, heads * (dim + rot_dim)], head by head [plain | rotated] (rotated in place); kv
        [T, rank + rot_dim] before its norm and rotation (None: the cache already holds this step's rows),
        gate [T, heads] (views with free row strides).  Returns [T, heads * vdim]."""
        assert (kv is not None) == self.own_latent
        if self.own_latent:
            D, Rr = self.head_dim, self.rot_dim
            ops.latent_rotary_write(q, D + Rr, D, self.num_heads, kv, self.latent_norm.data, self.eps, cache, batch.positions,
                                    batch.slot_mapping, self.inv_freq, self.magnitude, self.rot_dims, self.interleaved)
        stretches = None if batch.max_query_len < self.FORMED_FEW_ROWS else self._stretches(batch)
        if stretches is None or not ops.latent_prompt_supported(q, self.head_dim, self.rot_dim, self.value_dim, self.rank, cache):
            return self._attend_latent(q, cache, batch, gate)
        out = torch.empty((q.shape[0], self.num_heads * self.value_dim), dtype=q.dtype, device=q.device)
        for s0, s1, r0, r1, formed in stretches:
            if formed:
                self._attend_formed(out, q, cache, batch, s0, s1, r0, r1, gate)
            else:
                out[r0:r1] = self._attend_latent(q, cache, batch, gate, (s0, s1, r0, r1))
        return out

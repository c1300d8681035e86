"""Attention over a cached latent, with a sink in the softmax.

Queries come through a latent: ``c_q = rmsnorm(W_dq h) * w_dq``, ``q = W_uq c_q``, per head ``dim`` unrotated and
``rot_dim`` rotated numbers.  ``W_dkv h`` gives ``kv_rank`` numbers whose norm ``c = rmsnorm(.) * w_dkv`` is the token's
latent, and ``rot_dim`` more that are one rotated key part shared by all heads.  Per head the unrotated key is ``W_uk c``
and the value ``W_uv c``; the score of query ``t`` and key ``s <= t`` is ``(q_t . k_s + q_t^rot . k_s^rot) * scale``, the
softmax's denominator also holds ``exp(sink_head)`` (a term without key or value), and ``W_o`` follows on the heads' values.

Each of these is a field of the specification: without a query latent (``q_rank`` 0) the queries are ``W_q h``; without a rotated part
(``rot_dim`` 0) a score is ``q . k`` alone; with a window a query reads its last ``window`` keys, itself included, and pages that lie wholly
behind the window go back to the pool; with a gate head ``n``'s output is multiplied by ``sigmoid(W_g h)[n]`` (inside the attention kernel,
where the sums are divided by the softmax's denominator); with ``gate_values`` the heads' values are multiplied number by number by
``sigmoid(W_g h)`` (in the epilogue of the value up-projection).  The rotation pairs neighbours or halves, as its encoding says; without a query
latent the kernel that writes the cache row turns the queries' rotated parts as well.

Only ``c`` and the rotated key part are cached: one page plane whose rows hold ``kv_rank + rot_dim`` numbers.  The key
up-projection is taken to the query's side, ``q_t . (W_uk c_s) = (W_uk^T q_t) . c_s``, so a head's query becomes a vector
of the cache row's shape and all heads read the same rows: the attention kernel is one dot product per key and its
weighted sum runs over the latents; the value up-projection ``W_uv`` is applied to that sum.

Long portions of prompts (bfloat16, the head sizes the kernel is built for) go the other way: the cached rows that they read are brought side by side, keys
and values are projected up for all heads, and an ordinary attention runs over them.  A score then costs ``dim + rot_dim`` products instead of ``kv_rank +
rot_dim``, and a value ``vdim`` instead of ``kv_rank``; the projection costs ``kv_rank * (dim + vdim)`` for every key once, which a portion of _PROMPT_LEAST tokens or
more earns back where there is work enough.  The two ways differ in what is rounded between the products (the projected query and the mixed latent, or keys and values), not in what is
held in 32-bit: scores, softmax and sums.
"""
from __future__ import annotations

import torch

from ..config.base import ConfigError
from ..kernels import ops
from .base import KEEP_COMPUTE, KEEP_FLOAT32, KEEP_STORED, MIXERS, POSITION_ENCODINGS, Mixer, PagedNeed, WeightSpec

_MIN_KEYS_PER_SPLIT = 64        # two steps of the matrix-core kernel
_PROMPT_LEAST = 64              # tokens of a portion from which its keys and values may be projected up
# ... and the least work for which they are: (token, key) pairs times heads, a token itself counting like so many keys (its way through the two absorbed
# projections).  Measured with 32 / 16 / 8 heads, us of the whole mixer, absorbed against projected: 256 tokens after none 135 / 134, 92 / 105, 88 / 118; 512
# after none 221 / 131, 141 / 105, 112 / 116; 64 after 4000 193 / 193, 124 / 135; 128 after 4000 297 / 211, 177 / 138; 8 x 128 after none 215 / 132, 123 / 108, 117 / 117.
# Beside 31 decoded tokens, which then take kernels of their own, 256 after 2000 516 / 301, 282 / 205, 130 / 198.
_TOKEN_AS_KEYS, _UP_LEAST, _UP_LEAST_BESIDE = 256, 5 << 20, 8 << 20
# What a long context adds is not in those: every key is projected once, whatever the number of tokens that read it, and a portion's 128 tokens walk it in one work-group.
# So the absorbed way must also cost no less than the projected one up to _UP_SLACK, in the same unit (12 ps): its pairs, or the longest context over the splits that the
# step's tiles leave, 64 rows a tile; against a key's projection for a head and a key's way through the walk of the portion that reads the most, in steps of 32 keys (with
# a shared part) or 64.  Measured on the device with 32 / 16 / 8 heads, absorbed against projected: 64 tokens after 4000 188 / 197, 123 / 180, 82 / 162; after 8000 285 / 349,
# 168 / 287, 107 / 259; after 16000 477 / 649, 272 / 536, 156 / 468; 128 after 8000 490 / 361, 290 / 297, 178 / 270; 256 after 16000 1641 / 695, 876 / 562, 481 / 487; 64 after 8000 beside
# 31 decoded tokens after 2000 850 / 490, 400 / 367, 329 / 327.  The kernel that takes what the matrix cores' cannot costs 24 times as much.
_KEY_PROJECTED, _KEY_WALKED, _UP_SLACK, _GENERAL = 51, (1110, 1580), 1_700_000, 24


@MIXERS.register("latent_attention")
class LatentAttention(Mixer):
    graph_safe = True

    def __init__(self, spec, dtype, device):
        super().__init__(spec, dtype, device)
        if spec.kv_rank > ops.LATENT_MAX_RANK:
            raise ConfigError(f"latent attention is built for latents of up to {ops.LATENT_MAX_RANK} numbers, not {spec.kv_rank}")
        self.hidden, self.heads = spec.hidden, spec.heads
        self.dim, self.rot, self.vdim, self.rank, self.q_rank = spec.dim, spec.rot_dim, spec.vdim, spec.kv_rank, spec.q_rank
        self.row = spec.kv_rank + spec.rot_dim               # numbers of a cache row, and of a head's query against it
        self.scale = float(spec.scale)
        self.window = int(spec.window or 0)
        if spec.window is not None and spec.window < 1:
            raise ConfigError(f"latent attention: a window holds at least one key, got {spec.window}")
        if self.rot and spec.position is None:
            raise ConfigError("latent attention: a rotated part needs a position encoding")
        self.position = POSITION_ENCODINGS.build(spec.position, dtype, device) if spec.position is not None else None
        if self.position is not None and not hasattr(self.position, "inv_freq"):
            raise ConfigError("latent attention folds a rotation into its kernels; its position encoding must offer inv_freq")
        if self.position is not None and (not hasattr(self.position, "halves") or self.position.dims > self.rot):
            raise ConfigError(f"latent attention: the encoding {spec.position.kind!r} is not one over the first dimensions of a rotated part of {self.rot}")
        self.halves = bool(self.position.halves) if self.position is not None else False
        if spec.gate and spec.gate_values:
            raise ConfigError("latent attention: a gate is one number per head or one per value")
        if self.position is not None and getattr(self.position, "magnitude", 1.0) != 1.0:
            raise ConfigError("latent attention folds a plain rotation into its kernels; a magnitude on cosine and sine is not built there")
        # tiles of 64 rows where the matrix-core kernel is built for these sizes, of 16 for the general kernel
        on_matrix_cores = torch.device(device).type == "cuda" and ops.latent_attention_mfma_fits(dtype, self.heads, self.rank, self.rot)
        self.tile_tokens = ops.latent_tile_tokens(self.heads, ops.LATENT_MFMA_ROWS if on_matrix_cores else ops.LATENT_ATTENTION_ROWS)
        self.general_tile_tokens = ops.latent_tile_tokens(self.heads, ops.LATENT_ATTENTION_ROWS)
        self.compute_units = ops.compute_units()
        self.w_down = self.w_dq_norm = self.w_dkv_norm = self.w_uq = self.w_uk = self.w_uk_t = self.w_uv = self.sink = self.w_o = None
        # the columns of the fused first projection: [query latent, or the queries themselves | latent | rotated key part | gate], filled up with
        # zero rows of the matrix so that a token's row stays aligned
        self.q_cols = self.q_rank if self.q_rank else self.heads * (self.dim + self.rot)
        self.gate_at = self.q_cols + self.row
        self.gate_cols = self.heads if spec.gate else self.heads * self.vdim if spec.gate_values else 0
        self.down_cols = -(-(self.gate_at + self.gate_cols) // 8) * 8
        # long portions' keys and values are projected up where that attention is built for the sizes
        self.project_up = on_matrix_cores and self.rank % 64 == 0 and self.rot % 8 == 0 and self.scale > 0 and (not spec.gate_values or self.gate_at % 4 == 0) \
            and ops.prompt_rows_fits(dtype, self.dim, self.rot, self.vdim)

    def paged_need(self):
        return PagedNeed(num_heads=1, head_dim=self.row, planes=((1, self.row),), window=self.spec.window)

    def kernel_libraries(self):
        return ["latent", "experts", "local_attention"]

    def parts(self):
        yield self
        if self.position is not None:
            yield from self.position.parts()

    def weight_specs(self):
        H, n = self.hidden, self.heads
        # (the order of declaration is the order of the random-weights mode's draws)
        specs = {}
        if self.q_rank:
            specs.update({"dq": WeightSpec((self.q_rank, H)), "dq.norm": WeightSpec((self.q_rank,), keep=KEEP_STORED, init="one_plus_normal"),
                          "uq": WeightSpec((n * (self.dim + self.rot), self.q_rank))})
        else:
            specs["q"] = WeightSpec((n * (self.dim + self.rot), H))
        specs.update({
            "dkv": WeightSpec((self.row, H)), "dkv.norm": WeightSpec((self.rank,), keep=KEEP_STORED, init="one_plus_normal"),
            "uk": WeightSpec((n * self.dim, self.rank)), "uv": WeightSpec((n * self.vdim, self.rank)),
            "o": WeightSpec((H, n * self.vdim)),
        })
        if self.spec.sink:
            specs["sink"] = WeightSpec((n,), keep=KEEP_FLOAT32)
        if self.gate_cols:
            specs["g"] = WeightSpec((self.gate_cols, H))
        return specs

    def load_weights(self, tensors):
        n = self.heads
        first = [tensors["dq"] if self.q_rank else tensors["q"], tensors["dkv"]] + ([tensors["g"]] if self.gate_cols else [])
        first.append(first[0].new_zeros((self.down_cols - self.gate_at - self.gate_cols, self.hidden)))
        self.w_down = self._place(torch.cat(first, dim=0), KEEP_COMPUTE)    # one product reads h once
        self.w_dkv_norm = self._place(tensors["dkv.norm"], KEEP_STORED)
        if self.q_rank:
            self.w_dq_norm = self._place(tensors["dq.norm"], KEEP_STORED)
            self.w_uq = self._place(tensors["uq"], KEEP_COMPUTE)
        # per head the key up-projection transposed, [rank, dim]: it multiplies the unrotated query
        self.w_uk_t = self._place(tensors["uk"].view(n, self.dim, self.rank).transpose(1, 2).contiguous(), KEEP_COMPUTE)
        if self.project_up:
            self.w_uk = self._place(tensors["uk"], KEEP_COMPUTE)
        self.w_uv = self._place(tensors["uv"].view(n, self.vdim, self.rank).contiguous(), KEEP_COMPUTE)
        self.sink = self._place(tensors["sink"], KEEP_FLOAT32) if self.spec.sink else None
        self.w_o = self._place(tensors["o"], KEEP_COMPUTE)

    def _splits(self, ctx, tiles: int) -> int:
        """Work-groups that share a tile's keys: enough to give every compute unit one, no part under 64 keys."""
        groups = max(1, tiles * -(-self.heads // ops.LATENT_ATTENTION_ROWS))
        keys = ctx.max_total_len if not self.window else min(ctx.max_total_len, self.window + ctx.max_new_tokens - 1)
        return max(1, min(self.compute_units // groups, keys // _MIN_KEYS_PER_SPLIT, 64))

    def _portions(self, ctx, blocks: int = 0):
        """The step's long portions (``blocks``: the width of its block table) and the heads whose keys and values are held at once, or ``None``."""
        if not self.project_up or ctx.max_new_tokens < _PROMPT_LEAST:
            return None
        portions = ctx.long_portions(_PROMPT_LEAST, self.window)
        rows, pairs, tokens, longest = portions[4], portions[7], portions[8], portions[9]
        if (pairs + _TOKEN_AS_KEYS * tokens) * self.heads < (_UP_LEAST if portions[6] is None else _UP_LEAST_BESIDE):
            return None
        tiles = ctx.tile_count(self.tile_tokens)
        splits = self._splits(ctx, tiles)
        keys = ctx.max_total_len if not self.window else min(ctx.max_total_len, self.window + ctx.max_new_tokens - 1)
        absorbed = max(pairs * self.heads, keys // splits * 64 * min(self.compute_units, tiles * -(-self.heads // ops.LATENT_ATTENTION_ROWS) * splits)) + _TOKEN_AS_KEYS * tokens * self.heads
        if absorbed * (_GENERAL if blocks > ops.LATENT_MFMA_MAX_BLOCKS else 1) + _UP_SLACK < rows * self.heads * _KEY_PROJECTED + longest * _KEY_WALKED[self.rot > 0]:
            return None
        most = ops.PROMPT_ROWS_SCRATCH_BYTES // (rows * (self.dim + self.vdim) * 2)
        if most < 1:
            return None
        return portions, -(-self.heads // -(-self.heads // min(most, self.heads)))

    def _attend_up(self, q, values, down, plane, table, ctx, portions, at_once):
        """The long portions' rows of ``values``, from queries ``q`` whose rotated parts are turned."""
        rows, dev = portions[4], q.device
        latents = torch.empty((rows, self.rank), dtype=self.dtype, device=dev)
        keys = torch.empty(rows * (at_once * self.dim + self.rot), dtype=self.dtype, device=dev)
        up = torch.empty((at_once * self.vdim, rows), dtype=self.dtype, device=dev)
        w_uv = self.w_uv.view(self.heads * self.vdim, self.rank)
        gate = self._gates(down)
        width = self.dim + self.rot
        for a in range(0, self.heads, at_once):
            b = min(a + at_once, self.heads)
            own = rows * (b - a) * self.dim
            part = keys[: own + rows * self.rot]
            if a == 0 or b - a < at_once:      # (the rotated parts lie behind the heads' own)
                ops.latent_rows(plane, table, ctx.req_indptr, ctx.ctx_lens, portions, self.rank, self.rot, latents,
                                part[own:].view(rows, self.rot) if self.rot else None, self.window)
            ops.linear(latents, self.w_uk[a * self.dim: b * self.dim], None, part[:own].view(rows, (b - a) * self.dim))
            ops.linear(w_uv[a * self.vdim: b * self.vdim], latents, None, up[: (b - a) * self.vdim])
            ops.prompt_rows_attention(q[:, a * width: b * width], values[:, a * self.vdim: b * self.vdim], part, up[: (b - a) * self.vdim], rows, ctx.req_indptr,
                                      ctx.ctx_lens, portions, b - a, self.dim, self.rot, self.vdim, self.scale, self.sink[a:b] if self.sink is not None else None,
                                      self.window, gate[:, a:b] if self.spec.gate else None,
                                      gate[:, a * self.vdim: b * self.vdim] if self.spec.gate_values else None)

    def forward(self, h, ctx, cache):
        T, n = h.shape[0], self.heads
        dev = h.device
        inv_freq = self.position.inv_freq if self.position is not None else torch.zeros(0, dtype=torch.float32, device=dev)
        rot_dims = 2 * inv_freq.numel()
        plane = cache.planes[0]
        table = ctx.block_tables[cache.group]
        down = torch.empty((T, self.down_cols), dtype=self.dtype, device=dev)
        ops.linear(h, self.w_down, None, down)
        write = (ctx.token_req, table, plane, cache.page_size) if cache.writable else (None, None, None, 0)
        long = self._portions(ctx, table.shape[1])
        if self.q_rank:
            cq = torch.empty((T, self.q_rank), dtype=self.dtype, device=dev)
            ops.latent_prepare(down, self.q_rank, self.rank, self.rot, rot_dims, self.w_dq_norm, self.w_dkv_norm, float(self.spec.norm_eps),
                               ctx.positions, inv_freq, cq, *write, halves=self.halves)
            q = torch.empty((T, n * (self.dim + self.rot)), dtype=self.dtype, device=dev)
            ops.linear(cq, self.w_uq, None, q)
        else:                       # the queries are the first columns of the projection
            q = down[:, : self.q_cols]
        values = torch.empty((T, n * self.vdim), dtype=self.dtype, device=dev)
        # the query against a cache row: [W_uk^T q_unrotated, rotated part], head by head
        if long is None:
            qrow = torch.empty((T, n * self.row), dtype=self.dtype, device=dev)
            if not self.q_rank:
                ops.latent_prepare(down, 0, self.rank, self.rot, rot_dims, None, self.w_dkv_norm, float(self.spec.norm_eps),
                                   ctx.positions, inv_freq, None, *write, kv_off=self.q_cols, halves=self.halves,
                                   queries=(qrow, n, self.dim + self.rot, self.dim) if self.rot else None)
            elif self.rot:
                ops.rotate_pairs(q, self.dim + self.rot, self.dim, qrow, self.row, self.rank, ctx.positions, inv_freq, n, self.rot, self.halves)
            # (sequences whose block table the matrix-core kernel cannot keep in shared memory go to the general kernel and its tiles)
            general = table.shape[1] > ops.LATENT_MFMA_MAX_BLOCKS
            tq = self.general_tile_tokens if general else self.tile_tokens
            tile_req, tile_tok0, tiles = ctx.tiles(tq)
            if ctx.decode_only and tiles == T:          # one token per request: no tile list to look up
                tile_req = tile_tok0 = None
            self._attend_absorbed(q, self.dim + self.rot, qrow, self._gates(down), values, plane, table, ctx, ctx.req_indptr, tile_req, tile_tok0, tiles, tq, general,
                                  ctx.max_new_tokens)
        else:
            portions, at_once = long
            if not self.q_rank:
                ops.latent_prepare(down, 0, self.rank, self.rot, rot_dims, None, self.w_dkv_norm, float(self.spec.norm_eps),
                                   ctx.positions, inv_freq, None, *write, kv_off=self.q_cols, halves=self.halves)
            if self.rot:
                ops.rotate_pairs(q, self.dim + self.rot, self.dim, q, self.dim + self.rot, self.dim, ctx.positions, inv_freq, n, self.rot, self.halves)
            if portions[6] is not None:
                self._attend_others(q, values, down, plane, table, ctx, portions)
            self._attend_up(q, values, down, plane, table, ctx, portions, at_once)
        if self.dtype == torch.bfloat16 and ops.linear_partials_pay(T, self.hidden, n * self.vdim):
            return ops.linear_partials(values, self.w_o)      # few rows against a narrow matrix: the next norm adds the slabs up
        out = torch.empty((T, self.hidden), dtype=self.dtype, device=dev)
        ops.linear(values, self.w_o, None, out)
        return out

    def _attend_others(self, q, values, down, plane, table, ctx, portions):
        """The rows of ``values`` of the requests beside the long portions, their tokens taken out of the step, from queries whose rotated parts are turned."""
        general = table.shape[1] > ops.LATENT_MFMA_MAX_BLOCKS
        tq = self.general_tile_tokens if general else self.tile_tokens
        tile_req, tile_tok0, tiles, tokens, count, _ = ctx.tiles_by_length(tq, tq, _PROMPT_LEAST)[0]
        own = torch.empty((count, self.heads * self.dim), dtype=self.dtype, device=q.device)
        qrow = torch.empty((count, self.heads * self.row), dtype=self.dtype, device=q.device)
        gates = torch.empty((count, self.gate_cols), dtype=self.dtype, device=q.device) if self.gate_cols else None
        ops.latent_take(q, self.heads, self.dim, self.rot, tokens, own, qrow, self.rank, self._gates(down), gates)
        out = torch.empty((count, self.heads * self.vdim), dtype=self.dtype, device=q.device)
        most = 1 if count == ctx.num_requests - portions[3] else tq
        self._attend_absorbed(own, self.dim, qrow, gates, out, plane, table, ctx, portions[6], tile_req, tile_tok0, tiles, tq, general, most)
        ops.put_rows(out, tokens, values)

    def _gates(self, down):
        return down[:, self.gate_at: self.gate_at + self.gate_cols] if self.gate_cols else None

    def _attend_absorbed(self, q, q_head, qrow, gates, values, plane, table, ctx, indptr, tile_req, tile_tok0, tiles, tq, general, most_new):
        """``values`` of queries (``q_head`` numbers from one head's to the next one's) whose rotated parts lie in ``qrow`` already, against the cached rows as they are."""
        T, n = q.shape[0], self.heads
        ops.heads_linear(q, q_head, self.w_uk_t, qrow, self.row)
        mixed_latent = torch.empty((T, n * self.rank), dtype=self.dtype, device=q.device)
        ops.latent_attention(qrow, mixed_latent, plane, table, indptr, ctx.ctx_lens, tile_req, tile_tok0, tiles, tq,
                             n, self.rank, self.rot, plane.shape[2], self.scale, self.sink, self._splits(ctx, tiles),
                             general=general, max_new_tokens=most_new, window=self.window, gate=gates if self.spec.gate else None)
        ops.heads_linear(mixed_latent, self.rank, self.w_uv, values, self.vdim, gate=gates if self.spec.gate_values else None)

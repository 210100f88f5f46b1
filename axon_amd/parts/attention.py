"""Grouped-query attention over the paged cache: the mixer of this architecture.

q = Wq h + bq, k = Wk h + bk, v = Wv h + bv (bias after the product, before the rotation;
used iff the tensor exists: src/model.rs:2982-2991), rotate-half on q and k, k and v stored in
the request's pages, causal attention in which query head qh reads kv head qh // group with
scale 1/sqrt(head_dim) (src/model.rs:3373-3463), then the output projection, whose result is
added to the residual stream (src/model.rs:3031-3038).

The three projections run as one product over a fused [q_dim + 2 kv_dim, hidden] matrix
(fused when the weights are loaded; the reference fuses at launch: src/model.rs:2199-2238).

Parameters: `hidden_size`, `num_heads`, `num_kv_heads`, `head_dim`, `qkv_bias` (True, False
or "optional"), `out_bias`, `window` (0: all earlier positions), `position` (a PartSpec).
"""
from __future__ import annotations

import math
from typing import List, Optional

import torch

from ..config.base import ConfigError
from ..kernels import MODE_ADD_F32, MODE_STORE, PackedMatrix
from ..upload import upload
from .base import CacheBinding, CacheSpec, Mixer, PrecedingNorm, TensorDecl, build_part, register_mixer


# The float32 build has a kernel for tokens of any kind that needs no workspace (`attention`), with the bits of its
# prompt and decoding kernels; where the decoding kernel would want more memory than this, it is taken instead.
FLOAT32_PARTIAL = 1 << 27         # floats of the decoding kernel's partial results (512 MiB)


def float32_as_single_tokens(spans, window: int, n_heads: int, n_kv_heads: int):
    """The first tokens of the portions whose tokens the float32 decoding kernel takes one by one.  A block of the prompt
    kernel, one a head, takes 8 us for 64 positions of 128 dims whatever the number of its tokens and walks its positions in
    a row; a wave of the other, one a key head, takes one token's, side by side.  So portions of no more tokens than a group
    has heads go there (us, prompt / decoding kernel: 32 portions of 5 tokens, 28 heads over 4 31 / 14), and up to 64 tokens
    that see 256 positions or more, while tokens x key heads are few (28 over 4, 9 tokens at 4,000 positions 498 / 49, 64
    tokens at 600 86 / 49; 8 over 8, 40 at 4,000 276 / 138; 32 over 32, 16 at 600 79 / 86, 40 at 4,000 522 / 1,178)."""
    sees = lambda s: s.start_pos + s.q_len if window == 0 else min(s.start_pos + s.q_len, window + s.q_len)
    long_way = [s for s in spans if 1 < s.q_len <= 64 and sees(s) >= 256]
    few = sum(s.q_len for s in long_way) * n_kv_heads <= 256
    return {s.q_start for s in spans if 1 < s.q_len <= n_heads // n_kv_heads} | {s.q_start for s in long_way if few}


class AttentionPlan:
    """How the matrix-core kernels split a step: prompt portions (2 tokens or more) go to the
    prompt kernel in tiles of up to 128 tokens, single tokens to the decoding kernel, and the tokens
    of the portions in `as_singles` (their first tokens) too.  Made once per step and window, shared
    by all layers."""

    def __init__(self, ctx, window: int, n_heads: int, head_dim: int, as_singles=frozenset()):
        dev = ctx.rt.device
        self.tiles = None
        self.partial = None
        self.decode_work = None
        if ctx.decode_only:
            # every span is one token, in order: no index list; the engine has counted the chunks
            # and brought the list of them to the device (what a captured graph replays must not
            # come from the host)
            self.decode_tokens = ctx.n_tokens
            self.max_chunks = ctx.decode_shapes[("attention_chunks", window)]
            self.decode_work = ctx.decode_inputs[("attention_work", window)]
            n_single = ctx.n_tokens
        else:
            tiles, seen, singles, at = [], [], [], []
            tile = ctx.rt.k.attention_prefill_tile          # tokens of one request a tile of the prompt kernel holds
            for s in ctx.spans:
                if s.q_len == 1 or s.q_start in as_singles:
                    singles += range(s.q_start, s.q_start + s.q_len)
                    at += range(s.start_pos, s.start_pos + s.q_len)
                else:
                    for first in range(0, s.q_len, tile):
                        n = min(tile, s.q_len - first)
                        tiles.append((s.q_start + first, n))
                        last = s.start_pos + first + n              # positions the tile's last token sees
                        seen.append(min(last, window + n) if window > 0 else last)
            # the kernels trust these indices: check them here, on the host
            if (any(a < 0 or n < 1 or a + n > ctx.n_tokens for a, n in tiles)
                    or any(not 0 <= t < ctx.n_tokens for t in singles)):
                raise ValueError("attention plan: a span lies outside the tokens of the step")
            self.tiles = upload(pair_tiles(tiles, seen), dev) if tiles else None
            self.decode_tokens = upload(singles, dev) if singles else None
            self.max_chunks = max([1] + [decode_chunks_of(p, window, ctx.rt.k.attention_decode_chunk) for p in at])
            n_single = len(singles)
            if singles:
                work = ctx.rt.k.attention_decode_work(at, window)
                self.decode_work = upload(work, dev)
        if n_single:
            n = ctx.rt.k.attention_decode_workspace(n_single, n_heads, head_dim, self.max_chunks)
            lasting = ctx.decode_scratch.get(("attention_partial", window, n_heads, head_dim)) if ctx.decode_only else None
            if lasting is not None and lasting.numel() >= n:
                self.partial = lasting           # one workspace for every decoding step and graph
            else:
                self.partial = torch.empty(n, dtype=torch.float32, device=dev)


def pair_tiles(tiles, seen):
    """Two tiles a block, one that sees many positions with one that sees few: the tiles of a
    causal prompt see 1, 2, 3 ... blocks of positions, and blocks of equal work finish together.
    tiles: (first token, count); seen: positions each looks at.  Rows of (first, count, first,
    count), the second count 0 where a tile is left alone."""
    order = sorted(range(len(tiles)), key=lambda i: -seen[i])
    rows = []
    for k in range((len(order) + 1) // 2):
        a, b = order[k], order[len(order) - 1 - k]
        rows.append(tiles[a] + (tiles[b] if b != a else (0, 0)))
    return rows


def round_up_by_eighths(n: int) -> int:
    """n rounded up to a multiple of a power of two that is at most an eighth of it."""
    step = 1 << max(0, n.bit_length() - 4)
    return -(-n // step) * step


def decode_chunks_of(pos: int, window: int, chunk: int) -> int:
    """Chunks (of `chunk` positions, the kernel's constant) the decoding kernel cuts a token's range into."""
    lo = max(0, pos + 1 - window) if window > 0 else 0
    return (pos - lo // chunk * chunk) // chunk + 1


def attention_plan(ctx, window: int, n_heads: int, n_kv_heads: int, head_dim: int, page_size: int) -> Optional[AttentionPlan]:
    """The step's split, or None where the kernel for tokens of any kind takes them all."""
    key = ("attention_plan", window, n_heads, n_kv_heads, head_dim, page_size)
    if key not in ctx.shared:
        k = ctx.rt.k
        if k.attention_fast_ok(head_dim, page_size, n_heads, n_kv_heads):
            ctx.shared[key] = AttentionPlan(ctx, window, n_heads, head_dim)
        elif k.attention_blocks_ok(head_dim, page_size, n_heads, n_kv_heads):
            ctx.shared[key] = _float32_plan(ctx, window, n_heads, n_kv_heads, head_dim)
        else:
            ctx.shared[key] = None
    return ctx.shared[key]


def _float32_plan(ctx, window: int, n_heads: int, n_kv_heads: int, head_dim: int) -> Optional[AttentionPlan]:
    k = ctx.rt.k

    def floats(n_tokens: int, longest: int) -> int:
        chunks = decode_chunks_of(longest, window, k.attention_decode_chunk)
        return k.attention_decode_workspace(n_tokens, n_heads, head_dim, chunks)
    if ctx.decode_only:
        # a captured step is replayed at any context: what the engine's largest would want decides (see `decode_scratch`)
        most = decode_scratch_floats(k, window, n_heads, head_dim, ctx.cache.max_seqs, ctx.cache.max_seq_len)
        return AttentionPlan(ctx, window, n_heads, head_dim) if most <= FLOAT32_PARTIAL and ctx.n_tokens <= 65535 else None
    split = float32_as_single_tokens(ctx.spans, window, n_heads, n_kv_heads)
    for as_singles in (split, frozenset()):
        singles = [s for s in ctx.spans if s.q_len == 1 or s.q_start in as_singles]
        n = sum(s.q_len for s in singles)
        if n == 0 or n <= 65535 and floats(n, max(s.start_pos + s.q_len - 1 for s in singles)) <= FLOAT32_PARTIAL:
            return AttentionPlan(ctx, window, n_heads, head_dim, as_singles)
    return None


def decode_scratch_floats(k, window: int, n_heads: int, head_dim: int, max_seqs: int, max_seq_len: int) -> int:
    """The decoding kernel's partial results, laid out by the longest context in chunks rounded up to a power of two."""
    most = decode_chunks_of(max(0, max_seq_len - 1), window, k.attention_decode_chunk)
    return k.attention_decode_workspace(max_seqs, n_heads, head_dim, 1 << (most - 1).bit_length())


class GQAttention(Mixer):
    graph_safe = True
    def __init__(self, params, prefix=""):
        super().__init__(params, prefix)
        p = params
        self.hidden = int(p["hidden_size"])
        self.nh = int(p["num_heads"])
        self.nkv = int(p["num_kv_heads"])
        self.hd = int(p["head_dim"])
        self.window = int(p.get("window", 0))
        self.qkv_bias = p.get("qkv_bias", False)
        self.out_bias = bool(p.get("out_bias", False))
        if self.nh % self.nkv:
            raise ConfigError(f"{self.nh} query heads are not a multiple of {self.nkv} kv heads")
        if self.hd % 16 or not 16 <= self.hd <= 256:
            raise ConfigError(f"head_dim {self.hd} is not a multiple of 16 between 16 and 256: no kernel takes it")
        self.q_dim, self.kv_dim = self.nh * self.hd, self.nkv * self.hd
        self.scale = 1.0 / math.sqrt(self.hd)
        self.position = build_part("position", p["position"]) if p.get("position") is not None else None
        names = p.get("names", {})
        base = prefix + names.get("scope", "self_attn.")
        self.n = {k: base + names.get(k, k + "_proj") for k in ("q", "k", "v", "o")}
        self.w_qkv = self.b_qkv = self.w_o = self.b_o = None
        self._max_context = None
        self._kernels = None                 # those that want a workspace in decoding steps
        self.decode_chunk = 1 << 30          # until `load` has asked the kernels: one chunk
        self._work_list = lambda positions, window: list(range(len(positions)))

    # ------------------------------------------------------------------ declarations
    def tensors(self) -> List[TensorDecl]:
        t = [TensorDecl(self.n["q"] + ".weight", (self.q_dim, self.hidden)),
             TensorDecl(self.n["k"] + ".weight", (self.kv_dim, self.hidden)),
             TensorDecl(self.n["v"] + ".weight", (self.kv_dim, self.hidden)),
             TensorDecl(self.n["o"] + ".weight", (self.hidden, self.q_dim))]
        if self.qkv_bias:
            opt = self.qkv_bias == "optional"
            t += [TensorDecl(self.n["q"] + ".bias", (self.q_dim,), "bias", opt),
                  TensorDecl(self.n["k"] + ".bias", (self.kv_dim,), "bias", opt),
                  TensorDecl(self.n["v"] + ".bias", (self.kv_dim,), "bias", opt)]
        if self.out_bias:
            t.append(TensorDecl(self.n["o"] + ".bias", (self.hidden,), "bias"))
        return t

    def cache_spec(self) -> Optional[CacheSpec]:
        return CacheSpec(entries=2, heads=self.nkv, head_dim=self.hd, window=self.window)

    def max_context(self):
        return self._max_context

    def decode_shape(self, positions):
        """The decoding kernel's workspace is laid out by the longest context of the step, in
        chunks of the kernel's size, rounded up to a power of two so that few shapes exist (the
        blocks that are launched are those of `decode_input`, whatever this number)."""
        most = max(decode_chunks_of(p, self.window, self.decode_chunk) for p in positions)
        return ("attention_chunks", self.window), 1 << (most - 1).bit_length()

    def decode_input(self, positions):
        """The list of the chunks the decoding kernel computes, a block each: blocks are launched
        for the chunks that exist, not for the longest context times the tokens.  Padded in
        steps of an eighth or less."""
        work = self._work_list(positions, self.window)
        return ("attention_work", self.window), work + [-1] * (round_up_by_eighths(len(work)) - len(work))

    def decode_input_capacity(self, max_seqs: int, max_seq_len: int) -> int:
        return round_up_by_eighths(max_seqs * decode_chunks_of(max(0, max_seq_len - 1), 0, self.decode_chunk))

    def decode_scratch(self, max_seqs: int, max_seq_len: int):
        """The blocks' partial results of the decoding kernel (see `decode_shape`)."""
        if self._kernels is None:                # no kernel of this build and these sizes wants one
            return None
        floats = decode_scratch_floats(self._kernels, self.window, self.nh, self.hd, max_seqs, max_seq_len)
        if floats > FLOAT32_PARTIAL and not self._kernels.attention_fast_ok(self.hd, 64, self.nh, self.nkv):
            return None
        return ("attention_partial", self.window, self.nh, self.hd), floats

    def load(self, store, rt) -> None:
        self.decode_chunk = rt.k.attention_decode_chunk
        self._work_list = rt.k.attention_decode_work
        self._max_context = rt.k.attention_decode_max_context
        if rt.k.attention_blocks_ok(self.hd, 64, self.nh, self.nkv):
            self._kernels = rt.k
        self.w_qkv = rt.k.prepare_weight(store.fused_matrix([self.n[k] + ".weight" for k in ("q", "k", "v")]))
        biases = [store.vector(self.n[k] + ".bias", optional=True) for k in ("q", "k", "v")] if self.qkv_bias else []
        present = [b is not None for b in biases]
        if any(present):
            if not all(present):
                raise ConfigError(f"{self.prefix}: q, k and v biases must all be present or all absent")
            dt = torch.float32 if any(b.dtype == torch.float32 for b in biases) else biases[0].dtype
            self.b_qkv = torch.cat([b.to(dt) for b in biases]).contiguous()
        self.w_o = rt.k.prepare_weight(store.matrix(self.n["o"] + ".weight"))
        store.forget(self.n["o"] + ".weight")
        self.b_o = store.vector(self.n["o"] + ".bias") if self.out_bias else None
        if self.position is not None:
            self.position.load(store, rt)

    # ------------------------------------------------------------------ the step
    def finishes_following_norm(self, ctx) -> bool:
        return isinstance(self.w_o, PackedMatrix) and ctx.rt.k.gemm_then_norm_ok(ctx.n_tokens, self.hidden, self.q_dim)

    def applies_preceding_norm(self, ctx) -> bool:
        k = ctx.rt.k
        rows = self.q_dim + 2 * self.kv_dim
        return (isinstance(self.w_qkv, PackedMatrix) and self.position is not None
                and k.gemm_qkv_rope_ok(ctx.n_tokens, rows, self.hidden, self.hd, self.position.rotary_dim)
                and k.gemm_normed_ok(ctx.n_tokens, rows, self.hidden))

    def forward(self, ctx, binding: CacheBinding, h, residual, following=None) -> None:
        k = ctx.rt.k
        T = h.shape[0]
        group = ctx.cache.group(binding.group)
        k_cache, v_cache = group.layer(binding.index)
        # values are kept position-contiguous: a page of them is [heads, head_dim, page_size]
        v_cache = v_cache.view(v_cache.shape[0], self.nkv, self.hd, group.page_size)
        qkv = ctx.ws.take((T, self.q_dim + 2 * self.kv_dim), ctx.rt.dtype)
        if self.position is not None:
            table, rotary = self.position.tables(ctx), self.position.rotary_dim
        else:
            table, rotary = ctx.no_rotation(), 0
        if binding.writes:
            w, bias = self.w_qkv, self.b_qkv
        else:
            # reading another run's cache: only the queries are needed
            w, bias = self.w_qkv[:self.q_dim], None if self.b_qkv is None else self.b_qkv[:self.q_dim]
        in_one = isinstance(w, PackedMatrix) and k.gemm_qkv_rope_ok(T, w.shape[0], self.hidden, self.hd, rotary)
        cache = (group.block_table, k_cache, v_cache, self.nh, self.nkv, self.hd)
        if isinstance(h, PrecedingNorm) and not (in_one and k.gemm_normed_ok(T, w.shape[0], self.hidden, gain=h.gain)):
            h = h.apply(ctx)
        if isinstance(h, PrecedingNorm):
            # few rows: the norm, the product, the rotation and the store into the pages in one launch
            k.gemm_normed_qkv_rope(h.rows, h.gain, h.eps, w, bias, qkv, table, ctx.positions, ctx.seq_rows, *cache,
                                   group.page_size, binding.writes)
        elif in_one:
            # product, rotation and the store into the pages in one launch (a short step) or with the
            # rotation and the store done by the kernel that adds the sums of the product's segments
            k.gemm_qkv_rope(h, w, bias, qkv, table, ctx.positions, ctx.seq_rows, *cache, group.page_size, binding.writes)
        else:
            k.gemm(h, w, qkv[:, :w.shape[0]], bias, MODE_STORE)
            k.rope_kv_write(qkv, table, ctx.positions, ctx.seq_rows, *cache, rotary, group.page_size, binding.writes)
        att = ctx.ws.take((T, self.q_dim), ctx.rt.dtype)
        plan = attention_plan(ctx, self.window, self.nh, self.nkv, self.hd, group.page_size)
        if plan is not None:
            common = (k_cache, v_cache, group.block_table, ctx.positions, ctx.seq_rows, att)
            sizes = (self.nh, self.nkv, self.hd, group.page_size, self.window, self.scale)
            if plan.tiles is not None:
                k.attention_prefill(qkv, qkv.stride(0), *common, plan.tiles, *sizes)
            if plan.decode_tokens is not None:
                k.attention_decode(qkv, qkv.stride(0), *common, plan.decode_tokens, plan.partial, plan.max_chunks, *sizes,
                                   work=plan.decode_work)
        else:
            k.attention(qkv, qkv.stride(0), k_cache, v_cache, group.block_table, ctx.positions, ctx.seq_rows, att,
                        self.nh, self.nkv, self.hd, group.page_size, self.window, self.scale)
        k.gemm(att, self.w_o, residual, self.b_o, MODE_ADD_F32,
               following_norm=None if following is None else following.as_argument())


register_mixer("gqa_attention", GQAttention)

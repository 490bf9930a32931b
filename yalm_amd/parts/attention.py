"""Grouped-query self-attention over the cache, with a position encoding that
it owns and an optional window.

Per token (src/infer.cpp:278-338): q, k, v = W h; q and k rotated at the token's
position; k and v stored in the cache; per query head h with KV head h // group:
scores q.k / sqrt(head_dim) over the visible keys, softmax in float32, mix of
the values; the output projection is added to the residual stream.  Key j is
visible to the query at position i iff j <= i and (window == 0 or i - j <
window or j < sinks) (the reference's kv_len rows, src/infer.cpp:486-488).

Sinks (src/infer.cpp:305-319: with a context of n the reference keeps positions
0 and 1 and the last n - 2, and turns the kept keys one position further every
step past n): a sink j that the window no longer covers is scored as if it lay
window + sinks - 1 - j positions behind the query, whatever the query's
position.  Its key is stored as it was rotated at j and turned by
i - (window + sinks - 1) when it is read.

The three projections are one matrix [q; k; v] (the reference fuses them by
pointer, src/infer.cu:290-337); q/k rows are re-ordered at load if the folder
keeps them half-split (convert.py:145-158)."""
import math

import torch

from ..cache.manager import KVRequest
from ..ops import kernels
from ..weights.loader import ParamSpec, place
from .base import Part, build_part, part

# decode attention is split over pages so that about this many workgroups run
TARGET_WORKGROUPS = 256
RESIDENT_WORKGROUPS = 512       # decode-attention workgroups that the chip holds at once (two a compute unit)
# A prompt step of fewer tokens rotates and stores token by token: the kernel that works a page-shaped tile at a
# time has a workgroup per (tile, head), too few to fill the chip below this
ROPE_TILES_MIN_TOKENS = 320


def rope_by_tiles(T, n_heads, n_kv_heads, head_dim, slices):
    """Whether a step of whole prompts of T tokens rotates and stores by tiles of 64 positions.  With heads of 128 and more that takes the same
    time for few tokens as for some hundreds (12 us, two slices of K 15, four 16 to 25, heads of 256 20 and more), while token by token goes with the
    heads, a key and value head (whose values are stored turned) like ten of queries.  The two meet where tokens times such heads reach
    what is asked for here.  us token by token and by tiles:
      heads of 128, one slice    32 + 8: 360 tokens 11.7 11.9, 400 12.7 12.4   32 + 16: 320 15.7 11.3   48 + 8: 320 11.8 12.4, 360 13.0 12.2
                                 32 + 4: 576 12.0 12.4, 640 13.0 12.4   8 + 8: 448 11.3 11.7, 512 12.5 11.8   8 + 2: 1,024 9.4 11.7, 1,500 11.9 11.9
        two slices               32 + 8: 512 15.6 16.4, 640 20.8 20.1   32 + 16: 320 15.9 15.5   16 + 8: 576 14.9 15.5, 640 16.0 15.5
        four and eight slices    32 + 8: 448 23.1 24.2, 512 26.5 24.9   eight 512 35.2 39.1, 640 43.2 41.9   64 + 8: 320 24.1 24.8, 360 27.5 25.1
      heads of 144, one slice    32 + 8: 384 12.9 13.0   24 + 8: 448 14.1 13.2   two 32 + 8: 448 16.2 18.1   four 320 25.3 25.1, 384 30.6 26.3
      heads of 256, one slice    32 + 8: 448 19.0 21.2, 576 23.2 21.7   four 400 46.5 43.7   16 + 4: 768 17.1 20.8, 1,500 49.0 31.7
    Heads below 128 go by tiles from 320 tokens on (64: 512 tokens 11.6 7.6, two slices 11.7 9.0)."""
    if T < ROPE_TILES_MIN_TOKENS or head_dim < 128:
        return T >= ROPE_TILES_MIN_TOKENS
    if head_dim == 128:
        meet = 43000 if slices == 1 else 60000 if slices == 2 else 50000
    else:                 # for the narrowest of these: wider ones meet later
        meet = 43000 if slices <= 2 else 32000
    return T * (n_heads + 10 * n_kv_heads) >= meet


def one_tile_pays(n_seqs, longest, n_heads, n_kv_heads, head_dim, slices):
    """Whether a step of prompts of one tile each, the longest of `longest` tokens, is sooner done by kernels.attn_tile than by the rotation and
    the attention behind each other.  A workgroup takes in all slices of its rows, 98 KB for 64 tokens of heads of 128, at what a compute unit takes in
    (1 us), which the two launches spread over the chip; the launch less is worth 2 to 4 us inside a step, and 19 where the host is what
    the step waits for.  us a layer that the one launch takes more inside steps of eight layers:
      heads of 128, 32 + 8 at K 4,096: 64 tokens of 5 slices -2.1; 24 + 8 at K 8,192: 64 of 6 -1.8; 16 + 8 at 8,192: 48 of 8 -2.3, 64 of 8 0.3
                   8 + 2 at 8,192: 48 of 16 -5.4, 64 of 16 3.3; 16 + 4 at 12,288: 33 of 10 -2.3, 48 of 10 -0.6, 64 of 10 2.1
      heads of 64, 32 + 8 at 8,192: 64 of 10 -4.4; 8 + 2 at 8,192: 64 of 16 -12
    Every head of a group takes in the group's keys and values, with more than six heads most of the work once the chip is full.  us, the two launches and
    the one, back to back without a step around them:
      heads of 128, 64 + 8: 16 x 64 38.4 32.1, two slices 46.2 45.8; 24 x 64 48.3 46.2, 59.5 66.7; 64 x 64 108 117, 142 166
                   32 + 2:  32 x 64 35.6 27.9; 128 x 64 99.6 102, 130 141; 200 x 20 88.9 97.5   48 + 8: 256 x 64 325 288, two slices 426 413
      heads of 64, 64 + 8: 256 x 64 228 172, two slices 299 256"""
    if head_dim >= 128 and n_heads > 6 * n_kv_heads and n_heads * n_seqs * slices > 2560:
        return False
    return slices * longest * head_dim <= 480 * 128


def kv_tiles(n_tok):
    """The index tables a step of whole prompts needs for attention over its own keys and values, which are
    staged in page-shaped tiles of 64 positions: seq_tile0[B + 1], the first tile of each sequence (n_tiles in
    all), and tile_order, the order in which the attention kernel should take the tiles of queries."""
    import numpy as np
    tile0 = np.zeros(len(n_tok) + 1, dtype=np.int32)
    np.cumsum([(n + kernels.PAGE - 1) // kernels.PAGE for n in n_tok], out=tile0[1:])
    return {"seq_tile0": tile0, "tile_order": np.asarray(kernels.prefill_tile_order(n_tok), dtype=np.int32),
            "n_tiles": int(tile0[-1])}


kv_tiles.name = "kv_tiles"


def decode_splits(n_heads, n_kv_heads, head_dim, B, max_pages, ragged=False, shaped=False, own=False):
    """Into how many pieces a decode step's attention cuts every sequence, so that about TARGET_WORKGROUPS
    workgroups run.  shaped: the scores have a shape (a bias, a cap, ...), which the wide heads' kernels do not take.
    own: float32, whose kernel cuts every sequence by its own length: four pages and more a piece, whoever stands beside it.
    us below: bfloat16, 32 heads of 128 in 8 groups, all caches cold."""
    mfma = (head_dim in kernels.MFMA_HEAD_DIMS or (head_dim in kernels.MFMA_WIDE_HEAD_DIMS and not shaped)) \
        and not kernels.FORCE_SIMPLE
    if mfma:         # a workgroup of 4 waves per (split, KV head and up to 16 of its query heads, sequence), a page per wave at a time
        per = max(1, B * n_kv_heads * ((n_heads // n_kv_heads + 15) // 16))
        quarters = max(1, min((max_pages + 3) // 4, 4))
        # More workgroups than run at once: in quarters the last round is short, which pays while it is nearly empty; from half
        # a round on a split more is only another merge (96 rows of 1,000 tokens 70.2 in one, 82.1 in four; 80 of 3,000 158 and 169;
        # 128 of 300 31.4, in two 43.2; of 200 to 1,000 tokens 96 rows 48.0 and 65.9).  Of sequences of very unequal lengths the longest is then
        # one workgroup's alone, its pages one behind the other while the others are long done: up to 64 pages it ends in time (96 rows of 200 to
        # 3,200 tokens 119.6, in quarters 133.3; one of 2,500 and 95 of 100 to 600 41.4 and 46.9, one of 3,200 the same, one of 4,000 53.4
        # and 47.2, eight of 4,000 59.9 and 62.4), beyond that not (one of 8,000 90.0 and 50.5, of 24,000 237.8 and 84.2, eight of 6,000 81.8 and 73.3).
        if per > RESIDENT_WORKGROUPS:
            return quarters if own or 2 * per < 3 * RESIDENT_WORKGROUPS or (ragged and max_pages > 64) else 1
        if own or per > 64 or max_pages <= 4:
            even = max(1, min((max_pages + 3) // 4, TARGET_WORKGROUPS // per))
        else:
            # Few rows: a wave's pages come one behind the other, 2.3 us each, and a split more costs the merge 0.15 us, which is
            # least at the root of 3.8 pages; three pages of eight a split at the least (one row of 500 tokens in two splits 8.5, in three 7.5,
            # of 1,000 in four 8.4, in six 7.5; three rows of 1,000 9.4 and 8.2; eight of 500 in two 9.2, in three 8.8).
            # Beyond twelve the nearest multiple of eight, which deals a bucket's pages evenly to the waves (64 pages in 15 splits are 2 % slower than in 16, to
            # 17 %, over 72 steps of eight shapes of heads; 128 in 22 3 % than in 24, 256 in 31 3 % than in 32).
            # A workgroup on three quarters of the units reads as fast as one on each (one row of 28,000: 24 splits 23.6, 32 24.9).
            # One group for all heads is cut by the same rule (16 heads of 144, one row of 28,000 tokens in 40 22.9, in 110 and more 33.8).
            most = TARGET_WORKGROUPS // per if per > 8 else TARGET_WORKGROUPS * 3 // 4 // per
            root = math.isqrt(19 * max_pages // 5)
            even = max(1, min((3 * max_pages + 7) // 8, root if root <= 12 else (root + 3) // 8 * 8, most))
        # Sequences of very unequal lengths.  Where the workgroups stand two to a compute unit anyway, one split and
        # the rows in the order that pairs a long sequence with a short one; else splits of the longest sequence's
        # split size (the kernel cuts them so), enough of them that the long sequences' work spreads over the chip.  With a workgroup on more than
        # half of the units and up to 16 pages the longest one's rounds are few, and one split is sooner (32 rows of 200 to 1,000
        # tokens 19.1 in one, 25.7 in four; 17 of them 15.1 and 22.1; of 800 to 4,000 tokens 61 and 67 to 71, 17 of them 46 and 42).
        if ragged and per <= TARGET_WORKGROUPS and (own or 2 * per <= TARGET_WORKGROUPS or max_pages > 16):
            return max(even, quarters)
        return even
    return max(1, min(max_pages, TARGET_WORKGROUPS // max(1, B * n_heads)))


def decode_order(ctx, B, n_heads, n_kv_heads, n_splits, own=False):
    """The order in which a decode step's attention takes the rows, or None.  It pairs a long sequence's workgroup with a short one's, which
    holds where a row has one workgroup a KV head, or the workgroups of all its splits are few; with several splits of many rows the
    plain order spreads them better (24 rows of 50 to 4,000 tokens in four splits 49.5 us in this order, 44.9 in the plain one; 9 rows 21.1 and 29.0)."""
    per = B * n_kv_heads * ((n_heads // n_kv_heads + 15) // 16)
    return ctx.seq_order if own or n_splits == 1 or 2 * per <= TARGET_WORKGROUPS or per > RESIDENT_WORKGROUPS else None


def decode_counters(ctx, B, n_heads, n_kv_heads, n_splits):
    """What lets the attention kernel of a decode step merge its splits itself (None: there is nothing to merge)."""
    if n_splits == 1:
        return None
    return ctx.ws.get_zeroed("attn.counters", (kernels.attn_decode_counters(B, n_heads, n_kv_heads),), torch.int32)


@part("mixer", "gqa_attention")
class GQAttention(Part):
    prompt_tables = (kv_tiles,)

    def __init__(self, spec, dim, prefix):
        super().__init__(spec, dim, prefix)
        p = spec.params
        self.n_heads = int(p["n_heads"])
        self.n_kv_heads = int(p["n_kv_heads"])
        self.head_dim = int(p["head_dim"])
        self.window = int(p.get("window", 0) or 0)
        self.sinks = int(p.get("sinks", 0) or 0)
        if self.sinks and self.window < self.sinks:
            raise ValueError("%d attention sinks need a window at least as wide (window %d)" % (self.sinks, self.window))
        if not 0 <= self.sinks <= kernels.MAX_SINKS:
            raise ValueError("%d attention sinks asked for, at most %d are supported" % (self.sinks, kernels.MAX_SINKS))
        if self.n_heads % self.n_kv_heads:
            raise ValueError("n_heads %d is no multiple of n_kv_heads %d" % (self.n_heads, self.n_kv_heads))
        if self.head_dim % 2 or self.head_dim > kernels.MAX_HEAD_DIM:
            raise ValueError("head_dim %d is not supported (even, at most %d)" % (self.head_dim, kernels.MAX_HEAD_DIM))
        self.takes_prepared_prompts = self.head_dim % 16 == 0
        self.q_dim = self.n_heads * self.head_dim
        self.kv_dim = self.n_kv_heads * self.head_dim
        self.position = build_part("position", p["position"], dim, prefix)
        self.wqkv = None
        self.wo = None

    def children(self):
        return [self.position]

    @property
    def score_bias(self):
        """The position part's term for every score by the distance of query and key (float32 [n_heads, distances]
        on the device), if it has one: a position encoding that is no rotation."""
        bias = getattr(self.position, "score_bias", None)
        if bias is not None and self.sinks:
            raise ValueError("attention sinks are scored without a score bias: the two do not go together")
        return bias

    def param_specs(self):
        D = self.dim
        return [ParamSpec(self.prefix + "q_proj.weight", (self.q_dim, D), fan_in=D),
                ParamSpec(self.prefix + "k_proj.weight", (self.kv_dim, D), fan_in=D),
                ParamSpec(self.prefix + "v_proj.weight", (self.kv_dim, D), fan_in=D),
                ParamSpec(self.prefix + "o_proj.weight", (D, self.q_dim), fan_in=self.q_dim)]

    def load(self, get, compute_dtype, device):
        wq = self.position.arrange_projection_rows(get(self.prefix + "q_proj.weight"), self.n_heads)
        wk = self.position.arrange_projection_rows(get(self.prefix + "k_proj.weight"), self.n_kv_heads)
        wv = get(self.prefix + "v_proj.weight")
        self.wqkv = place(torch.cat([wq, wk, wv], dim=0), compute_dtype, device)
        self.wo = place(get(self.prefix + "o_proj.weight"), compute_dtype, device)

    def weight_bytes(self):
        return (self.wqkv.numel() + self.wo.numel()) * self.wqkv.element_size()

    def cache_request(self):
        return KVRequest(self.n_kv_heads, self.head_dim, self.window, self.sinks)

    def row_elements(self):
        """The widest buffer a token has in this part: q, k and v side by side."""
        return self.q_dim + 2 * self.kv_dim

    def describe(self, compute_dtype):
        what = "attention, %d heads in %d groups of head size %d%s" % (
            self.n_heads, self.n_kv_heads, self.head_dim,
            (", window %d" % self.window if self.window else "") + (" + %d sinks" % self.sinks if self.sinks else ""))
        if compute_dtype != torch.bfloat16:
            return what + ": float32-arithmetic kernels", False
        if self.head_dim in kernels.MFMA_HEAD_DIMS or (self.head_dim in kernels.MFMA_WIDE_HEAD_DIMS
                                                       and not hasattr(self.position, "score_bias")):
            return what + ": matrix-core kernels", False
        return what + ": float32-arithmetic kernels on bfloat16 storage (the matrix-core kernels take head sizes " \
                      "of 16 to 256 in steps of 16, to 128 with a score bias, not %d): correct, many times slower" % self.head_dim, True

    def decode_splits(self, B, max_pages, ragged=False):
        return decode_splits(self.n_heads, self.n_kv_heads, self.head_dim, B, max_pages, ragged, shaped=hasattr(self.position, "score_bias"),
                             own=self.wo is not None and self.wo.dtype == torch.float32)

    def fuses_norm(self, norm, x, ctx):
        if not hasattr(norm, "fused") or self.head_dim % 16:
            return False
        T = x.shape[0]
        if ctx.mode == "prefill":             # takes the norm where the product before has left or prepared it
            return kernels.can_add_norm(T, self.dim, self.wo.dtype) or kernels.can_chain(T, self.dim, self.wo.dtype)
        if ctx.mode != "decode":
            return False
        if self.wo.dtype == torch.float32:
            return kernels.fuse_norm_pays(T, self.dim, torch.float32, self.q_dim + 2 * self.kv_dim, qkv=True)
        return kernels.can_chain(T, self.dim, self.wo.dtype) or kernels.can_add_norm(T, self.dim, self.wo.dtype)

    def forward_prenorm(self, x, norm, ctx, line, writes_cache=True, emit_for=None):
        """A decode step from the residual stream: norm, q/k/v, rotation and cache write in
        one kernel, attention over the cache, output projection added to x (which may
        prepare the activations of the next norm, emit_for)."""
        if ctx.mode == "prefill":                 # whole prompts: the norm, unless its output is ready or prepared, then the plain way
            src = ctx.normed.pop(id(norm), None)
            if src is not None and src[1] is None:
                h = src[0]
            elif src is not None and kernels.can_chain(x.shape[0], self.dim, self.wo.dtype):
                return self.forward(src[0], x, ctx, line, writes_cache, emit_for=emit_for, scale_from=src[1:])
            else:
                h = ctx.ws.get("block.h", (x.shape[0], self.dim), ctx.act_dtype)
                norm.forward(x, h, ctx)
            return self.forward(h, x, ctx, line, writes_cache, emit_for=emit_for)
        if not writes_cache:                      # a reader of another entry's line: the plain way
            ctx.normed.pop(id(norm), None)
            h = ctx.ws.get("block.h", (x.shape[0], self.dim), ctx.act_dtype)
            norm.forward(x, h, ctx)
            return self.forward(h, x, ctx, line, writes_cache)
        T = x.shape[0]
        pos = self.position
        if pos.table is not None and ctx.max_position >= pos.n_positions:
            raise ValueError("position %d is beyond the %d positions the rotation table holds"
                             % (ctx.max_position, pos.n_positions))
        group = ctx.cache.group_of(line)
        k_pages, v_pages = group.line_pages(line)
        q = ctx.ws.get("attn.q", (T, self.q_dim), self.wo.dtype)
        src = ctx.normed.pop(id(norm), None)
        if src is not None and src[1] is not None and kernels.can_chain(T, self.dim, self.wo.dtype):
            xn, ss, eps = src
            kernels.gemm_chain_qkv_rope(xn, (ss, eps), self.wqkv, q, k_pages, v_pages, group.table, group.ring_pages,
                                        ctx.tok_pos, ctx.seq_slot, pos.table, self.n_heads, self.n_kv_heads,
                                        self.head_dim, pos.rotary_dim)
        elif src is None and kernels.fuse_norm_pays(T, self.dim, self.wo.dtype, self.q_dim + 2 * self.kv_dim, qkv=True):
            nw, eps = norm.fused()
            kernels.gemm_norm_qkv_rope(x, nw, eps, self.wqkv, q, k_pages, v_pages, group.table, group.ring_pages,
                                       ctx.tok_pos, ctx.seq_slot, pos.table, self.n_heads, self.n_kv_heads,
                                       self.head_dim, pos.rotary_dim)
        else:             # the norm's output is ready or prepared, or the rows are too many for one kernel
            scale = None
            if src is not None and src[1] is not None:        # prepared: the product's sums are scaled row by row
                h, scale = src[0], (src[1], src[2])
            elif src is not None:
                h = src[0]
            else:
                h = ctx.ws.get("block.h", (T, self.dim), ctx.act_dtype)
                norm.forward(x, h, ctx)
            n_qkv = self.q_dim + 2 * self.kv_dim
            if kernels.can_gemm_partial(T, self.dim, h.dtype):
                # the GEMM's K slices go to the rotation kernel as they are, which adds them: no kernel in between
                qkv = ctx.ws.get("gemm.partial", (kernels.fused_workspace_floats(T, n_qkv, self.dim),), torch.float32)
                slices = kernels.gemm_partial(h, self.wqkv, qkv, scale_from=scale)
            else:
                qkv = ctx.ws.get("attn.qkv", (T, n_qkv), torch.float32)
                self._gemm(ctx, h, self.wqkv, qkv, kernels.EPI_STORE_F32, scale_from=scale)
                slices = 1
            kernels.rope_kv_write(qkv, q, None, None, None, k_pages, v_pages, group.table, group.ring_pages,
                                  ctx.tok_seq, ctx.tok_pos, ctx.seq_slot, ctx.seq_len, pos.table, self.n_heads,
                                  self.n_kv_heads, self.head_dim, pos.rotary_dim, slices=slices)
        o = ctx.ws.get("attn.o", (T, self.q_dim), self.wo.dtype)
        self._decode_attention(q, o, ctx, group, line, k_pages, v_pages, True)
        emit = self._emit_args(emit_for, ctx, x)
        prepared = self._add_emit_args(emit_for, ctx, T, self.dim, self.q_dim) if emit is None else None
        ready = self._add_norm_args(emit_for, ctx, T, self.dim, self.q_dim) if emit is None and prepared is None else None
        if emit is not None and kernels.can_chain(T, self.q_dim, o.dtype):
            nw2, xn2, ss2, eps2 = emit
            kernels.gemm_chain(o, self.wo, x, kernels.EPI_ADD_F32, emit=(nw2, xn2, ss2))
            ctx.normed[id(emit_for)] = (xn2, ss2, eps2)
        elif prepared is not None:                # 17..128 rows: the K slices are added and the next norm prepared at once
            nw2, eps2, xn2, ss2, ws2 = prepared
            kernels.gemm_add_emit(o, self.wo, x, nw2, xn2, ss2, ws2)
            ctx.normed[id(emit_for)] = (xn2, ss2, eps2)
        elif ready is not None and kernels.can_add_norm(T, self.q_dim, o.dtype):
            nw2, eps2, h2, ws2 = ready
            kernels.gemm_add_norm(o, self.wo, x, nw2, eps2, h2, ws2)
            ctx.normed[id(emit_for)] = (h2, None, None)
        else:
            self._gemm(ctx, o, self.wo, x, kernels.EPI_ADD_F32)

    def _decode_attention(self, q, o, ctx, group, line, k_pages, v_pages, writes_cache):
        T = q.shape[0]
        n_splits = self.decode_splits(T, min(group.ring_pages, ctx.pages_bucket), ctx.ragged)
        partial = ctx.ws.get("attn.partial",
                             (kernels.attn_decode_workspace_floats(T, self.n_heads, self.head_dim, n_splits),),
                             torch.float32)
        sinks = None
        if self.sinks:       # taken in where the splits are merged; a sequence still at its first positions
            sink_k, sink_v = group.line_sinks(line)        # has just written a sink, which is stored on the way
            sinks = (sink_k, sink_v, self.position.table, self.position.rotary_dim, writes_cache)
        kernels.attn_decode(q, k_pages, v_pages, group.table, group.ring_pages, ctx.seq_slot, ctx.seq_len, o, partial,
                            self.n_heads, self.n_kv_heads, self.head_dim, self.window, n_splits, sinks=sinks,
                            step_max_len=ctx.step_max_len, seq_order=decode_order(ctx, T, self.n_heads, self.n_kv_heads, n_splits, q.dtype == torch.float32),
                            score_bias=self.score_bias,
                            counters=decode_counters(ctx, T, self.n_heads, self.n_kv_heads, n_splits))

    def forward(self, h, x, ctx, line, writes_cache=True, emit_for=None, scale_from=None):
        """scale_from: h is a norm that is prepared and not finished (a step of at most CHAIN_MAX_ROWS tokens); the product's
        sums are scaled row by row."""
        T = h.shape[0]
        act = h.dtype
        ws = ctx.ws
        pos = self.position
        if pos.table is not None and ctx.max_position >= pos.n_positions:
            raise ValueError("position %d is beyond the %d positions the rotation table holds"
                             % (ctx.max_position, pos.n_positions))
        prefill = ctx.mode == "prefill"
        n_qkv = self.q_dim + 2 * self.kv_dim
        slices = 1
        if prefill and kernels.can_gemm_partial(T, self.dim, act):
            # the product's K slices (a short prompt's has some) go to the rotation kernel as they are, which adds them
            qkv = ws.get("gemm.partial", (kernels.fused_workspace_floats(T, n_qkv, self.dim),), torch.float32)
            slices = kernels.gemm_partial(h, self.wqkv, qkv)
        else:
            qkv = ws.get("attn.qkv", (T, n_qkv), torch.float32)
            if scale_from is not None:
                kernels.gemm_chain(h, self.wqkv, qkv, kernels.EPI_STORE_F32, scale_from=scale_from)
            else:
                self._gemm(ctx, h, self.wqkv, qkv, kernels.EPI_STORE_F32)
        group = ctx.cache.group_of(line)
        k_pages, v_pages = group.line_pages(line)
        o = ws.get("attn.o", (T, self.q_dim), act)
        # short prompts, every sequence one tile of keys that nobody reads again in this step: rotation, cache write and attention
        # are one kernel
        n_seqs, n_tiles = ctx.seq_slot.shape[0], ctx.tables["kv_tiles"]["n_tiles"] if prefill else 0
        if prefill and writes_cache and n_tiles == n_seqs and not self.sinks and self.score_bias is None and not ctx.line_is_shared(line) \
                and kernels.attn_tile_fits(qkv, o, k_pages, v_pages, self.head_dim, self.window, n_seqs) \
                and one_tile_pays(n_seqs, ctx.max_position + 1, self.n_heads, self.n_kv_heads, self.head_dim, slices):
            kernels.attn_tile(qkv, o, k_pages, v_pages, group.table, group.ring_pages, ctx.cu_seqlens, ctx.seq_slot, pos.table,
                              self.n_heads, self.n_kv_heads, self.head_dim, pos.rotary_dim, slices=slices, n_tiles=n_tiles)
        else:
            self._rotate_and_attend(qkv, slices, o, ctx, group, line, k_pages, v_pages, writes_cache)
        emit = self._emit_args(emit_for, ctx, x) if prefill and kernels.can_chain(T, self.q_dim, act) else None
        ready = self._add_norm_args(emit_for, ctx, T, self.dim, self.q_dim) if prefill and emit is None else None
        if emit is not None:                      # up to 16 tokens: the product prepares the next norm, as in a decode step
            nw2, xn2, ss2, eps2 = emit
            kernels.gemm_chain(o, self.wo, x, kernels.EPI_ADD_F32, emit=(nw2, xn2, ss2))
            ctx.normed[id(emit_for)] = (xn2, ss2, eps2)
        elif ready is not None:                   # the product's K slices (or the product) are added with the next norm behind
            nw2, eps2, h2, ws2 = ready
            kernels.gemm_add_norm(o, self.wo, x, nw2, eps2, h2, ws2)
            ctx.normed[id(emit_for)] = (h2, None, None)
        else:
            self._gemm(ctx, o, self.wo, x, kernels.EPI_ADD_F32)

    def _rotate_and_attend(self, qkv, slices, o, ctx, group, line, k_pages, v_pages, writes_cache):
        """From the q/k/v product's sums (or its K slices) to the heads' results o, with keys and values staged for the
        step's own attention (whole prompts) or read from the cache."""
        T, act, ws, pos = o.shape[0], o.dtype, ctx.ws, self.position
        prefill = ctx.mode == "prefill"
        q = ws.get("attn.q", (T, self.q_dim), act)
        if prefill:
            # the step's own keys and values in page format; a line that later entries read
            # keeps them for those entries
            tiles = ctx.tables["kv_tiles"]
            seq_tile0, n_tiles = tiles["seq_tile0"], tiles["n_tiles"]
            tag = "attn.stage%d" % line if ctx.line_is_shared(line) else "attn.stage"
            kst = ws.get(tag + ".k", (n_tiles, self.n_kv_heads, kernels.PAGE, self.head_dim), act)
            vst = ws.get(tag + ".v", (n_tiles, self.n_kv_heads, self.head_dim, kernels.PAGE), act)
        else:
            kst = vst = seq_tile0 = None
        if writes_cache:
            done = prefill and rope_by_tiles(T, self.n_heads, self.n_kv_heads, self.head_dim, slices) and kernels.rope_kv_write_tiles(
                qkv, q, kst, vst, ctx.cu_seqlens, seq_tile0, k_pages, v_pages, group.table, group.ring_pages,
                ctx.seq_slot, ctx.seq_len, pos.table, self.n_heads, self.n_kv_heads, self.head_dim, pos.rotary_dim,
                slices=slices)
            if not done:
                kernels.rope_kv_write(qkv, q, kst, vst, seq_tile0, k_pages, v_pages, group.table,
                                      group.ring_pages, ctx.tok_seq, ctx.tok_pos, ctx.seq_slot, ctx.seq_len, pos.table,
                                      self.n_heads, self.n_kv_heads, self.head_dim, pos.rotary_dim, slices=slices)
        else:
            kernels.rope_kv_write(qkv, q, None, None, None, None, None, None, 0, ctx.tok_seq, ctx.tok_pos,
                                  ctx.seq_slot, ctx.seq_len, pos.table, self.n_heads, self.n_kv_heads, self.head_dim,
                                  pos.rotary_dim, slices=slices)
        if prefill:
            lse = ws.get("attn.lse", (T, self.n_heads), torch.float32) if self.sinks else None
            # with sinks the result is kept unrounded too, so that the row with the sinks mixed in is rounded once
            o32 = ws.get("attn.o32", (T, self.q_dim), torch.float32) if self.sinks and act != torch.float32 else None
            if self.sinks and writes_cache:
                sink_k, sink_v = group.line_sinks(line)
                kernels.sink_store(kst, vst, seq_tile0, ctx.seq_slot, ctx.seq_len, sink_k, sink_v)
            kernels.attn_prefill(q, kst, vst, o, ctx.cu_seqlens, seq_tile0, ctx.tok_seq, ctx.tok_pos,
                                 self.n_heads, self.n_kv_heads, self.head_dim, self.window, tiles.get("tile_order"),
                                 lse=lse, out_f32=o32, score_bias=self.score_bias)
            if self.sinks:
                sink_k, sink_v = group.line_sinks(line)
                kernels.attn_sink_mix(q, o, lse, sink_k, sink_v, ctx.tok_seq, ctx.tok_pos, ctx.seq_slot, pos.table,
                                      self.n_heads, pos.rotary_dim, self.window, src_f32=o32)
        else:
            self._decode_attention(q, o, ctx, group, line, k_pages, v_pages, writes_cache)

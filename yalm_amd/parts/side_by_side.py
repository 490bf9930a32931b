"""Two mixers side by side as one mixer: both read the same input, each result is normed over the model's width
(RMS, a plain weight of its own), and `weight` times their sum goes to the stream (`weight` 1/2: their mean).  With `scales`
(left, right) the results are not normed: the mixer's result is left * (the left one's) + right * (the right one's).  The two
(JoinableMixer, both joinable) then share one product in front and one behind: their first matrices stand one below the other,
their last ones side by side, and a side's scale rides on what it puts in front of the last product (in float32, before that is
rounded to the compute dtype).  Normed ones share the product in front where both can (a product of 10,240 weight rows and one of
12,288 are one of 22,528: a launch less, and rows that deal evenly to the compute units).

The two are any registered mixers that offer forward_to (which writes a result instead of adding it); each keeps what
it keeps (keys and values in pages, a fixed-size state) under a cache line of its own: this mixer's cache request is
the pair {"left": ..., "right": ...}, and the cache manager gives line (l, "left") and (l, "right") to the members
of line l."""
import torch

from ..ops import kernels
from ..weights.loader import ParamSpec, place
from .base import JoinableMixer, Part, build_part, part


@part("mixer", "side_by_side")
class SideBySide(Part):
    emits_norm = True                 # forward takes emit_for

    def __init__(self, spec, dim, prefix):
        super().__init__(spec, dim, prefix)
        p = spec.params
        self.left = build_part("mixer", p["left"], dim, prefix)
        self.right = build_part("mixer", p["right"], dim, prefix)
        for m in (self.left, self.right):
            if not hasattr(m, "forward_to"):
                raise ValueError("a %s cannot stand beside another mixer: it has no forward_to" % type(m).__name__)
        self.eps = float(p.get("eps", 1e-6))
        self.weight = float(p.get("weight", 0.5))
        names = p.get("tensors") or {}
        self.left_norm = self.prefix + str(names.get("left_norm", "left.out"))
        self.right_norm = self.prefix + str(names.get("right_norm", "right.out"))
        self.w_left = self.w_right = None
        self.scales = tuple(float(s) for s in p["scales"]) if p.get("scales") else None
        self.w_in = self.wo = None
        self.shares_front = self.scales is None and all(hasattr(m, "front_shared") for m in (self.left, self.right))
        if self.shares_front:
            for m in (self.left, self.right):
                m.front_shared = True
        # whether a step of few rows may run the two last products, of one shape, as one launch: results that wait in buffers of their own
        self.products_together = all(hasattr(m, "mixed") for m in (self.left, self.right)) and self.left.mixed_in != self.right.mixed_in
        if self.scales is not None:
            for m, scale in zip((self.left, self.right), self.scales):
                if not isinstance(m, JoinableMixer) or not m.joinable:
                    raise ValueError("a %s cannot share its products with another mixer" % type(m).__name__)
                m.joined, m.share = True, scale

    @property
    def late_bias(self):
        """The bias that the joined result lacks: the members' (they have loaded them times their scales)."""
        biases = [m.late_bias for m in (self.left, self.right) if self.scales is not None and m.late_bias is not None]
        return None if not biases else (biases[0] if len(biases) == 1 else biases[0] + biases[1])

    def children(self):
        return [self.left, self.right]

    @property
    def prompt_tables(self):
        return tuple(getattr(self.left, "prompt_tables", ())) + tuple(getattr(self.right, "prompt_tables", ()))

    def param_specs(self):
        if self.scales is not None:
            return []
        return [ParamSpec(self.left_norm, (self.dim,), init="norm"), ParamSpec(self.right_norm, (self.dim,), init="norm")]

    def load(self, get, compute_dtype, device):
        if self.scales is not None or self.shares_front:
            self.w_in = place(torch.cat([m.in_rows(get) for m in (self.left, self.right)], dim=0), compute_dtype, device)
        if self.scales is not None:
            self.wo = place(torch.cat([m.out_columns(get) for m in (self.left, self.right)], dim=1), compute_dtype, device)
            return                        # the members load the rest themselves
        # the share of each side rides on its norm's weight (exact for a power of two)
        self.w_left = (get(self.left_norm).to(torch.float32) * self.weight).to(device).contiguous()
        self.w_right = (get(self.right_norm).to(torch.float32) * self.weight).to(device).contiguous()

    def weight_bytes(self):
        if self.scales is not None:
            return (self.w_in.numel() + self.wo.numel()) * self.w_in.element_size()
        return 2 * self.dim * 4 + (self.w_in.numel() * self.w_in.element_size() if self.w_in is not None else 0)

    def cache_request(self):
        return {"left": self.left.cache_request(), "right": self.right.cache_request()}

    def describe(self, compute_dtype):
        if self.scales is not None:
            return "two mixers side by side, one product in front of both and one behind", False
        if self.shares_front:
            return "two mixers side by side, one product in front of both, each result normed over the width", False
        return "two mixers side by side, each normed over the width", False

    def row_elements(self):
        if self.scales is not None:
            return max(self.left.n_in + self.right.n_in, self.left.n_out + self.right.n_out)
        return max(self.dim, self.left.n_in + self.right.n_in) if self.shares_front else self.dim

    def forward_to(self, h, y, ctx, line, writes_cache=True, late_bias_taken=False):
        """Writes the mixer's result to y (float32 [T, dim]), without its late_bias."""
        if self.scales is None:
            raise ValueError("two mixers that are normed add to the stream only")
        if self.late_bias is not None and not late_bias_taken:
            raise ValueError("this mixer's result lacks a bias that nobody adds")
        self._joint(h, y, ctx, line, writes_cache, kernels.EPI_STORE_F32)

    def _joint(self, h, x, ctx, line, writes_cache, epilogue):
        T, l, r = h.shape[0], self.left, self.right
        proj = ctx.ws.get("side.proj", (T, l.n_in + r.n_in), torch.float32)
        self._gemm(ctx, h, self.w_in, proj, kernels.EPI_STORE_F32)
        o = ctx.ws.get("side.o", (T, l.n_out + r.n_out), h.dtype)
        l.between(h, proj[:, :l.n_in], o[:, :l.n_out], ctx, (line, "left"), writes_cache, l.share)
        r.between(h, proj[:, l.n_in:], o[:, l.n_out:], ctx, (line, "right"), writes_cache, r.share)
        self._gemm(ctx, o, self.wo, x, epilogue)

    def forward(self, h, x, ctx, line, writes_cache=True, emit_for=None):
        """emit_for: the norm that reads the stream next; two normed results leave its output for whoever takes it."""
        T = h.shape[0]
        if self.scales is not None:
            if self.late_bias is not None:
                raise ValueError("a mixer whose last product has a bias writes its result (forward_to); it does not add to the stream")
            return self._joint(h, x, ctx, line, writes_cache, kernels.EPI_ADD_F32)
        # both results whole: a second float32 [T, dim] beside the first (64 MB for 4,096 tokens of width 4,096), added in one pass
        y, y2 = (ctx.ws.get(name, (T, self.dim), torch.float32) for name in ("side.y", "side.y2"))
        front = ({}, {})
        if self.shares_front:
            n = self.left.n_in
            proj = ctx.ws.get("side.proj", (T, n + self.right.n_in), torch.float32)
            self._gemm(ctx, h, self.w_in, proj, kernels.EPI_STORE_F32)
            front = ({"proj": proj[:, :n]}, {"proj": proj[:, n:]})
        if T <= kernels.CHAIN_MAX_ROWS and self.products_together and all(getattr(m, "late_bias", None) is None for m in (self.left, self.right)) \
                and kernels.gemm_pair_fits(
                ctx.ws.get(self.left.mixed_in, (T, self.left.wo.shape[1]), h.dtype), self.left.wo,
                ctx.ws.get(self.right.mixed_in, (T, self.right.wo.shape[1]), h.dtype), self.right.wo):
            # the left result's gate waits for nothing that the right one does not wait for, and goes along with it
            together = getattr(self.left, "leaves_gate", False) and getattr(self.right, "takes_gate", False)
            left_over = [] if together else None
            o = self.left.mixed(h, ctx, (line, "left"), writes_cache, **front[0], **({"gate_left": left_over} if together else {}))
            o2 = self.right.mixed(h, ctx, (line, "right"), writes_cache, **front[1], **({"gate": left_over[0]} if left_over else {}))
            kernels.gemm_pair(o, self.left.wo, y, o2, self.right.wo, y2)
        else:
            self.left.forward_to(h, y, ctx, (line, "left"), writes_cache, **front[0])
            self.right.forward_to(h, y2, ctx, (line, "right"), writes_cache, **front[1])
        if emit_for is None or not hasattr(emit_for, "fused"):
            kernels.norm_add_pair(y, self.w_left, y2, self.w_right, self.eps, x)
            return
        ahead = ctx.ws.get("block.h", (T, self.dim), ctx.act_dtype)           # both members have read what lay there
        kernels.norm_add_pair(y, self.w_left, y2, self.w_right, self.eps, x, ahead, emit_for.fused())
        ctx.normed[id(emit_for)] = (ahead, None, None)

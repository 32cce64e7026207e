"""Grouped-query causal attention over the paged cache.

Reference mini_llm/nn/attention.py:141-254: q/k/v projections of the normed input, head
split (head h owns columns h*d..(h+1)*d), optional per-head RMSNorm of q and k over head_dim
with one weight for all q heads and one for all k heads (Qwen3, 291-302), rotation of q and k
by the token's absolute position, write of k and v into the cache, softmax(q k^T * scale) v
over cached positions j <= p (mask rule 231-235; scale 1/sqrt(d) unless given, 95-99), kv head
h // (nq/nkv) for query head h (18-33), then the output projection without bias.

q, k and v come from one stacked [nq*d + 2*nkv*d, H] product.  When `kv_shared` is set the
layer owns no keys or values: it projects queries only and attends to the cache of the layer
it is told to read.  `window` keeps keys with p - window < j <= p.  With `values_from_keys` there is no
value projection: a position's value is its key as projected, before the per-head norm and the rotation; the
key matrix is stacked a second time where the value matrix would be, so that every kernel after the product sees
the usual row of q, k and v heads (the product makes those columns twice, from the same weights and inputs).
`forward(..., accumulate=False)` stores the output projection into the float32 rows it is given instead of adding to them.

Further forms, each a parameter: `norm_over="projection"` normalises q and k over the whole projection (all heads of a token
at once, a weight per column) instead of per head; `value_dim` gives the values a size of their own; `keep_first` keeps the
first positions of a sequence visible behind a window (token i sees j <= i with i - j < window or j < keep_first; the kept
keys keep their positions); `output_gate` multiplies the heads' outputs by sigmoid(W_g x) before the output projection (the
gate's matrix is stacked behind q, k and v).  A layer with any of them prepares its heads with `qkv_norm_prep`; its attention
runs on the matrix cores where the shape allows (bfloat16, values as wide as keys; the kept positions' keys are then one more
partial result beside those of the window's splits, which the merge of the splits adds in) and in the any-shape kernel otherwise.

And these, served by the same path: `unit_norm_after_rotation` divides every q and k head by its own root mean square (no
weight, `qk_norm_eps`) after the rotation instead of a weighted norm before it (`rotate_unit_prep` prepares the heads; the
position part says whether a pair is (i, i + rot/2) or (2i, 2i + 1)); `sink` adds a learned term exp(sink_h) per head to the
softmax's denominator, which has no key and no value; `score_cap` passes the scaled scores through cap * tanh(score / cap);
`output_gate="head"` gates with one number a head, sigmoid(W_g x)_h, in the attention kernel that finishes a query or the merge
of its partial results, where `True` gates every value by a kernel of its own; `bias` with any of these
adds the stacked biases to q, k and v: in the product's epilogue, or, where `rotate_unit_prep` prepares the heads, in that kernel
as it reads the rows (in float32; the product then runs without a bias, through the vendor's library for many rows).

And with the norm over the projection: `query_temperature` (coef, every) multiplies a query at position p by
1 + coef * ln(floor((p + 1) / every) + 1); `value_mix` mixes a layer's values with those of an earlier layer of the same token,
v <- (1 - lambda) v + lambda v_first with a learned lambda, before they are cached ("first": the layer whose values the others take,
"later": a layer that takes them; they stay in a buffer of the step); `distance_bias` takes rate_h * ln(1 + reach_h * (i - j)) off
head h's score of query i and key j (`"linear"`: slope_h * (i - j) with the fixed slopes 2^(-8 (h + 1) / heads)); a number for `sink` is a sink of that score in every head instead of a learned one.  Values
narrower than keys (a multiple of 16) run on the matrix cores too.

`chunk` in place of a window: position i sees position j <= i only in its own chunk of that many positions, counted from position 0.
Heads that need no preparation at all (no norm, rotation, bias, temperature or mixed values) stay where the product left them:
only their keys and values pass through a kernel on their way into the pages, and in decode steps of few rows the attention kernel
stores those too.
"""

from __future__ import annotations

import math

import torch

from ..kernels import ops
from .base import PagedKVNeed, Part, PartSpec, TensorSpec, create, length_class, reach_of, register
from .linear import ScaledRows, kernels_of, linear, materialize, rows_of, workspace_of


class GQAAttention(Part):
    graph_safe = True  # launches only library kernels on arena buffers
    plan_safe = True   # ... and nothing but this package's kernels, with arguments that follow the step's shape alone
    takes_lazy_norm = True
    begins_next_norm = True
    wants_query_groups = True   # ragged steps go to a kernel that walks groups of a request's consecutive tokens
    can_overwrite = True        # forward(..., accumulate=False) stores its output

    @property
    def carries_rows(self) -> bool:
        return self.whole_rows

    def __init__(self, hidden_size: int, num_heads: int, num_kv_heads: int, head_dim: int, *,
                 position: PartSpec = PartSpec("none"), qk_norm: bool = False, qk_norm_eps: float = 1e-6,
                 bias: bool = False, scale: float | None = None, window: int | None = None,
                 kv_shared: bool = False, values_from_keys: bool = False, norm_over: str = "head", value_dim: int | None = None,
                 keep_first: int = 0, output_gate: bool | str = False, unit_norm_after_rotation: bool = False,
                 sink: bool | float = False, score_cap: float | None = None, query_temperature: tuple | None = None,
                 value_mix: str | None = None, distance_bias: bool | str = False, chunk: int | None = None):
        for name, value in (("hidden_size", hidden_size), ("num_heads", num_heads), ("num_kv_heads", num_kv_heads), ("head_dim", head_dim)):
            if value <= 0:
                raise ValueError(f"{name} must be positive, got {value}")
        if num_heads % num_kv_heads != 0:
            raise ValueError(f"num_heads must be divisible by num_kv_heads, got {num_heads} and {num_kv_heads}")
        if scale is not None and (not math.isfinite(scale) or scale <= 0):
            raise ValueError(f"scale must be finite and positive, got {scale}")
        # what a query sees: the kernels' word for it, and the most positions that can be (None: all)
        self.reach, self.chunk, self.span = reach_of(window, chunk), chunk, window if chunk is None else chunk
        if qk_norm and qk_norm_eps <= 0:
            raise ValueError(f"qk_norm_eps must be positive, got {qk_norm_eps}")
        self.hidden_size, self.num_heads, self.num_kv_heads, self.head_dim = hidden_size, num_heads, num_kv_heads, head_dim
        self.position = create("position", position)
        self.qk_norm, self.qk_norm_eps, self.bias = qk_norm, qk_norm_eps, bias
        self.scale = 1.0 / math.sqrt(head_dim) if scale is None else scale
        if values_from_keys and kv_shared:
            raise ValueError("a layer that owns no keys has no values to take from them")
        self.window, self.kv_shared, self.values_from_keys = window, kv_shared, values_from_keys
        if norm_over not in ("head", "projection"):
            raise ValueError(f"norm_over must be 'head' or 'projection', got {norm_over!r}")
        if value_dim is not None and value_dim <= 0:
            raise ValueError(f"value_dim must be positive when given, got {value_dim}")
        if keep_first < 0 or (keep_first and window is None):
            raise ValueError(f"keep_first must not be negative and needs a window, got {keep_first}")
        if output_gate not in (False, True, "head"):
            raise ValueError(f"output_gate must be False, True (a gate a value) or 'head' (a gate a head), got {output_gate!r}")
        if score_cap is not None and (not math.isfinite(score_cap) or score_cap <= 0):
            raise ValueError(f"score_cap must be finite and positive when given, got {score_cap}")
        if unit_norm_after_rotation and qk_norm:
            raise ValueError("heads are normalised before the rotation with a weight (qk_norm) or after it without one, not both")
        if unit_norm_after_rotation and qk_norm_eps <= 0:
            raise ValueError(f"qk_norm_eps must be positive, got {qk_norm_eps}")
        self.norm_over, self.value_dim, self.keep_first, self.output_gate = norm_over, value_dim or head_dim, keep_first, output_gate
        self.unit_after, self.has_sink, self.score_cap = unit_norm_after_rotation, sink is True, score_cap
        self.sink_score = None if isinstance(sink, bool) else float(sink)        # a sink of one known score in every head
        if query_temperature is not None and query_temperature[1] <= 0:
            raise ValueError(f"the query temperature's step must be positive, got {query_temperature[1]}")
        if value_mix not in (None, "first", "later"):
            raise ValueError(f"value_mix must be None, 'first' or 'later', got {value_mix!r}")
        if distance_bias not in (False, True, "linear"):
            raise ValueError(f"distance_bias must be False, True (learned, with a logarithm) or 'linear' (fixed slopes), got {distance_bias!r}")
        self.query_temperature, self.value_mix, self.distance_bias = query_temperature, value_mix, distance_bias
        self.neighbours = getattr(self.position, "pairing", "halves") == "interleaved"
        # the forms that the kernels preparing whole rows serve (see the module's text)
        self.whole_rows = bool((qk_norm and norm_over == "projection") or self.value_dim != head_dim or keep_first > 0 or output_gate
                               or unit_norm_after_rotation or self.has_sink or self.sink_score is not None or score_cap is not None or self.neighbours
                               or query_temperature is not None or value_mix is not None or distance_bias)
        # heads that no kernel has to touch between the product and the attention (see the module's text)
        self.heads_as_projected = bool(self.whole_rows and not (qk_norm or bias or unit_norm_after_rotation or query_temperature is not None
                                                               or value_mix is not None) and position.kind == "none")
        if (unit_norm_after_rotation or self.neighbours) and (query_temperature is not None or value_mix is not None):
            raise ValueError("a query temperature and mixed values are made by the kernel that normalises over the projection")
        if self.whole_rows and (kv_shared or values_from_keys or (qk_norm and norm_over == "head")):
            raise ValueError("a norm over the projection or after the rotation, values of their own size, kept first positions, a sink, "
                             "capped scores and an output gate come without shared or key-made values and per-head norms before the rotation")
        if self.neighbours and qk_norm:
            raise ValueError("neighbouring pairs are rotated by the kernel that normalises after the rotation or not at all")
        self.b_late = None
        self.gate_width = 0 if not output_gate else num_heads if output_gate == "head" else num_heads * self.value_dim
        self.sinks = self.distance = self.mix = None
        self.w_qkv = self.b_qkv = self.w_o = self.q_norm = self.k_norm = None

    # ------------------------------------------------------------------ weights
    def tensors(self):
        h, d = self.hidden_size, self.head_dim
        names = ("q_proj",) if self.kv_shared else ("q_proj", "k_proj") if self.values_from_keys else ("q_proj", "k_proj", "v_proj")
        widths = {"q_proj": self.num_heads * d, "k_proj": self.num_kv_heads * d, "v_proj": self.num_kv_heads * self.value_dim}
        specs = {f"{n}.weight": TensorSpec((widths[n], h)) for n in names}
        if self.bias:
            specs.update({f"{n}.bias": TensorSpec((widths[n],), role="bias") for n in names})
        if self.output_gate:
            specs["g_proj.weight"] = TensorSpec((self.gate_width, h))
        if self.has_sink:
            specs["sink"] = TensorSpec((self.num_heads,), role="bias")
        if self.value_mix is not None:      # (the layer the others take their values from has no use for its own)
            specs["value_mix"] = TensorSpec((), role="bias", optional=self.value_mix == "first")
        if self.distance_bias is True:      # drawn around one at random: a reach must not be negative
            specs["distance_rate"] = TensorSpec((self.num_heads,), role="norm")
            specs["distance_reach"] = TensorSpec((self.num_heads,), role="norm")
        specs["o_proj.weight"] = TensorSpec((h, self.num_heads * self.value_dim))
        if self.qk_norm:
            over = d if self.norm_over == "head" else None
            specs["q_norm.weight"] = TensorSpec((over or widths["q_proj"],), role="norm")
            if not self.kv_shared:
                specs["k_norm.weight"] = TensorSpec((over or widths["k_proj"],), role="norm")
        return specs

    def bind(self, weights, dtype):
        names = ("q_proj",) if self.kv_shared else ("q_proj", "k_proj", "k_proj") if self.values_from_keys else ("q_proj", "k_proj", "v_proj")
        if self.output_gate:
            names += ("g_proj",)
        stacked = [weights[f"{n}.weight"] for n in names]
        biases = [weights[f"{n}.bias"] if n != "g_proj" else weights["g_proj.weight"].new_zeros(self.gate_width) for n in names] if self.bias else None
        self.w_qkv = self.stack_rows(stacked, dtype) if self.whole_rows else torch.cat(stacked, 0).to(dtype).contiguous()
        self.b_qkv = torch.cat(biases, 0).to(dtype).contiguous() if self.bias and not self.whole_rows else None
        # the kernels that prepare whole rows add the biases themselves, in float32, as they read the rows
        self.b_late = torch.cat(biases, 0).float().contiguous() if self.bias and self.whole_rows else None
        if self.has_sink:
            self.sinks = weights["sink"].float().contiguous()
        elif self.sink_score is not None:
            self.sinks = torch.full((self.num_heads,), self.sink_score, dtype=torch.float32, device=self.w_qkv.device)
        if self.value_mix == "later":
            self.mix = weights["value_mix"].float().reshape(1).contiguous()
        if self.distance_bias == "linear":
            slopes = 2.0 ** (-8.0 * torch.arange(1, self.num_heads + 1, dtype=torch.float64) / self.num_heads)
            self.distance = slopes.float().to(self.w_qkv.device)
        elif self.distance_bias:
            self.distance = torch.stack((weights["distance_rate"].float(), weights["distance_reach"].float())).contiguous()
        self.w_o = weights["o_proj.weight"].to(dtype).contiguous()
        if self.qk_norm:
            self.q_norm = weights["q_norm.weight"]
            self.k_norm = weights["k_norm.weight"] if not self.kv_shared else self.q_norm
            if self.whole_rows:
                self.q_norm, self.k_norm = self.q_norm.float().contiguous(), self.k_norm.float().contiguous()

    def weight_bytes(self):
        return (self.w_qkv.numel() + self.w_o.numel()) * self.w_o.element_size()

    def flops(self, tokens, pairs):
        if self.span is not None:
            pairs = min(pairs, tokens * self.span)
        # the projections, then scores and weighted values: two products of head_dim per pair and query head
        return super().flops(tokens, pairs) + 2.0 * pairs * self.num_heads * (self.head_dim + self.value_dim)

    def cache_need(self):
        if self.kv_shared:
            return None
        return PagedKVNeed(self.num_kv_heads, self.head_dim, self.window, value_dim=None if self.value_dim == self.head_dim else self.value_dim,
                           keep_first=self.keep_first, chunk=self.chunk)

    @staticmethod
    def _decode_splits(workgroups: int, longest: int, bound: int, page_size: int) -> int:
        """Into how many workgroups the keys of one decode token are divided: enough to give every
        compute unit two when the batch alone does not (measured on MI355X inside the 8-request
        decode step at 2,048 tokens of context: 8 splits 4.58 ms, 4 splits 4.61 ms), but at least
        256 keys each (a power of two that follows the length's class, not the length); and enough
        that the block table entries of one workgroup (at most 4,096) fit its LDS for contexts up
        to `bound`."""
        units = ops.compute_units()
        # from five workgroups for every eight units on, the batch alone does as well or better, and there is nothing
        # to merge (2,048 tokens of context, batch 20 / 24 / 32: 37.8 / 42.0 / 52.7 us undivided against 40.1 / 45 /
        # 54.4 us with the 4 / 3 / 2 parts that two workgroups a unit would ask for; the same at 8,192 tokens)
        wanted = 1 if 8 * workgroups >= 5 * units else -(-2 * units // workgroups)
        # between one and one and a half workgroups a unit some units have two where the others have one, and with
        # contexts of 2,048 tokens and more the second round costs more than a merge: two parts (40 query heads on 8:
        # batch 33 / 40 / 44 / 48 at 2,048 tokens 72.6 / 75.1 / 77.9 / 79.7 us undivided, 66.5 / 71.5 / 73.3 / 78.2 in two parts;
        # at 4,096 tokens 140 / 144 / 148 / 151 against 122 / 129 / 134 / 144; at 1,024 tokens and from batch 52 on nothing
        # is gained; four parts are better still up to batch 40 and worse from 44 on, and a graph serves both)
        if units < workgroups <= units + units // 2 and length_class(longest) >= 2048:
            wanted = 2
        return max(1, min(wanted, length_class(longest) // 256, 64), -(-bound // (4096 * page_size)))

    @classmethod
    def _decode_shape(cls, workgroups: int, longest: int, bound: int, page_size: int, head_dim: int) -> tuple[int, int]:
        """(splits, form) of attention_decode(): workgroups of four waves, two a unit (form 1), divided as _decode_splits says;
        or, while the batch alone has no more than one workgroup a unit, of eight waves (form 2; heads of up to 128), one a unit.
        A unit streams its workgroup's keys at some 40 GB/s whatever is on its way at once, and a merge costs 3-4 us and the gap
        before it, so eight waves finish a short context sooner than a merge would.  us with four waves / with eight, parts in
        brackets, merge counted, 32 heads on 8: batch 1 at 2,048 tokens 14.5 [8] / 13.2 [8], batch 8 24.5 [8] / 23.4 [4], batch 8 at 8,192
        58.2 [8] / 56.1 [4]; but batch 40 at 600 28.3 / 32.6 and batch 64 at 1,500 73.1 / 75.9.
          * As many parts as one round of workgroups has room for: a second round that is partly empty costs more than the shorter walks
            give (192 workgroups at 1,500: 34.9 [1] / 32.7 [1], 40.9 [2]; 96: 24.1 [4] / 20.8 [2], 29.8 [3], 27.3 [4]).
          * Two rounds over contexts long enough for a request that is far longer than the others, which a step waits for, to count, where
            one round is not full: from 4,096 tokens on, from 2,048 where one round has room for two parts and less, from 1,024 where it
            has for one (while the four waves' rule divides).  96 workgroups at 3,000 40.3 [6] / 37.1 [5], 35.2 [2], at 8,000 88.7 [6] / 77.8 [5], 75.5 [2]; of 12
            requests one at 32,000 and the others at 500 85 [6] / 86 [5], 190 [2]; 136 workgroups at 1,500 33.2 [4] / 32.9 [3], 28.2 [1].
          * Two or three beyond that, the fuller, from 8,192 tokens on (192 workgroups: of 24 requests one at 32,000 430 [1] / 105 [4], 364 [1];
            all at 8,000 146 [1] / 144 [4], 138 [1]).
          * Four waves again from 4,096 tokens on where one round is full: a unit's stream is the limit, so one long context among short
            ones wants units, not waves (64 workgroups, one request of 8 at 32,000 67 [8] / 102 [4]; all at 8,000 52.8 [8] / 51.6 [4]).
          * At least 256 keys each (batch 1 at 900: 14.1 [2] / 12.5 [2], 15.1 [1]; batch 16 at 520, 640, 768 and 900 15.5 / 14.4 [2] 13.4 [1],
            16.8 / 15.5 16.1, 18.2 / 17.3 18.6, 20.5 / 19.1 21.9), and under 1,024 tokens undivided for smaller heads, whose keys are
            fewer bytes (64 dims, batch 4 at 520 and 768 10.2 [2] / 8.4 [1] 8.9 [2] and 10.4 / 9.1 9.8)."""
        units = ops.compute_units()
        if workgroups > units or head_dim > 128:
            return cls._decode_splits(workgroups, longest, bound, page_size), 1
        reach = length_class(longest)
        most = min(reach // 256, 64)
        wanted, twice, few = units // workgroups, 2 * units // workgroups, 8 * workgroups <= 5 * units
        if head_dim < 128 and reach < 1024:
            wanted = 1
        elif units % workgroups == 0:
            if reach >= 4096 and 8 * workgroups >= units and 2 * workgroups <= units:
                return cls._decode_splits(workgroups, longest, bound, page_size), 1
        elif few:
            # (160 workgroups, the last that the other rule divides, are as well off undivided under 2,048 tokens)
            counts = reach >= 4096 or (reach >= 2048 and wanted < 3) or (reach >= 1024 and wanted < 2 and 8 * workgroups < 5 * units)
            wanted = twice if counts and twice <= min(most, 32) else wanted
        elif reach >= 8192:
            thrice = 3 * units // workgroups
            wanted = thrice if 2 * thrice > 3 * twice else twice
        return max(1, min(wanted, most), -(-bound // (4096 * page_size))), 2

    def _keys_read_once(self, splits: int, form: int, longest: int, page_size: int) -> int:
        """`form` of a shape that _decode_shape() gave, 3 in place of 1 where keys and values are better loaded with the hint that they are read
        once (csrc/common.h, load_once).  us without / with it, keys that no cache holds, heads of 128 on 8 kv heads unless it says otherwise:
          * Workgroups that walk 128 keys and more, as their contexts' class or the window says: waves without a tile of their own bring
            their workgroup's last once more, which the hint has them fetch again.  Contexts of a half up to all of 64, 150, 300 and 450 tokens:
            batch 128 13.0 / 14.6, 18.1 / 17.4, 27.6 / 26.6, 38.1 / 36.6, batch 33 6.4 / 6.9, 8.4 / 8.5, 11.8 / 12.1, 16.4 / 16.8; batch 64 seeing 128 of 4,000
            tokens 11.8 / 11.1, 512 29.7 / 27.6; batch 8 at 8,000 in 8 parts 52.0 / 47.9; heads of 64, batch 64 at 1,000 42.6 / 39.6.  (So many keys
            of as many workgroups as go with four waves are tens of MB a layer: no cache keeps them until the next step.)
          * Pages of up to 32, whose tiles have the lines of values to themselves; of larger ones the next tile, another wave's, has the other
            half: batch 64 at 2,048 in pages of 16, 32, 64 and 256 99.1 / 87.1, 100.1 / 90.0, 105.8 / 110.1 and 107.2 / 114.4.
          * Heads of up to 128: those of 192 bring a tile at a time (batch 40 at 600 31.1 / 33.7, batch 16 at 4,000 in 4 parts 68.5 / 65.5, one
            request at 1,000 in 3 of 28 layers' keys 13.8 / 15.3).
        Workgroups of eight waves walk contexts of few requests, which the last-level cache keeps from step to step unless they are
        loaded so (one request at 509 tokens, 0.6B sizes, 1,035 us a step / 1,078)."""
        seen = length_class(longest) if self.span is None else min(length_class(longest), self.span)
        return 3 if form == 1 and self.head_dim <= 128 and page_size <= 32 and seen // splits >= 128 else form

    @staticmethod
    def _walks_in_pairs(ctx, heads_per_group: int, head_dim: int) -> bool:
        """Whether the kernel for ragged steps lets two neighbouring query groups walk their keys together (attention_prefill's
        `one_request`): two heads a kv group, groups of more than 16 tokens, all of one request."""
        return heads_per_group == 2 and head_dim == 128 and ctx.max_qblock > 16 and ctx.R - ctx.single_rows == 1

    @staticmethod
    def _one_launch(workgroups: int, splits: int, rest: int, group_size: int, heads_per_group: int, longest: int) -> bool:
        """Whether a mixed step's single tokens (`workgroups`, divided into `splits` by themselves) and the portion behind them (`rest`
        workgroups) go in one launch (attention_mixed), the single tokens' keys undivided: neither fills the chip by itself, and two
        launches wait for each other.  us a layer in two launches / in one, `a` beside `b` tokens after `c`: 32 heads on 8, 24 at 1,500 beside
        488 after 488 77 / 43; 40 on 8 78 / 60; 64 on 8 80 / 63; 20 at 8,192 beside 2,028 after 0 254 / 163, 295 / 206 and 306 / 213.
        Not so
          * single tokens that would be divided, unless they are half a workgroup a unit and more, which the portion's workgroups
            fill up, and no context is much longer than the others need be: 17 on 8 kv heads, one at 8,192 and the others at 500, beside
            2,028 145 / 120; at 16,000 171 / 206, at 32,000 224 / 380 (all 17 at 16,000: 348 / 253);
          * five heads a group and more beside a long portion in groups of 32, whose launch alone has a wave for every head and
            walks its keys once (csrc/attention.hip, MANY_WAVES), while no context is longer than that walk: 32 on 4, 33 at 500, 1,500
            and 4,000 beside 2,028 115 / 130, 141 / 130 and 178 / 134, 64 at 500 and 1,500 112 / 138 and 146 / 152."""
        units = ops.compute_units()
        if heads_per_group > 4 and group_size > 16 and rest <= units and longest <= 3072:
            return False
        return splits == 1 or (2 * workgroups > units and longest <= 8192)

    @staticmethod
    def _prefill_splits(workgroups: int, longest: int, outputs: int, heads_per_group: int = 4, tokens: int = 0, paired: bool = False) -> int:
        """Into how many workgroups the keys of every query group of a ragged step are divided: one, unless
        the groups alone leave compute units idle (a last portion of a prompt, a short portion after a long
        context), and never from two workgroups a unit on.  Partial results (float32, `outputs` values per split)
        stay within 256 MB.  Measured on
        MI355X, 32 query heads on 8 kv heads:
          * contexts of 16,384 tokens and more: towards eight workgroups a unit, at least 1,024 keys each
            (32,768 tokens of context: 1 token 1,161 -> 57 us with 32 splits, 64 tokens 1,165 -> 105 us with
            16, 512 tokens 1,186 -> 576 us with 8);
          * shorter contexts: towards two workgroups a unit, at least 256 keys each (2,048 tokens of context: 64 tokens 42.5 -> 18.6 us with 8 splits, 256 tokens 43.2 -> 32.4 with
            4, 512 tokens 87.5 -> 76.4 with 2, but 1,024 tokens 96.8 -> 127 and 2,032 tokens 111 -> 173 with 2:
            what the merge reads and writes grows with the tokens, what a split saves with the context).  So under
            16,384 tokens of context the keys are divided only where the longest context is at least four times the
            step's `tokens` (undivided against 2 splits with their merge: 512 tokens after 0 / 512 / 1,024 / 1,536:
            16.9 / 26.6 / 36.2 / 45.8 against 24.4 / 30.5 / 36.9 / 42.9 us; 256 tokens after 256 / 512 / 768 / 1,024:
            16.5 / 21.1 / 25.7 / 30.2 against 18.8 / 20.3 / 23.1 / 25.6 us; 128 tokens after 0 / 256 / 512: 14.4 / 14.1 /
            18.5 against 16.2 / 16.8 / 17.1 us).
        A kv group of five to eight heads walks the keys once with a wave for every head while the launch is at
        most two workgroups a unit; that walk is short enough that one workgroup a unit is the aim (40 heads on
        8: 512 tokens after 1,536 54 us undivided against 72 with 2; 256 tokens 51 -> 43 with 2, 128 tokens
        after 8,064 177 -> 59 with 4, 64 tokens after 2,000 50 -> 22 with 8); from 16,384 tokens of context on the rule
        for long contexts holds for them too (512 tokens after 32,256: 697 us undivided, 617 with 8)."""
        units = ops.compute_units()
        within = (64 << 20) // max(outputs, 1)
        if paired:
            # Two heads a kv group, groups of 32 that walk in pairs (csrc/attention.hip, SPREAD_PAIRS): a walk is as long as its keys
            # whatever it works on, so two workgroups a unit are the aim behind any context (16 heads on 8: 2,048 tokens after 14,336
            # 567 us undivided, 322 with 2, 382 with 3, 313 with 4; after 2,048 136 / 100 / - / 103; 1,024 after 15,360 551 us
            # undivided, 290 / 178 / 184 with 2 / 4 / 8; but 8,192 tokens, two a unit without, 390 and 404 with 2)
            if workgroups >= 2 * units:
                return 1
            return max(1, min(-(-2 * units // workgroups), longest // 256, 32, within))
        if workgroups >= 2 * units:      # (2,048 tokens in groups of 32 after 30,720: 1,071 us undivided, 1,115 with 2)
            return 1
        if longest < 16384 and longest < 4 * tokens:
            return 1
        if heads_per_group > 4 and workgroups <= units and longest < 16384:
            return max(1, min(-(-units // workgroups), longest // 256, 32, within))
        if longest >= 16384:
            return max(1, min(-(-8 * units // workgroups), longest // 1024, 32, within))
        return max(1, min(-(-2 * units // workgroups), longest // 256, 32, within))

    PREPARE_INSIDE_ROWS = 16     # rows of a decode step up to which the attention kernel prepares q, k and v itself

    # ------------------------------------------------------------------ forward
    def forward(self, ctx, x, residual, cache, then_norm=None, accumulate: bool = True):
        if cache is None:
            raise ValueError("attention needs a paged cache (its own, or the one it is told to read)")
        t, d, nq = rows_of(x), self.head_dim, self.num_heads
        nkv = 0 if self.kv_shared else self.num_kv_heads
        group = ctx.group(cache.group)
        tables = self.position.tables(ctx)
        cos, sin = tables if tables is not None else (None, None)
        if self.whole_rows:
            return self._forward_whole_rows(ctx, x, residual, cache, group, cos, sin, then_norm, accumulate)
        qkv = ctx.scratch("attn_qkv", (t, (nq + 2 * nkv) * d), ctx.dtype)
        # 17..128 rows of a decode step: the q/k/v product and the preparation of its heads as two kernels, the
        # second adding up the sums of the product's K splits (no kernel of its own for that)
        together = (ctx.all_decode and self.b_qkv is None and ctx.dtype == torch.bfloat16 and t > self.PREPARE_INSIDE_ROWS
                    and ops.gemm_mid_qk_prep_takes(self.w_qkv.dtype, t, nq, nkv, d, self.w_qkv.shape[1], 0 if cos is None else cos.shape[1],
                                                   kernels_of(ctx)))
        begun = plain = None
        if together:
            begun = x if isinstance(x, ScaledRows) else None          # a norm that the product before began
            plain = begun.x if begun is not None else materialize(ctx, x)
            together = plain.dtype == torch.bfloat16 and plain.is_contiguous()
        if together:
            ops.gemm_mid_qk_prep(qkv, plain, self.w_qkv, None if begun is None else begun.sumsq, 0.0 if begun is None else begun.eps,
                                 nq, nkv, d, self.q_norm, self.k_norm, self.qk_norm_eps, cos, sin, cache.k_pages, cache.v_pages,
                                 group.slots, group.page_size, choice=kernels_of(ctx), workspace=workspace_of(ctx))
        else:
            linear(ctx, qkv, x if plain is None or begun is not None else plain, self.w_qkv, self.b_qkv)
        out = ctx.scratch("attn_out", (t, nq * d), ctx.dtype)
        kv_heads = cache.k_pages.shape[1]
        decode = ctx.all_decode and ops.attention_decode_supported(ctx.dtype, nq, kv_heads, d, group.page_size)
        # a decode step's attention kernel normalises and rotates q and k and writes the new key and
        # value itself, when the rotation covers the whole head or there is none; beyond 16 rows a kernel
        # before it does that once a token (measured: 98 against 108 us for the attention kernel at 64 rows)
        whole_head = cos is None or cos.shape[1] * 2 == d
        prepare = queries_raw = None
        if together:
            pass
        elif decode and whole_head and ops.decode_prepare_supported(d, cos is not None) and t <= self.PREPARE_INSIDE_ROWS:
            prepare = ops.DecodePrepare(self.q_norm, self.k_norm, self.qk_norm_eps, cos, sin, nkv)
        else:
            # a ragged step of heads of 128: the attention kernel normalises and rotates the q heads on their way into its
            # registers, so that only the k and v heads pass through a kernel before it (a third of the rows' bytes;
            # measured at 2,048 tokens, 32 q heads on 8: 19-22 -> 10.4 us for the kernel before attention, 66 -> 68 us
            # for attention itself)
            if (not decode and nkv > 0 and whole_head and ops.attention_prefill_prepares(d)
                    and ops.attention_decode_supported(ctx.dtype, nq, kv_heads, d, group.page_size)):
                queries_raw = ops.DecodePrepare(self.q_norm, None, self.qk_norm_eps, cos, sin, 0)
            ops.qk_prep(qkv, nq, nkv, d, self.q_norm, self.k_norm, self.qk_norm_eps, cos, sin,
                        cache.k_pages, cache.v_pages, group.slots, group.page_size, skip_q=queries_raw is not None)
        if decode:
            longest, bound = ctx.max_k, ctx.max_k_bound
            if self.span is not None:
                longest, bound = min(longest, self.span + 32), min(bound, self.span + 64)
            splits, form = self._decode_shape(t * kv_heads, longest, bound, group.page_size, d)
            part_o = part_ml = None
            if splits > 1:
                part_o = ctx.scratch("attn_part_o", (t, nq * splits * d), torch.float32)
                part_ml = ctx.scratch("attn_part_ml", (t, nq * splits * 2), torch.float32)
            ops.attention_decode(out, qkv, cache.k_pages, cache.v_pages, group.block_table, ctx.token_slot, ctx.positions,
                                 nq, self.scale, self.reach, splits, part_o, part_ml, ctx.max_k_bound, prepare,
                                 form=self._keys_read_once(splits, form, ctx.max_k, group.page_size))   # the next tile on its way while one is worked on, the first one before the query is prepared (measured: 0.6 % of a step)
        elif ops.attention_decode_supported(ctx.dtype, nq, kv_heads, d, group.page_size):
            # sized by the step's coarse bound of the longest context, the same for every step of one shape
            longest = ctx.max_k_bound if self.span is None else min(ctx.max_k_bound, self.span + 64)
            singles = ctx.single_rows
            paired = self._walks_in_pairs(ctx, nq // kv_heads, d)
            rest_splits = self._prefill_splits((-(-ctx.num_qblocks // 2) if paired else ctx.num_qblocks) * kv_heads, longest, (t - singles) * nq * d,
                                               nq // kv_heads, t - singles, paired)
            splits, form = self._decode_shape(singles * kv_heads, longest, ctx.max_k_bound, group.page_size, d) if singles else (1, 1)
            if (singles and d == 128 and rest_splits == 1 and ctx.max_k_bound <= 4096 * group.page_size
                    and self._one_launch(singles * kv_heads, splits, ctx.num_qblocks * kv_heads, ctx.max_qblock, nq // kv_heads, longest)):
                ops.attention_mixed(out, qkv, cache.k_pages, cache.v_pages, group.block_table, ctx.token_slot, ctx.positions, singles, ctx.qblock_token0,
                                    ctx.qblock_count, nq, self.scale, self.reach, ctx.max_qblock, ctx.max_k_bound, queries_raw, one_request=paired)
                return linear(ctx, residual, out, self.w_o, accumulate=accumulate, then_norm=then_norm)
            if singles:
                # the single tokens at the head of a mixed step (decoding requests beside a prompt portion) go to the
                # kernel of decode steps, which divides one token's keys between waves and workgroups; as rows of
                # the other kernel each would walk its whole context in one workgroup
                part_o = part_ml = None
                if splits > 1:
                    part_o = ctx.scratch("attn_single_part_o", (singles, nq * splits * d), torch.float32)
                    part_ml = ctx.scratch("attn_single_part_ml", (singles, nq * splits * 2), torch.float32)
                first = None
                if queries_raw is not None:      # the decode kernel prepares the q heads of its rows likewise
                    parted = None
                    if cos is not None:          # the tables' rows of the single tokens and of the rest, cut once a step
                        parted = ctx.memo.get(("rotation_rows", id(cos)))
                        if parted is None:
                            parted = ctx.memo[("rotation_rows", id(cos))] = (cos[:singles], sin[:singles], cos[singles:], sin[singles:])
                    first = ops.DecodePrepare(self.q_norm, self.k_norm, self.qk_norm_eps, None if parted is None else parted[0],
                                              None if parted is None else parted[1], 0)
                ops.attention_decode(out[:singles], qkv[:singles], cache.k_pages, cache.v_pages, group.block_table, ctx.token_slot,
                                     ctx.positions, nq, self.scale, self.reach, splits, part_o, part_ml, ctx.max_k_bound, first,
                                     form=self._keys_read_once(splits, form, ctx.max_k_bound, group.page_size))
            rest = ctx.memo.get("rows_after_singles")
            if rest is None:
                rest = ctx.memo["rows_after_singles"] = (ctx.token_slot[singles:], ctx.positions[singles:])
            if queries_raw is not None and singles and cos is not None:
                queries_raw = ops.DecodePrepare(self.q_norm, None, self.qk_norm_eps, parted[2], parted[3], 0)
            splits = rest_splits
            part_o = part_ml = None
            if splits > 1:
                part_o = ctx.scratch("attn_part_o", (t - singles, nq * splits * d), torch.float32)
                part_ml = ctx.scratch("attn_part_ml", (t - singles, nq * splits * 2), torch.float32)
            ops.attention_prefill(out[singles:], qkv[singles:], cache.k_pages, cache.v_pages, group.block_table, rest[0], rest[1],
                                  ctx.qblock_token0, ctx.qblock_count, nq, self.scale, self.reach, ctx.max_qblock, ctx.max_k_bound,
                                  splits, part_o, part_ml, queries_raw, one_request=paired)
        else:
            self._attend(ctx, out, qkv, cache, group)
        return linear(ctx, residual, out, self.w_o, accumulate=accumulate, then_norm=then_norm)

    # floats, 128 MB, that the results of pieces of keys may take before a launch stays undivided (of the buffers a step keeps, which grow by doubling)
    PIECE_RESULTS = 1 << 25

    @staticmethod
    def _piece_splits(workgroups: int, longest: int) -> int:
        """Into how many workgroups of one wave attention_f32_divided() divides the keys of a row (1: attention(), which gives a row of a kv head a
        workgroup of eight waves).  A class of lengths has one answer: at most as many parts as the longest of them has pieces (where a row has fewer,
        some have nothing to do), at most two to a unit, which are a full chip.
        us, rows of 8 kv heads with two query heads each, attention() / divided into what the rule says [parts], merge counted:
          * up to a workgroup for every four units, 128 dims: one row at 256 tokens 10.3 / 9.4 [8], at 300 14.2 / 9.4, at 511 14.9 / 9.7, at 700 22.0 / 10.6 [16], at
            2,000 50.9 / 13.8 [32], at 4,000 99 / 23 [64]; eight at 256 11.0 / 10.0 [8], at 300 14.7 / 11.5, at 511 15.9 / 13.3, at 700 23.1 / 19.7, at 1,000 28.2 / 21.4,
            at 4,000 116 / 72; 64 dims: one at 256 7.3 / 7.8, at 300 9.4 / 7.9, at 511 9.9 / 8.4, eight at 256 7.8 / 8.1, at 300 9.9 / 8.7, at 4,000 73 / 50 (at 256 itself,
            four pieces, attention() has one trip; from 257 on two);
          * up to one for every two units, over long contexts: 12 rows at 4,000 126 / 104 [10], 16 133 / 128 [8], of 64 dims 80 / 70; at 509 and 1,000 tokens 96
            and 128 workgroups lost by it (16.7 / 19.7, 36.9 / 39.3);
          * beyond that attention() fills the chip: 256 workgroups at 4,000 185 / 237 [8].
        One, three and four query heads a kv head take the same times to 0.5 us (16 rows at 4,000 133 / 126, 131 and 133)."""
        units, reach = ops.compute_units(), length_class(longest)
        if reach >= 256 and 4 * workgroups <= units:
            return min(reach // 32, 2 * units // workgroups)
        if reach >= 2048 and 2 * workgroups <= units:
            return 4 * units // workgroups
        return 1

    def _attend_divided(self, ctx, out, qkv, cache, group) -> bool:
        """Float32 attention of rows of a request each with the keys of a row divided between workgroups, if that is the faster way."""
        rows, nq, d = qkv.shape[0], self.num_heads, self.head_dim
        if d % 64 != 0 or nq > 4 * cache.k_pages.shape[1] or length_class(ctx.max_k) == 0 or qkv.stride(0) % 4 != 0 or qkv.data_ptr() % 16 != 0:
            return False
        longest, slots = ctx.max_k, -(-ctx.max_k_bound // 64)              # pieces of 64 positions, the most that a row sees
        if self.span is not None:
            longest, slots = min(longest, self.span + 32), min(slots, self.span // 64 + 2)
        splits = self._piece_splits(rows * cache.k_pages.shape[1], longest)
        if splits == 1 or rows * nq * slots * (d + 2) > self.PIECE_RESULTS:
            return False
        part_o = ctx.scratch("attn_piece_o", (rows * nq * slots, d), torch.float32)        # (rows of the buffer: one, not one for every bound)
        part_ml = ctx.scratch("attn_piece_ml", (rows * nq * slots, 2), torch.float32)
        ops.attention_f32_divided(out, qkv, cache.k_pages, cache.v_pages, group.block_table, ctx.token_slot, ctx.positions, nq, self.scale, self.reach,
                                  splits, slots, part_o, part_ml)
        return True

    def _attend(self, ctx, out, qkv, cache, group, gates=None, **more):
        """Attention by the kernels for any shape and dtype; where tokens can share a workgroup, the single tokens at the head of a
        mixed step (each of a request of its own) go in a launch of their own, so that a prompt's tokens behind them do."""
        singles = 0 if ctx.all_decode else ctx.single_rows
        reach = length_class(ctx.max_k)
        longest = 2 * reach - 1 if reach else ctx.max_k                   # at most; of long contexts their class's, which a shape's steps share
        plain = gates is None and not self.keep_first and not more.get("softcap") and more.get("sinks") is None and more.get("distance") is None
        shares = ops.attention_shares(ctx.dtype, self.num_heads, cache.k_pages.shape[1], self.head_dim, self.value_dim, group.page_size, plain)
        alone = qkv.shape[0] if ctx.all_decode else singles               # rows of a request of their own
        if alone and shares and self._attend_divided(ctx, out[:alone], qkv[:alone], cache, group):
            if alone == qkv.shape[0]:
                return
        elif not singles or not shares:
            ops.attention(out, qkv, cache.k_pages, cache.v_pages, group.block_table, ctx.token_slot, ctx.positions, self.num_heads, self.scale,
                          self.reach, self.keep_first, gates=gates, together=1 if ctx.all_decode else 16, longest=longest, **more)
            return
        else:
            ops.attention(out[:singles], qkv[:singles], cache.k_pages, cache.v_pages, group.block_table, ctx.token_slot, ctx.positions, self.num_heads,
                          self.scale, self.reach, together=1, longest=longest)
        rest = ctx.memo.get("rows_after_singles")
        if rest is None:
            rest = ctx.memo["rows_after_singles"] = (ctx.token_slot[singles:], ctx.positions[singles:])
        ops.attention(out[singles:], qkv[singles:], cache.k_pages, cache.v_pages, group.block_table, *rest, self.num_heads, self.scale, self.reach, together=16,
                      longest=longest)

    def _forward_whole_rows(self, ctx, x, residual, cache, group, cos, sin, then_norm, accumulate):
        """The forms whose heads `qkv_norm_prep` prepares: one product for q, k, v (and the gate), the norms over the whole
        projection, rotation and the write into the pages in one kernel, attention, the gate, the output projection."""
        t, d, dv, nq, nkv = rows_of(x), self.head_dim, self.value_dim, self.num_heads, self.num_kv_heads
        gate_at = (nq + nkv) * d + nkv * dv
        qkv = ctx.scratch("attn_qkvg", (t, self.w_qkv.shape[0]), ctx.dtype)
        linear(ctx, qkv, x, self.w_qkv)
        self.hand_out_carried(ctx, qkv)
        cores = ops.attention_decode_supported(ctx.dtype, nq, nkv, d, group.page_size, dv)
        prepare = None
        if self.heads_as_projected and cores and ctx.all_decode and t <= self.PREPARE_INSIDE_ROWS and dv == d and not self.keep_first:
            prepare = ops.DecodePrepare(None, None, 0.0, None, None, nkv)        # the attention kernel stores the new keys and values
        elif self.heads_as_projected:
            ops.qkv_norm_prep(qkv[:, nq * d:], 0, nkv, d, dv, None, None, 0.0, None, None, cache.k_pages, cache.v_pages, group.slots, group.page_size)
        elif self.unit_after or self.neighbours:
            ops.rotate_unit_prep(qkv, nq, nkv, d, dv, self.qk_norm_eps, self.unit_after, cos, sin, self.neighbours, cache.k_pages, cache.v_pages,
                                 group.slots, group.page_size, bias=self.b_late)
        else:
            first = None if self.value_mix is None else ctx.scratch("attn_first_values", (t, nkv * dv), ctx.dtype)
            ops.qkv_norm_prep(qkv, nq, nkv, d, dv, self.q_norm, self.k_norm, self.qk_norm_eps, cos, sin, cache.k_pages, cache.v_pages,
                              group.slots, group.page_size, bias=self.b_late, temperature=self.query_temperature, positions=ctx.positions,
                              first_values=first, value_mix=self.mix)
        more = {"sinks": self.sinks, "softcap": self.score_cap or 0.0, "distance": self.distance}
        # a gate a head is applied by the attention kernel that finishes a query (or by the merge of its partial results); a
        # gate a value by a kernel of its own behind them
        gates = qkv[:, gate_at:gate_at + nq] if self.output_gate == "head" else None
        out = ctx.scratch("attn_out", (t, nq * dv), ctx.dtype)
        extra = 1 if self.keep_first else 0      # the kept first positions' share is one more partial result for the merge
        if cores and ctx.all_decode:
            longest, bound = ctx.max_k, ctx.max_k_bound
            if self.span is not None:
                longest, bound = min(longest, self.span + 32), min(bound, self.span + 64)
            splits, form = self._decode_shape(t * nkv, longest, bound, group.page_size, d)
            part_o = part_ml = None
            if splits + extra > 1:
                part_o = ctx.scratch("attn_part_o", (t, nq * (splits + extra) * dv), torch.float32)
                part_ml = ctx.scratch("attn_part_ml", (t, nq * (splits + extra) * 2), torch.float32)
            ops.attention_decode(out, qkv, cache.k_pages, cache.v_pages, group.block_table, ctx.token_slot, ctx.positions,
                                 nq, self.scale, self.reach, splits, part_o, part_ml, ctx.max_k_bound, prepare,
                                 form=self._keys_read_once(splits, form, ctx.max_k, group.page_size),
                                 keep_first=self.keep_first, gates=gates, **more)
        elif cores:
            longest = ctx.max_k_bound if self.span is None else min(ctx.max_k_bound, self.span + 64)
            singles = ctx.single_rows
            if singles:
                splits, form = self._decode_shape(singles * nkv, longest, ctx.max_k_bound, group.page_size, d)
                part_o = part_ml = None
                if splits + extra > 1:
                    part_o = ctx.scratch("attn_single_part_o", (singles, nq * (splits + extra) * dv), torch.float32)
                    part_ml = ctx.scratch("attn_single_part_ml", (singles, nq * (splits + extra) * 2), torch.float32)
                ops.attention_decode(out[:singles], qkv[:singles], cache.k_pages, cache.v_pages, group.block_table, ctx.token_slot,
                                     ctx.positions, nq, self.scale, self.reach, splits, part_o, part_ml, ctx.max_k_bound, None,
                                     form=self._keys_read_once(splits, form, ctx.max_k_bound, group.page_size),
                                     keep_first=self.keep_first, gates=None if gates is None else gates[:singles], **more)
            rest = ctx.memo.get("rows_after_singles")
            if rest is None:
                rest = ctx.memo["rows_after_singles"] = (ctx.token_slot[singles:], ctx.positions[singles:])
            paired = self._walks_in_pairs(ctx, nq // nkv, d)
            splits = self._prefill_splits((-(-ctx.num_qblocks // 2) if paired else ctx.num_qblocks) * nkv, longest, (t - singles) * nq * dv,
                                          nq // nkv, t - singles, paired)
            part_o = part_ml = None
            if splits + extra > 1:
                part_o = ctx.scratch("attn_part_o", (t - singles, nq * (splits + extra) * dv), torch.float32)
                part_ml = ctx.scratch("attn_part_ml", (t - singles, nq * (splits + extra) * 2), torch.float32)
            ops.attention_prefill(out[singles:], qkv[singles:], cache.k_pages, cache.v_pages, group.block_table, rest[0], rest[1],
                                  ctx.qblock_token0, ctx.qblock_count, nq, self.scale, self.reach, ctx.max_qblock, ctx.max_k_bound,
                                  splits, part_o, part_ml, None, keep_first=self.keep_first, gates=None if gates is None else gates[singles:],
                                  one_request=paired, **more)
        else:
            self._attend(ctx, out, qkv, cache, group, gates=gates, **more)
        if self.output_gate is True:
            ops.sigmoid_gate(out, qkv[:, gate_at:gate_at + self.gate_width])
        return linear(ctx, residual, out, self.w_o, accumulate=accumulate, then_norm=then_norm)


register("mixer", "gqa_attention", GQAAttention)

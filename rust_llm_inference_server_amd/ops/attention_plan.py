"""Host-side planning of the attention kernels' work for one step.

The step builder knows nothing of these kernels: a mixer that uses them names an
``AttentionPlanner`` as its ``step_planner()``, and the builder carries what ``plan`` returns
(int32 arrays and a few launch sizes) to the device with the rest of the step's metadata.

Every choice here follows from a sequence's *own* lengths and from the constants below, never
from how many other sequences or tiles the batch holds, so that the order of a row's sums (and
with it the rounding of its result) is the same alone and among neighbours:

* a sequence that brings one token is cut into partitions of ``DECODE_PART_KEYS`` keys (a
  multiple of that beyond ``DECODE_MAX_PARTS`` partitions) by the decode kernels themselves;
  the plan only says how deep the grid must be for the longest of them;
* a sequence that brings a portion of a prompt takes tiles of 128 queries where the kernel for whole heads serves it
  (``whole_heads``), or when its own context is long or its own tiles are plenty, else tiles of 64;
* the keys of its tiles are cut into runs (one workgroup each, merged afterwards) when its own
  tiles are too few to fill the chip and its context is long.

The reference cuts decode contexts by a rule of the same kind
(crates/model/src/paged_attention.rs:21-36), though from the batch's longest context."""
from __future__ import annotations

from typing import Any, List, Tuple

import numpy as np

from ..stepplan import HostPlan, StepLengths, StepPlanner

# Keys per partition of a decode context and the most partitions a context is cut into.
DECODE_PART_KEYS = 1024
DECODE_MAX_PARTS = 16
PREFILL_TILE = 64     # new tokens per workgroup of the matrix-core prefill attention
WIDE_TILE = 128       # ... of its form with two query blocks per wave, and of the kernel for whole heads
# Tiles of 128 queries of whole heads of these sizes (attention_prefill.h) are ahead of tiles of 64 at every length (us, 64
# -> 128: 1B shape 2 new tokens 4.7 -> 3.7, on 1,000 cached 18.8 -> 12.5, 17 on 8,000 23.8 -> 20.1, 512 12.2 -> 9.3, 2,048 42
# -> 31; 3B shape 1,024 31.8 -> 24.7, 464 on 2,000 49 -> 34.7; one portion of 2 to 100 tokens on 0 to 8,000 0.64 to 0.87,
# batches of 8, 32 and 63 portions of 2 to 64 tokens 0.63 to 0.99, but 63 of 2 to 17 tokens on 500 of 24 heads of 128
# 1.04 to 1.06: a rule on a sequence's own lengths does not see the others).
WHOLE_HEADS = (64, 128)
# Their keys are walked by two groups of waves in turn where a sequence makes at most this many workgroups, by head size,
# and has this many positions (us, one group -> two: heads of 64, 16 x 32 workgroups 36.6 -> 31.3, 8 x 32 19.6 -> 16.9, 4 x 32 x 6
# runs 58.3 -> 57.0, 64 x 32 314 -> 320, three prompts of up to 190 tokens 5.85 -> 6.23; heads of 128, 8 x 24 28.3 -> 24.3, 4 x
# 24 x 2 runs 39.6 -> 34.4, 4 x 32 x 4 runs 88.3 -> 93.1, 16 x 32 53.0 -> 57.8, 64 x 32 547 -> 584).
SHARED_KEYS_MAX_GROUPS = {64: 512, 128: 256}
SHARED_KEYS_MIN_CONTEXT = 256
# Otherwise a sequence takes tiles of 128 queries when they make this many workgroups (tiles x heads; 5/3
# as many up to head size 64), or when its context is long (4096 positions after the step, or
# 2048 cached ones); 1 << 30: never.
PREFILL_WIDE_MIN_GROUPS = 768
# A sequence whose tiles make at most this many workgroups has the keys of its tiles cut into
# runs: as many as keep the compute units' resident workgroups busy, with at least
# PREFILL_SPLIT_MIN_KEYS keys a run and at most PREFILL_MAX_RUNS runs (0 units: never).
PREFILL_SPLIT_UNITS = 256
PREFILL_SPLIT_MIN_KEYS = 1024
PREFILL_MAX_RUNS = 16


def decode_parts(context: int, window: int = 0) -> int:
    """Live partitions of a decode context of ``context`` positions (what the kernels'
    ``decode_part_len`` gives); with a window only its keys count (rounded as the matrix-core
    kernel rounds their start, down to a multiple of 32)."""
    lo = max(0, context - window) if window else 0
    n = context - (lo & ~31)
    span = DECODE_PART_KEYS * DECODE_MAX_PARTS
    part = DECODE_PART_KEYS * max(1, -(-n // span))
    return max(1, -(-n // part))


def decode_depth(max_context: int) -> int:
    """Grid depth (and stride of the partial results) that covers every context up to
    ``max_context``."""
    return max(1, min(DECODE_MAX_PARTS, -(-max_context // DECODE_PART_KEYS)))


def decode_walk_room(group: int, head_dim: int) -> int:
    """Partitions whose parked sums (eight waves, ``group`` heads, ``head_dim`` + 2 floats) a
    decode workgroup has LDS for: 64 KB up to head size 64, where two workgroups share a compute
    unit's 160 KB, 159 KB beyond, where a compute unit holds one."""
    lds = 64 * 1024 if head_dim <= 64 else 159 * 1024
    return lds // (8 * group * (head_dim + 2) * 4)


def decode_shares(num_seqs: int, num_kv_heads: int, depth: int, group: int, head_dim: int,
                  compute_units: int) -> Tuple[int, int]:
    """(groups, cap) for the matrix-core decode kernel under a grid ``depth`` partitions deep:
    a sequence's partitions are dealt out evenly to ``groups`` workgroups, none of which takes
    more than ``cap`` (a sequence with more partitions than that gets more workgroups); cap 1:
    a workgroup per partition.  This is the one choice here that looks at the batch, and it
    may: the partitions and the order of their sums stay what a sequence's own length makes
    them, only the workgroups that share them change, and the kernel gives the same floats
    however they are dealt out.  Sequences times KV heads that fill the compute units by
    themselves take one workgroup each; fewer take as many each as bring them to about what the
    compute units hold at once (two workgroups each up to head size 64, one beyond).  The
    eight waves' sums of every partition in a share must fit the LDS (``decode_walk_room``),
    and the kernel takes shares of whole pairs of chunks only (partitions of a multiple of 512
    keys)."""
    if depth <= 1 or DECODE_PART_KEYS % 512 != 0:
        return depth, 1
    resident = 2 if head_dim <= 64 else 1
    each = max(1, compute_units * resident // max(1, num_seqs * num_kv_heads))
    groups = min(depth, each)
    cap = min(decode_walk_room(group, head_dim), -(-depth // groups))
    return (groups, cap) if cap > 1 else (depth, 1)


class AttentionPlanner(StepPlanner):
    """Plans for ``ops.paged_attention`` with ``num_heads`` query heads of ``head_dim``.

    ``matrix``: the batch can take the matrix-core kernels (bfloat16, head size in steps of 16
    up to 256); without it only the depth of the decode grid is planned.  ``singles_apart``:
    sequences that bring one token beside portions of prompts take the decode kernel (they
    lead the step); otherwise they get tiles like everyone else.  ``span``: the most keys one
    query sees (chunked attention), 0: all earlier ones; work that cannot be is not cut into
    pieces.  ``whole_heads`` (set by a mixer that knows): queries see every earlier key and scores are only scaled,
    which with pages of 16 positions and more and heads of ``WHOLE_HEADS`` dims the kernel for whole heads takes."""

    whole_heads = False

    def __init__(self, num_heads: int, num_kv_heads: int, head_dim: int, matrix: bool = True,
                 singles_apart: bool = True, span: int = 0):
        self.span = int(span)
        self.nh, self.nkv, self.d = int(num_heads), int(num_kv_heads), int(head_dim)
        self.matrix = bool(matrix) and self.d % 16 == 0 and self.d <= 256
        g = self.nh // max(1, self.nkv)
        # what the matrix-core decode kernel takes: at most 16 query heads per KV head, whose
        # merge buffer fits the LDS
        self.singles_apart = (bool(singles_apart) and self.matrix and g <= 16
                              and g * (self.d + 2) * 32 <= 65536)

    def key(self) -> Any:
        return ("attention", self.nh, self.nkv, self.d, self.matrix, self.singles_apart, self.span,
                self.whole_heads)

    def _reach(self, context: int) -> int:
        """Keys that a decoded token of ``context`` positions may walk (the matrix-core kernel
        starts at a multiple of 32)."""
        return min(context, self.span + 31) if self.span else context

    @staticmethod
    def pages_fit(page_size: int) -> bool:
        """Page sizes the matrix-core kernels take: powers of two from 8 on."""
        return page_size >= 8 and page_size & (page_size - 1) == 0

    # ------------------------------------------------------------------ per sequence
    def tile_queries(self, cached: int, new: int, page_size: int = 0) -> int:
        """64 or 128: the tile form of a sequence with ``cached`` positions and ``new`` tokens."""
        if self.d > 128 or PREFILL_WIDE_MIN_GROUPS >= (1 << 30):
            return PREFILL_TILE
        if self.whole_heads and not self.span and self.d in WHOLE_HEADS and page_size >= 16:
            return WIDE_TILE
        cached = min(cached, self.span) if self.span else cached
        groups = -(-new // WIDE_TILE) * self.nh
        enough = PREFILL_WIDE_MIN_GROUPS if self.d > 64 else PREFILL_WIDE_MIN_GROUPS * 5 // 3
        if groups >= enough or cached + new >= 4096 or cached >= 2048:
            return WIDE_TILE
        return PREFILL_TILE

    def key_groups(self, new: int, context: int, runs: int, page_size: int) -> int:
        """Groups of waves that share the keys of a tile of 128 queries (the kernel for whole heads)."""
        if not (self.whole_heads and not self.span and page_size >= 16):
            return 1
        groups = -(-new // WIDE_TILE) * self.nh * runs
        return 2 if groups <= SHARED_KEYS_MAX_GROUPS.get(self.d, 0) and context >= SHARED_KEYS_MIN_CONTEXT else 1

    def key_runs(self, cached: int, new: int, tile: int) -> int:
        """Runs the keys of this sequence's tiles are cut into (1: none)."""
        cached = min(cached, self.span) if self.span else cached
        groups = -(-new // tile) * self.nh
        if PREFILL_SPLIT_UNITS <= 0 or groups > PREFILL_SPLIT_UNITS:
            return 1
        # resident workgroups per compute unit: 4 up to head size 64, 3 with tiles of 128
        # queries, 2 beyond (of the general form; the kernel for whole heads has 4 and 2, half of
        # that where two groups of waves share keys, and takes these numbers as they are)
        resident = 2 if self.d > 64 else (3 if tile == WIDE_TILE else 4)
        return max(1, min(PREFILL_SPLIT_UNITS * resident // groups,
                          (cached + new) // PREFILL_SPLIT_MIN_KEYS, PREFILL_MAX_RUNS))

    # ----------------------------------------------------------------------- a step
    def plan(self, lengths: StepLengths) -> HostPlan:
        start = np.asarray(lengths.start, dtype=np.int64)
        new = np.asarray(lengths.new, dtype=np.int64)
        S = len(new)
        matrix = self.matrix and self.pages_fit(lengths.page_size)
        all_single = lengths.num_single == S
        singles = lengths.num_single if (self.singles_apart and matrix) or all_single else 0
        runs = np.ones(S, dtype=np.int32)
        units: dict = {"units64": [], "units128": [], "units128x2": []}
        for s in range(singles if matrix else S, S):
            c, n = int(start[s]), int(new[s])
            tile = self.tile_queries(c, n, lengths.page_size)
            r = self.key_runs(c, n, tile)
            runs[s] = r
            qb = np.arange(0, n, tile, dtype=np.int64)
            keys = c + np.minimum(n, qb + tile)                # keys a tile walks
            if self.span:
                keys = np.minimum(keys, (c + qb) % self.span + tile)
            u = np.empty((len(qb), r, 5), dtype=np.int64)
            u[:, :, 0] = s
            u[:, :, 1] = qb[:, None]
            u[:, :, 2] = np.arange(r)[None, :]
            u[:, :, 3] = r
            u[:, :, 4] = (keys[:, None] + r - 1) // r          # work of a unit
            name = "units64" if tile == PREFILL_TILE else \
                "units128x2" if self.key_groups(n, c + n, r, lengths.page_size) == 2 else "units128"
            units[name].append(u.reshape(-1, 5))
        arrays, values = {"seq_runs": runs}, {}
        for name, listed in units.items():
            if listed:
                u = np.concatenate(listed)
                u = u[np.argsort(-u[:, 4], kind="stable")]     # longest first
                arrays[name] = u[:, :4].astype(np.int32).reshape(-1)
                values["num_" + name] = len(u)
            else:
                arrays[name] = np.zeros(0, dtype=np.int32)
                values["num_" + name] = 0
        values["max_runs"] = int(runs.max()) if S else 1
        values["tile_row0"] = int(new[:singles].sum())         # rows before the tiles' rows
        values["num_decode"] = singles
        ctx = start + new
        values["decode_depth"] = decode_depth(self._reach(int(ctx[:singles].max()))
                                              if singles else 1)
        return HostPlan(arrays, values)

    def plan_captured(self, num_seqs: int, max_context: int, page_size: int) -> HostPlan:
        return HostPlan({}, {"decode_depth": decode_depth(self._reach(max_context)),
                             "num_decode": num_seqs,
                             "max_runs": 1, "tile_row0": num_seqs, "num_units64": 0,
                             "num_units128": 0, "num_units128x2": 0})


def plan_for(lens_cached: List[int], lens_new: List[int], planner: AttentionPlanner,
             page_size: int) -> Tuple[HostPlan, StepLengths]:
    """The plan of a batch given as plain lists, single tokens first (for tests and probes)."""
    num_single = 0
    for n in lens_new:
        if n != 1:
            break
        num_single += 1
    lengths = StepLengths(np.asarray(lens_cached, dtype=np.int64),
                          np.asarray(lens_new, dtype=np.int64), num_single, page_size)
    return planner.plan(lengths), lengths

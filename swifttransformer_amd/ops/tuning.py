"""Thresholds that were fitted by measurement, in one place.

None of them decides whether a result is right: each chooses between two kernels, or two shapes
of one kernel, that compute the same thing.  They were fitted on an MI355X (256 compute units)
at the layer sizes named beside them, and a sweep over other sizes has already moved some of
them once; on another device or model family they are the first thing to measure again.  The
parts read them from ``tuning`` when they run, so changing a field takes effect at the next step
(steps recorded before keep the shapes they were recorded with).

The thresholds that live in the kernel library have setters of the same kind:
``ops.kernels.gemm_library_rule`` (from how many rows, and for how large and deep a matrix, a
product goes to the vendor library) and ``ops.kernels.gemm_wide_workgroups``."""
from __future__ import annotations

from dataclasses import dataclass


@dataclass
class Tuning:
    # A product takes the norm of its input rows as its prologue (instead of a norm kernel before
    # it) up to this many rows and this width.  Every workgroup of such a product normalises all
    # rows again, so the kernel it saves is paid back as rows and width grow.  Recorded decode
    # steps of 24 layers: at width 2048 the fused form wins up to the 16 rows the product kernel
    # takes (14 rows: 6,710 tokens/s against 6,390; 16 rows: 7,150 against 7,050); at width 4096
    # it loses at every row count (a layer at 8 rows: 169 us fused against 155 us).
    fused_norm_max_rows: int = 16
    fused_norm_max_width: int = 2048
    # The decode attention splits a row's keys over workgroups until there is a workgroup for
    # every compute unit, at least this many keys a split (two workgroups a unit were 0-2 %
    # slower at batch 2 to 12, OPT-1.3B sizes).
    min_keys_per_split: int = 256
    # Decode steps of requests with contexts of up to this many tokens have recordings of their own, in which few rows' keys are split
    # less than in those for all contexts.  What a mixer does with them is its own rule (``PagedAttention._short_splits`` and the
    # ``_splits`` of the others).  Whole steps of four layers, us, for all contexts and for short ones, at 30 and at 185 tokens: one request,
    # opt-125m 132 -> 125, 132 -> 130; gisedra-125m (shared entries of 160, window) 359 -> 356, 367 -> 363; zimorax-1.3b (sinks) 469 ->
    # 453, 476 -> 461; pupalix-125m 278 -> 254, 278 -> 265; four, gisedra-1.3b 720 -> 691, 735 -> 711; eight, fefozen-125m (gated
    # latent) 206 -> 201, 205 -> 202.  Whole keys and splits that the output projection merges meet at about 200 (heads of 64).
    short_span: int = 192
    # A step that is not plain decoding is recorded when its shape comes up for this many-th time.
    record_after: int = 2
    # Recordings of up to this many rows have the vendor library's kernels timed (20 to 100 ms a
    # product shape, once).  Up to 256 rows the fastest candidate is 10 to 25 % ahead of the
    # library's first suggestion at the OPT-1.3B sizes (a layer's four products: 92 -> 76 us at 256
    # rows) and within 3 % beyond; at the 13B sizes the first suggestion is off at prompt sizes too
    # (FC2 at 512 rows 202 -> 156 us, FC1 at 2,048 rows 465 -> 365 us: a layer 8 to 10 % faster),
    # so every recording times them.
    tune_products_up_to_rows: int = 1 << 20
    # Key channels a wave of the gated-linear-attention scan takes (4, 8 or 16): in steps of single
    # tokens, where the requests are many and the states' traffic counts, and in steps with prompt
    # portions, where a portion's tokens come one after the other and more parts a head are more
    # compute units at work on them (every part writes a plane of partial results, which the head
    # norm sums).
    gla_part_dim_decode: int = 16
    gla_part_dim_prompt: int = 8
    # Pairs an expert from which bfloat16 experts go in tiles of 64 and of 128 places through LDS instead of 16 (csrc/moe.hip).  All
    # kernels of a call with tiles of 16 / 64 / 128 places, us: 64 experts of 2,048 x 1,024, four a token, 188 / 171 / 177 at 6 pairs an
    # expert, 374 / 182 / 188 at 31, 1,092 / 258 / 226 at 100, 1,173 / 276 / 265 at 112; 8 of 4,096 x 4,096, two a token, 181 / 176 / 204
    # at 6, 445 / 180 / 205 at 31, 1,105 / 231 / 221 at 100, 1,138 / 274 / 271 at 112; 16 of 2,048 x 2,048, two a token, 100 / 94 / 109 at
    # 6, 376 / 124 / 116 at 64, 592 / 129 / 123 at 112, - / 197 / 166 at 200; of 1,024 x 1,024 37 / 36 / 45 at 6, 164 / 47 / 57 at 112, - / 70 / 63
    # at 200; of 768 x 768 30 / 31 / 35 at 6, 106 / 42 / 47 at 112, - / 56 / 52 at 200; 8 of 768 x 768 23 / 28 / 33 at 6, 29 / 30 / 34 at 20, 61 /
    # 32 / 42 at 112, - / 39 / 44 at 200.  How large the matrices are moves the lines: tiles of 64 win from 4 to 20 pairs on, of 128 from 64 to
    # 200 and more.
    moe_staged_64_pairs: int = 7
    moe_staged_128_pairs: int = 112
    # Window attention of bfloat16 rows goes by tiles of 16 rows from so many rows of a step on (csrc/sink_tiles.hip), by rows below.
    # 32 heads of 64 on 8 key heads, window 1,024, by rows and by tiles in us, mixed and not: a prompt of 64 rows 28 and 29, 24 and 13;
    # of 128 28 and 35, 24 and 25; of 256 72 and 37, 60 and 27.  Beside single tokens of 900 keys a row costs more by rows than a whole
    # tile: 64 and a portion of 64 173 and 89, 148 and 52; 100 and 28 173 and 133, 149 and 78.  At 60 keys the same 100 and 28 take 27
    # and 34, 24 and 24: what the kernel for rows gains there is less than what it loses at long contexts, which a recorded step's host
    # does not see.
    sink_tiles_rows: int = 128
    # The additive recurrence of heads with more than 64 key channels goes by chunks from so many rows on, and so many more for
    # each item of the step (figures beside csrc/state_chunks.hip: 32 heads of 128 x 128, one prompt of 64 rows 38 us row by row
    # and 43 by chunks, 96 rows 52 and 44; 104 rows beside 24 single ones 78 and 83, 200 rows 100 and 86).
    state_chunks_wide_rows: int = 80
    state_chunks_wide_rows_per_item: int = 4


tuning = Tuning()

"""Flattened strategy / placement encoding: the object graph
``dict[Node, OpStrategy] -> OpSpec -> DTensorSpec`` that the reference walks in
``ShardingOptimizer.build_ds`` (autoparallel/optimize_sharding.py:270-380; types at
torch/distributed/tensor/_op_schema.py:94-141) laid out as CSR arrays over tensors,
specs, strategies, edges and entries, ready to sit in HBM.

Layout
------
tensor table   one row per distinct (shape, stride, dtype): ``tensor_rank``,
               ``tensor_itemsize``, ``tensor_shape[T, 8]``, ``tensor_stride[T, 8]``.
spec table     one row per DTensorSpec occurrence: ``spec_codes`` (uint32, byte i =
               placement code of mesh dim i) and ``spec_tensor`` (row of the tensor
               table, -1 for "not a DTensorSpec": ``None`` outputs, scalars).
strategy table one row per (node, strategy): ``strat_flops``, ``strat_rw_bytes``,
               ``strat_dtype``, ``strat_zero_cost``, ``strat_num_args``;
               ``node_strat_begin[N + 1]`` is its CSR pointer.
edge table     one row per (consumer node, argument): producer output specs are spec
               rows ``[edge_src_begin, +edge_n_src)``, consumer input specs are
               ``[edge_tgt_begin, +edge_n_tgt)``; the edge's cost matrix occupies
               entries ``[edge_entry_begin[e], edge_entry_begin[e + 1])``, row-major by
               consumer strategy (= ``redistribute_cost[argi][ii]`` of strategy ``ss``).
pt_values      rule-provided costs that survive where either side is not a
               DTensorSpec (optimize_sharding.py:336-355).
tiles          rectangles of edge matrices, one per workgroup.

Placement codes: 0x00 Replicate; 0x40|op Partial(op) (op 0 = sum); 0x80|v<<4|d Shard(d)
with v a variant id (0 = plain ``Shard``).
"""

from __future__ import annotations

from dataclasses import dataclass, fields
from typing import Optional

import numpy as np

from . import _native
from ._native import APC_MAX_RANK, APC_PACKED_MAX_DUPS, APC_TILE_MAX_COLS, APC_TILE_MAX_DUPS, APC_TILE_MAX_ROWS

REPLICATE = 0x00
PARTIAL_SUM = 0x40
KIND_REPLICATE, KIND_PARTIAL, KIND_SHARD = 0, 1, 2

# reduce ops of Partial; index = code payload
PARTIAL_OPS = ("sum", "avg", "min", "max", "product", "band", "bor", "bxor")

EDGE_GRAD_RESCALE = _native.EDGE_GRAD_RESCALE
EDGE_NO_PRODUCER = _native.EDGE_NO_PRODUCER

# Tiling chosen when the caller names no tile size (measured on one MI355X).  Identical edges: as many copies
# per tiled edge as leave at most AUTO_MAX_STORED_PER_TILE values for a tile to store, in small tiles: a
# value computed once is stored to all copies, and a long workgroup is the launch's tail.  66 M entries on (8, 8, 8),
# 80 layers, tile of about 512 entries and 8 copies (3 236 values) 131 us; 2048 / 4 137, 4096 / 4 145, 512 / 4 145, 512 / 16
# (6 472 values) 161, 4096 / 16 195.  11 M on (32, 8), 40 layers: 512 / 8 (2 638 values) 26.6, 1024 / 8 27.3, 512 / 16 27.0,
# 512 / 4 36.5, 2048 / 2 53.9; Llama-3-70B on (8, 8, 8), 73 M entries: 512 / 8 (3 638 values) 124, 512 / 4 133, 2048 / 4 126;
# 6 M on (8, 8, 8), 10 layers: 512 / 16 (3 500) 18.2, 512 / 8 23.9, 2048 / 2 34.5 us.  The line lies where large tables have
# it; tables of up to 14 M entries would gain above it: 16 / 8 copies, 10 M, 48 strategies at most, 4 603 / 2 301 values 22.4 /
# 24.1, 14 M 5 936 / 2 968 values 28.4 / 28.9 us.
# Few or no copies: larger tiles, until one stores AUTO_MIN_STORED_PER_TILE (its specs and cost terms are staged once).
# Tiles of 1024 / 2048 / 4096 entries, no edge like another, the matrices alone: 5.5 M entries on (32, 8) 29.4 / 29.7 (869
# values) / 33.6 us, on (16, 8, 4) 25.5 / 24.0 / 27.1; 21 M 78 / 77 / 84, 64 / 60 / 62.  (Where the tiles take the row minima
# too, as they do of the 5.5 M, 1024 are faster: 45.1 / 48.4 / 57.2.)
# With more than AUTO_MANY_TILES of those tiles there are workgroups for the chip however large they are, and the largest
# win: tiles of 2048 / 4096 entries, 59 M entries (70 662 / 61 636 tiles) on (32, 8) 202 / 205, on (16, 8, 4) 183 / 182 us;
# 123 M (145 062 tiles of 2048) 404 / 402, 367 / 364; 228 M 722 / 713, 659 / 648; 464 M on (16, 8, 4) 1263 / 1228.
AUTO_MIN_TILE_ENTRIES = 512
AUTO_MIN_STORED_PER_TILE = 800
AUTO_MAX_STORED_PER_TILE = 4000
AUTO_MANY_TILES = 100_000
# Tiles in the order of their size, the largest first: the launch ends with short workgroups instead of whichever edge is
# last.  Neighbouring tiles then meet a line of the output between them from different dies at different times, and beyond
# the caches every such line is written twice in part: what that costs goes by stored bytes, so not for tables with
# many copies or many entries, and not where a tile is less than a pass of a wavefront anyway.  us a pass, edge by edge / by size: 6.1 M
# entries on (64, 4) 36.5 / 30.0, 5.2 M on (12, 6) 36.2 / 28.1, 5.3 M on (2, 4, 2, 2) 39.4 / 31.6, 2.6 M on (12, 6) 13.5 / 12.7,
# 488 k, packed, 17.6 / 16.5, 587 k on (6, 4, 2) 15.2 / 14.3, 20 M on (16, 8, 4) 69.8 / 64.2, 27 M 88 / 83; two layers 23.7 /
# 21.7, four layers 19.0 / 18.6; the other way: 39 M entries 111 / 122, six layers 14.6 / 15.1, nineteen 18.5 / 19.2, 73 M in
# eighty 127 / 204; 30 entries a tile 14.8 / 15.9.
ORDERED_MAX_ENTRIES = 32_000_000
ORDERED_MAX_COPIES = 4
ORDERED_MIN_PER_TILE = 64
# Their largest tiles are no tail, and may be larger than AUTO_MIN_STORED_PER_TILE would have them: 2048 / 4096 entries, 20 M on
# (16, 8, 4) 66.5 (924 values) / 63.9 us, on (64, 4) 63.4 / 66.9, 30 M 92.1 (928) / 86.6 and 90.2 / 84.3, 14 M 59.6 (934) / 57.0 and
# 57.0 / 53.8, 5.2 M 25.0 (952) / 23.6 and 22.5 / 23.8, on (2, 4, 2, 2) 27.5 / 26.8; 1024 / 2048 / 4096, 5.3 M in two layers on (64, 4)
# 21.7 (960) / 20.9 (1 240) / 24.1.  (While there are tiles for more than a round or two.)  Only in that order: the same tables edge by
# edge, which is how one that is launched once goes, 71.5 / 78.4 us, 70.0 / 76.2, 94.1 / 98.2, 93.1 / 96.6, 64.2 / 64.9, 62.1 / 63.7,
# 29.8 / 33.9, 27.8 / 31.6, 34.0 / 39.9, with all three arrays written 95.9 / 103.7, 93.8 / 102.8 and so on; the planner's one launch, on
# what has just been uploaded, 5.2 M 42.2 / 46.1, 40.0 / 45.0 and on (8, 8, 8) 42.4 / 46.9, 20 M 67.7 / 74.7, 69.2 / 76.6, 74.2 / 78.6, 14 M
# 75.7 / 77.9, 72.9 / 73.3, 75.7 / 77.4; the other way 9.4 M, 61.9 / 61.0, 59.3 / 58.1, 63.1 / 61.1.
ORDERED_MIN_STORED_PER_TILE, ORDERED_SOME_ROUNDS = 1000, 4000
# A table this small is bound by the latency of one workgroup, not by work: it keeps the largest
# tiles and up to 16 copies per tiled edge (Llama-3-8B on (32, 8), 1.8 M entries: 13.3 us with
# 840 tiles of 16 copies against 14.6 us with 1 616 tiles of 8 and 17.7 us with 3 168 of 4).
AUTO_SMALL_TABLE_ENTRIES = 4_000_000
# ... over packed tiles, where it is all copies or next to nothing to compute.  A packed tile costs a record of 2.7 KB from
# memory and evaluates every entry directly; a staged tile evaluates the terms once and looks them up, and where there are no copies
# to store wins from the second round of workgroups on.  Whole pass, packed (tiles of four rows per wavefront) / staged, us:
#   computed entries, no copies, from STAGED_MIN_COMPUTED: 366 k in 7 884 tiles on (32, 8) 16.9 / 11.4, 149 k 6.8 / 5.6, 54 k 4.9 / 4.4,
#   409 k on (8, 8, 8) 16.0 / 10.0, 53 k 6.3 / 5.5, 836 k on (2, 4, 2, 2) 34.2 / 14.8, 337 k on (6, 4, 2) 15.8 / 12.1; about equal at
#   46 k 4.4 / 4.4, 4 copies of 54 k 5.2 / 5.1; the other way 26 k 4.9 / 5.2, 19 k 4.0 / 4.3, 13 k 3.9 / 4.3, 2 k 3.6 / 4.2;
#   more than STAGED_MANY_EDGES tiled edges, on meshes of one or two dims of at most STAGED_MAX_STORED_PER_EDGE values with their copies (the round of packed workgroups behind the first costs more on meshes of more
#   dims: the line lies where it does on those of one): on (6,) 11 k in 2 025 4.8 / 5.0, 4 copies 5.5 / 5.4, 16 7.3 / 7.5, 20 k in 3 353 6.6 / 6.1, 24 k in
#   4 080 7.6 / 6.3, on (64,) 15 k in 2 906 6.3 / 5.5, 16 copies 9.1 / 7.8, on (32, 8) 16 k in 2 027 5.4 / 5.0, 16 copies 7.7 / 7.2, 28 k in 3 354 7.2 / 6.3, on
#   (8, 8, 8) 16 k in 2 030 6.0 / 5.3, 8 copies 7.1 / 6.2, on (2, 4, 2, 2) 7.0 / 5.3; the other way 5 copies of 34 k in 2 244 on (6,) 5.6 / 6.1, 337
#   values each in 2 582 on (32, 8) 8.4 / 8.9, on (12, 6) 9.1 / 9.8, 449 9.1 / 9.8 and 9.6 / 10.6, 310 in 4 478 12.0 / 12.6 and 12.8 / 13.7 (on (8, 8, 8) 337 in 2 582
#   9.9 / 8.9, on (2, 4, 2, 2) 12.1 / 9.6);
#   more than STAGED_MAX_COPIES copies: 8 of 54 k in 474 5.6 / 6.1, 16 7.0 / 8.5, 16 of 109 k on (32, 8) 8.4 / 10.3, 10 of 119 k on
#   (8, 8, 8) 7.6 / 8.7; then staged from this many computed entries on, in tiles that hold this many each, as (measured before the staging
#   got cheaper) 901 k on (32, 8) 23.2 / 15.5, on (8, 8, 8) 28.4 / 14.7, 575 k 18.4 / 15.5, 190 k on (8, 8, 8) 9.1 / 7.1;
#   a 3-D mesh with a size that is no power of two, whose 72 states a tile stages, from STAGED_MIN_PER_EDGE_OF_STATES computed entries a tiled edge
#   on: (6, 4, 2), 37 in 1 981 7.3 / 6.3, 38 in 4 857 13.5 / 11.6, 36 in 901 5.7 / 5.6; the other way 22 in 3 312 9.1 / 9.3, 4 copies 9.6 / 10.2, 14 in
#   4 885 11.3 / 11.5, 8 in 3 357 8.7 / 9.2, 4 copies 9.2 / 9.9 (on (3, 8), whose tiles stage less, 22 in 3 311 8.2 / 7.2, 14 in 4 884 10.1 / 8.2);
#   a 4-D mesh with a size that is no power of two, whose states cost most to stage, by the last line alone: 430 k in tiles of 91 entries
#   25.0 / 25.7, 149 k of 94 11.3 / 11.6, 81 k of 17 15.7 / 25.2.
STAGED_MIN_COMPUTED, STAGED_MAX_COPIES, STAGED_MANY_EDGES, STAGED_MIN_PER_EDGE_OF_STATES = 40_000, 6, 2048, 30
STAGED_MAX_STORED_PER_EDGE = 304
# Packed tiles of few entries.  A workgroup of four wavefronts a tile (256 lanes) leaves lanes idle where the rows of every tile are
# evaluated at once by fewer: then 64, and from more than PACKED_MANY_TILES on, where at most PACKED_MAX_SMALL_COPIES values are stored for one
# computed, 32 or 16.  us, 256 / 64 / 32 / 16 lanes: tiles of at most 16 entries, 436 on (64,) 3.3 / 3.4 / 3.7 / 3.6, 1 928 4.7 / 3.7 / 3.8 / 3.8,
# 2 906 6.2 / 4.2 / 4.2 / 3.7, 3 488 in two layers on (6,) 7.1 / 5.2 / 4.7 / 4.0, 3 158 of nine copies 7.5 / 5.9 / - / 6.3, 926 of sixteen 5.7 / 5.2 / 6.0 / 6.0; of at
# most 25, 1 446 on (16, 8, 4) 5.1 / 4.4 / 4.4, 4 644 10.8 / 8.0 / 6.4, 4 693 on (3, 2, 2, 2) 15.1 / 11.4 / 9.5, 2 596 of twenty copies on (3, 8) 8.1 / 7.0 / 7.4; of
# at most 64, 944 of sixteen copies on (32, 8) 5.9 / 5.3, 4 297 on (8, 8, 8) 10.0 / 7.8, 5 571 on (3, 2, 2, 2) 17.2 / 12.8.  Where a wavefront
# goes over its tile twice it loses (944 tiles of at most 81 entries on (32, 8) 6.1 / 6.9, 4 297 of 100 9.3 / 8.0 with 7.3 staged), except on
# meshes whose states are staged one by one, for tables that go over packed tiles anyway (2 910 of at most 100 on (3, 2, 2, 2) 11.9 / 10.1, 3 720 of 81 on (6, 4, 2)
# 12.2 / 11.1).
# (A launch of 256 lanes a tile runs at one of two speeds from process to process, one of 64 at one in between or as fast: 436 tiles on (64,) 3.3 or 4.2 /
# 3.3 or 3.75, 126 of eleven copies on (6, 4, 2) 4.5 or 5.0 / 4.7.)
# They beat staged tiles (same cases: 5.4 / 3.7 for 2 906 tiles of 16 entries, 7.3 / 6.4 for 4 644 of 25, 7.4 / 6.0 for 2 188 of 64 and ten copies, 12.7 / 9.7
# for 5 571 of 64 on (6, 4, 2)) except, with 64 lanes, PACKED_MANY_TILES_OF_64 and more without copies on power-of-two meshes of
# three dims or four (staged / packed: 2 910 6.2 / 6.1 on (2, 4, 2, 2), 5.9 / 5.4 on (16, 8, 4); then 4 297 7.3 / 7.8 on (8, 8, 8), 7.5 / 9.3 on (2, 4, 2, 2)).
PACKED_MANY_TILES, PACKED_MAX_SMALL_COPIES, PACKED_MANY_TILES_OF_64 = 2048, 4, 3072
STAGED_MIN_COMPUTED_OF_COPIES, STAGED_MIN_COMPUTED_PER_TILE = 150_000, {1: 100, 2: 100, 3: 100, 4: 180}
# Its tiles are cut until there are this many: enough workgroups for the chip, few enough stagings.  But no smaller than what
# a STAGED_SMALLEST_SHARE-th of the entries to compute is (its power of two), at least 512: a launch is as long as its largest tile, and larger
# tables last longer.  Tiles of about 512 / 1024 / 2048 / 4096 entries, by size:
# 399 k entries on (8, 8, 8) 6.6 (1 181 tiles) / 6.7 / 7.7 / 8.4 us, 850 k 9.4 / 8.6 / 8.7 (1 270 tiles) / 9.3; 420 k on
# (12, 6) 7.0 (1 265) / 7.1 / 7.9 / 8.3, 2.6 M 15.2 / 12.5 / 11.6 (2 431) / 11.9; 1.6 M on (32, 8) 16.2 / 13.6 / 13.5 (2 718) /
# 13.3, on (6, 4, 2), without the minima, 2048 (2 930) 13.7, 4096 14.4; 587 k in 3 353 edges on (6, 4, 2) 14.8 (3 500) / 14.3.
# Edge by edge they lose little where they lose: 512 / 1024, 1.1 M on (12, 6) 11.2 / 11.3, on (32, 8) 10.7 / 11.2, on (6, 4, 2) 13.6 /
# 12.3, 1.3 M 10.2 / 9.2, 9.6 / 9.1, 11.7 / 10.2; 1024 / 2048, 2.6 M on (12, 6) 12.7 / 13.8.
STAGED_TILES, STAGED_SMALLEST_SHARE, STAGED_MIN_TILE_ENTRIES = 2800, 750, 512
# On a 4-D mesh with a size that is no power of two a tile stages 304 states: fewer, larger tiles.  On both sides of the
# 900, with row minima in the tiles: (3, 2, 2, 2), 530 k entries, whole edges (979 tiles) 19.4, 1024 17.5; 1.8 M, 39.8, 41.7; 658 k
# (676 whole) 1024 18.3, 2048 16.6, 4096 20.2; 900 k 512 27.5, 1024 20.4, 4096 (1 230) 18.8.
STAGED_TILES_OF_MANY_STATES, STAGED_MIN_TILE_ENTRIES_OF_MANY_STATES = 900, 1024

# numpy mirror of the C struct apc_tile (64 bytes)
TILE_DTYPE = np.dtype([
    ("edge", "<i4"), ("row_begin", "<i4"), ("col_begin", "<i4"), ("counts", "<i4"),
    ("src_begin", "<i4"), ("n_src", "<i4"), ("tgt_begin", "<i4"), ("flags", "<i4"), ("strat_begin", "<i4"),
    ("tensor", "<i4"), ("entry_begin", "<i8"), ("pt_begin", "<i8"), ("dup_begin", "<i4"), ("dup_count", "<i4"),
])
assert TILE_DTYPE.itemsize == 64


# numpy mirror of the C struct apc_packed_tile: everything one tile reads, in one record
PACKED_MIXED = 0x100
PACKED_TILE_DTYPE = np.dtype([
    ("rows", "<i4"), ("cols", "<i4"), ("flags", "<i4"), ("dup_count", "<i4"), ("tensor", "<i4"), ("tensor_rank", "<i4"),
    ("tensor_itemsize", "<i4"), ("edge", "<i4"), ("entry_begin", "<i8"), ("row_begin", "<i8"), ("pt_begin", "<i8"),
    ("reserved", "<i8"), ("tensor_shape", "<i8", (APC_MAX_RANK,)), ("tensor_stride", "<i8", (APC_MAX_RANK,)),
    ("dup_entry_begin", "<i8", (APC_PACKED_MAX_DUPS,)), ("dup_row_begin", "<i8", (APC_PACKED_MAX_DUPS,)),
    ("col_codes", "<u4", (APC_TILE_MAX_COLS,)), ("col_tensor", "<i4", (APC_TILE_MAX_COLS,)),
    ("row_codes", "<u4", (APC_TILE_MAX_ROWS,)), ("row_tensor", "<i4", (APC_TILE_MAX_ROWS,)),
    ("row_flops", "<i8", (APC_TILE_MAX_ROWS,)), ("row_rw_bytes", "<i8", (APC_TILE_MAX_ROWS,)),
    ("row_meta", "<i4", (APC_TILE_MAX_ROWS,)),
])
assert PACKED_TILE_DTYPE.itemsize == 2752


def shard_code(dim: int, variant: int = 0) -> int:
    if not 0 <= dim < 16:
        raise ValueError(f"Shard dim {dim} outside [0, 16)")
    if not 0 <= variant < 4:
        raise ValueError(f"Shard variant {variant} outside [0, 4)")
    return 0x80 | (variant << 4) | dim


def partial_code(op: int | str = 0) -> int:
    if isinstance(op, str):
        op = PARTIAL_OPS.index(op)
    if not 0 <= op < 64:
        raise ValueError(f"Partial op id {op} outside [0, 64)")
    return 0x40 | op


def code_kind(code: int) -> int:
    return code >> 6


def code_dim(code: int) -> int:
    return code & 0x0F


def pack_codes(codes) -> int:
    out = 0
    for i, c in enumerate(codes):
        out |= (int(c) & 0xFF) << (8 * i)
    return out


def unpack_codes(packed: int, ndim: int) -> tuple:
    return tuple((int(packed) >> (8 * i)) & 0xFF for i in range(ndim))


def _i32(x):
    return np.ascontiguousarray(x, dtype=np.int32)


def _i64(x):
    return np.ascontiguousarray(x, dtype=np.int64)


@dataclass
class CostTables:
    mesh_sizes: tuple
    tensor_rank: np.ndarray
    tensor_itemsize: np.ndarray
    tensor_shape: np.ndarray
    tensor_stride: np.ndarray
    spec_codes: np.ndarray
    spec_tensor: np.ndarray
    strat_flops: np.ndarray
    strat_rw_bytes: np.ndarray
    strat_dtype: np.ndarray
    strat_zero_cost: np.ndarray
    strat_num_args: np.ndarray
    node_strat_begin: np.ndarray
    edge_node: np.ndarray
    edge_arg: np.ndarray
    edge_src_begin: np.ndarray
    edge_n_src: np.ndarray
    edge_tgt_begin: np.ndarray
    edge_n_tgt: np.ndarray
    edge_flags: np.ndarray
    edge_pt_begin: np.ndarray
    edge_entry_begin: np.ndarray
    edge_strat_begin: np.ndarray
    pt_values: np.ndarray
    tile_edge: np.ndarray = None
    tile_row_begin: np.ndarray = None
    tile_row_count: np.ndarray = None
    tile_col_begin: np.ndarray = None
    tile_col_count: np.ndarray = None
    tile_records: np.ndarray = None
    edge_canonical: np.ndarray = None  # edge -> the identical edge that is tiled (itself unless de-duplicated)
    dup_entry_begin: np.ndarray = None  # entry offsets of the duplicates, grouped by canonical edge
    dup_row_begin: np.ndarray = None  # their first matrix rows (rows numbered as in ``row_ptr()``)
    edge_dup_begin: np.ndarray = None
    edge_dup_count: np.ndarray = None
    tiling: dict = None  # tile size and copies per tiled edge of the current tiling

    _DTYPES = {
        "tensor_rank": np.int32, "tensor_itemsize": np.int32, "tensor_shape": np.int64,
        "tensor_stride": np.int64, "spec_codes": np.uint32, "spec_tensor": np.int32,
        "strat_flops": np.int64, "strat_rw_bytes": np.int64, "strat_dtype": np.int8,
        "strat_zero_cost": np.uint8, "strat_num_args": np.int32, "node_strat_begin": np.int64,
        "edge_node": np.int32, "edge_arg": np.int32, "edge_src_begin": np.int32,
        "edge_n_src": np.int32, "edge_tgt_begin": np.int32, "edge_n_tgt": np.int32,
        "edge_flags": np.int32, "edge_pt_begin": np.int64, "edge_entry_begin": np.int64,
        "edge_strat_begin": np.int32, "pt_values": np.float64, "tile_edge": np.int32,
        "tile_row_begin": np.int32, "tile_row_count": np.int32, "tile_col_begin": np.int32,
        "tile_col_count": np.int32, "edge_canonical": np.int64, "dup_entry_begin": np.int64,
        "dup_row_begin": np.int64, "edge_dup_begin": np.int64, "edge_dup_count": np.int64,
    }
    _DTYPES = {name: np.dtype(t) for name, t in _DTYPES.items()}

    def __post_init__(self):
        self.mesh_sizes = tuple(int(x) for x in self.mesh_sizes)
        for name, dt in self._DTYPES.items():
            v = getattr(self, name)
            if v is not None:
                setattr(self, name, np.ascontiguousarray(v, dtype=dt))
        if self.tensor_shape.ndim != 2 or self.tensor_shape.shape[1] != APC_MAX_RANK:
            raise ValueError(f"tensor_shape must be [T, {APC_MAX_RANK}]")
        if self.tensor_stride.shape != self.tensor_shape.shape:
            raise ValueError("tensor_stride must have the shape of tensor_shape")
        if self.tile_edge is None:
            self.build_tiles()
        elif self.tile_records is None:
            self.pack_tile_records()

    def _rows(self, n: int, *names, exact: bool = False) -> list:
        """The named arrays as the library's host entry points read them, which see an address and not where its
        array ends: contiguous, of the table's dtype, with ``n`` rows at least (``exact``: just as many)."""
        out = []
        for name in names:
            a = np.ascontiguousarray(getattr(self, name), self._DTYPES[name])
            if name in ("tensor_shape", "tensor_stride"):
                if a.shape[1:] != (APC_MAX_RANK,):
                    raise ValueError(f"{name} must be [T, {APC_MAX_RANK}]")
            elif a.ndim != 1:
                if name not in ("spec_codes", "pt_values"):  # (whose rows are runs of values, whatever their shape)
                    raise ValueError(f"{name} has the shape {a.shape}")
                a = a.reshape(-1)
            if len(a) < n or (exact and len(a) != n):
                raise ValueError(f"{name} must have {n} rows, it has {len(a)}")
            out.append(a)
        return out

    def _strategy_rows(self, exact: bool = False) -> list:
        return self._rows(self.n_strategies, "strat_flops", "strat_rw_bytes", "strat_dtype", "strat_zero_cost", "strat_num_args",
                          exact=exact)

    def _matrix_sizes(self, exact: bool = True) -> list:
        return self._rows(self.n_edges, "edge_n_src", "edge_n_tgt", exact=exact)

    @staticmethod
    def _records(records, n: int, dtype) -> np.ndarray:
        a = np.ascontiguousarray(records)
        if a.nbytes < n * dtype.itemsize:
            raise ValueError(f"{n} records of {dtype.itemsize} bytes are needed, there are {a.nbytes} bytes")
        return a

    # ---- sizes -------------------------------------------------------------------------
    @property
    def n_tensors(self) -> int:
        return len(self.tensor_rank)

    @property
    def n_specs(self) -> int:
        return len(self.spec_codes)

    @property
    def n_strategies(self) -> int:
        return len(self.strat_flops)

    @property
    def n_nodes(self) -> int:
        return len(self.node_strat_begin) - 1

    @property
    def n_edges(self) -> int:
        return len(self.edge_n_src)

    @property
    def n_entries(self) -> int:
        return int(self.edge_entry_begin[-1])

    @property
    def n_tiles(self) -> int:
        return len(self.tile_edge)

    def algorithmic_bytes(self, comm=True, transition=True, cost=True) -> int:
        """Bytes one table build must move at minimum: the outputs written per entry,
        the placement codes of both spec lists of every edge and a 64-byte edge header."""
        per_entry = 8 * int(comm) + 1 * int(transition) + 8 * int(cost)
        m = len(self.mesh_sizes)
        per_edge = (self.edge_n_src.astype(np.int64) + self.edge_n_tgt.astype(np.int64)) * m + 64
        return per_entry * self.n_entries + int(per_edge.sum())

    def shape_width(self) -> int:
        """Values per row of the local shape / stride tables: the largest tensor rank, rounded up
        to even (rows leave the kernel as 16-byte pairs), at least 2."""
        top = int(self.tensor_rank.max()) if self.n_tensors else 0
        return max(2, top + (top & 1))

    def algorithmic_bytes_input_tables(self, spec_table: bool = True) -> int:
        """Bytes the tensor, spec and compute-cost tables must move at minimum: per tensor 136 B
        read (rank, itemsize, shape, stride) and 9 B written; per spec 8 B read and 24 B + two
        rows of ``shape_width()`` values written (shard count, local element and byte counts,
        local shape and stride); per strategy 22 B read and 16 B written."""
        spec = (32 + 16 * self.shape_width()) * self.n_specs if spec_table else 0
        return 145 * self.n_tensors + spec + 38 * self.n_strategies

    def algorithmic_bytes_priced_per_unit(self, row_minima: bool = True) -> int:
        """The same pass priced by fixed per-unit figures, whatever arrays a launch happens to
        write: 8 B (one fp64 cost) + 1 B (transition flag) per entry; per edge its two spec lists
        (one byte per mesh dim and spec) and a 64-byte header; 8 B written + 17 B read per
        (node, strategy) compute cost; 12 B written per row minimum."""
        m = len(self.mesh_sizes)
        per_edge = (self.edge_n_src.astype(np.int64) + self.edge_n_tgt.astype(np.int64)) * m + 64
        return 9 * self.n_entries + int(per_edge.sum()) + 25 * self.n_strategies + (12 * self.n_rows if row_minima else 0)

    @property
    def n_rows(self) -> int:
        """Matrix rows over all edges: one per (edge, consumer strategy)."""
        return int(self.edge_n_tgt.astype(np.int64).sum())

    def validate_row_minima(self) -> None:
        """Raises unless every matrix row lies inside one tile (the precondition of the
        ``apc_*_row_min`` entry points), through the library's host-side check."""
        _native.host_call("apc_validate_row_minima_host", self.n_edges, *self._matrix_sizes(exact=False), self.n_tiles,
                          self._records(self.tile_records, self.n_tiles, TILE_DTYPE))

    # ---- tiles -------------------------------------------------------------------------
    def edge_classes(self) -> np.ndarray:
        """For every edge the first edge whose matrix depends on the same bytes: both spec lists
        (codes and tensor rows), flags, the consumer strategies' compute-cost inputs and the
        pass-through values.  Equal edges have bit-identical comm / transition / cost."""
        first_same = np.empty(self.n_edges, np.int64)
        n_src, n_tgt = self._matrix_sizes()
        src_begin, tgt_begin, flags, pt_begin, strat_begin = self._rows(
            self.n_edges, "edge_src_begin", "edge_tgt_begin", "edge_flags", "edge_pt_begin", "edge_strat_begin")
        _native.host_call(
            "apc_edge_classes_host", self.n_specs, *self._rows(self.n_specs, "spec_codes", "spec_tensor"), self.n_strategies,
            *self._strategy_rows(exact=True), self.n_edges, src_begin, n_src, tgt_begin, n_tgt, flags, pt_begin, strat_begin,
            len(self.pt_values), *self._rows(0, "pt_values"), first_same)
        return first_same

    def edge_signatures(self) -> list:
        """One digest per edge over what ``edge_classes`` compares, for comparing edges of several tables, or in a
        program of one's own: equal digests = bit-identical comm / transition / cost."""
        import hashlib

        sb, ns = self.edge_src_begin.astype(np.int64), self.edge_n_src.astype(np.int64)
        tb, nt = self.edge_tgt_begin.astype(np.int64), self.edge_n_tgt.astype(np.int64)
        st = self.edge_strat_begin.astype(np.int64)
        codes, tensor = self.spec_codes, self.spec_tensor
        strat = np.rec.fromarrays([self.strat_flops, self.strat_rw_bytes, self.strat_dtype, self.strat_zero_cost,
                                   self.strat_num_args])
        out = []
        for e in range(self.n_edges):
            h = hashlib.blake2b(digest_size=16)
            h.update(np.array([ns[e], nt[e], self.edge_flags[e]], np.int64).tobytes())
            h.update(codes[sb[e]:sb[e] + ns[e]].tobytes())
            h.update(tensor[sb[e]:sb[e] + ns[e]].tobytes())
            h.update(codes[tb[e]:tb[e] + nt[e]].tobytes())
            h.update(tensor[tb[e]:tb[e] + nt[e]].tobytes())
            h.update(strat[st[e]:st[e] + nt[e]].tobytes())
            if self.edge_pt_begin[e] >= 0:
                b = int(self.edge_pt_begin[e])
                h.update(self.pt_values[b:b + int(ns[e] * nt[e])].tobytes())
            out.append(h.digest())
        return out

    def build_tiles(self, tile_entries: Optional[int] = None, dedupe: bool = False, max_copies: int = 16,
                    signatures=None, rows_per_wavefront_pass: Optional[int] = None, repeated: bool = True) -> None:
        """Cuts every edge matrix into rectangles of about ``tile_entries`` entries:
        whole rows when a row fits the LDS column budget, column chunks otherwise.  With
        ``dedupe`` only the first of every group of identical edges is tiled; its tiles
        store their values to all copies.  (Call it after the strategy table is final:
        the compute-cost inputs are part of an edge's identity.)  One tiled edge serves at
        most ``max_copies - 1`` duplicates, so a long run of identical edges still spreads
        over many workgroups.  ``tile_entries=None`` chooses tile size and copies per tiled
        edge from the table (``tiling`` records the choice).  ``rows_per_wavefront_pass = w``: a
        tile of whole rows holds at most ``w * (64 // columns)`` of them, what ``w`` wavefronts that
        each walk ``64 // columns`` whole rows at a time cover in one pass (the packed-tile launch
        of a small table, whose slowest workgroup decides the launch; the automatic choice sets it
        to 4 for such a table unless ``staging_pays`` or its rows are too wide to pack).
        ``signatures``: with a tile size and ``dedupe``, one value per edge, equal where matrices are
        (as of ``edge_signatures``); without, edges are compared by content.  ``repeated=False``: tile sizes for launches that
        go edge by edge (a pass that runs once, a report); the default ones are for a repeated pass, which takes the tiles of
        some tables by size (``largest_tiles_first_pays``)."""
        self._build_tiles(self.edge_classes, tile_entries, dedupe, max_copies, signatures, rows_per_wavefront_pass, repeated)

    def _build_tiles(self, edge_classes, tile_entries, dedupe, max_copies=16, signatures=None, rows_per_wavefront_pass=None,
                     repeated=True) -> None:
        """``edge_classes``: what finds the identical edges."""
        classes = None
        if dedupe and self.n_edges and signatures is not None and tile_entries is not None:
            first: dict = {}
            classes = np.arange(self.n_edges, dtype=np.int64)
            for e, signature in enumerate(signatures):
                classes[e] = first.setdefault(signature, e)
        elif dedupe and self.n_edges:
            classes = edge_classes()
        canonical = np.empty(self.n_edges, np.int64)
        n_src, n_tgt = self._matrix_sizes()

        def count(te, mc, rows):
            return _native.host_counts("apc_count_tiles_host", self.n_edges, n_src, n_tgt, classes, te, mc, rows, canonical)

        def computed():  # (of the last count)
            return int((n_src.astype(np.int64) * n_tgt)[canonical == np.arange(self.n_edges)].sum())

        automatic = tile_entries is None
        if automatic:
            te, mc = APC_TILE_MAX_ROWS * APC_TILE_MAX_COLS, int(max_copies)
            small = self.n_entries <= AUTO_SMALL_TABLE_ENTRIES
            if small:
                n, n_dups = packed_cut = count(te, mc, 4)
                whole_edges = n, computed()
                tiled_edges = int(np.count_nonzero((canonical == np.arange(self.n_edges)) & (n_src > 0) & (n_tgt > 0)))
                fits = n == 0 or int(n_src.max()) <= APC_TILE_MAX_COLS
                rows_per_wavefront_pass = 4
                if n and (not fits or self._staging_may_pay(whole_edges[1], tiled_edges, repeated)):
                    n, n_dups = count(te, mc, 0)
                    wanted, least = STAGED_TILES, max(STAGED_MIN_TILE_ENTRIES, whole_edges[1] // STAGED_SMALLEST_SHARE)
                    if self._many_states():
                        wanted, least = STAGED_TILES_OF_MANY_STATES, STAGED_MIN_TILE_ENTRIES_OF_MANY_STATES
                    while n < wanted and te // 2 >= 1 << (least.bit_length() - 1):
                        te //= 2
                        n, n_dups = count(te, mc, 0)
                    if not fits or self.staging_pays(whole_edges[1], n, tiled_edges, repeated):
                        rows_per_wavefront_pass = None
                    else:
                        te, (n, n_dups) = APC_TILE_MAX_ROWS * APC_TILE_MAX_COLS, packed_cut
            else:
                n, n_dups = count(te, mc, 0)
                whole_edges = n, computed()
                te = AUTO_MIN_TILE_ENTRIES
                n, n_dups = count(te, mc, 0)
                while self.n_entries > n * AUTO_MAX_STORED_PER_TILE and mc > 2 and n_dups:
                    mc //= 2
                    n, n_dups = count(te, mc, 0)
                ordered = repeated and self._orders(computed(), n)
                while te < APC_TILE_MAX_ROWS * APC_TILE_MAX_COLS:
                    stored = ORDERED_MIN_STORED_PER_TILE if ordered and n > ORDERED_SOME_ROUNDS else AUTO_MIN_STORED_PER_TILE
                    if self.n_entries >= n * stored and not (te > AUTO_MIN_TILE_ENTRIES and n > AUTO_MANY_TILES):
                        break
                    te *= 2
                    n, n_dups = count(te, mc, 0)
        else:
            te, mc = max(int(tile_entries), 1), int(max_copies)  # (below 1: one row a tile, as 1)
            n, n_dups = count(te, mc, int(rows_per_wavefront_pass or 0))
        self.tiling = {"tile_entries": te if automatic else int(tile_entries), "max_copies": mc if dedupe else 1}
        if automatic:
            self.tiling["whole_edges"] = whole_edges
            if small:
                self.tiling["tiled_edges"] = tiled_edges
        if rows_per_wavefront_pass:
            self.tiling["rows_per_wavefront_pass"] = int(rows_per_wavefront_pass)
        self.edge_canonical = canonical
        self.edge_dup_begin, self.edge_dup_count = np.empty(self.n_edges, np.int64), np.empty(self.n_edges, np.int64)
        self.dup_entry_begin, self.dup_row_begin = np.empty(n_dups, np.int64), np.empty(n_dups, np.int64)
        self.tile_edge, self.tile_row_begin, self.tile_row_count, self.tile_col_begin, self.tile_col_count = (
            np.empty(n, np.int32) for _ in range(5))
        _native.host_call(
            "apc_fill_tiles_host", self.n_edges, n_src, n_tgt, *self._rows(self.n_edges + 1, "edge_entry_begin"), canonical, te,
            int(rows_per_wavefront_pass or 0), n, n_dups, self.edge_dup_begin, self.edge_dup_count, self.dup_entry_begin,
            self.dup_row_begin, self.tile_edge, self.tile_row_begin, self.tile_row_count, self.tile_col_begin, self.tile_col_count)
        self.pack_tile_records()

    def pack_tile_records(self) -> None:
        """The tile rectangles plus the fields of their edge, as the packed records the
        table kernel reads (C struct ``apc_tile``)."""
        if self.edge_canonical is None or len(self.edge_canonical) != self.n_edges:
            self.edge_canonical = np.arange(self.n_edges, dtype=np.int64)
            self.dup_entry_begin = _i64([])
            self.dup_row_begin = _i64([])
            self.edge_dup_count = np.zeros(self.n_edges, np.int64)
            self.edge_dup_begin = np.zeros(self.n_edges, np.int64)
        rec = np.empty(self.n_tiles, TILE_DTYPE)
        _native.host_call(
            "apc_tile_records_host", self.n_specs, *self._rows(self.n_specs, "spec_tensor"), self.n_edges,
            *self._rows(self.n_edges, "edge_src_begin", "edge_n_src", "edge_tgt_begin", "edge_flags", "edge_pt_begin"),
            *self._rows(self.n_edges + 1, "edge_entry_begin"),
            *self._rows(self.n_edges, "edge_strat_begin", "edge_dup_begin", "edge_dup_count"),
            self.n_tiles, *self._rows(self.n_tiles, "tile_edge", "tile_row_begin", "tile_row_count", "tile_col_begin",
                                      "tile_col_count"), rec)
        self.tile_records = rec

    # ---- packed tiles ------------------------------------------------------------------
    def _many_states(self) -> bool:
        return len(self.mesh_sizes) == 4 and any(m & (m - 1) for m in self.mesh_sizes)

    def _staging_may_pay(self, computed: int, tiled_edges: int, repeated: bool) -> bool:
        """``staging_pays`` of some number of tiles."""
        return computed >= STAGED_MIN_COMPUTED_OF_COPIES or self.staging_pays(computed, computed + 1, tiled_edges, repeated)

    def staging_pays(self, computed: int, n_tiles: int, tiled_edges: Optional[int] = None, repeated: bool = True) -> bool:
        """Whether tiles staged in LDS beat packed ones on a small table (above: STAGED_MIN_COMPUTED).  ``tiled_edges``: the edges
        that have tiles, by default those of the current tiling where it was chosen from the table.  A pass that runs once
        (``repeated=False``, a planner's) goes over packed tiles unless much is computed: their records hold the tables as the
        host has them, which a planner may have written there, where staged tiles read the device's; a few us are nothing to it.  A
        repeated one compares the two (``DeviceCostTables.prepare_step``)."""
        if tiled_edges is None:
            tiled_edges = (self.tiling or {}).get("tiled_edges", 0)
        M = len(self.mesh_sizes)
        states = self._states_one_by_one()
        if repeated and (not states or (M == 3 and computed >= STAGED_MIN_PER_EDGE_OF_STATES * (tiled_edges or n_tiles))):
            stored = M >= 3 or self.n_entries <= STAGED_MAX_STORED_PER_EDGE * tiled_edges
            if (tiled_edges > STAGED_MANY_EDGES and stored) or (computed >= STAGED_MIN_COMPUTED and self.n_entries <= STAGED_MAX_COPIES * computed):
                return True
        return computed >= STAGED_MIN_COMPUTED_OF_COPIES and computed >= n_tiles * STAGED_MIN_COMPUTED_PER_TILE[M]

    def packed_lanes(self, records: Optional[np.ndarray] = None) -> int:
        """Lanes a packed tile is evaluated by (above: PACKED_MANY_TILES), for the tiling's records or the ``records`` given."""
        return self._packed_lanes_and_rounds(records)[0]

    def _packed_lanes_and_rounds(self, records: Optional[np.ndarray] = None) -> tuple:
        """-> (``packed_lanes``, rounds in which a wavefront takes the tile that needs most)"""
        counts = (self.tile_records if records is None else records)["counts"]
        rows, cols = counts & 0xFFFF, np.maximum(counts >> 16, 1)
        n, stored = len(counts), self.n_entries

        def rounds(lanes):
            per_round = lanes // cols
            return int((-(-rows // np.maximum(per_round, 1))).max()) if per_round.all() else n + APC_TILE_MAX_ROWS

        if n == 0:
            return 256, 0
        most = rounds(64)
        if most > 1:
            return 64 if most == 2 and n > PACKED_MANY_TILES and self._states_one_by_one() else 256, most
        if n > PACKED_MANY_TILES and stored <= PACKED_MAX_SMALL_COPIES * int((rows.astype(np.int64) * cols).sum()):
            for lanes in (16, 32):
                if rounds(lanes) == 1:
                    return lanes, 1
        return 64, most

    def small_packing_pays(self) -> bool:
        """Whether packed tiles, a few lanes each and in one round, beat staged ones (above: PACKED_MANY_TILES)."""
        return self.small_packing_lanes() > 0

    def small_packing_lanes(self) -> int:
        """``packed_lanes`` where ``small_packing_pays``, else 0."""
        lanes, rounds = self._packed_lanes_and_rounds()
        if lanes == 256 or rounds != 1:
            return 0
        pays = lanes < 64 or self._states_one_by_one() or len(self.mesh_sizes) < 3 or self.n_tiles < PACKED_MANY_TILES_OF_64 or \
            2 * self.n_entries >= 3 * self.computed_entries()
        return lanes if pays else 0

    def _states_one_by_one(self) -> bool:
        """Whether a staged tile works out the running-bytes states of a mesh of three dims or four one by one."""
        return len(self.mesh_sizes) >= 3 and any(m & (m - 1) for m in self.mesh_sizes)

    def largest_tiles_first_pays(self) -> bool:
        """Whether a launch takes the tiles by size instead of edge by edge (above: ORDERED_MAX_ENTRIES)."""
        return self.n_entries <= ORDERED_MAX_ENTRIES and self.n_tiles > 0 and self._orders(self.computed_entries(), self.n_tiles)

    def _orders(self, computed: int, n_tiles: int) -> bool:
        return self.n_entries <= ORDERED_MAX_ENTRIES and ORDERED_MIN_PER_TILE * n_tiles <= computed \
            and self.n_entries <= ORDERED_MAX_COPIES * computed

    def launch_records(self, records: Optional[np.ndarray] = None) -> np.ndarray:
        """``tile_records``, or the ``records`` of an earlier tiling, in the order in which a launch takes them."""
        if records is None:
            records, n, pays = self.tile_records, self.n_tiles, self.largest_tiles_first_pays()
        else:
            n = len(records)
            computed = int(((records["counts"] & 0xFFFF).astype(np.int64) * (records["counts"] >> 16)).sum())
            pays = n > 0 and self._orders(computed, n)
        if not pays:
            return records
        ordered = np.empty(n, TILE_DTYPE)
        _native.host_call("apc_order_tiles_host", n, self._records(records, n, TILE_DTYPE), ordered)
        return ordered

    def computed_entries(self) -> int:
        """Entries the tiles compute: those of identical edges once for all their copies."""
        return int((self.tile_row_count.astype(np.int64) * self.tile_col_count.astype(np.int64)).sum())

    def packable(self) -> bool:
        """Every tile holds whole rows of at most APC_TILE_MAX_COLS columns and serves at most
        APC_PACKED_MAX_DUPS identical edges: the table can be built from packed tiles."""
        if self.n_tiles == 0 or not self.rows_fit_tiles():
            return False
        if int(self.tile_records["dup_count"].max()) > APC_PACKED_MAX_DUPS:
            return False
        return bool(self.n_strategies == 0 or int(self.strat_num_args.max()) <= 0x7FFF)

    def _packed_sources(self, records=None) -> list:
        """What a packed tile is copied out of, as the library takes it."""
        self._matrix_sizes()  # (the rows of all edges come from their sizes)
        return [self.n_tensors, *self._rows(self.n_tensors, "tensor_rank", "tensor_itemsize", "tensor_shape", "tensor_stride"),
                self.n_specs, *self._rows(self.n_specs, "spec_codes", "spec_tensor"),
                self.n_strategies, *self._strategy_rows(), self.n_edges, self.edge_row_begin(), self.n_tiles,
                self._records(self.tile_records if records is None else records, self.n_tiles, TILE_DTYPE), len(self.dup_entry_begin),
                *self._rows(len(self.dup_entry_begin), "dup_entry_begin", "dup_row_begin")]

    def pack_tiles(self, records=None) -> np.ndarray:
        """One ``apc_packed_tile`` record per tile (of ``records``, the table's own by default): the tile's header, its tensor's row, the
        first entries / rows of its identical edges, its producer and consumer specs and its
        consumer strategies' rows of the strategy table, copied out of the tables (after the
        strategy table is final).  A workgroup then loads nothing whose address depends on
        another load."""
        if not self.packable():
            raise RuntimeError("packed tiles need whole rows in every tile and at most "
                               f"{APC_PACKED_MAX_DUPS} identical edges per tile")
        pk = np.empty(self.n_tiles, PACKED_TILE_DTYPE)
        _native.host_call("apc_pack_tiles_host", *self._packed_sources(records), pk)
        return pk

    def validate_packed(self, packed: np.ndarray) -> None:
        """Packed records against the tables, through the library's host-side check: for records that were kept or came
        from elsewhere (``pack_tiles`` refuses the tables whose records this would refuse)."""
        _native.host_call("apc_validate_packed_tiles_host", *self._packed_sources(),
                          self._records(packed, self.n_tiles, PACKED_TILE_DTYPE))

    # ---- checks ------------------------------------------------------------------------
    def validate(self, params) -> None:
        """Structural check through the library's host-side validator; raises
        RuntimeError naming the first malformed row."""
        self._validate(params, None)

    def _validate(self, params, on_device) -> None:
        """``on_device``: called where lengths and types are right; -> what needs no check of the host's any more, ``"tiles"``
        (with the copies' offsets), ``"tables"`` (those and every row) or nothing."""
        if tuple(params.mesh_sizes) != self.mesh_sizes:
            raise RuntimeError(f"tables were encoded for mesh {self.mesh_sizes}, params describe {params.mesh_sizes}")
        if len(self.edge_entry_begin) != self.n_edges + 1:
            raise RuntimeError("edge_entry_begin must have n_edges + 1 rows")
        for name in ("edge_src_begin", "edge_tgt_begin", "edge_flags", "edge_pt_begin", "edge_strat_begin",
                     "edge_n_tgt"):
            if len(getattr(self, name)) != self.n_edges:
                raise RuntimeError(f"{name} must have n_edges rows")
        if len(self.spec_tensor) != self.n_specs:
            raise RuntimeError("spec_tensor must have n_specs rows")
        for name in ("strat_rw_bytes", "strat_dtype", "strat_zero_cost", "strat_num_args"):
            if len(getattr(self, name)) != self.n_strategies:
                raise RuntimeError(f"{name} must have n_strategies rows")
        if self.tile_records is None or len(self.tile_records) != self.n_tiles:
            raise RuntimeError("tile_records must have one record per tile (call pack_tile_records())")
        rank, itemsize, shape = self._rows(self.n_tensors, "tensor_rank", "tensor_itemsize", "tensor_shape", exact=True)
        codes, spec_tensor = self._rows(self.n_specs, "spec_codes", "spec_tensor")
        flops, rw_bytes, *_, num_args = self._strategy_rows()
        n_src, n_tgt = self._matrix_sizes()
        src_begin, tgt_begin, flags, pt_begin, strat_begin, canonical, dup_count = self._rows(
            self.n_edges, "edge_src_begin", "edge_tgt_begin", "edge_flags", "edge_pt_begin", "edge_strat_begin", "edge_canonical",
            "edge_dup_count")
        (dup_entry_begin,) = self._rows(0, "dup_entry_begin")
        (entry_begin,) = self._rows(self.n_edges + 1, "edge_entry_begin")
        records = self._records(self.tile_records, self.n_tiles, TILE_DTYPE)
        held = on_device() if on_device is not None else None
        if held != "tables":
            _native.host_call(
                "apc_validate_tables_host", params.to_c(), self.n_tensors, rank, self.n_specs, codes, spec_tensor, self.n_edges,
                src_begin, n_src, tgt_begin, n_tgt, flags, pt_begin, entry_begin, strat_begin,
                len(self.pt_values), self.n_strategies, 0 if held == "tiles" else self.n_tiles, records, len(dup_entry_begin), dup_entry_begin)
        # what the kernels cannot check: every edge is tiled completely or a duplicate of an edge that is; flop and
        # byte counts convert to fp64 exactly (the kernels divide them as doubles)
        _native.host_call(
            "apc_validate_tiling_host", self.n_tensors, rank, itemsize, shape, self.n_strategies, flops, rw_bytes, num_args,
            self.n_edges, n_src, n_tgt, canonical, dup_count, len(dup_entry_begin), self.n_tiles,
            *self._rows(self.n_tiles, "tile_edge", "tile_row_count", "tile_col_count", exact=True))

    def as_dict(self) -> dict:
        """Plain-data view (numpy arrays) of every table."""
        out = {"mesh_sizes": self.mesh_sizes}
        for f in fields(self):
            if f.name != "mesh_sizes":
                out[f.name] = getattr(self, f.name)
        return out

    # ---- derived index arrays ------------------------------------------------------------
    def strategy_bound_index(self) -> dict:
        """Index arrays of the per-strategy lower bounds (C entry ``apc_strategy_bounds``):
        the node of every strategy, every node's edges (as consumer) in edge order, and the
        first matrix row of every edge in the order of ``row_ptr()``."""
        n_nodes = self.n_nodes
        n_strat = np.diff(self.node_strat_begin).astype(np.int64)
        node = self.edge_node.astype(np.int64)
        if self.n_edges and (node.min() < 0 or node.max() >= n_nodes):
            raise RuntimeError("edge_node outside the node table")
        if not np.array_equal(self.edge_n_tgt.astype(np.int64), n_strat[node]):
            raise RuntimeError("an edge's row count differs from its consumer node's strategy count")
        order = np.argsort(node, kind="stable")
        node_edge_begin = np.zeros(n_nodes + 1, np.int64)
        np.cumsum(np.bincount(node, minlength=n_nodes), out=node_edge_begin[1:])
        edge_row_begin = np.cumsum(self.edge_n_tgt.astype(np.int64)) - self.edge_n_tgt
        return {
            "strat_node": _i32(np.repeat(np.arange(n_nodes, dtype=np.int64), n_strat)),
            "node_edge_begin": node_edge_begin,
            "edges_by_node": _i32(order),
            "edge_row_begin": _i64(edge_row_begin),
        }

    def edge_row_begin(self) -> np.ndarray:
        """First matrix row of every edge: rows are numbered edge by edge, one per consumer
        strategy (the order of ``row_ptr()``)."""
        nt = self.edge_n_tgt.astype(np.int64)
        return _i64(np.cumsum(nt) - nt)

    def rows_fit_tiles(self) -> bool:
        """Every matrix row lies inside one tile (and none is empty), so the launch that writes
        the cost matrices can take the row minima itself."""
        ns = self.edge_n_src.astype(np.int64)
        nt = self.edge_n_tgt.astype(np.int64)
        with_rows = nt > 0
        if not bool(((ns[with_rows] >= 1) & (ns[with_rows] <= APC_TILE_MAX_COLS)).all()):
            return False
        te = self.tile_edge.astype(np.int64)
        return bool((self.tile_col_begin == 0).all() and (self.tile_col_count == ns[te]).all())

    def row_copies(self):
        """-> (selected, copy_ptr, copy_rows, n_values_selected): the matrix rows of the edges that
        are tiled, and for each of them the rows of the identical edges that receive the same
        values (rows numbered as in ``row_ptr()``).  A minimum taken over ``selected`` and
        stored to the copies covers every row while reading each distinct row once."""
        nt = self.edge_n_tgt.astype(np.int64)
        ns = self.edge_n_src.astype(np.int64)
        rb = self.edge_row_begin()
        canon = np.nonzero(self.edge_canonical == np.arange(self.n_edges))[0]
        ntc = nt[canon]
        n_sel = int(ntc.sum())
        first = np.cumsum(ntc) - ntc
        r = np.arange(n_sel, dtype=np.int64) - np.repeat(first, ntc)  # consumer strategy of every selected row
        selected = np.repeat(rb[canon], ntc) + r
        per_row = np.repeat(self.edge_dup_count[canon].astype(np.int64), ntc)
        copy_ptr = np.zeros(n_sel + 1, np.int64)
        np.cumsum(per_row, out=copy_ptr[1:])
        which = np.repeat(np.arange(n_sel, dtype=np.int64), per_row)
        k = np.arange(int(copy_ptr[-1]), dtype=np.int64) - copy_ptr[which]
        dup_first = np.repeat(self.edge_dup_begin[canon].astype(np.int64), ntc)
        copy_rows = self.dup_row_begin[dup_first[which] + k] + r[which] if len(which) else _i64([])
        return _i64(selected), _i64(copy_ptr), _i64(copy_rows), int((ns[canon] * ntc).sum())

    def row_ptr(self) -> np.ndarray:
        """CSR pointer of matrix rows over the entry array: one segment per
        (edge, consumer strategy), length = that edge's producer count."""
        ns = self.edge_n_src.astype(np.int64)
        nt = self.edge_n_tgt.astype(np.int64)
        lens = np.repeat(ns, nt)
        out = np.zeros(len(lens) + 1, np.int64)
        np.cumsum(lens, out=out[1:])
        return out

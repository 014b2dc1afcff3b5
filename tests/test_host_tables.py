"""The library's host-side table passes (identical edges, tilings, packed records, transfers)
against plain restatements of what they are: CPU except where marked."""

import numpy as np
import pytest

from autoparallel_amd import CostModelParams
from autoparallel_amd._native import APC_TILE_MAX_COLS, APC_TILE_MAX_DUPS, APC_TILE_MAX_ROWS
from autoparallel_amd.synthetic import stress_dag
from test_abi_and_encoding import twin_graph


def _content(tb, e):
    """Everything edge e's matrix depends on, as bytes."""
    ns, nt, sb, tg, st = (int(a[e]) for a in (tb.edge_n_src, tb.edge_n_tgt, tb.edge_src_begin, tb.edge_tgt_begin, tb.edge_strat_begin))
    parts = [np.int64([ns, nt, tb.edge_flags[e], tb.edge_pt_begin[e] >= 0])]
    parts += [a[sb:sb + ns] for a in (tb.spec_codes, tb.spec_tensor)] + [a[tg:tg + nt] for a in (tb.spec_codes, tb.spec_tensor)]
    parts += [a[st:st + nt] for a in (tb.strat_flops, tb.strat_rw_bytes, tb.strat_dtype, tb.strat_zero_cost, tb.strat_num_args)]
    if tb.edge_pt_begin[e] >= 0:
        b = int(tb.edge_pt_begin[e])
        parts.append(tb.pt_values[b:b + ns * nt])
    return b"|".join(p.tobytes() for p in parts)


@pytest.mark.parametrize("seed,nodes,hi", [(0, 1, 2), (1, 40, 3), (2, 300, 24), (3, 60, 100)])
def test_edge_classes_are_the_edges_of_equal_content(seed, nodes, hi):
    tb = twin_graph(stress_dag(seed=seed, n_nodes=nodes, mesh_sizes=(4, 2), min_strategies=1, max_strategies=hi))
    rng = np.random.default_rng(seed)
    for e in rng.integers(0, tb.n_edges, tb.n_edges // 4):  # some twins differ in one value each, in any part
        which = rng.integers(0, 4)
        if which == 0:
            tb.spec_tensor[tb.edge_tgt_begin[e]] = -1
        elif which == 1:
            tb.strat_rw_bytes[tb.edge_strat_begin[e] + tb.edge_n_tgt[e] - 1] += 1
        elif which == 2:
            tb.edge_flags[e] ^= 1
        elif tb.edge_pt_begin[e] >= 0:
            tb.pt_values[tb.edge_pt_begin[e]] = np.inf
    first, want = {}, []
    for e in range(tb.n_edges):
        want.append(first.setdefault(_content(tb, e), e))
    assert np.array_equal(tb.edge_classes(), want)


@pytest.mark.parametrize("te,copies,rows", [(1, 2, None), (64, 1, None), (300, 5, 3), (4096, 16, 4), (4096, 100, None)])
@pytest.mark.parametrize("hi", [3, 64, 65, 130])
def test_tilings_follow_their_definition(te, copies, rows, hi):
    tb = twin_graph(twin_graph(stress_dag(seed=hi, n_nodes=30, mesh_sizes=(4, 2), min_strategies=1, max_strategies=hi)))
    tb.build_tiles(te, dedupe=True, max_copies=copies, rows_per_wavefront_pass=rows)
    tb.validate(CostModelParams.from_mesh((4, 2)))
    # duplicates: each class of equal edges in runs of one tiled edge and at most copies - 1 others
    room = min(APC_TILE_MAX_DUPS, max(copies - 1, 0))
    open_edge, want = {}, []
    for e, f in enumerate(tb.edge_classes().tolist()):
        c, n = open_edge.get(f, (e, room))
        c, n = (e, 0) if n >= room else (c, n + 1)
        open_edge[f] = (c, n)
        want.append(c)
    assert np.array_equal(tb.edge_canonical, want)
    row_begin = tb.edge_row_begin()
    tiles = []
    for e in range(tb.n_edges):
        ns, nt = int(tb.edge_n_src[e]), int(tb.edge_n_tgt[e])
        dups = [d for d in range(tb.n_edges) if want[d] == e and d != e]
        at = slice(int(tb.edge_dup_begin[e]), int(tb.edge_dup_begin[e] + tb.edge_dup_count[e]))
        assert np.array_equal(tb.dup_entry_begin[at], tb.edge_entry_begin[dups]) and np.array_equal(tb.dup_row_begin[at], row_begin[dups])
        if want[e] != e or ns == 0 or nt == 0:
            continue
        chunks = -(-ns // APC_TILE_MAX_COLS)
        width = -(-ns // chunks)
        most = min(max(te // width, 1), APC_TILE_MAX_ROWS)
        if rows and chunks == 1:
            most = min(most, rows * max(64 // width, 1))
        n = -(-nt // most)
        per = -(-nt // n)
        tiles += [(e, r * per, min(per, nt - r * per), c * width, min(width, ns - c * width)) for r in range(n) for c in range(chunks)]
    got = np.stack([tb.tile_edge, tb.tile_row_begin, tb.tile_row_count, tb.tile_col_begin, tb.tile_col_count], 1)
    assert np.array_equal(got, np.asarray(tiles).reshape(-1, 5))


def test_packed_records_repeat_the_tables():
    tb = twin_graph(stress_dag(seed=4, n_nodes=200, mesh_sizes=(4, 2), min_strategies=1, max_strategies=40, frac_nonspec_nodes=0.1))
    tb.build_tiles(None, dedupe=True)
    tb.validate_packed(tb.pack_tiles())  # (the validator compares field by field)
    tb.tile_records["strat_begin"][3] = tb.n_strategies
    with pytest.raises(RuntimeError, match="tile 3: rows outside the tables"):
        tb.pack_tiles()


@pytest.mark.parametrize("field,value", [("num_args", 0), ("col_begin", 1), ("n_src", 63)])
def test_tables_whose_packed_records_the_validator_refuses_are_not_packed(field, value):
    """The planner's pass takes the packed records as they come from ``pack_tiles``."""
    tb = stress_dag(seed=4, n_nodes=200, mesh_sizes=(4, 2), min_strategies=1, max_strategies=40)
    if field == "num_args":
        tb.strat_num_args[tb.edge_strat_begin[tb.tile_edge[3]]] = value
    else:
        tb.tile_records[field][3] += value
    with pytest.raises(RuntimeError, match="tile [0-3]:"):
        tb.pack_tiles()


def test_tilings_from_signatures_and_of_less_than_one_entry():
    want, tb = _two_layers(), _two_layers()
    assert tb.edge_signatures() == want.edge_signatures() and len(tb.edge_signatures()) == tb.n_edges
    tb.build_tiles(512, True, 16, tb.edge_signatures())
    assert tb.tile_records.tobytes() == want.tile_records.tobytes()
    tb.build_tiles(512, dedupe=True, signatures=range(tb.n_edges))  # no edge is like another
    assert np.array_equal(tb.edge_canonical, np.arange(tb.n_edges))
    tb.build_tiles(512, dedupe=True, signatures=["same"] * 3)  # (an edge without a signature stands for itself)
    assert tb.edge_canonical.tolist() == [0, 0, 0, *range(3, tb.n_edges)]
    want.build_tiles(1)
    for te in (0, -7):
        tb.build_tiles(te)
        assert tb.tile_records.tobytes() == want.tile_records.tobytes() and tb.tiling["tile_entries"] == te


# what each host pass reads of the tables, besides the array whose length gives the number of rows
READS = {
    "edge_classes": ("spec_tensor", "strat_rw_bytes", "strat_dtype", "strat_zero_cost", "strat_num_args", "edge_src_begin",
                     "edge_tgt_begin", "edge_n_tgt", "edge_flags", "edge_pt_begin", "edge_strat_begin"),
    "build_tiles": ("edge_n_tgt", "edge_entry_begin", "spec_tensor", "edge_src_begin", "edge_tgt_begin", "edge_flags",
                    "edge_pt_begin", "edge_strat_begin"),
    "pack_tile_records": ("spec_tensor", "edge_src_begin", "edge_tgt_begin", "edge_flags", "edge_pt_begin", "edge_entry_begin",
                          "edge_strat_begin", "edge_dup_begin", "edge_dup_count", "tile_row_begin", "tile_row_count",
                          "tile_col_begin", "tile_col_count"),
    "pack_tiles": ("tensor_itemsize", "tensor_shape", "tensor_stride", "spec_tensor", "strat_rw_bytes", "strat_dtype",
                   "strat_zero_cost", "strat_num_args", "edge_n_tgt", "tile_records", "dup_row_begin"),
    "validate_row_minima": ("edge_n_tgt", "tile_records"),
    "validate": ("tensor_itemsize", "tensor_shape", "spec_tensor", "strat_rw_bytes", "strat_dtype", "strat_zero_cost",
                 "strat_num_args", "edge_n_tgt", "edge_src_begin", "edge_tgt_begin", "edge_flags", "edge_pt_begin",
                 "edge_entry_begin", "edge_strat_begin", "edge_canonical", "edge_dup_count", "tile_records", "tile_row_count",
                 "tile_col_count"),
}


def _read(tb, method):
    return getattr(tb, method)(*([CostModelParams.from_mesh((4, 2))] if method == "validate" else []))


def _two_layers():
    tb = twin_graph(stress_dag(seed=4, n_nodes=60, mesh_sizes=(4, 2), min_strategies=1, max_strategies=10))
    tb.build_tiles(512, dedupe=True)
    return tb


@pytest.mark.parametrize("method,name", [(m, n) for m, names in READS.items() for n in names])
def test_an_array_that_ends_early_is_refused_before_it_is_read(method, name):
    """The library sees addresses: an array shorter than the table it belongs to must not reach it."""
    for keep in (-1, 0):  # one row short; empty
        tb = _two_layers()
        setattr(tb, name, getattr(tb, name)[:keep])
        with pytest.raises((ValueError, RuntimeError, IndexError)):
            _read(tb, method)


def test_tables_that_are_too_long_or_of_another_shape_are_refused_where_they_were():
    """Where lengths have to agree, not only to suffice."""
    for method, name in (("build_tiles", "edge_n_tgt"), ("edge_classes", "strat_flops"), ("edge_classes", "strat_num_args"),
                         ("validate", "tensor_shape"), ("validate", "tile_row_count")):
        tb = _two_layers()
        a = getattr(tb, name)
        setattr(tb, name, np.concatenate([a, a[-1:]]))
        with pytest.raises(ValueError):
            _read(tb, method)
    for method, name in (("build_tiles", "edge_n_src"), ("pack_tiles", "spec_tensor"), ("edge_classes", "strat_dtype")):
        tb = _two_layers()
        setattr(tb, name, getattr(tb, name).reshape(-1, 1))
        with pytest.raises(ValueError):
            _read(tb, method)
    want, tb = _two_layers(), _two_layers()
    tb.pt_values, tb.spec_tensor = tb.pt_values.reshape(-1, 1), np.concatenate([tb.spec_tensor, [0]])
    assert np.array_equal(tb.edge_classes(), want.edge_classes())
    tb.build_tiles(512, dedupe=True)
    assert tb.tile_records.tobytes() == want.tile_records.tobytes()


@pytest.mark.parametrize("method", READS)
def test_arrays_of_other_types_and_strides_are_read_by_value(method):
    want, tb = _two_layers(), _two_layers()
    for name in READS[method] + ("strat_flops", "edge_n_src"):
        a = getattr(tb, name)
        if a.dtype.names is None and a.ndim == 1:
            other = np.int64 if a.dtype.itemsize < 8 or a.max(initial=0) > 2**31 - 1 else np.int32
            spread = np.zeros(2 * len(a), other)
            spread[::2] = a
            setattr(tb, name, spread[::2])
        else:
            setattr(tb, name, np.repeat(a, 2, axis=0)[::2])
    got = _read(tb, method)
    assert (got is None) == (_read(want, method) is None)
    if got is not None:
        assert got.tobytes() == _read(want, method).tobytes()
    elif method != "validate":
        assert tb.tile_records.tobytes() == want.tile_records.tobytes()


_NO_MEMORY = """
import sys
sys.path.insert(0, {root!r})
import numpy as np
from autoparallel_amd import _native
i64, i32 = (lambda *v: np.asarray(v, np.int64)), (lambda *v: np.asarray(v, np.int32))
try:
    if sys.argv[1] == "entry":  # (the vectors come before any array is read)
        _native.host_counts("apc_count_tiles_host", 1 << 61, i32(1), i32(1), i64(0), 64, 2, 0, i64(0))
    else:  # 1 M elements: several threads; one of them meets a class of 2**61 labels (and takes its memory first)
        _native.host_call("apc_prune_masks_host", 3, i64(0, 1024, 2048, 2048 + (1 << 61)), i64(0, 1, 2, 2), i32(0, 0),
                          np.asarray([0, 1], np.uint8), 1, i64(0, 1 << 20), i32(0), i32(1), np.zeros(1 << 20), np.zeros(2048),
                          np.zeros(3), np.zeros(1), 0.0, 1.0, np.zeros(2048, bool), np.zeros(1 << 20, bool))
except RuntimeError as e:
    print(e, flush=True)
"""


@pytest.mark.parametrize("where", ["entry", "thread"])
def test_memory_that_cannot_be_had_is_an_error_and_not_the_end_of_the_process(where):
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", _NO_MEMORY.format(root=root), where], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and "failed (-4)" in out.stdout, (out.returncode, out.stderr[-500:])


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[0], [1, 0, 3], [4 << 20], [(4 << 20) + 1, 255, 0, 257], [1, 40 << 20, 7, 9 << 20],
                                   [1 << 20, (1 << 20) + 1, (1 << 20) - 1, 0] * 9, [5 << 20, (1 << 20) + 1, 100, 4 << 20]])
def test_transfers_bring_back_the_bytes(gpu_device, sizes):
    """Sizes around the pinned chunk (4 MiB) and beyond the chunks in flight, arrays that share a buffer (up to 1 MiB)
    and arrays that do not."""
    import torch

    from autoparallel_amd import _native

    ops = _native.torch_ops()
    host = [torch.randint(0, 256, (n,), dtype=torch.uint8) for n in sizes] + [torch.arange(5, dtype=torch.float64).reshape(5, 1)]
    dev = ops.upload(host, gpu_device)
    back = ops.download(dev)
    for h, d, b in zip(host, dev, back):
        assert d.is_cuda and d.shape == h.shape and d.dtype == h.dtype and torch.equal(b, h)
        assert d.numel() == 0 or d.data_ptr() % 256 == 0
    assert ops.upload([], gpu_device) == [] and ops.download([]) == []


@pytest.mark.gpu
def test_an_array_that_was_replaced_is_given_back(gpu_device):
    """However long the arrays live that were uploaded with it."""
    import torch

    from autoparallel_amd import _native

    big = torch.zeros(8 << 20, dtype=torch.uint8)
    before = torch.cuda.memory_allocated(gpu_device)
    a, small, b = _native.torch_ops().upload([big, torch.zeros(9), big], gpu_device)
    del a, b
    assert torch.cuda.memory_allocated(gpu_device) - before < 1 << 20 and not small.any()


@pytest.mark.gpu
def test_what_a_large_transfer_brings_is_an_ordinary_tensor(gpu_device):
    """Arrays of 32 MiB and more, cut over the threads' parts: in memory that torch can resize, as every other."""
    import torch

    from autoparallel_amd import _native

    sizes = [(32 << 20) - 1, 32 << 20, (40 << 20) + 3, 100]
    dev = [torch.randint(0, 256, (n,), dtype=torch.uint8, device=gpu_device) for n in sizes]
    for back, there in zip(_native.torch_ops().download(dev), dev):
        want = there.cpu()
        assert torch.equal(back, want) and back.untyped_storage().resizable()
        grown = back.resize_(len(back) + 5)
        assert torch.equal(grown[:-5], want)

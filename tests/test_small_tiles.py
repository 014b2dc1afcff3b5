"""Packed tiles by few lanes each: 16, 32 or 64 instead of a workgroup (``CostTables.packed_lanes``)."""

import ctypes

import numpy as np
import pytest
import torch

from autoparallel_amd import CostModelParams, _native
from autoparallel_amd.device_tables import DeviceCostTables
from autoparallel_amd.encoding import PACKED_MANY_TILES
from autoparallel_amd.graphs.cost_inputs import StrategyRecipes
from autoparallel_amd.synthetic import stress_dag
from oracle import c_oracle
from oracle import cost_oracle as po
from test_abi_and_encoding import twin_graph

MESHES = [(64,), (6,), (32, 8), (12, 6), (8, 8, 8), (6, 4, 2), (2, 4, 2, 2), (3, 2, 2, 2)]


def _tables(mesh, nodes, lo, hi, seed=3):
    odd = int(np.lcm.reduce([m // (m & -m) for m in mesh]))
    tb = stress_dag(seed=seed, n_nodes=nodes, mesh_sizes=tuple(1 << (m - 1).bit_length() for m in mesh), min_strategies=lo, max_strategies=hi)
    tb.mesh_sizes = mesh
    live = np.arange(tb.tensor_shape.shape[1])[None, :] < tb.tensor_rank[:, None]
    tb.tensor_shape[live] *= odd
    # a third of the tensors with the strides of another layout, some with an empty dim
    tb.tensor_stride[::3] = tb.tensor_stride[::3, ::-1]
    tb.tensor_shape[5::11, 0] = 0
    tb.build_tiles(None, dedupe=True)
    return tb


@pytest.mark.parametrize("mesh", [(64,), (3, 2, 2, 2)])
def test_lanes_are_those_that_take_a_tile_at_once(mesh):
    few, many = (_tables(mesh, n, 1, 4) for n in (100, 3000))
    assert few.packed_lanes() == 64 and many.n_tiles > PACKED_MANY_TILES and many.packed_lanes() == 16
    assert _tables(mesh, 3000, 5, 5).packed_lanes() == 32  # 5 x 5: three rows of 16 lanes, six of 32
    assert _tables(mesh, 300, 1, 8).packed_lanes() == 64  # 8 x 8
    assert _tables(mesh, 300, 1, 11).packed_lanes() == 256  # 11 x 11: three rounds of five rows
    # 10 x 10: two rounds of six rows, by a wavefront on meshes of many states; no reason to leave staged tiles
    twice = _tables(mesh, 2500, 1, 10)
    assert twice.packed_lanes() == (64 if len(mesh) > 1 else 256) and not twice.small_packing_pays()
    assert few.small_packing_pays() and many.small_packing_pays()
    many.tile_records = many.tile_records[:0]
    assert many.packed_lanes() == 256


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", MESHES)
@pytest.mark.parametrize("nodes,lo,hi", [(37, 1, 4), (90, 2, 5), (61, 1, 8), (150, 1, 16)])
def test_every_number_of_lanes_has_the_oracles_bits(gpu_device, monkeypatch, mesh, nodes, lo, hi):
    """Tiles of one round of lanes and of several, numbers of tiles that leave the last wavefront partly empty, copies, pass-through
    entries, layouts and empty dims: the oracle's costs, row minima, compute costs and tensor bytes."""
    tb = _with_copies(_tables(mesh, nodes, lo, hi))
    tb.build_tiles(None, dedupe=True)
    assert len(np.unique(tb.tile_records["dup_count"])) > 3
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"]
    lowest, where = c_oracle.segmented_min(want, tb.row_ptr())
    kept = None
    for lanes in (256, 64, 32, 16):
        monkeypatch.setattr(tb, "packed_lanes", lambda: lanes)
        d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
        step = d.prepare_step(fused_inputs=True, one_launch=True, row_min_in_tiles=True, outputs=("cost",), spec_table=False, packed=True)
        for t in (d.cost, d.row_min, d.row_argmin):
            t.fill_(-1)
        for launch in step.values():
            launch()
        torch.cuda.synchronize()
        for got, expected in ((d.cost, want), (d.row_min, lowest), (d.row_argmin, where)):
            assert np.array_equal(got.cpu().numpy(), expected), lanes
        rest = [t.cpu().numpy() for t in (d.compute_cost, d.compute_cost_per_arg, d.tensor_bytes, d.tensor_contiguous)]
        kept = kept or rest
        assert all(np.array_equal(a, b) for a, b in zip(rest, kept))


def _packed_pass(tb, mesh, device, monkeypatch, lanes):
    monkeypatch.setattr(tb, "packed_lanes", lambda: lanes)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=device)
    step = d.prepare_step(fused_inputs=True, one_launch=True, row_min_in_tiles=True, outputs=("cost",), spec_table=False, packed=True)
    for t in (d.cost, d.row_min, d.row_argmin):
        t.fill_(-1)
    for launch in step.values():
        launch()
    torch.cuda.synchronize()
    return d


def _with_copies(tb, seed=1):
    """Eight copies of every node and edge, of which some have another strategy table: from none to seven identical edges to a tile."""
    for _ in range(3):
        tb = twin_graph(tb)
    nodes = np.random.default_rng(seed).random(tb.n_nodes) < np.linspace(0, 0.6, tb.n_nodes)
    changed = np.repeat(nodes, np.diff(tb.node_strat_begin))
    tb.strat_rw_bytes[changed] += 1 + np.arange(tb.n_strategies)[changed] // 3
    return tb


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", [(64,), (12, 6), (8, 8, 8), (3, 2, 2, 2)])
@pytest.mark.parametrize("most", [16, 32])
def test_copies_and_sides_up_to_the_lanes(gpu_device, monkeypatch, mesh, most):
    """Single rows of up to as many columns as lanes (over both halves of 32), single columns and tiles between, next to each other in a
    wavefront with different numbers of copies."""
    tb = _with_copies(_tables(mesh, 40, 1, most, seed=most))
    tb.build_tiles(most, dedupe=True)
    rows, cols, copies = tb.tile_row_count, tb.tile_col_count, tb.tile_records["dup_count"]
    assert rows.max() == cols.max() == most and (rows == 1).any() and (cols == 1).any() and len(np.unique(copies)) >= 6
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"]
    lowest, where = c_oracle.segmented_min(want, tb.row_ptr())
    wide = where[np.isfinite(lowest) & (np.diff(tb.row_ptr()) > 16)]
    assert most == 16 or ((wide >= 16).any() and (wide < 16).any())
    for lanes in (256, 64, 32, 16)[:4 if most == 16 else 3]:
        d = _packed_pass(tb, mesh, gpu_device, monkeypatch, lanes)
        for got, expected in ((d.cost, want), (d.row_min, lowest), (d.row_argmin, where)):
            assert np.array_equal(got.cpu().numpy(), expected), lanes


@pytest.mark.gpu
@pytest.mark.parametrize("lanes", [16, 32])
def test_a_tile_larger_than_its_lanes_is_reported(gpu_device, monkeypatch, lanes):
    """The entries of the others are the oracle's, those of the larger ones are left alone, and the error flag says so."""
    mesh = (12, 6)
    tb = _tables(mesh, 60, 1, lanes + 8)
    tb.build_tiles(lanes, dedupe=False)
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"]
    large = np.zeros(tb.n_entries, bool)
    counts = tb.tile_records["counts"]
    for e, row, n in zip(tb.tile_edge, tb.tile_row_begin, counts):
        cols, first = n >> 16, tb.edge_entry_begin[e] + row * (n >> 16)
        large[first:first + (n & 0xFFFF) * cols] = max(n & 0xFFFF, cols) > lanes
    assert large.any() and not large.all()
    d = _packed_pass(tb, mesh, gpu_device, monkeypatch, lanes)
    got = d.cost.cpu().numpy()
    assert np.array_equal(got[~large], want[~large]) and (got[large] == -1).all()
    with pytest.raises(RuntimeError, match="fewer lanes"):
        d._check_flag(int(d._step_error_flag.item()))
    d = _packed_pass(tb, mesh, gpu_device, monkeypatch, 64)
    d._check_flag(int(d._step_error_flag.item()))
    assert np.array_equal(d.cost.cpu().numpy(), want)


@pytest.mark.parametrize("lanes,through_the_operator", [(0, False), (8, False), (128, False), (-16, False), (8, True), ((1 << 32) + 16, True)])
def test_other_numbers_of_lanes_are_refused(lanes, through_the_operator):
    """On the CPU; 2^32 + 16 is not 16."""
    params = CostModelParams.from_mesh((4,)).to_c()
    if through_the_operator:
        t = torch.empty(0)
        with pytest.raises(RuntimeError, match="lanes a tile"):
            _native.torch_ops().bind_cost_tables_packed(_native.params_tensor(params), *[t] * 16, 0, 0, *[t] * 3, lanes)
        return
    null, none = ctypes.c_void_p(None), ctypes.c_int64(0)
    call = lambda n: _native.lib().apc_build_tables_packed_small(  # noqa: E731
        ctypes.byref(params), none, *[null] * 6, none, *[null] * 9, none, null, none, *[null] * 3, ctypes.c_int32(n), null)
    assert call(lanes) != 0 and b"lanes a tile" in _native.lib().apc_last_error()
    assert [call(n) for n in (16, 32, 64, 256)] == [0] * 4


@pytest.mark.gpu
def test_small_tiles_under_capture(gpu_device):
    """A table that goes over few lanes a tile: a captured pass finds the tiles of an earlier preparation, or, where that was over staged
    tiles, goes over those."""
    mesh = (64,)
    tb = _tables(mesh, 2200, 1, 4)
    assert tb.small_packing_pays() and tb.staging_pays(tb.computed_entries(), tb.n_tiles)
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"]
    for before in (None, False):
        d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
        assert d.row_min_in_tiles_pays()
        d.planner_pass(packed=before)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step = d.planner_pass()
            for launch in step.values():
                launch()
        assert list(step) == ["build_tables" if before is False else "build_tables_packed"]
        for _ in range(3):
            d.cost.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(d.cost.cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("change", ["tiling", "tables", "tables of two lengths", "strategy inputs", "changed on the host", "prepared for one run"])
def test_a_capture_after_a_change_of_small_tiles(gpu_device, change):
    """A table that goes over few lanes a tile though it could be staged, one of whose tables or whose tiling is another before a pass is
    captured, with no preparation between the two: it has the costs of the tables as they are then."""
    mesh = (64,)
    tb = _tables(mesh, 2200, 1, 4)
    assert tb.small_packing_pays() and tb.staging_pays(tb.computed_entries(), tb.n_tiles)
    op = po.make_params(mesh, rescale=2.2)
    before = c_oracle.build_tables(tb.as_dict(), op)["cost"]
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    if change == "changed on the host":  # (not uploaded: the pass is of the host's tables, and staged tiles are no way out)
        tb.strat_rw_bytes *= 2
    d.planner_pass()
    repeated = change != "prepared for one run"
    if not repeated:
        d.planner_pass(repeated=False)
    packed = d._packed_cache
    assert packed is not None and (change == "changed on the host") == (d._edge_rows is None)
    if change == "tiling":
        tb.build_tiles(None, dedupe=True, max_copies=2)
        d.refresh("tile_records", "dup_entry_begin", "dup_row_begin")
    elif change == "strategy inputs":  # (the device counts, and the host's table receives the result)
        recipes = StrategyRecipes(tb.n_nodes)
        recipes.node_kind[:] = 1
        recipes.node_row_begin[:] = np.arange(tb.n_nodes + 1)
        recipes.byte_rows = np.zeros(tb.n_nodes, np.int32)
        for name, t in zip(("strat_flops", "strat_rw_bytes", "strat_dtype", "strat_zero_cost"), d.run_strategy_inputs(recipes)):
            getattr(tb, name)[:] = t.cpu().numpy()
    else:
        tb.strat_flops[:] = 0
        if change == "tables of two lengths":
            kept, tb.strat_flops = tb.strat_flops, np.append(tb.strat_flops, 0)
            d.refresh("strat_flops")
            tb.strat_flops = kept
        d.refresh("strat_flops")
    # what a pass has no choice but to go over is made again at once, and nothing where staged tiles are one
    assert (d._packed_cache is not None) == (change in ("changed on the host", "prepared for one run"))
    want = c_oracle.build_tables(tb.as_dict(), op)["cost"]
    assert change == "tiling" or not np.array_equal(want, before)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step = d.planner_pass(repeated=repeated)
        for launch in step.values():
            launch()
    assert list(step) == ["build_tables" if d._packed_cache is None else "build_tables_packed"]
    for _ in range(3):
        d.cost.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(d.cost.cpu().numpy(), want)
    step = d.planner_pass()  # the next preparation is over packed tiles again
    assert list(step) == ["build_tables_packed"]
    for launch in step.values():
        launch()
    torch.cuda.synchronize()
    assert np.array_equal(d.cost.cpu().numpy(), want)


@pytest.mark.gpu
def test_a_tiling_that_is_refused_leaves_the_small_tiles_as_they_were(gpu_device, monkeypatch):
    monkeypatch.setattr(DeviceCostTables, "CHECK_ON_DEVICE_MIN_ROWS", 0)
    tb = _tables((64,), 2200, 1, 4)
    d = DeviceCostTables(tb, CostModelParams.from_mesh((64,), rescale=2.2), device=gpu_device)
    d.planner_pass()
    packed = d._packed_cache
    assert packed is not None and d._packed_stands_in
    tb.tile_records["row_begin"][3] += 10**6
    with pytest.raises(RuntimeError):
        d.refresh_tiling("tile_records", "dup_entry_begin", "dup_row_begin")
    tb.tile_records["row_begin"][3] -= 10**6
    assert d._packed_cache is packed and d._packed_stands_in
    d.refresh("strat_flops")
    assert d._packed_cache is None

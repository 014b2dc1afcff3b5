"""Tilings chosen from the table: every entry is computed once, the cut follows the rules, and the
pass over it gives the oracle's bits."""

import numpy as np
import pytest
import torch

from autoparallel_amd import CostModelParams, encoding
from autoparallel_amd.device_tables import DeviceCostTables
from autoparallel_amd.optimize_sharding import DeviceBackend
from autoparallel_amd.synthetic import stress_dag
from oracle import c_oracle
from oracle import cost_oracle as po
from test_abi_and_encoding import twin_graph

# mesh, nodes, largest strategy count, twin graphs made one table (identical edges)
TABLES = [((8, 4), 40, 8, 0), ((8, 4), 400, 48, 0), ((12, 6), 300, 64, 0), ((12, 6), 60, 90, 0), ((4, 2, 2), 400, 48, 1),
          ((6, 4, 2), 200, 65, 0), ((3, 2, 2, 2), 300, 48, 0), ((2, 4, 2, 2), 60, 130, 0), ((64,), 300, 4, 0)]


def _table(mesh, nodes, hi, twins):
    tb = stress_dag(seed=hi, n_nodes=nodes, mesh_sizes=mesh, min_strategies=1, max_strategies=hi, frac_nonspec_nodes=0.02,
                    frac_noncontiguous=0.2)
    for _ in range(twins):
        tb = twin_graph(tb)
    return tb


@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("mesh,nodes,hi,twins", TABLES)
def test_automatic_cut_follows_its_rules(mesh, nodes, hi, twins, large, monkeypatch):
    if large:  # (the rules of large tables on tables of the test's size)
        monkeypatch.setattr(encoding, "AUTO_SMALL_TABLE_ENTRIES", 0)
    tb = _table(mesh, nodes, hi, twins)
    tb.build_tiles(None, dedupe=True)
    tb.validate(CostModelParams.from_mesh(mesh))
    seen = np.zeros(tb.n_entries, np.int32)
    for e, r0, nr, c0, nc in zip(tb.tile_edge, tb.tile_row_begin, tb.tile_row_count, tb.tile_col_begin, tb.tile_col_count):
        at = slice(int(tb.edge_dup_begin[e]), int(tb.edge_dup_begin[e] + tb.edge_dup_count[e]))
        within = (np.arange(r0, r0 + nr)[:, None] * int(tb.edge_n_src[e]) + np.arange(c0, c0 + nc)[None, :]).ravel()
        for begin in (int(tb.edge_entry_begin[e]), *tb.dup_entry_begin[at].tolist()):
            seen[begin + within] += 1
    assert (seen == 1).all()
    computed = tb.computed_entries()
    fits = int(tb.edge_n_src.max()) <= encoding.APC_TILE_MAX_COLS
    packed = tb.tiling.get("rows_per_wavefront_pass") == 4
    te = tb.tiling["tile_entries"]
    if large:
        assert not packed and (tb.n_entries >= tb.n_tiles * encoding.AUTO_MIN_STORED_PER_TILE or te == 4096)
    else:
        assert packed == (fits and not tb.staging_pays(computed, tb.n_tiles))
    # what a planner finds taken does not depend on how the edges were cut further
    other = _table(mesh, nodes, hi, twins)
    other.build_tiles(4096, dedupe=True, rows_per_wavefront_pass=None if large else 4)
    assert tb.tiling["whole_edges"] == (other.n_tiles, other.computed_entries())


@pytest.mark.parametrize("many,te", [(100_000, 2048), (100, 4096)])
def test_tiles_are_cut_larger_when_there_are_many_anyway(many, te, monkeypatch):
    monkeypatch.setattr(encoding, "AUTO_SMALL_TABLE_ENTRIES", 0)
    monkeypatch.setattr(encoding, "AUTO_MANY_TILES", many)
    tb = stress_dag(seed=3, n_nodes=400, mesh_sizes=(16, 8, 4))  # (what the stress table is a larger one of)
    tb.build_tiles(None, dedupe=True)
    assert tb.tiling["tile_entries"] == te and tb.n_tiles > 100
    tb.validate(CostModelParams.from_mesh((16, 8, 4)))


def test_tile_sizes_for_launches_that_go_edge_by_edge(monkeypatch):
    """The larger tiles of a table whose repeated pass takes them by size are not for a pass that runs once, which the
    planner's is."""
    monkeypatch.setattr(encoding, "AUTO_SMALL_TABLE_ENTRIES", 0)
    monkeypatch.setattr(encoding, "ORDERED_SOME_ROUNDS", 100)
    mesh = (16, 8, 4)
    tb = stress_dag(seed=3, n_nodes=300, mesh_sizes=mesh, min_strategies=4, max_strategies=64, fanout_lambda=2.0)
    tb.build_tiles(None, dedupe=True)
    assert tb.largest_tiles_first_pays() and tb.tiling["tile_entries"] == 4096
    whole = tb.tiling["whole_edges"]
    tb.build_tiles(None, dedupe=True, repeated=False)
    assert tb.tiling["tile_entries"] == 2048 and tb.tiling["whole_edges"] == whole
    tb.validate(CostModelParams.from_mesh(mesh))
    asked = tb.tile_records.copy()

    class Device:
        params = CostModelParams.from_mesh(mesh)

        def refresh(self, *names):
            pass

    tb.build_tiles(None, dedupe=True)
    backend = object.__new__(DeviceBackend)
    backend.dev = Device()
    backend.upload_strategy_inputs(tb)
    assert np.array_equal(tb.tile_records, asked)


@pytest.mark.gpu
@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("mesh,nodes,hi,twins", TABLES)
def test_pass_over_the_automatic_cut_matches_the_oracle(gpu_device, mesh, nodes, hi, twins, large, monkeypatch):
    if large:
        monkeypatch.setattr(encoding, "AUTO_SMALL_TABLE_ENTRIES", 0)
    tb = _table(mesh, nodes, hi, twins)
    tb.build_tiles(None, dedupe=True)
    op = po.make_params(mesh, rescale=2.2)
    want = c_oracle.build_tables(tb.as_dict(), op)
    params = CostModelParams.from_mesh(mesh, rescale=2.2)
    for limit in (0, DeviceCostTables.ONE_LAUNCH_MAX_BYTES):  # input tables in front, or everything in one launch
        monkeypatch.setattr(DeviceCostTables, "ONE_LAUNCH_MAX_BYTES", limit)
        d = DeviceCostTables(tb, params, device=gpu_device)
        step = d.planner_pass()
        assert len(step) == (1 if limit else 2)
        for launch in step.values():
            launch()
        torch.cuda.synchronize()
        assert np.array_equal(d.cost.cpu().numpy(), want["cost"])
        assert np.array_equal(d.compute_cost_per_arg.cpu().numpy(), c_oracle.compute_costs(tb.as_dict(), op)[1])
        if d.row_min is not None:
            mins, args = c_oracle.segmented_min(want["cost"], tb.row_ptr())
            assert np.array_equal(d.row_min.cpu().numpy(), mins) and np.array_equal(d.row_argmin.cpu().numpy(), args)


@pytest.mark.parametrize("mesh,limit,of_many", [((64,), 344, 128), ((32, 8), 344, 128), ((8, 8, 8), 192, 128), ((2, 4, 2, 2), 192, 128),
                                                ((3, 2, 2, 2), 128, 128)])
def test_bytes_of_the_largest_pass_in_one_launch(mesh, limit, of_many):
    d = object.__new__(DeviceCostTables)
    d.tables = _table(mesh, 40, 4, False)
    assert d.one_launch_limit() == limit << 20
    assert d.one_launch_limit(row_min_in_tiles=True) == min(limit, 256) << 20
    d.ONE_LAUNCH_MANY_TILES = d.tables.n_tiles
    assert d.one_launch_limit() == limit << 20
    d.ONE_LAUNCH_MANY_TILES -= 1
    assert d.one_launch_limit() == of_many << 20
    for asked in (0, 1 << 20, 1 << 40):  # (what a program sets is the limit on every mesh)
        d.ONE_LAUNCH_MAX_BYTES = asked
        assert d.one_launch_limit() == d.one_launch_limit(row_min_in_tiles=True) == asked


@pytest.mark.parametrize("mesh,at_30,below", [((6, 4, 2), True, False), ((8, 4, 2), True, True), ((12, 6), True, True), ((3, 2, 2, 2), False, False),
                                              ((2, 4, 2, 2), True, True)])
def test_staging_of_small_matrices(mesh, at_30, below):
    """Many tiled edges of few entries each, with and without copies; a pass that runs once is over packed tiles either way."""
    tb = _table(mesh, 40, 4, False)
    edges = 3000
    for copies in (1, 5):
        tb.edge_entry_begin[-1] = 30 * edges * copies
        for computed, want in ((30 * edges, at_30), (30 * edges - 1, below)):
            assert tb.staging_pays(computed, edges, edges) == tb._staging_may_pay(computed, edges, True) == want
            assert tb.staging_pays(computed, edges, 0) == (want if copies == 1 or computed * 6 >= tb.n_entries else False)
            assert not tb.staging_pays(computed, edges, edges, repeated=False)

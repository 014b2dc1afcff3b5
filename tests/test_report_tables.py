"""The launches of a report: first rows of the edges, greedy strategies in one launch, both tables' launches behind one wait."""

import numpy as np
import pytest
import torch

from autoparallel_amd import CostModelParams, _native
from autoparallel_amd.device_tables import DeviceCostTables
from autoparallel_amd.optimize_sharding import DeviceBackend
from autoparallel_amd.synthetic import stress_dag

from oracle import c_oracle
from oracle import cost_oracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 2, 1023, 1024, 1025, 4095, 4096, 4097, 8195, 16_383, 16_384, 16_385, 32_771, 210_003])
def test_first_rows_of_the_edges(gpu_device, n):
    """Sums beyond 32 bits within a thread's edges, across a wavefront, across the wavefronts and from block to block."""
    n_tgt = np.random.default_rng(n).integers(0, 90, n).astype(np.int32)
    n_tgt[n // 3:n // 3 + 4] = 2**31 - 1
    n_tgt[n // 2::37] = 1 << 30
    n_tgt[-1:] = 0
    want = np.cumsum(n_tgt.astype(np.int64)) - n_tgt
    assert n < 1000 or (want > 2**33).sum() > n // 3
    got = _native.torch_ops().edge_rows(torch.from_numpy(n_tgt).to(gpu_device))
    assert got.dtype == torch.int64 and np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("group", [None, 1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("most", [1, 3, 40, 700])
def test_greedy_strategies_are_the_two_launches(gpu_device, group, most, monkeypatch):
    """Nodes without strategies or edges, odd counts, ties, infinities and NaN: the bits of bounds and segmented minimum."""
    if group:
        monkeypatch.setenv("APC_SEGMIN_GROUP", str(group))
    rng = np.random.default_rng(most)
    n_nodes = 301
    n_strat = rng.integers(0, most + 1, n_nodes)
    n_edges_of = rng.integers(0, 4, n_nodes)
    begin = np.concatenate([[0], np.cumsum(n_strat)])
    edge_begin = np.concatenate([[0], np.cumsum(n_edges_of)])
    owner = np.repeat(np.arange(n_nodes), n_edges_of)
    rows = np.cumsum(n_strat[owner]) - n_strat[owner]
    order = rng.permutation(len(owner))  # (edges numbered in another order than the nodes')
    row_begin = np.empty(len(owner), np.int64)
    row_begin[order] = rows
    row_min = rng.integers(0, 5, int(n_strat[owner].sum())).astype(np.float64)
    row_min[rng.random(len(row_min)) < 0.1] = np.inf
    row_min[rng.random(len(row_min)) < 0.02] = np.nan
    on = [torch.from_numpy(np.ascontiguousarray(a)).to(gpu_device) for a in (
        begin.astype(np.int64), edge_begin.astype(np.int64), order.astype(np.int32), row_begin, row_min)]
    ops = _native.torch_ops()
    strat_node = torch.from_numpy(np.repeat(np.arange(n_nodes, dtype=np.int32), n_strat)).to(gpu_device)
    want = ops.strategy_bounds(strat_node, *on)
    want_min, want_arg = ops.segmented_min(want, on[0])
    bound, node_min, node_arg = ops.greedy_strategies(*on, int(begin[-1]))
    for got, ref in ((bound, want), (node_min, want_min)):
        assert torch.equal(got.view(torch.int64), ref.view(torch.int64))
    assert torch.equal(node_arg, want_arg)


@pytest.mark.parametrize("group", [None, 1, 8])
@pytest.mark.parametrize("most,edges", [(2, 9), (4, 5), (9, 13), (70, 6)])
def test_greedy_strategies_of_nodes_of_many_edges(gpu_device, group, most, edges, monkeypatch):
    """Sums over more edges than a lane has in flight, in their order: magnitudes of which another order has other bits."""
    if group:
        monkeypatch.setenv("APC_SEGMIN_GROUP", str(group))
    rng = np.random.default_rng(most + edges)
    n_nodes = 97
    n_strat, n_edges_of = rng.integers(0, most + 1, n_nodes), rng.integers(0, edges + 1, n_nodes)
    begin, edge_begin = (np.concatenate([[0], np.cumsum(a)]).astype(np.int64) for a in (n_strat, n_edges_of))
    owner = np.repeat(np.arange(n_nodes), n_edges_of)
    row_begin = (np.cumsum(n_strat[owner]) - n_strat[owner]).astype(np.int64)
    row_min = 10.0 ** rng.uniform(-9, 9, int(n_strat[owner].sum()))
    row_min[rng.random(len(row_min)) < 0.05] = np.nan
    on = [torch.from_numpy(a).to(gpu_device) for a in (begin, edge_begin, np.arange(len(owner), dtype=np.int32), row_begin, row_min)]
    want = np.zeros(int(begin[-1]))
    for n in range(n_nodes):
        for e in range(edge_begin[n], edge_begin[n + 1]):
            want[begin[n]:begin[n + 1]] += row_min[row_begin[e]:row_begin[e] + n_strat[n]]
    ops = _native.torch_ops()
    bound, node_min, node_arg = ops.greedy_strategies(*on, int(begin[-1]))
    assert np.array_equal(bound.cpu().numpy(), want, equal_nan=True)
    for got, ref in zip((node_min, node_arg), ops.segmented_min(bound, on[0])):
        assert np.array_equal(got.cpu().numpy(), ref.cpu().numpy(), equal_nan=got.is_floating_point())


@pytest.mark.parametrize("n_nodes", [2, 60, 1100])
@pytest.mark.parametrize("row_min", [False, True])
def test_inputs_of_a_report_are_those_of_the_single_launches(gpu_device, n_nodes, row_min, monkeypatch):
    """Tensors and strategies below and beyond a workgroup, with and without the edges' first rows; the flag of the last strategy alone."""
    tb = stress_dag(seed=8, n_nodes=n_nodes, mesh_sizes=(4, 2))
    tb.build_tiles(None, dedupe=True)
    d = DeviceCostTables(tb, CostModelParams.from_mesh((4, 2)), device=gpu_device)
    monkeypatch.setattr(d, "row_min_in_tiles_pays", lambda: row_min)
    d.build_all()
    got = [d.tensor_bytes, d.tensor_contiguous, d.compute_cost, d.compute_cost_per_arg]
    for a, b in zip(got, (*d.run_tensor_tables(), *d.run_compute_costs())):
        assert torch.equal(a, b)
    if row_min:
        for a, b in zip((d.row_min, d.row_argmin), d.segmented_min(d.cost, tb.row_ptr())):
            assert torch.equal(a, b)
    tb.strat_flops[-1], tb.strat_dtype[-1], tb.strat_zero_cost[-1] = 1, 7, 0
    d.refresh("strat_flops", "strat_dtype", "strat_zero_cost")
    with pytest.raises(ValueError, match="dtype not supported"):
        d.build_all()


def test_an_unsupported_dtype_is_refused(gpu_device):
    tb = stress_dag(seed=5, n_nodes=200, mesh_sizes=(4, 2))
    params = CostModelParams.from_mesh((4, 2))
    d = DeviceCostTables(tb, params, device=gpu_device)
    kept = d.build_all()
    tb.strat_dtype[tb.strat_flops > 0] = 7
    tb.strat_zero_cost[:] = 0
    d.refresh("strat_dtype", "strat_zero_cost")
    with pytest.raises(ValueError, match="dtype not supported"):
        d.build_all()
    assert d.cost is kept[2] and bool(torch.isnan(d.compute_cost).any())


EDGE_ARRAYS = ("edge_src_begin", "edge_n_src", "edge_tgt_begin", "edge_n_tgt", "edge_flags", "edge_strat_begin")


@pytest.mark.parametrize("how", ["build_all", "run_redistribute_tables", "upload_strategy_inputs"])
def test_edge_arrays_of_another_integer_type(gpu_device, how, monkeypatch):
    """Set after the construction: the host converts them where it reads them, and no kernel reads them."""
    monkeypatch.setattr(DeviceCostTables, "CHECK_ON_DEVICE_MIN_ROWS", 0)
    mesh = (4, 2)
    tb = stress_dag(seed=5, n_nodes=200, mesh_sizes=mesh)
    tb.build_tiles(None, dedupe=True)
    backend = DeviceBackend(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    d = backend.dev
    for name in EDGE_ARRAYS:
        setattr(tb, name, getattr(tb, name).astype(np.int64))
    d.refresh(*EDGE_ARRAYS)
    if how == "build_all":
        d.build_all()
    elif how == "run_redistribute_tables":
        d.run_redistribute_tables(row_min=True)
    else:
        backend.upload_strategy_inputs(tb)
        backend.launch_tables()
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"]
    assert np.array_equal(d.cost.cpu().numpy(), want)
    want_min, want_arg = c_oracle.segmented_min(want, tb.row_ptr())
    assert d.row_min is not None
    assert np.array_equal(d.row_min.cpu().numpy(), want_min) and np.array_equal(d.row_argmin.cpu().numpy(), want_arg)


def test_the_rows_of_a_report_from_the_host_and_the_device(gpu_device):
    mesh = (4, 2)
    tb = stress_dag(seed=5, n_nodes=200, mesh_sizes=mesh)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh), device=gpu_device)

    def report(n_tgt, n_rows):
        return d.ops.report_tables(
            d.p, *d._tensor_table(), d.d["spec_codes"], d.d["spec_tensor"], *d._strategy_table(), d.d["pt_values"], d.d["tile_records"],
            d.d["dup_entry_begin"], tb.n_entries, n_tgt, d.d["dup_row_begin"], n_rows)[0]

    on_host = torch.from_numpy(tb.edge_n_tgt)
    for a, b in zip(report(on_host, tb.n_rows), report(on_host.to(gpu_device), tb.n_rows)):
        assert torch.equal(a, b)
    for n_tgt, n_rows in ((on_host.long(), tb.n_rows), (on_host, tb.n_rows - 1), (on_host[:-1], tb.n_rows)):
        with pytest.raises(RuntimeError, match="edge_n_tgt"):
            report(n_tgt, n_rows)

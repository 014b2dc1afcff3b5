"""The launches of a report: first rows of the edges, greedy strategies in one launch, both tables' launches behind one wait."""

import numpy as np
import pytest
import torch

from autoparallel_amd import CostModelParams, _native
from autoparallel_amd.device_tables import DeviceCostTables
from autoparallel_amd.synthetic import stress_dag

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 2, 1023, 1024, 1025, 70_001])
def test_first_rows_of_the_edges(gpu_device, n):
    n_tgt = np.random.default_rng(n).integers(0, 90, n).astype(np.int32)
    if n > 2:
        n_tgt[n // 2] = 1 << 22  # (sums beyond 32 bits)
        n_tgt[-1] = 0
    n_tgt = np.tile(n_tgt, 1 if n < 2000 else 3)
    got = _native.torch_ops().edge_rows(torch.from_numpy(n_tgt).to(gpu_device))
    assert got.dtype == torch.int64 and np.array_equal(got.cpu().numpy(), np.cumsum(n_tgt.astype(np.int64)) - n_tgt)


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

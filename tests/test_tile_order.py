"""Which workgroup takes which tile: every tile once, whatever their number."""

import numpy as np
import pytest
import torch

from autoparallel_amd import CostModelParams, _native
from autoparallel_amd.device_tables import DeviceCostTables
from autoparallel_amd.encoding import TILE_DTYPE, partial_code, shard_code
from autoparallel_amd.synthetic import stress_dag
from oracle import c_oracle
from oracle import cost_oracle as po
from test_abi_and_encoding import twin_graph
from test_gpu_parity import _run_and_compare, _two_node_tables


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 7, 8, 9, 255, 256, 257, 263, 264, 511, 513, 1023, 1025, 2049])
def test_every_tile_has_a_workgroup(gpu_device, n):
    """Tile counts around a round of runs (32 tiles for each of the 8 XCDs) and around the XCDs, over the three kinds of launch."""
    tgt = [(shard_code(0), 0), (0, partial_code(0)), (shard_code(1), shard_code(0))]
    tb = _two_node_tables((4, 2), [64, 64], [64, 1], 2, [(0, shard_code(1))], [tgt[k % 3] for k in range(n)], flops=1000, rw=500)
    tb.build_tiles(1)
    assert tb.n_tiles == n
    _run_and_compare(tb, (4, 2), 1.0, gpu_device)


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 17, 255, 256, 257, 263, 264, 265, 300, 511, 512, 1000, 2049])
def test_tiles_by_size_are_dealt_one_by_one(n):
    """Every tile keeps its fields; the workgroups in the order of their start meet the tiles by size, as the launch deals them."""
    rng = np.random.default_rng(n)
    records = np.zeros(n, TILE_DTYPE)
    records["edge"], records["counts"] = np.arange(n), rng.integers(1, 65, n) | rng.integers(1, 65, n) << 16
    got = np.empty_like(records)
    _native.host_call("apc_order_tiles_host", n, records, got)
    assert np.array_equal(got, records[got["edge"]]) and np.array_equal(np.sort(got["edge"]), np.arange(n))
    dealt = []  # (tile_of_block)
    for b in range(-(-n // 8) * 8):
        full = n // 256 * 256
        per, within, base = (32, b % 256, b - b % 256) if b < full else (-(-(n - full) // 8), b - full, full)
        dealt.append(base + within % 8 * per + within // 8)
    dealt = [t for t in dealt if t < n]
    assert sorted(dealt) == list(range(n))
    sizes = ((got["counts"] & 0xFFFF) * (got["counts"] >> 16))[dealt]
    assert (np.diff(sizes) <= 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("mesh,nodes,hi", [((12, 6), 200, 64), ((8, 4), 100, 90), ((4, 2, 2), 60, 40)])
def test_passes_over_tiles_by_size(gpu_device, mesh, nodes, hi):
    tb = stress_dag(seed=nodes, n_nodes=nodes, mesh_sizes=mesh, min_strategies=8, max_strategies=hi, frac_nonspec_nodes=0.02)
    tb.build_tiles(None, dedupe=True)
    assert tb.largest_tiles_first_pays() and not np.array_equal(tb.launch_records(), tb.tile_records)
    _run_and_compare(tb, mesh, 2.2, gpu_device)


class _CopyOnly:
    @staticmethod
    def upload(arrays, device):
        return [a.clone() for a in arrays]


def _tiled_twice(mesh):
    """-> (a table, what tiles it a second time, with copies' offsets of its own)."""
    tb = twin_graph(stress_dag(seed=8, n_nodes=150, mesh_sizes=mesh, min_strategies=8, max_strategies=40))
    tb.build_tiles(512, dedupe=True, max_copies=2)
    return tb, lambda: tb.build_tiles(1024, dedupe=False)


@pytest.mark.parametrize("again_first", [False, True])
def test_launch_order_is_of_the_uploaded_tiling(again_first):
    """A table that is tiled anew and not uploaded again: the records a repeated pass takes are the uploaded ones, whose
    copies' offsets are on the device, and the other way round (offsets that the old records do not name)."""
    tb, again = _tiled_twice((12, 6))
    if again_first:
        again()
        again = lambda: tb.build_tiles(512, dedupe=True, max_copies=2)  # noqa: E731
    d = object.__new__(DeviceCostTables)
    d.tables, d.device, d.d, d.ops = tb, torch.device("cpu"), {}, _CopyOnly
    d.refresh("tile_records", "dup_entry_begin", "dup_row_begin")
    uploaded = d.d["tile_records"].numpy().copy().view(TILE_DTYPE).ravel()
    again()
    got = d._tile_records(True).numpy().view(TILE_DTYPE).ravel()
    assert len(got) == len(uploaded) and not np.array_equal(got, uploaded)
    assert np.array_equal(np.sort(got, order=("entry_begin", "row_begin", "col_begin")),
                          np.sort(uploaded, order=("entry_begin", "row_begin", "col_begin")))
    assert int((got["dup_begin"] + got["dup_count"]).max()) <= d.d["dup_entry_begin"].numel()
    assert np.array_equal(d._tile_records(False).numpy().view(TILE_DTYPE).ravel(), uploaded)
    d.refresh("tile_records", "dup_entry_begin", "dup_row_begin")  # ... and of the new one from then on
    assert np.array_equal(d._tile_records(True).numpy().view(TILE_DTYPE).ravel(), tb.launch_records())


@pytest.mark.gpu
@pytest.mark.parametrize("one_launch", [True, False])
def test_passes_over_the_uploaded_tiling(gpu_device, one_launch):
    mesh = (12, 6)
    tb, again = _tiled_twice(mesh)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    again()
    step = d.prepare_step(row_min=True, fused_inputs=True, one_launch=one_launch, row_min_in_tiles=True, outputs=("cost",),
                          spec_table=False, packed=False)
    for launch in step.values():
        launch()
    torch.cuda.synchronize()
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"]
    assert np.array_equal(d.cost.cpu().numpy(), want)
    mins, args = c_oracle.segmented_min(want, tb.row_ptr())
    assert np.array_equal(d.row_min.cpu().numpy(), mins) and np.array_equal(d.row_argmin.cpu().numpy(), args)

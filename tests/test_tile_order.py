"""Which workgroup takes which tile: every tile once, whatever their number."""

import numpy as np
import pytest

from autoparallel_amd import _native
from autoparallel_amd.encoding import TILE_DTYPE, partial_code, shard_code
from autoparallel_amd.synthetic import stress_dag
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

"""Which workgroup takes which tile: every tile once, whatever their number."""

import pytest

from autoparallel_amd.encoding import partial_code, shard_code
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

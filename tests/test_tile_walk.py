"""The walk of a staged tile's lanes over its entries: every width and height where a step, the shift to a line of the output or the
last pass can go wrong, over tables of several edges so that tiles begin anywhere."""

import itertools

import pytest

from autoparallel_amd.encoding import partial_code, shard_code
from test_abi_and_encoding import twin_graph
from test_gpu_parity import _run_and_compare, _two_node_tables


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", [(8,), (4, 2), (3, 2), (2, 3, 2), (2, 2, 2, 2), (3, 2, 2, 2)])
@pytest.mark.parametrize("threads", [64, 128, 256])
def test_tiles_of_every_width(gpu_device, mesh, threads, monkeypatch):
    monkeypatch.setenv("APC_TILE_THREADS", str(threads))
    placements = [0, partial_code(0), shard_code(0), shard_code(1), shard_code(2)]
    every = list(itertools.islice(itertools.cycle(itertools.product(placements, repeat=len(mesh))), 700))
    for k, (ns, nt) in enumerate([(1, 1), (1, 65), (2, 33), (3, 64), (5, 7), (31, 5), (32, 2), (33, 64), (63, 3), (64, 1), (64, 64), (65, 9),
                                  (90, 64), (128, 3), (129, 66)]):
        tb = _two_node_tables(mesh, [96, 48, 36], [1728, 36, 1] if k % 3 else [1, 96, 4608], 2, every[k:k + ns], every[3 * k:3 * k + nt],
                              flags=k % 2, flops=10**9, rw=10**6)
        tb = twin_graph(tb)  # (the second edge begins behind the first one's entries, on no boundary)
        tb.build_tiles((64, 512, 4096)[k % 3], dedupe=k % 2 == 0)
        _run_and_compare(tb, mesh, 2.2, gpu_device)

"""Bytes and contiguity as a tile takes them from the tensor's shape rows (the scan over lanes in doubles, and the integers behind it):
in the launch of all tables, whose tiles derive them, and in the packed one."""

import itertools

import pytest

from autoparallel_amd.encoding import partial_code, shard_code
from test_gpu_parity import _run_and_compare, _two_node_tables


def _contiguous(shape):
    stride, n = [], 1
    for x in reversed(shape):
        stride.append(n)
        n *= max(x, 1)
    return stride[::-1]


def _tensors():
    yield [], [], 8
    yield [5], [1], 2
    yield [1, 64, 1, 32], [7, 32, 9, 1], 4  # (a dim of one element has any stride)
    # up to the last exact product, in bytes and in a stride that the product's neighbour would equal
    for top in (0, 1):
        yield [2**26, 2**26], [2**26 + top, 1], 1
        yield [2, 2**51], [2**51 + top, 1], 1
        yield [2, 2**51], [2**62 + top, 1], 1
        # an empty dim: the stride in front of it is what is behind it, or nothing
        yield [2**30, 0, 2**20], [2**20 + top, 2**20, 1], 2
        yield [2**30, 0, 2**20], [0, 2**20 + top, 1], 2
        yield [2**30, 2**28, 0, 2**30], [2**58 + top, 2**30, 2**30, 1], 2
    eight = [3, 2, 5, 4, 7, 6, 9, 8]
    yield eight, _contiguous(eight), 4
    for k in range(8):  # one stride that does not fit
        stride = _contiguous(eight)
        stride[k] += 1
        yield eight, stride, 4


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", [(8,), (4, 2), (3, 2), (2, 4, 2), (3, 2, 2, 2)])
def test_bytes_and_contiguity_in_tiles(gpu_device, mesh):
    for shape, stride, itemsize in _tensors():
        placements = [0, partial_code(0)] + [shard_code(d) for d in range(min(len(shape), 2))]
        every = list(itertools.islice(itertools.product(placements, repeat=len(mesh)), 24))
        print(mesh, shape, stride, flush=True)
        _run_and_compare(_two_node_tables(mesh, shape, stride, itemsize, every, every[::-1], flops=10**9, rw=10**6), mesh, 2.2, gpu_device)

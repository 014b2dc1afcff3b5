"""The 2-D walk that takes mesh dim 1 first, (Partial, Partial) -> all Shard (collective_runtime_estimation.py:146-151), in the
tiles that look their terms up."""

import itertools

import pytest

from autoparallel_amd.encoding import partial_code, shard_code
from test_gpu_parity import _run_and_compare, _two_node_tables


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", [(4, 8), (5, 3), (6, 1), (1, 7), (65536, 32768)])
@pytest.mark.parametrize("contiguous", [True, False])
@pytest.mark.parametrize("threads,general", [(64, False), (128, False), (256, False), (128, True)])
def test_partial_partial_to_all_shard(gpu_device, mesh, contiguous, threads, general, monkeypatch):
    """Sum and other Partials (only the former's codes flip), consumers that shard every dim, one or none, Shard(0) and others in
    either place; every state the words can name, on the smallest dims, uneven ones and 31 exponents."""
    monkeypatch.setenv("APC_TILE_THREADS", str(threads))
    if general:
        monkeypatch.setenv("APC_GENERAL_TERMS", "1")
    P, A, S0, S1, S2 = partial_code(0), partial_code(1), shard_code(0), shard_code(1), shard_code(2)
    src = [(P, P), (A, P), (P, A), (P, 0), (0, P), (P, S0), (S1, P), (P, P)]
    tgt = list(itertools.product([S0, S1, S2, 0, P], repeat=2))
    shape, stride = [96, 64, 32], [2048, 32, 1] if contiguous else [1, 96, 6144]
    for flags, rescale in ((0, 1.0), (1, 2.2)):
        _run_and_compare(_two_node_tables(mesh, shape, stride, 2, src, tgt, flags=flags), mesh, rescale, gpu_device)

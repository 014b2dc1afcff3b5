"""Row minima taken by the tile kernels themselves: a row is read back by one to sixteen lanes, some rows of a wavefront at a
time, and the result stored to every identical edge by a lane of its own."""

import dataclasses

import numpy as np
import pytest
import torch

from autoparallel_amd import CostModelParams
from autoparallel_amd.device_tables import DeviceCostTables
from autoparallel_amd.encoding import EDGE_NO_PRODUCER, shard_code
from oracle import c_oracle
from oracle import cost_oracle as po
from test_abi_and_encoding import twin_graph
from test_gpu_parity import _two_node_tables

MESH = (4, 2)


def _special(values, rng):
    """Ties, infinities, zeros of both signs, the type's lowest value, and NaN in a row's first column (which no value compares
    below) and in others (which are then passed over)."""
    v = values.copy()
    v[:, :] = np.where(rng.random(v.shape) < 0.5, np.round(v), v)
    for what in (np.inf, -np.inf, np.nan, 0.0, -0.0, np.finfo(np.float64).min):
        v[rng.random(v.shape) < 0.05] = what
    v[rng.random(len(v)) < 0.1] = np.inf
    v[rng.random(len(v)) < 0.1, 0] = np.nan
    v[rng.random(len(v)) < 0.05] = np.nan
    return v


def _same_bits(got, want):
    return np.array_equal(got.view(np.int64), want.view(np.int64))


@pytest.mark.gpu
@pytest.mark.parametrize("threads", [64, 128, 256])
@pytest.mark.parametrize("twins", [0, 1, 4])
def test_row_minima_of_any_values(gpu_device, threads, twins, monkeypatch):
    """Every row length from one entry to a tile's widest, row counts around what a wavefront takes at once and around a
    tile's height, no copies to sixteen: the bits of a scan from left to right."""
    monkeypatch.setenv("APC_TILE_THREADS", str(threads))
    rng = np.random.default_rng(threads + twins)
    for ns, nt in [(1, 1), (1, 130), (2, 64), (3, 1), (4, 257), (7, 65), (8, 63), (15, 40), (16, 34), (17, 33), (31, 17), (32, 64),
                   (33, 9), (47, 5), (62, 66), (63, 16), (64, 1), (64, 64), (64, 129)]:
        tb = _two_node_tables(MESH, [64, 64], [64, 1], 2, [(0, 0)] * ns, [(shard_code(0), 0)] * nt, flags=EDGE_NO_PRODUCER)
        values = _special(100 * rng.standard_normal((nt, ns)), rng)
        tb = dataclasses.replace(tb, pt_values=values.ravel(), edge_pt_begin=np.zeros(1, np.int64))
        for _ in range(twins):
            tb = twin_graph(tb)
        tb.build_tiles(4096, dedupe=True)
        d = DeviceCostTables(tb, CostModelParams.from_mesh(MESH), device=gpu_device)
        # (the values plus a compute cost of 0.0, which makes 0.0 of -0.0: no minimum has a choice of zeros)
        want = c_oracle.build_tables(tb.as_dict(), po.make_params(MESH))["cost"]
        assert np.array_equal(want, np.tile(values.ravel(), 1 << twins), equal_nan=True) and not np.signbit(want[want == 0]).any()
        mins, args = c_oracle.segmented_min(want, tb.row_ptr())
        for one_launch in (True, False):
            step = d.prepare_step(row_min=True, fused_inputs=True, one_launch=one_launch, row_min_in_tiles=True, outputs=("cost",),
                                  spec_table=False, packed=False)
            for launch in step.values():
                launch()
            torch.cuda.synchronize()
            what = (ns, nt, one_launch)
            assert _same_bits(d.cost.cpu().numpy(), want), what
            assert _same_bits(d.row_min.cpu().numpy(), mins), what
            assert np.array_equal(d.row_argmin.cpu().numpy(), args), what

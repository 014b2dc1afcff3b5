"""Launches whose arguments are kept in device memory (``apc_keep_next_launch`` / ``apc_run_kept``, ``BoundLaunch.keep_arguments``)
against the same launches with their arguments passed by value."""

import ctypes
import gc
import os
import re
import shutil
import subprocess
import weakref

import numpy as np
import pytest
import torch

from autoparallel_amd import CostModelParams, _native
from autoparallel_amd.device_tables import DeviceCostTables
from autoparallel_amd.graphs.cost_inputs import StrategyRecipes
from autoparallel_amd.synthetic import stress_dag
from oracle import c_oracle
from oracle import cost_oracle as po


_HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "include", "apcost.h")
_BLOCK_BYTES = int(re.search(r"#define APC_KEPT_BLOCK_BYTES (\d+)", open(_HEADER).read()).group(1))


class _Kept(ctypes.Structure):  # include/apcost.h: apc_kept_launch
    _fields_ = [("kernel", ctypes.c_void_p), ("what", ctypes.c_char_p), ("grid", ctypes.c_uint32), ("threads", ctypes.c_uint32),
                ("lds_bytes", ctypes.c_uint32), ("block_bytes", ctypes.c_uint32), ("work", ctypes.c_void_p),
                ("n_tiles", ctypes.c_int32), ("xcd_shift", ctypes.c_int32), ("tile_blocks", ctypes.c_int64),
                ("cost_out", ctypes.c_void_p), ("block", ctypes.c_int64 * (_BLOCK_BYTES // 8)), ("kernel_by_value", ctypes.c_void_p)]


def _redistribute(lib, params, n_tiles, per_arg):
    one = ctypes.c_void_p(8)  # (a placeholder that is never read: a recorded call launches nothing)
    return lib.apc_redistribute_tables(ctypes.byref(params), one, one, one, one, None, per_arg, ctypes.c_int64(n_tiles), one, None,
                                       ctypes.c_int64(1), None, None, one, None)


def test_recording_a_launch_checks_it_and_ends_with_it():
    """The call after ``apc_keep_next_launch`` is checked as ever; a refused or an empty one leaves nothing to run, and the
    recording ends with that call either way."""
    lib = _native.lib()
    params = CostModelParams.from_mesh((4, 2)).to_c()
    assert lib.apc_keep_next_launch(None) != 0
    kept = _Kept()
    one = ctypes.c_void_p(8)
    assert lib.apc_keep_next_launch(ctypes.byref(kept)) == 0
    assert _redistribute(lib, params, 3, None) != 0 and b"compute_cost_per_arg" in lib.apc_last_error()  # refused
    assert kept.kernel is None
    assert lib.apc_run_kept(ctypes.byref(kept), None, None) == 0  # nothing to launch
    assert _redistribute(lib, params, 0, one) == 0 and kept.kernel is None  # (not recorded: the recording has ended)
    assert lib.apc_keep_next_launch(ctypes.byref(kept)) == 0
    assert _redistribute(lib, params, 0, one) == 0 and kept.kernel is None  # no tiles
    assert lib.apc_keep_next_launch(ctypes.byref(kept)) == 0
    assert _redistribute(lib, params, 3, one) == 0
    assert kept.kernel and kept.what == b"apc_redistribute_tables" and kept.n_tiles == 3 and kept.grid == 8
    assert 0 < kept.block_bytes <= _BLOCK_BYTES and kept.kernel_by_value == kept.kernel  # (a kernel with one form)
    assert lib.apc_run_kept(ctypes.byref(kept), ctypes.c_void_p(8), None) != 0  # the block's alignment
    assert b"64-byte" in lib.apc_last_error()


def test_the_kept_launch_mirrors_the_header(tmp_path):
    fields = [name for name, _ in _Kept._fields_]
    source = "#include <stdio.h>\n#include <stddef.h>\n#include \"apcost.h\"\nint main(void) {\n" + "".join(
        f'printf("%zu ", offsetof(apc_kept_launch, {name}));\n' for name in fields) + 'printf("%zu", sizeof(apc_kept_launch));\nreturn 0; }\n'
    (tmp_path / "layout.c").write_text(source)
    subprocess.run([shutil.which("gcc") or "cc", f"-I{os.path.dirname(_HEADER)}", "-o", str(tmp_path / "layout"), str(tmp_path / "layout.c")],
                   check=True)
    got = [int(x) for x in subprocess.run([str(tmp_path / "layout")], check=True, capture_output=True, text=True).stdout.split()]
    assert got == [getattr(_Kept, name).offset for name in fields] + [ctypes.sizeof(_Kept)]


@pytest.mark.gpu
@pytest.mark.parametrize("form", [dict(packed=True, row_min=True, row_min_in_tiles=True), dict(one_launch=True, packed=False),
                                  dict(one_launch=False, packed=False)])
def test_kept_launches_without_a_block(gpu_device, form):
    """``apc_run_kept`` with a NULL block: the recorded arguments by value, through the form of the kernel that takes them."""
    mesh, lib = (16, 8, 4), _native.lib()
    tb = stress_dag(seed=10, n_nodes=250, mesh_sizes=mesh, max_strategies=20)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    step = d.prepare_step(**dict(dict(row_min=False, fused_inputs=True, outputs=("cost",), spec_table=False), **form), repeated=False)
    d.cost.zero_()
    for launch in step.values():
        kept = _Kept()
        assert lib.apc_keep_next_launch(ctypes.byref(kept)) == 0
        launch()  # (recorded and not enqueued)
        assert kept.kernel and kept.kernel_by_value
        for _ in range(2):
            assert lib.apc_run_kept(ctypes.byref(kept), None, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    torch.cuda.synchronize()
    assert np.array_equal(d.cost.cpu().numpy(), c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"])


def _outputs(d):
    torch.cuda.synchronize()
    arrays = (d.comm, d.transition, d.cost, d.tensor_bytes, d.tensor_contiguous, d.compute_cost, d.compute_cost_per_arg, d.row_min,
              d.row_argmin)
    return [None if t is None else t.cpu().numpy().copy() for t in arrays]


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", [(6,), (32, 8), (12, 6), (16, 8, 4), (2, 3, 2, 2)])
def test_kept_launches_write_what_launches_by_value_write(gpu_device, mesh):
    """Every form of the pass, from the current stream, from another one and from a captured graph (replayed with eager work
    between the replays)."""
    tb = stress_dag(seed=9, n_nodes=250, mesh_sizes=mesh, max_strategies=30, frac_nonspec_nodes=0.05, frac_noncontiguous=0.2)
    p = CostModelParams.from_mesh(mesh, rescale=2.2)
    all_three = ("comm", "transition", "cost")
    forms = [dict(outputs=("cost",), spec_table=False, packed=True), dict(outputs=("cost",), spec_table=False, one_launch=True, packed=False),
             dict(outputs=all_three, one_launch=True), dict(outputs=all_three, one_launch=False),
             dict(outputs=("cost",), spec_table=False, one_launch=False, row_min_in_tiles=False)]
    for form in forms:
        want = None
        for repeated in (False, True):
            d = DeviceCostTables(tb, p, device=gpu_device)
            step = d.prepare_step(**dict(dict(row_min=True, fused_inputs=True, row_min_in_tiles=True), **form), repeated=repeated)
            for launch in step.values():
                launch()
            got = _outputs(d)
            if want is None:
                want = got
                continue
            assert all((g is None) == (w is None) and (g is None or np.array_equal(g, w)) for g, w in zip(got, want)), form
            side = torch.cuda.Stream(device=d.device)
            d.cost.zero_()
            side.wait_stream(torch.cuda.current_stream())
            for launch in step.values():
                launch(side)
            assert np.array_equal(_outputs(d)[2], want[2]), form
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                for launch in step.values():
                    launch()
            for _ in range(3):
                d.cost.zero_()
                graph.replay()
                assert np.array_equal(_outputs(d)[2], want[2]), form


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [dict(one_launch=True, packed=False), dict(one_launch=False, packed=False),
                                  dict(packed=True, row_min=True, row_min_in_tiles=True)])
def test_a_graph_holds_what_its_launches_read(gpu_device, kind):
    """``step`` and then the tables' device object are dropped: a graph of the pass still has the blocks of its launches."""
    mesh = (16, 8, 4)
    tb = stress_dag(seed=4, n_nodes=300, mesh_sizes=mesh, max_strategies=20)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    form = dict(dict(row_min=False, fused_inputs=True, outputs=("cost",), spec_table=False), **kind)
    step = d.prepare_step(**form)
    launches = [weakref.ref(launch) for launch in step.values()]
    graph = d.capture_step_graph(step)
    del step
    gc.collect()
    assert all(launch() is not None for launch in launches)
    cost = d.cost
    d.prepare_step(**form)  # (the device object holds the launches of its latest step only)
    del d
    gc.collect()
    assert all(launch() is not None for launch in launches)
    others = [torch.full((n,), 7, dtype=torch.int64, device=gpu_device) for n in (64, 128, 256, 383) for _ in range(8)]
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"]
    for _ in range(3):
        cost.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(cost.cpu().numpy(), want)
    assert all(bool((t == 7).all()) for t in others)


@pytest.mark.gpu
def test_the_device_object_holds_the_launches_of_its_latest_step(gpu_device):
    mesh = (32, 8)
    tb = stress_dag(seed=4, n_nodes=300, mesh_sizes=mesh, max_strategies=20)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    for _ in range(2):
        step = d.planner_pass()
        bound = [weakref.ref(launch.bound) for launch in step.values()]
        del step
        gc.collect()
        assert all(b() is not None for b in bound)


@pytest.mark.gpu
@pytest.mark.parametrize("as_current", [True, False])
def test_what_a_launch_on_another_stream_uses_is_not_given_out_before_it_ran(gpu_device, as_current):
    """Launches behind other work of a second stream; everything is dropped, and arrays of the same sizes are allocated before
    that stream gets to them."""
    mesh = (16, 8, 4)
    tb = stress_dag(seed=6, n_nodes=400, mesh_sizes=mesh, max_strategies=30)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    step = d.prepare_step(row_min=False, fused_inputs=True, outputs=("cost",), spec_table=False, packed=False)
    arrays = (d.cost, d.compute_cost, d.compute_cost_per_arg, d.tensor_bytes)
    used = {t.data_ptr() for t in arrays}
    sizes = [t.numel() for t in arrays]
    side = torch.cuda.Stream(device=d.device)
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.cuda._sleep(1_000_000_000)  # (half a second)
        for launch in step.values():
            launch() if as_current else launch(side)
    del d, step, launch, arrays
    others = [torch.empty(n, dtype=torch.int64, device=gpu_device) for n in sizes for _ in range(3)]
    assert not side.query()  # (it had not got to the launches)
    assert used.isdisjoint(t.data_ptr() for t in others)
    for t in others:
        t.fill_(7)
    torch.cuda.synchronize()
    assert all(bool((t == 7).all()) for t in others)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [dict(one_launch=True, packed=False), dict(one_launch=False, packed=False), dict(fused_inputs=False, spec_table=True),
                                  dict(packed=True, row_min=True, row_min_in_tiles=True)])
def test_a_pass_is_prepared_while_the_stream_captures(gpu_device, form):
    """Without copies: of packed tiles, those of an earlier preparation are taken."""
    mesh = (16, 8, 4)
    tb = stress_dag(seed=12, n_nodes=250, mesh_sizes=mesh, max_strategies=20)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    form = dict(dict(row_min=False, fused_inputs=True, outputs=("cost",), spec_table=False), **form)
    if form.get("packed"):
        d.prepare_step(**form)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step = d.prepare_step(**form)
        for launch in step.values():
            launch()
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"]
    for _ in range(3):
        d.cost.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(d.cost.cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("before", [None, True])
def test_the_default_pass_is_prepared_while_the_stream_captures(gpu_device, before):
    """A small table that staged tiles are faster for, with the row minima: over staged tiles after a preparation by default,
    over packed ones where only those were prepared before."""
    mesh = (16, 8, 4)
    tb = stress_dag(seed=13, n_nodes=250, mesh_sizes=mesh, max_strategies=24)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    assert d.packed_pass_pays() and d.row_min_in_tiles_pays() and tb.staging_pays(tb.computed_entries(), tb.n_tiles)
    d.planner_pass(packed=before)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step = d.planner_pass()
        for launch in step.values():
            launch()
    assert list(step) == ["build_tables_packed" if before else "build_tables"]
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"]
    lowest = np.minimum.reduceat(want, tb.row_ptr()[:-1])
    for _ in range(3):
        for t in (d.cost, d.row_min):
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(d.cost.cpu().numpy(), want) and np.array_equal(d.row_min.cpu().numpy(), lowest)


def _small_packed(gpu_device):
    mesh = (32, 8)
    tb = stress_dag(seed=5, n_nodes=120, mesh_sizes=mesh, max_strategies=12)
    tb.build_tiles(None, dedupe=True)
    return tb, DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device), po.make_params(mesh, rescale=2.2)


@pytest.mark.gpu
@pytest.mark.parametrize("change", ["refresh", "refresh, captured", "strategy inputs"])
def test_packed_tiles_are_of_the_tables_uploaded_last(gpu_device, change):
    """A packed pass, then another strategy table on the same tiling: the next pass has its costs, and the launches bound
    before keep theirs."""
    tb, d, op = _small_packed(gpu_device)
    first = d.planner_pass(packed=True)
    first_cost = d.cost
    before = c_oracle.build_tables(tb.as_dict(), op)["cost"]
    if change == "strategy inputs":  # (the device counts, and the host's table receives the result)
        recipes = StrategyRecipes(tb.n_nodes)
        recipes.node_kind[:] = 1  # (bytes of the specs from the first on)
        recipes.node_row_begin[:] = np.arange(tb.n_nodes + 1)
        recipes.byte_rows = np.zeros(tb.n_nodes, np.int32)
        counts = [t.cpu().numpy() for t in d.run_strategy_inputs(recipes)]
        for name, a in zip(("strat_flops", "strat_rw_bytes", "strat_dtype", "strat_zero_cost"), counts):
            getattr(tb, name)[:] = a
    else:
        tb.strat_rw_bytes[:] = tb.strat_rw_bytes * 3 + (1 << 30)
        d.refresh("strat_rw_bytes")
    want = c_oracle.build_tables(tb.as_dict(), op)["cost"]
    assert not np.array_equal(want, before)
    if change.endswith("captured"):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for launch in d.planner_pass(packed=True).values():
                launch()
        runs = [graph.replay] * 3
    else:
        runs = list(d.planner_pass(packed=True).values())
    for run in runs:
        d.cost.zero_()
        run()
        torch.cuda.synchronize()
        assert np.array_equal(d.cost.cpu().numpy(), want)
    for launch in first.values():
        launch()
    assert np.array_equal(first_cost.cpu().numpy(), before)


@pytest.mark.gpu
def test_host_tables_between_two_lengths_can_be_refreshed(gpu_device):
    """Packed tiles are not made again of tables of which some have been replaced; a pass prepared then says so."""
    tb, d, op = _small_packed(gpu_device)
    d.planner_pass(packed=True)
    kept = tb.strat_flops
    tb.strat_flops = np.append(kept, 0)
    d.refresh("strat_flops")
    tb.strat_flops = kept
    d.refresh("strat_flops")
    for launch in d.planner_pass(packed=True).values():
        launch()
    assert np.array_equal(d.cost.cpu().numpy(), c_oracle.build_tables(tb.as_dict(), op)["cost"])


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["strat_rw_bytes", "spec_codes", "tensor_shape", None])
def test_the_default_pass_is_of_the_hosts_tables(gpu_device, name):
    """A small table that staged tiles are faster for, one of whose tables was changed on the host after the upload: over packed
    tiles, as every small table; over staged ones, captured ones too, where it was uploaded again or nothing was changed."""
    mesh = (16, 8, 4)
    tb = stress_dag(seed=13, n_nodes=250, mesh_sizes=mesh, max_strategies=24)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    op = po.make_params(mesh, rescale=2.2)
    assert d.packed_pass_pays() and tb.staging_pays(tb.computed_entries(), tb.n_tiles) and not tb.staging_pays(
        tb.computed_entries(), tb.n_tiles, repeated=False)
    if name is not None:
        a, row = getattr(tb, name), int(tb.edge_tgt_begin[-1])
        if name == "spec_codes":
            a[row:row + tb.edge_n_tgt[-1]] = a[row:row + tb.edge_n_tgt[-1]][::-1].copy()
        else:
            a[:] *= 2
    want = c_oracle.build_tables(tb.as_dict(), op)["cost"]
    lowest = np.minimum.reduceat(want, tb.row_ptr()[:-1])

    def check(runs, kind):
        assert list(step) == [kind]
        for run in runs:
            for t in (d.cost, d.row_min):
                t.zero_()
            run()
            torch.cuda.synchronize()
            assert np.array_equal(d.cost.cpu().numpy(), want) and np.array_equal(d.row_min.cpu().numpy(), lowest)

    step = d.planner_pass()
    check(step.values(), "build_tables" if name is None else "build_tables_packed")
    tb.strat_flops[:] += 1 << 40  # (what is prepared later on the same tiling, without an upload, is of the same tables)
    step = d.planner_pass()
    check(step.values(), "build_tables" if name is None else "build_tables_packed")
    tb.strat_flops[:] -= 1 << 40
    if name is not None:
        d.refresh(name)
        step = d.planner_pass()
        check(step.values(), "build_tables")
        d.refresh(name)  # (no preparation between this and the capture)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step = d.planner_pass()
        for launch in step.values():
            launch()
    check([graph.replay] * 3, "build_tables" if name is None else "build_tables_packed")

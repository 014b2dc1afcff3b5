"""The structural check of tables that are on the device (``apc_check_tables``) against the host's (``apc_validate_tables_host``).
Every index is checked before it is used, on either side."""
import numpy as np
import pytest

from autoparallel_amd import CostModelParams, _native
from autoparallel_amd.device_tables import _UPLOAD, DeviceCostTables
from autoparallel_amd.encoding import EDGE_GRAD_RESCALE
from autoparallel_amd.optimize_sharding import DeviceBackend
from autoparallel_amd.synthetic import stress_dag

from oracle import c_oracle
from oracle import cost_oracle as po
from test_abi_and_encoding import twin_graph

MESHES = [(8,), (12, 6), (4, 2, 2), (2, 2, 2, 2)]


@pytest.fixture(autouse=True)
def always_on_device(monkeypatch):
    monkeypatch.setattr(DeviceCostTables, "CHECK_ON_DEVICE_MIN_ROWS", 0)
    monkeypatch.setattr(DeviceCostTables, "PACK_ON_DEVICE_MIN_TILES", 0)


def _tables(mesh, seed=8):
    tb = twin_graph(stress_dag(seed=seed, n_nodes=60, mesh_sizes=mesh, max_strategies=10))
    tb.build_tiles(256, dedupe=True)
    return tb


def _refused(f):
    try:
        f()
    except RuntimeError as e:
        return str(e)
    return None


def _set(name, row, value):
    def mutate(t):
        a = getattr(t, name)
        a[row % len(a)] = value(t, a[row % len(a)]) if callable(value) else value
    return mutate


def _set_record(field, row, change):
    def mutate(t):
        t.tile_records[field][row % t.n_tiles] += change
    return mutate


MUTATIONS = (
    [_set("tensor_rank", 0, 9), _set("tensor_rank", 1, -1), _set("spec_tensor", 3, 10**6), _set("spec_tensor", 5, -2), _set("spec_tensor", 7, -1),
     _set("edge_entry_begin", 0, 1), _set("edge_entry_begin", 2, lambda t, v: v + 1), _set("edge_entry_begin", -1, 0)]
    + [_set("spec_codes", k, c) for k, c in enumerate((0xC0, 0x01, 0x8F, 0x80, 0x82, 0x40, 0x8000, 0x800000, 0xC0000000, 0x80000000, 0))]
    + [_set(n, e, lambda t, v, d=d: v + d) for n in ("edge_src_begin", "edge_tgt_begin", "edge_strat_begin", "edge_n_src", "edge_n_tgt")
       for e, d in ((1, 1), (4, -1), (6, 10**6), (2, -10**6))]
    + [_set("edge_pt_begin", e, v) for e in range(0, 60, 7) for v in (-1, 10**9, 0)]
    + [_set("edge_flags", e, lambda t, v: v ^ 1) for e in (0, 5, 9)]
    + [_set_record(f, t, d) for f in ("edge", "row_begin", "col_begin", "counts", "src_begin", "n_src", "tgt_begin", "flags", "strat_begin",
                                      "tensor", "entry_begin", "pt_begin", "dup_begin", "dup_count") for t, d in ((0, 1), (5, -1), (-1, 10**6))]
    + [_set("dup_entry_begin", k, lambda t, v, d=d: v + d) for k in (0, 3, -1) for d in (1, -10**7, 10**7)]
    + [_set("dup_entry_begin", 0, lambda t, v: t.tile_records["entry_begin"][t.tile_records["dup_count"] > 0][0])]
)


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", MESHES)
def test_the_device_refuses_what_the_host_refuses(gpu_device, mesh):
    params = CostModelParams.from_mesh(mesh)
    sound = _tables(mesh)
    d = DeviceCostTables(sound, params, device=gpu_device)
    assert d._refresh_and_check(("tile_records",), "tables") == "tables" and d._refresh_and_check((), "tiles") == "tiles"
    refused = 0
    for k, mutate in enumerate(MUTATIONS):
        tb = _tables(mesh)
        mutate(tb)
        want = _refused(lambda: tb.validate(params))
        d.tables = tb
        held = d._refresh_and_check([n for n in d.d if n not in ("strat_flops",)], "tables")
        rows_hold = _refused(lambda: tb._validate(params, lambda: "tiles")) is None
        # (what only the host checks, the tiling, is checked either way)
        structure = _refused(lambda: tb._validate(params, lambda: "tables"))
        assert (held == "tables") == (want is None or want == structure), (k, want)
        if rows_hold:  # the records alone, of tables whose rows hold
            assert (d._refresh_and_check((), "tiles") == "tiles") == (held == "tables"), (k, want)
        got = _refused(lambda: DeviceCostTables(tb, params, device=gpu_device))
        assert got == want, k
        refused += want is not None
    assert refused > len(MUTATIONS) // 2


@pytest.mark.gpu
def test_a_tiling_that_is_refused_leaves_the_old_one_on_the_device(gpu_device):
    mesh = (4, 2, 2)
    tb = _tables(mesh)
    backend = DeviceBackend(tb, CostModelParams.from_mesh(mesh), device=gpu_device)
    before = dict(backend.dev.d)
    tb._build_tiles = lambda *a, **k: tb.dup_entry_begin.__setitem__(0, 1)
    with pytest.raises(RuntimeError, match="duplicate offset"):
        backend.upload_strategy_inputs(tb)
    assert all(backend.dev.d[k] is before[k] for k in before)


@pytest.mark.gpu
def test_long_runs_of_edges_without_entries_are_left_to_the_host(gpu_device):
    """A copy whose edge lies behind more edges without entries than a lane passes over: the host finds it sound."""
    mesh, n = (4, 2), 70
    tb = _tables(mesh)
    at = int(np.nonzero((tb.edge_entry_begin[:-1] == tb.dup_entry_begin[-1]) & (tb.edge_n_src > 0))[0][0])
    for name in ("edge_node", "edge_arg", "edge_src_begin", "edge_n_src", "edge_tgt_begin", "edge_n_tgt", "edge_flags", "edge_pt_begin",
                 "edge_entry_begin", "edge_strat_begin"):
        a = getattr(tb, name)
        setattr(tb, name, np.insert(a, at, np.full(n, 0 if name == "edge_n_src" else a[at], a.dtype)))
    tb.build_tiles(256, dedupe=True)
    assert tb.edge_entry_begin[at + n] in tb.dup_entry_begin
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh), device=gpu_device)
    assert d._refresh_and_check((), "tiles") is None


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", MESHES)
@pytest.mark.parametrize("max_strategies", [1, 10, 90])  # (lists shorter and longer than a wavefront)
def test_identical_edges_are_the_same_on_the_device(gpu_device, mesh, max_strategies):
    """Twins of every edge, some of them then changed in one value each of what a matrix depends on."""
    tb = twin_graph(stress_dag(seed=21, n_nodes=80, mesh_sizes=mesh, min_strategies=1, max_strategies=max_strategies))
    rng = np.random.default_rng(max_strategies)
    for name in ("strat_flops", "strat_rw_bytes", "strat_dtype", "strat_num_args", "spec_codes"):
        a = getattr(tb, name)
        a[rng.integers(len(a) // 2, len(a), 3)] += 1
    zero = tb.strat_zero_cost[-1:]
    zero[:] = 1 - zero
    if len(tb.pt_values):
        tb.pt_values[-1] = np.nan  # (compared by its bits, as -0.0)
        tb.pt_values[0], tb.pt_values[len(tb.pt_values) // 2] = 0.0, -0.0
    tb.edge_flags[-3] ^= 2
    tb.edge_src_begin[-1] = tb.n_specs  # (outside the tables: stands for itself)
    d = object.__new__(DeviceCostTables)
    d.ops, d.tables, d.device, d.d = _native.torch_ops(), tb, gpu_device, {}
    d._refresh(_UPLOAD)
    got = d.edge_classes()
    assert np.array_equal(got, tb.edge_classes())
    assert 0 < np.count_nonzero(got != np.arange(tb.n_edges)) < tb.n_edges // 2


@pytest.mark.gpu
def test_the_planner_tiles_by_the_classes_of_the_device(gpu_device):
    mesh = (4, 2, 2)
    tb = _tables(mesh)
    tb.build_tiles(None, dedupe=True, repeated=False)
    want = tb.tile_records.copy()
    backend = DeviceBackend(tb, CostModelParams.from_mesh(mesh), device=gpu_device)
    backend.upload_strategy_inputs(tb)
    assert np.array_equal(tb.tile_records, want) and np.array_equal(backend.dev.d["tile_records"].cpu().numpy().view(np.uint8).ravel(), want.view(np.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", MESHES)
@pytest.mark.parametrize("max_strategies", [1, 10, 64])
def test_tiles_packed_on_the_device_are_the_hosts(gpu_device, mesh, max_strategies):
    """Byte for byte, in the table's order and in launch order; with pass-through edges, twins and specs of no tensor."""
    tb = twin_graph(stress_dag(seed=31, n_nodes=80, mesh_sizes=mesh, min_strategies=1, max_strategies=max_strategies))
    tb.build_tiles(None, dedupe=True)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh), device=gpu_device)
    assert tb.packable() and (tb.tile_records["dup_count"] > 0).any()
    for repeated in (False, True):
        want = tb.pack_tiles(tb.launch_records() if repeated else None)
        dev, packed = d.ops.pack_tiles(*d._tensor_table(), d.d["spec_codes"], d.d["spec_tensor"], *d._strategy_table(), d.d["edge_n_tgt"],
                                       d._tile_records(repeated), d.d["dup_entry_begin"], d.d["dup_row_begin"])
        assert packed and dev.cpu().numpy().tobytes() == want.tobytes()
    # a strategy with more arguments than a record holds, and a record that leaves the tables
    many = d.d["strat_num_args"].clone()
    many[int(tb.tile_records["strat_begin"][0] + tb.tile_records["row_begin"][0])] = 0x8000
    records = d.d["tile_records"].clone()
    records[0, 4] = tb.n_specs  # (src_begin)
    for strategies, tiles in (((*d._strategy_table()[:4], many), d.d["tile_records"]), (d._strategy_table(), records)):
        assert not d.ops.pack_tiles(*d._tensor_table(), d.d["spec_codes"], d.d["spec_tensor"], *strategies, d.d["edge_n_tgt"], tiles,
                                    d.d["dup_entry_begin"], d.d["dup_row_begin"])[1]


@pytest.mark.gpu
def test_classes_and_packed_tiles_are_of_the_hosts_strategy_table(gpu_device):
    """A strategy table changed on the host after the upload."""
    mesh = (4, 2, 2)
    tb = _tables(mesh)
    tb.build_tiles(None, dedupe=True)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh), device=gpu_device)
    tb.strat_flops[:] = tb.strat_rw_bytes
    assert d._packed_tiles(False).cpu().numpy().tobytes() == tb.pack_tiles().tobytes()
    tb.strat_num_args[::3] += 1
    assert np.array_equal(d.edge_classes(), tb.edge_classes())


@pytest.mark.gpu
def test_a_pass_that_runs_once_is_of_the_hosts_strategy_table(gpu_device):
    """A small table that a repeated pass takes over staged tiles, built once by a planner that has changed the strategy table."""
    mesh = (16, 8, 4)
    tb = stress_dag(seed=13, n_nodes=250, mesh_sizes=mesh, max_strategies=24)
    assert tb.staging_pays(tb.computed_entries(), tb.n_tiles) and not tb.staging_pays(tb.computed_entries(), tb.n_tiles, repeated=False)
    backend = DeviceBackend(tb, CostModelParams.from_mesh(mesh), device=gpu_device)
    backend._strategy_inputs_on_device = True
    tb.strat_flops[:] = tb.strat_rw_bytes
    backend.upload_strategy_inputs(tb)
    backend.launch_tables()
    assert backend.launches == ("build_tables_packed",)
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh))["cost"]
    assert np.array_equal(backend.dev.cost.cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["edge_flags", "edge_src_begin", "edge_tgt_begin", "edge_strat_begin", "edge_pt_begin", "spec_codes",
                                  "spec_tensor", "pt_values"])
def test_classes_are_of_the_hosts_edges_and_specs(gpu_device, name):
    """Twins that were changed on the host after the upload."""
    mesh = (4, 2, 2)
    tb = _tables(mesh)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh), device=gpu_device)
    before = tb.edge_classes()
    a = getattr(tb, name)
    if name == "edge_flags":
        a[len(a) // 2::2] ^= EDGE_GRAD_RESCALE
    elif name == "pt_values":
        a[len(a) // 2:] = np.arange(len(a) - len(a) // 2)
    else:
        a[len(a) // 2:] = a[len(a) // 2:][::-1]
    want = tb.edge_classes()
    assert not np.array_equal(want, before) and np.array_equal(d.edge_classes(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("mesh", MESHES)
def test_a_twin_that_was_changed_after_the_upload_gets_its_own_costs(gpu_device, mesh):
    """Every other twin with the other gradient rescale, set on the host between the backend's construction and the tiling."""
    tb = _tables(mesh)
    backend = DeviceBackend(tb, CostModelParams.from_mesh(mesh, rescale=2.2), device=gpu_device)
    tb.edge_flags[tb.n_edges // 2::2] ^= EDGE_GRAD_RESCALE
    backend.upload_strategy_inputs(tb)
    want_classes = tb.edge_classes()
    assert np.array_equal(want_classes[tb.edge_canonical], want_classes)  # (a copy is a copy of its like)
    backend.launch_tables()
    want = c_oracle.build_tables(tb.as_dict(), po.make_params(mesh, rescale=2.2))["cost"]
    assert np.array_equal(backend.dev.cost.cpu().numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["spec_codes", "spec_tensor", "tensor_rank", "tensor_itemsize", "tensor_shape", "tensor_stride", "strat_rw_bytes",
                                  "edge_n_tgt", "tile_records", "dup_entry_begin", "dup_row_begin"])
def test_packed_tiles_are_of_the_hosts_tables(gpu_device, name):
    """Tables that were changed on the host after the upload, and one of them to another integer type."""
    mesh = (4, 2, 2)
    tb = _tables(mesh)
    tb.build_tiles(None, dedupe=True)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh), device=gpu_device)
    before = tb.pack_tiles().tobytes()
    a = getattr(tb, name)
    a[:] = a[::-1].copy()
    want = tb.pack_tiles().tobytes()
    assert want != before or name == "tensor_itemsize"  # (of which there is one)
    if a.dtype == np.int32:
        setattr(tb, name, a.astype(np.int64))
    for repeated in (False, True):
        d._packed_cache = None
        want = tb.pack_tiles(tb.launch_records() if repeated else None).tobytes()
        assert d._packed_tiles(repeated).cpu().numpy().tobytes() == want


@pytest.mark.gpu
@pytest.mark.parametrize("least", [0, 1 << 30])
def test_packed_by_the_host_or_on_the_device(gpu_device, least, monkeypatch):
    monkeypatch.setattr(DeviceCostTables, "PACK_ON_DEVICE_MIN_TILES", least)
    mesh = (4, 2, 2)
    tb = _tables(mesh)
    tb.build_tiles(None, dedupe=True)
    d = DeviceCostTables(tb, CostModelParams.from_mesh(mesh), device=gpu_device)
    on_device = []
    monkeypatch.setattr(d, "_pack_on_device", lambda repeated: on_device.append(1) or DeviceCostTables._pack_on_device(d, repeated))
    for repeated in (False, True):
        want = tb.pack_tiles(tb.launch_records() if repeated else None).tobytes()
        assert d._packed_tiles(repeated).cpu().numpy().tobytes() == want
    assert bool(on_device) == (least == 0)

"""Device-resident cost tables: uploads a ``CostTables`` encoding to HBM once and
runs the HIP kernels of libapcost.so over it through the operators of the torch layer
(``torch.ops.apcost``, csrc/apcost_torch.cpp: tensors in, tensors out, argument checks,
current stream and device guard on the C++ side).

torch is used for device memory and streams only; every computation is a kernel of the
library.  Without a HIP device (or without the built libraries) construction raises: there
is no CPU path.

Every method that allocates, launches or copies runs on the package's device thread
(``_device_thread``), where no dispatch mode of the caller (a graph capture's fake-tensor
mode) is active; the launchers of ``prepare_step`` enqueue from whichever thread calls them.
"""

from __future__ import annotations

import numpy as np
import torch

from . import _native
from ._device_thread import on_device_thread as _guarded
from .cost_model import CostModelParams
from .encoding import TILE_DTYPE, CostTables
from .pruning import index_arrays

_UPLOAD = (
    "tensor_rank", "tensor_itemsize", "tensor_shape", "tensor_stride", "spec_codes", "spec_tensor",
    "strat_flops", "strat_rw_bytes", "strat_dtype", "strat_zero_cost", "strat_num_args",
    "edge_src_begin", "edge_n_src", "edge_tgt_begin", "edge_n_tgt", "edge_flags", "edge_pt_begin",
    "edge_entry_begin", "edge_strat_begin", "pt_values", "tile_records", "dup_entry_begin",
    "dup_row_begin",
)


_CHECKED = (
    "tensor_rank", "spec_codes", "spec_tensor", "edge_src_begin", "edge_n_src", "edge_tgt_begin", "edge_n_tgt", "edge_flags",
    "edge_pt_begin", "edge_entry_begin", "edge_strat_begin", "tile_records", "dup_entry_begin",
)


# what makes two edges identical (``CostTables.edge_classes``), in the order of the operator
_CLASSED = (
    "spec_codes", "spec_tensor", "strat_flops", "strat_rw_bytes", "strat_dtype", "strat_zero_cost", "strat_num_args", "edge_src_begin",
    "edge_n_src", "edge_tgt_begin", "edge_n_tgt", "edge_flags", "edge_pt_begin", "edge_strat_begin", "pt_values",
)


# what packed tiles are made of (``_pack_on_device``)
_PACKED = (
    "tensor_rank", "tensor_itemsize", "tensor_shape", "tensor_stride", "spec_codes", "spec_tensor", "strat_flops", "strat_rw_bytes",
    "strat_dtype", "strat_zero_cost", "strat_num_args", "edge_n_tgt", "tile_records", "dup_entry_begin", "dup_row_begin",
)


_ONE_LAUNCH_MAX_BYTES = 192 << 20


def _as_tensor(a: np.ndarray) -> torch.Tensor:
    """The array as a CPU tensor over the same memory."""
    if a.dtype == np.uint32:  # same bits; torch's uint32 support is partial
        a = a.view(np.int32)
    if a.dtype.names is not None:  # packed records travel as raw int32 words
        a = np.ascontiguousarray(a).view(np.int32).reshape(len(a), a.dtype.itemsize // 4)
    if not a.flags.c_contiguous:
        a = np.ascontiguousarray(a)
    if a.size == 0:
        return torch.empty(a.shape, dtype=_TORCH_DTYPE[a.dtype.type])
    return torch.from_numpy(a)


def _to_device(a: np.ndarray, device) -> torch.Tensor:
    """One array on ``device`` (or the CPU): a copy of its own."""
    t = _as_tensor(a)
    device = torch.device(device)
    if device.type != "cuda":
        return t.clone()
    return _native.torch_ops().upload([t], device)[0]


_TORCH_DTYPE = {np.int32: torch.int32, np.int64: torch.int64, np.uint8: torch.uint8, np.float64: torch.float64,
                np.int8: torch.int8, np.uint32: torch.int32}


class DeviceCostTables:
    @_guarded
    def __init__(self, tables: CostTables, params: CostModelParams, device="cuda:0", validate=True):
        if not torch.cuda.is_available():
            raise RuntimeError("DeviceCostTables needs a HIP device; there is no CPU path")
        self.ops = _native.torch_ops()
        self.tables = tables
        self.params = params
        self.device = torch.device(device)
        self.c_params = params.to_c()
        self.p = _native.params_tensor(self.c_params)  # struct apc_params as the operators take it
        self.d = {}
        if validate and self._check_on_device_pays():
            tables._validate(params, lambda: self._refresh_and_check(_UPLOAD, "tables"))
        else:
            if validate:
                tables.validate(params)
            self._refresh(_UPLOAD)
        self.tensor_bytes = None
        self.tensor_contiguous = None
        self.compute_cost = None
        self.compute_cost_per_arg = None
        self.comm = None
        self.transition = None
        self.cost = None
        self.row_min = None  # minima / first argmins of the rows of ``cost``, when a table launch took them
        self.row_argmin = None

    @_guarded
    def refresh(self, *names):
        """Re-uploads host tables that changed after construction (strategy inputs filled in
        from the shard-shape table, tiles rebuilt with de-duplication)."""
        self._refresh(names)

    def _refresh(self, names):
        arrays = [getattr(self.tables, k) for k in names]
        self.d.update(zip(names, self._upload(*arrays)))
        if "tile_records" in names:
            # (the host's table may be tiled anew before it is uploaded again: what is on the device stays one tiling)
            self._tiles = self.d["tile_records"], arrays[names.index("tile_records")]
            self._ordered_tiles = None
        if "edge_n_tgt" in names:
            self._edge_rows = None
        if not set(_PACKED).isdisjoint(names):
            self._host_on_device = None
            self._drop_stand_ins()
            if self._packed_cache is not None:
                self._pack_again()

    # Tables of fewer rows (specs + 4 edges) are checked, and tiled by classes found, on the host; a re-tiling sends the rows for both
    # (``send_rows``).  us, by the host / on the device, with the rows sent once for classes and check: 3.5 k rows 60 / 140, 23 k 200 / 150, 47 k
    # 370 / 180, 94 k 600 / 215, 187 k 840 / 290, 375 k (15 104 edges, 14 160 copies) 1 350 / 470; a new table's check alone 31 / 46, 67 / 51, 110 / 57,
    # 280 / 68, 460 / 91, 850 / 140.  The two meet at some 15 k rows; the line leaves tables with a few tenths of a ms at stake to the host, which
    # says which row is malformed without a second look.
    CHECK_ON_DEVICE_MIN_ROWS = 60_000

    def _check_on_device_pays(self) -> bool:
        tb = self.tables
        return tb.n_specs + 4 * tb.n_edges >= self.CHECK_ON_DEVICE_MIN_ROWS

    def _refresh_and_check(self, names, what, rows=None):
        """Uploads ``names``; -> ``what`` ("tables" or "tiles") where the device finds it well formed, else nothing.  ``rows``: of
        ``send_rows``, checked in place of the tables of later launches."""
        tb = self.tables
        self._refresh(names)
        d = {**self.d, **(rows or {})}
        longs = ("edge_pt_begin", "edge_entry_begin", "dup_entry_begin")
        if any(d[k].dtype != (torch.int64 if k in longs else torch.int32) for k in _CHECKED):
            return None  # (arrays of other types, which the host converts)
        hold = self.ops.tables_hold(
            self.p, what == "tables", *(d[k] for k in _CHECKED[:-2]), len(tb.pt_values), tb.n_strategies, d["tile_records"],
            d["dup_entry_begin"])
        return what if hold else None

    @_guarded
    def send_rows(self) -> dict:
        """What a tiling is made of and checked against, as the host has it: copies on the device beside the tables that launches
        read, which a program may have left behind its host tables.  (315 k specs, 15 104 edges and 129 k strategies 0.27 ms, 428 k, 8 564
        and 136 k 0.33.)"""
        tb = self.tables
        n, n_src_tgt = tb.n_edges, tb._matrix_sizes()
        spec = [a[:tb.n_specs] for a in tb._rows(tb.n_specs, "spec_codes", "spec_tensor")]
        edge_names = ("edge_src_begin", "edge_tgt_begin", "edge_flags", "edge_pt_begin", "edge_strat_begin")
        rows = dict(zip(_CLASSED[:7], spec + tb._strategy_rows(exact=True)), edge_n_src=n_src_tgt[0], edge_n_tgt=n_src_tgt[1],
                    **{k: a[:n] for k, a in zip(edge_names, tb._rows(n, *edge_names))})
        rows["pt_values"] = tb._rows(0, "pt_values")[0][:len(tb.pt_values)]
        rows["tensor_rank"] = tb._rows(tb.n_tensors, "tensor_rank", exact=True)[0]
        rows["edge_entry_begin"] = tb._rows(n + 1, "edge_entry_begin")[0][:n + 1]
        return dict(zip(rows, self._upload(*rows.values())))

    @_guarded
    def edge_classes(self, rows=None):
        """``CostTables.edge_classes`` (host array) of the host's tables, found on the device; ``rows``: of ``send_rows``."""
        rows = rows or self.send_rows()
        return self.ops.download([self.ops.edge_classes(*(rows[k] for k in _CLASSED))])[0].numpy()

    @_guarded
    def refresh_tiling(self, *names, rows=None):
        """``CostTables.validate``, and a re-upload of ``names``, the tiling among them; where the check raises, the device keeps
        what it had.  ``rows``: of ``send_rows`` since the host's tables last changed."""
        if not self._check_on_device_pays():
            self.tables.validate(self.params)
            self._refresh(names)
            return
        kept = "_tiles", "_ordered_tiles", "_edge_rows", "_packed_cache", "_packed_current", "_packed_stands_in"
        before = dict(self.d), [getattr(self, k) for k in kept]
        try:
            self.tables._validate(self.params, lambda: self._refresh_and_check(names, "tables", rows or self.send_rows()))
        except BaseException:
            self.d, values = before
            for k, v in zip(kept, values):
                setattr(self, k, v)
            raise

    # ---- helpers -------------------------------------------------------------------------
    def _upload(self, *arrays):
        """Host arrays as device tensors, in one transfer."""
        return self.ops.upload([_as_tensor(a) for a in arrays], self.device)

    def _empty(self, shape, dtype):
        return torch.empty(shape, dtype=dtype, device=self.device)

    # (for the entry points of the C ABI that have no operator: raw pointers and the stream handle)
    @property
    def lib(self):
        return _native.lib()

    def _stream(self):
        return _native.vp(torch.cuda.current_stream(self.device).cuda_stream)

    def _p(self, key):
        t = self.d[key] if isinstance(key, str) else key
        return _native.vp(t.data_ptr() if t is not None and t.numel() else 0)

    def _tensor_table(self):
        d = self.d
        return d["tensor_rank"], d["tensor_itemsize"], d["tensor_shape"], d["tensor_stride"]

    def _strategy_table(self):
        d = self.d
        return d["strat_flops"], d["strat_rw_bytes"], d["strat_dtype"], d["strat_zero_cost"], d["strat_num_args"]

    # ---- integer tables ------------------------------------------------------------------
    @_guarded
    def run_tensor_tables(self):
        self.tensor_bytes, self.tensor_contiguous = self.ops.tensor_tables(*self._tensor_table())
        return self.tensor_bytes, self.tensor_contiguous

    @_guarded
    def run_spec_tables(self):
        width = self.tables.shape_width()  # rows as wide as the largest rank needs, not APC_MAX_RANK
        names = ("num_shards", "local_shape", "local_stride", "local_numel", "local_bytes")
        out = dict(zip(names, self.ops.shard_shapes_bytes(self.p, self.d["spec_codes"], self.d["spec_tensor"],
                                                          *self._tensor_table(), width)))
        self.spec_out = out
        return out

    # ---- per-strategy flop / byte counts -----------------------------------------------------
    @_guarded
    def run_strategy_inputs(self, recipes):
        """Flop and byte counts of every (node, strategy) from the spec table and the per-node
        ``recipes`` (``graphs.cost_inputs.StrategyRecipes``), on the device; the strategy table
        of later launches reads the results where they are.  -> (flops, rw_bytes, dtype_code,
        zero_cost) device tensors."""
        tb = self.tables
        spec = getattr(self, "spec_out", None) or self.run_spec_tables()
        n_nodes = tb.n_nodes
        for name in ("node_kind", "node_dtype", "node_const_bytes"):
            if len(getattr(recipes, name)) != n_nodes:
                raise ValueError(f"recipes.{name} must have one row per node")
        # every row a recipe names, plus the node's strategies, lies inside the spec table; the
        # tensors of a flop formula have the rank it reads
        n_strat = np.diff(tb.node_strat_begin).astype(np.int64)
        per_node = np.repeat(n_strat, np.diff(recipes.node_row_begin))
        if len(recipes.byte_rows) and int((recipes.byte_rows.astype(np.int64) + per_node).max()) > tb.n_specs:
            raise ValueError("a recipe's spec rows run past the spec table")
        with_formula = recipes.node_kind >= 2
        if with_formula.any():
            if int((recipes.node_flop_rows[with_formula].astype(np.int64).max(axis=1) + n_strat[with_formula]).max()) > tb.n_specs:
                raise ValueError("a flop formula's spec rows run past the spec table")
            need = 4 if (recipes.node_kind >= 4).any() else 3 if (recipes.node_kind == 3).any() else 2
            if spec["local_shape"].shape[1] < need:
                raise ValueError("the spec table's shape rows are narrower than a flop formula's tensors")
        out = self.ops.strategy_inputs(*self._upload(
            np.repeat(np.arange(n_nodes, dtype=np.int32), n_strat), np.ascontiguousarray(tb.node_strat_begin, np.int64),
            recipes.node_kind, recipes.node_dtype, recipes.node_const_bytes, recipes.node_row_begin, recipes.byte_rows,
            recipes.node_flop_rows.reshape(-1)), spec["local_shape"], spec["local_bytes"])
        for key, t in zip(("strat_flops", "strat_rw_bytes", "strat_dtype", "strat_zero_cost"), out):
            self.d[key] = t
        self._packed_current, self._host_on_device = False, None  # (the host's strategy table is about to change)
        self._drop_stand_ins()
        return out

    # ---- per-strategy compute cost ---------------------------------------------------------
    @_guarded
    def run_compute_costs(self):
        self.compute_cost, self.compute_cost_per_arg, err = self.ops.compute_cost(self.p, *self._strategy_table())
        self._check_flag(int(err.item()))
        return self.compute_cost, self.compute_cost_per_arg

    # ---- redistribution-cost matrices ------------------------------------------------------
    @_guarded
    def alloc_outputs(self, comm=True, transition=True, cost=True):
        n = self.tables.n_entries
        self.comm = self._empty((n,), torch.float64) if comm else None
        self.transition = self._empty((n,), torch.uint8) if transition else None
        self.cost = self._empty((n,), torch.float64) if cost else None

    def _bind_redistribute_tables(self, comm, transition, cost, rows=None, repeated=False):
        """A bound launch of the table kernel over the tables already built, writing the given
        per-entry arrays (None: not written) and, with ``rows = (edge_row_begin, row_min,
        row_argmin)``, the row minima."""
        d = self.d
        erb, rmin, rarg = rows if rows is not None else (None, None, None)
        return self.ops.bind_redistribute_tables(
            self.p, self.tensor_bytes, self.tensor_contiguous, d["spec_codes"], d["spec_tensor"], d["pt_values"],
            self.compute_cost_per_arg, self._tile_records(repeated), d["dup_entry_begin"], self.tables.n_entries, comm, transition, cost,
            erb, d["dup_row_begin"] if rows is not None else None, rmin, rarg)

    @_guarded
    def launch_redistribute_tables(self, row_min=False):
        """One enqueue of the table kernel over pre-allocated outputs.  ``row_min``: the launch
        also writes ``row_min`` / ``row_argmin`` (allocated by ``run_redistribute_tables``)."""
        rows = None
        if row_min:
            rows = (_to_device(self.tables.edge_row_begin(), self.device), self.row_min, self.row_argmin)
        self._bind_redistribute_tables(self.comm, self.transition, self.cost, rows).run()

    @_guarded
    def run_redistribute_tables(self, comm=True, transition=True, cost=True, row_min=None):
        """``row_min``: also take the row minima of ``cost`` in the same launch (``None``: when all
        three outputs are wanted and ``row_min_in_tiles_pays``)."""
        if self.tensor_bytes is None:
            self.run_tensor_tables()
        if cost and self.compute_cost_per_arg is None:
            self.run_compute_costs()
        self.alloc_outputs(comm, transition, cost)
        if row_min is None:
            row_min = self.row_min_in_tiles_pays()
        if row_min:
            self.tables.validate_row_minima()  # raises when some matrix row is spread over tiles
        self.row_min = self.row_argmin = None
        if row_min:
            n_rows = self.tables.n_rows
            self.row_min = self._empty((n_rows,), torch.float64)
            self.row_argmin = self._empty((n_rows,), torch.int32)
        self.launch_redistribute_tables(row_min=bool(row_min))
        return self.comm, self.transition, self.cost

    @_guarded
    def build_all(self):
        """tensor tables and compute costs -> cost matrices (with the row minima when ``row_min_in_tiles_pays``), all on
        the current stream, in two launches.  A strategy with flops and an unsupported dtype raises, as in
        ``run_compute_costs``; the matrices are not kept then."""
        tb, d = self.tables, self.d
        row_min = self.row_min_in_tiles_pays()
        if row_min:
            tb.validate_row_minima()  # raises when some matrix row is spread over tiles
        n_tgt = tb._rows(tb.n_edges, "edge_n_tgt", exact=True)[0] if row_min else None
        out, unsupported = self.ops.report_tables(
            self.p, *self._tensor_table(), d["spec_codes"], d["spec_tensor"], *self._strategy_table(), d["pt_values"], d["tile_records"],
            d["dup_entry_begin"], tb.n_entries, *((_as_tensor(n_tgt), d["dup_row_begin"], int(n_tgt.sum(dtype=np.int64))) if row_min else
                                                  (None, None, 0)))
        self.tensor_bytes, self.tensor_contiguous, self.compute_cost, self.compute_cost_per_arg = out[:4]
        self._check_flag(int(unsupported))
        self.comm, self.transition, self.cost = out[4:7]
        self.row_min, self.row_argmin = out[7:] if row_min else (None, None)
        return self.comm, self.transition, self.cost

    # ---- one full device-side pass with pre-bound arguments -------------------------------------
    # One launch for all tables saves a ramp-up and drain, about 6 us; the tiles' own derivation of what they would otherwise read costs 0.1
    # to 0.15 ns a tile beside the work that both have.  The cost alone, us in one launch / two:
    #   up to ONE_LAUNCH_MAX_BYTES on 3-D and 4-D meshes, (16, 8, 4), 16 M entries (136 MiB) 33.3 / 34.5, 21.7 M (183 MiB) 44.1 / 44.6, on
    #   (6, 4, 2) 49.3 / 49.7, on (2, 4, 2, 2) 53.7 / 54.4, with three states in turn 28 M 78.6 / 74.3, 42 M 125 / 120;
    #   up to ONE_LAUNCH_MAX_BYTES_FLAT on meshes of one or two dims, where a tile stages less: on (64, 4) 32.7 M (274 MiB) 84.5 / 85.2, 40 M
    #   (336 MiB) 109 / 114, 37.8 M in eight layers (331 MiB) 83.4 / 83.2, on (32, 8) 41.7 M (350 MiB) 112.5 / 118, 32.3 M in 40 layers 70.4 / 78.6,
    #   on (12, 6) 41.7 M 116 / 121; with three states in turn 47 M in eight layers on (64, 4) (376 MiB) 129 / 124;
    #   with the row minima in the tiles there up to ONE_LAUNCH_MAX_BYTES_FLAT_MINIMA, three states in turn, on (32, 8) 16.3 M in 300 layers (203 MiB)
    #   62.6 / 64.8, 18.7 M in 40 (172 MiB) 49.9 / 50.7, 25.3 M (230 MiB) 64.3 / 63.8, then 30 M (272 MiB) 75.2 / 74.0, on (64, 4) 37 M in four (324 MiB) 92.8 / 89.6, 37.8 M
    #   in eight (331 MiB) 87.8 / 84.4;
    #   beyond ONE_LAUNCH_MAX_BYTES_OF_MANY_TILES not in more than ONE_LAUNCH_MANY_TILES, where the tiles cost what the launch saves: 44 850 tiles
    #   (above) and 46 056 116 / 121, then 49 238 on (32, 8) 55.6 / 54.5, 70 738 63.5 / 60.9, 96 217 77.8 / 72.5, 427 120 on (64, 4) 263 / 238, on (16, 8, 4)
    #   45 064 54.6 / 53.5, 70 737 61.4 / 59.4, on (6, 4, 2) 96.9 / 89.3; nor on a 4-D mesh with a size that is no power of two, whose states cost most
    #   to stage, 20 016 tiles (184 MiB) 89.8 / 88.4, 42 860 (177 MiB) 152 / 141.  Smaller tables are one launch whatever their tiles: it decides
    #   whether they can go over packed ones (5.3 M entries in 162 354 tiles lose by it, 179 / 107, measured when both took longer).
    ONE_LAUNCH_MAX_BYTES = _ONE_LAUNCH_MAX_BYTES
    ONE_LAUNCH_MAX_BYTES_FLAT = 344 << 20
    ONE_LAUNCH_MAX_BYTES_FLAT_MINIMA = 256 << 20
    ONE_LAUNCH_MAX_BYTES_OF_MANY_TILES = 128 << 20
    ONE_LAUNCH_MANY_TILES = 48 << 10

    def one_launch_limit(self, row_min_in_tiles: bool = False) -> int:
        """Bytes of the largest pass that is one launch: ``ONE_LAUNCH_MAX_BYTES`` where a program has set it, else by the mesh, the
        tiles and whether they take the row minima."""
        tb, limit = self.tables, self.ONE_LAUNCH_MAX_BYTES
        if limit != _ONE_LAUNCH_MAX_BYTES:
            return limit
        if tb.n_tiles > self.ONE_LAUNCH_MANY_TILES or tb._many_states():
            return self.ONE_LAUNCH_MAX_BYTES_OF_MANY_TILES
        if len(tb.mesh_sizes) <= 2:
            return self.ONE_LAUNCH_MAX_BYTES_FLAT_MINIMA if row_min_in_tiles else self.ONE_LAUNCH_MAX_BYTES_FLAT
        return limit

    def row_min_in_tiles_pays(self) -> bool:
        """Whether the launch that writes the cost matrices should take the row minima itself.
        Priced inside the tiles: 0.5 ns per tile and 1.6 ps per entry a tile computes (identical edges are computed, and
        reduced, once for all their copies); as a ``segmented_min`` launch: 4 us and every stored entry read back at 4.5 TB/s.
        The first two are what minima across the lanes of a wavefront and a barrier a tile took.  With the rows of a wavefront
        joined through its LDS the minima of tables that compute every entry cost 1.0 - 1.4 ps an entry, so the rule
        is early to leave them to the separate launch.  Cost alone, us a pass without minima / in tiles / separate, by size:
        5.2 M entries on (12, 6) 21.0 / 27.8 / 30.3, 9.4 M on (16, 8, 4) 29.0 / 42.3 / 50.7, on (2, 4, 2, 2) 35.4 / 46.2 / 52.7; where the
        rule says separate: 20 M on (16, 8, 4) 65.1 / 85.0 / 96.6, 3.6 M on (64, 4) 17.3 / 22.3 / 25.5 (edge by edge 20.3 / 30.2 /
        28.5).  It decides whether a planner finds the minima taken, and stays."""
        tb = self.tables
        if tb.n_tiles == 0 or not tb.rows_fit_tiles():
            return False
        # (of the edges cut as little as they can be, where the tiling was chosen from the table: how it is cut further
        # does not decide whether a planner finds the minima taken)
        n_tiles, computed = (tb.tiling or {}).get("whole_edges") or (tb.n_tiles, tb.computed_entries())
        return 0.5e-3 * n_tiles + 1.6e-6 * computed < 4.0 + 8.0 * tb.n_entries / 4.5e6

    def _alloc_input_tables(self, spec_table: bool):
        """Allocates (does not fill) the outputs of the tensor, compute-cost and, when wanted,
        spec tables."""
        tb = self.tables
        self.tensor_bytes = self._empty((tb.n_tensors,), torch.int64)
        self.tensor_contiguous = self._empty((tb.n_tensors,), torch.uint8)
        self.compute_cost = self._empty((tb.n_strategies,), torch.float64)
        self.compute_cost_per_arg = self._empty((tb.n_strategies,), torch.float64)
        if not spec_table:
            return None
        n, width = tb.n_specs, tb.shape_width()
        self.spec_out = {
            "num_shards": self._empty((n,), torch.int64),
            "local_shape": self._empty((n, width), torch.int64),
            "local_stride": self._empty((n, width), torch.int64),
            "local_numel": self._empty((n,), torch.int64),
            "local_bytes": self._empty((n,), torch.int64),
        }
        return self.spec_out

    def pass_bytes(self, outputs=("comm", "transition", "cost"), spec_table=True, row_min_in_tiles=False) -> int:
        """Bytes a pass with these outputs must move at minimum (what its launches write, plus
        the spec lists and edge headers the tiles read)."""
        tb = self.tables
        total = tb.algorithmic_bytes(comm="comm" in outputs, transition="transition" in outputs, cost="cost" in outputs)
        total += tb.algorithmic_bytes_input_tables(spec_table=spec_table)
        if row_min_in_tiles:
            total += 12 * tb.n_rows
        return total

    # A table up to this many entries is bound by the latency of one workgroup: its planner pass
    # runs over packed tiles (every wavefront on its own, one round of loads, no LDS staging).
    # Above, the per-entry arithmetic of that kernel (direct evaluation) costs more than the
    # staging it saves; so it does below for the tables of which ``CostTables.staging_pays`` says so.
    PACKED_MAX_ENTRIES = 4_000_000

    def packed_pass_pays(self) -> bool:
        tb = self.tables
        return tb.n_entries <= self.PACKED_MAX_ENTRIES and tb.packable()

    # Fewer tiles are packed by the host: 93 take it 56 us with their transfer and the device 80, 437 128 / 80.
    PACK_ON_DEVICE_MIN_TILES = 200

    # (tile records, whether in launch order, the packed ones on the device, lanes that take one), and whether those are of the tables as
    # they are now
    _packed_cache, _packed_current = None, True

    def _packed_tiles(self, repeated):
        """``CostTables.pack_tiles()`` on the device, made once per tiling and again when a table it is made of was uploaded anew; in launch
        order for a pass that is repeated (the order costs the host more than it saves one launch, which takes a copy that is there in
        either)."""
        tb, cached = self.tables, self._packed_cache
        if cached is not None and cached[0] is tb.tile_records and (cached[1] or not repeated) and (
                self._packed_current or torch.cuda.is_current_stream_capturing()):
            return cached[2]
        lanes = tb.packed_lanes()
        dev, packed = self._pack_on_device(repeated) if tb.n_tiles >= self.PACK_ON_DEVICE_MIN_TILES else (None, False)
        if not packed:  # (the host packs them, or says which it cannot)
            dev = _to_device(tb.pack_tiles(tb.launch_records() if repeated else None), self.device)
        self._packed_cache, self._packed_current = (tb.tile_records, repeated, dev, lanes), True
        return dev

    def _pack_on_device(self, repeated):
        """-> (packed tiles of the host's tables, whether all could be packed): put together on the device, the tables sent beside those that
        launches read (0.32 ms for the 314 k specs and 129 k strategies of 15 104 edges, 0.35 by the host; 0.38 / 1.47 for 10 022 tiles
        of 428 k and 136 k, 0.085 / 0.15 for 436 of 1 766 and 730)."""
        return self.ops.pack_tiles(*self._upload(*self._packed_of(repeated)))

    def _packed_of(self, repeated) -> list:
        """The host's tables that packed tiles are made of (``_PACKED``)."""
        tb = self.tables
        records = tb.launch_records() if repeated else tb.tile_records
        n_dups = len(tb.dup_entry_begin)
        return [
            *(a[:tb.n_tensors] for a in tb._rows(tb.n_tensors, "tensor_rank", "tensor_itemsize", "tensor_shape", "tensor_stride")),
            *(a[:tb.n_specs] for a in tb._rows(tb.n_specs, "spec_codes", "spec_tensor")),
            *(a[:tb.n_strategies] for a in tb._strategy_rows()), tb._matrix_sizes()[1], tb._records(records, tb.n_tiles, TILE_DTYPE),
            *(a[:n_dups] for a in tb._rows(n_dups, "dup_entry_begin", "dup_row_begin"))]

    _host_on_device = None  # (tile records, whether a preparation over them found the host's tables on the device), since the last upload

    def _staged_is_as_packed(self, capturing, sent) -> bool:
        """Whether a pass over staged tiles, which read the tables on the device, has the results of one over packed ones, which are
        the host's: whether no table was changed on the host and not uploaded.  Found once per tiling, as those are made (0.1 to 0.4 ms);
        ``sent``, a list, then receives the copies of the host's tables (``_packed_of``) and of the edges' first rows.  While the stream captures, as
        an earlier preparation found it, or left it without packed tiles."""
        tb, known = self.tables, self._host_on_device
        if known is not None and known[0] is tb.tile_records:
            return known[1]
        if capturing:
            return self._packed_cache is None or self._packed_cache[0] is not tb.tile_records
        *tables, edge_rows = self._upload(*self._packed_of(False), tb.edge_row_begin())
        sent[:] = tables, edge_rows
        there = [self.d[k] for k in _PACKED]

        def joined(arrays):
            return torch.cat([a.reshape(-1).view(torch.uint8) for a in arrays])

        same = all(a.dtype == b.dtype and a.shape == b.shape for a, b in zip(tables, there)) and torch.equal(joined(tables), joined(there))
        self._host_on_device = tb.tile_records, same
        return same

    # Whether the packed tiles are there in place of staged ones only.  What a pass over staged tiles would have left behind, the edges' first
    # rows, is there then too, and where a table changes they go: the next preparation makes others with its look at the
    # host's tables, and while a stream captures staged tiles take the pass.  (Made again with every upload, as those that a pass has
    # no choice but to go over, they cost it 0.1 to 0.4 ms for the 1 to 3 us that they save a pass.)
    _packed_stands_in = False

    def _packed_for_staged(self, capturing, sent) -> bool:
        """Whether packed tiles, a few lanes each, take a pass that staged ones could take; ``sent``: of ``_staged_is_as_packed``."""
        tb, cached = self.tables, self._packed_cache
        there = cached is not None and cached[0] is tb.tile_records
        if there and self._packed_stands_in:
            return True
        if capturing and not (there and self._packed_current):
            return False
        lanes = tb.small_packing_lanes()
        if not lanes or capturing:
            return bool(lanes)
        tables, self._edge_rows = sent or (None, self._edge_rows)
        if self._edge_rows is None:
            self._edge_rows = _to_device(tb.edge_row_begin(), self.device)
        if not there:
            self._packed_stands_in = True
            if tables and tb.n_tiles >= self.PACK_ON_DEVICE_MIN_TILES and not tb.largest_tiles_first_pays():
                dev, packed = self.ops.pack_tiles(*tables)
                if packed:
                    self._packed_cache, self._packed_current = (tb.tile_records, True, dev, lanes), True
        return True

    def _drop_stand_ins(self):
        if self._packed_stands_in:
            self._packed_cache, self._packed_stands_in = None, False

    def _pack_again(self):
        """The packed tiles anew where a table they are made of was uploaded: a pass that is prepared next, also while the stream
        captures, finds them.  (Launches bound earlier keep theirs.)"""
        records, repeated, *_ = self._packed_cache
        self._packed_cache = None
        if records is not self.tables.tile_records:
            return
        lanes = self.tables.packed_lanes()
        try:
            dev, packed = self._pack_on_device(repeated)
        except ValueError:  # (host tables of different lengths: one of several that are being replaced)
            return
        if packed:
            self._packed_cache, self._packed_current = (records, repeated, dev, lanes), True

    def _tile_records(self, repeated):
        """The device copy of the tile records, in launch order for a pass that is repeated: of the tiling that is on the
        device with its copies' offsets."""
        on_device, records = self._tiles
        if not repeated or self.d["tile_records"] is not on_device:
            return self.d["tile_records"]
        if self._ordered_tiles is None:
            ordered = self.tables.launch_records(records)
            self._ordered_tiles = on_device if ordered is records else _to_device(ordered, self.device)
        return self._ordered_tiles

    @_guarded
    def prepare_step(self, row_min=True, fused_inputs=False, one_launch=None, row_min_in_tiles=None,
                     outputs=("comm", "transition", "cost"), spec_table=True, packed=None, repeated=True):
        """Allocates every output once and returns ``{kernel name: zero-argument launcher}``
        in launch order.  A launcher only enqueues (no allocation, no synchronisation), so a
        timed loop measures the kernels and not Python argument marshalling.  With
        ``fused_inputs`` the tensor, spec and compute-cost tables are one launch
        (``input_tables``) instead of three; with ``one_launch`` they and the cost matrices
        are one (``build_tables``); ``one_launch=None`` takes one launch for tables up to
        ``one_launch_limit()`` when ``fused_inputs`` is set.  ``row_min_in_tiles``: the launch
        that writes the cost matrices takes the row minima too (no ``segmented_min`` launch, no
        second read of the matrices); it needs every row inside one tile
        (``CostTables.rows_fit_tiles``), and ``None`` takes it when ``row_min_in_tiles_pays``.
        ``outputs``: which of the per-entry arrays the pass writes; ``spec_table=False`` leaves
        the local shard shapes out (a planner has computed them before it could fill in the
        flop / byte counts this pass reads).  ``packed``: the one launch runs over packed tiles
        (``apc_build_tables_packed``: the assembled cost and the row minima, no spec table);
        ``None`` takes them when the pass is of that kind, ``packed_pass_pays`` and staged tiles
        (``CostTables.staging_pays``, ``small_packing_lanes``) are not faster still.  Packed tiles hold the host's tables as they are at the first
        preparation after a tiling or an upload; where staged tiles are faster for the repeated pass of a small table, they are taken if the tables on the device, which
        they read, are the same.  ``repeated=False``: the pass will run once, and the arguments
        of its launches are not laid out in device memory first (``apc_kept_launch``: one copy, for 0.75 us less a launch over packed
        tiles or a large table, nothing where staged tiles wait for other loads at that time), nor its tiles put
        into launch order (``CostTables.launch_records``: 10 ns a tile on the host).  Those copies, one a launch
        and one of the tiles, are waited for.  So are the uploads of row indices and packed tiles; while the current stream
        captures, a pass is prepared as with ``repeated=False`` and takes the edges' first rows, or the packed tiles, of an earlier preparation
        (a table that staged tiles are faster for goes over packed ones where only those are there, and one that packed tiles are faster for over
        staged ones where a table or the tiling was uploaded since)."""
        tb = self.tables
        capturing, runs_once = torch.cuda.is_current_stream_capturing(), not repeated
        repeated = bool(repeated) and not capturing
        outputs = tuple(outputs)
        if not outputs or any(o not in ("comm", "transition", "cost") for o in outputs):
            raise ValueError(f"outputs must name some of comm, transition, cost: {outputs}")
        if not spec_table and not fused_inputs:
            raise ValueError("a pass without the spec table is built with fused_inputs")
        fits = self.tables.rows_fit_tiles()
        if row_min_in_tiles is None:
            row_min_in_tiles = self.row_min_in_tiles_pays()
        row_min_in_tiles = bool(row_min_in_tiles) and bool(row_min)
        if row_min_in_tiles and not fits:
            raise ValueError("row minima inside the table launch need every matrix row inside one tile")
        if row_min and not row_min_in_tiles and "cost" not in outputs:
            raise ValueError("a segmented_min launch over the rows reads the cost array: ask for it")
        total = self.pass_bytes(outputs, spec_table, row_min_in_tiles)
        if one_launch is None:
            one_launch = bool(fused_inputs) and total <= self.one_launch_limit(row_min_in_tiles)
        packed_kind = bool(one_launch) and row_min_in_tiles and outputs == ("cost",) and not spec_table
        stands_in = False
        if packed is None:
            packed = packed_kind and self.packed_pass_pays()
            if packed and (self._edge_rows is not None or not capturing):
                of_tiles, sent = (tb.computed_entries(), tb.n_tiles), []
                packed = not (tb.staging_pays(*of_tiles, repeated=False) or (
                    not runs_once and tb.staging_pays(*of_tiles) and self._staged_is_as_packed(capturing, sent)))
                stands_in = not packed and self._packed_for_staged(capturing, sent)
                packed = packed or stands_in
        elif packed and not (packed_kind and self.tables.packable()):
            raise ValueError("a pass over packed tiles is one launch that writes the assembled cost and the row minima, "
                             "without the spec table, over tiles of whole rows")
        spec = self._alloc_input_tables(spec_table)
        self.alloc_outputs("comm" in outputs, "transition" in outputs, "cost" in outputs)
        self.row_min = self.row_argmin = None
        ops, d = self.ops, self.d
        err = torch.zeros((1,), dtype=torch.int32, device=self.device)
        self._step_keepalive = [err, spec]
        spec_outputs = [spec[k] for k in ("num_shards", "local_shape", "local_stride", "local_numel", "local_bytes")] \
            if spec_table else []
        width = spec["local_shape"].shape[1] if spec_table else tb.shape_width()
        input_tables = (self.p, *self._tensor_table(), self.tensor_bytes, self.tensor_contiguous, d["spec_codes"],
                        d["spec_tensor"], spec_outputs, width, *self._strategy_table(), self.compute_cost,
                        self.compute_cost_per_arg, err)

        def bind(bound):
            # a launcher only looks up the current stream (or takes the given one) and enqueues
            if repeated:
                bound.keep_arguments()
            (run, run_on), handle = _native.bound_runners(), bound.handle()

            def launch(on_stream=None):
                if run(handle) if on_stream is None else run_on(
                        handle, int(on_stream.cuda_stream), int(getattr(on_stream, "stream_id", on_stream.cuda_stream))):
                    raise _native.bound_error()
            launch.bound = bound  # (what the handle names lives as long as its launcher)
            return launch

        rows = None
        if row_min:
            self.row_min = self._empty((tb.n_rows,), torch.float64)
            self.row_argmin = self._empty((tb.n_rows,), torch.int32)
        if row_min_in_tiles and not packed:  # (packed tiles hold their rows' numbers themselves)
            if self._edge_rows is None or not capturing:
                self._edge_rows = _to_device(tb.edge_row_begin(), self.device)
            rows = (self._edge_rows, self.row_min, self.row_argmin)
        erb, rmin, rarg = rows if rows is not None else (None, None, None)
        dup_rows = d["dup_row_begin"] if rows is not None else None
        if packed:
            if not stands_in and not capturing:
                self._packed_stands_in = False
            tiles = self._packed_tiles(repeated)
            step = {"build_tables_packed": bind(ops.bind_cost_tables_packed(
                self.p, *self._tensor_table(), self.tensor_bytes, self.tensor_contiguous, *self._strategy_table(),
                self.compute_cost, self.compute_cost_per_arg, err, d["pt_values"], tiles, tb.n_entries, tb.n_rows,
                self.cost, self.row_min, self.row_argmin, self._packed_cache[3]))}
        elif one_launch:
            step = {"build_tables": bind(ops.bind_cost_tables(
                *input_tables, d["pt_values"], self._tile_records(repeated), d["dup_entry_begin"], tb.n_entries, self.comm,
                self.transition, self.cost, erb, dup_rows, rmin, rarg))}
        elif fused_inputs:
            step = {"input_tables": bind(ops.bind_input_tables(*input_tables))}
        else:
            step = {
                "tensor_tables": bind(ops.bind_tensor_tables(*self._tensor_table(), self.tensor_bytes,
                                                             self.tensor_contiguous)),
                "spec_tables": bind(ops.bind_spec_tables(self.p, d["spec_codes"], d["spec_tensor"],
                                                         *self._tensor_table(), spec_outputs, width)),
                "compute_costs": bind(ops.bind_compute_costs(self.p, *self._strategy_table(), self.compute_cost,
                                                             self.compute_cost_per_arg, err)),
            }
        if not one_launch and not packed:
            step["redistribute_tables"] = bind(self._bind_redistribute_tables(self.comm, self.transition, self.cost, rows, repeated))
        if row_min and not row_min_in_tiles:
            row_ptr = _to_device(tb.row_ptr(), self.device)
            assert row_ptr.numel() - 1 == self.row_min.numel()
            copies = self._row_copies()
            if copies is not None:  # identical edges: every distinct row is read once, its minimum stored to all
                selected, copy_ptr, copy_rows, n_read = copies
                step["segmented_min"] = bind(ops.bind_segmented_min(self.cost, row_ptr, selected, copy_ptr, copy_rows,
                                                                    n_read, self.row_min, self.row_argmin))
            else:
                step["segmented_min"] = bind(ops.bind_segmented_min(self.cost, row_ptr, None, None, None, 0,
                                                                    self.row_min, self.row_argmin))
        self._step_error_flag = err
        # (a program may drop ``step`` once it has enqueued or captured its launches, which read more than the arrays above)
        self._step_keepalive.append([launch.bound for launch in step.values()])
        return step

    # ---- the planner's table build -------------------------------------------------------------
    PLANNER_OUTPUTS = ("cost",)

    def planner_pass(self, packed=None, repeated=True):
        """The launches ``ShardingOptimizer.build_ds`` issues once the flop / byte counts are in
        the strategy table (optimize_sharding.py:270-380 in one pass): the tensor and
        compute-cost tables and the assembled cost of every entry, the array the ILP objective
        is summed from, in one launch for tables up to ``one_launch_limit()`` (else the input
        tables, then the matrices); the launch also takes the row minima when that is cheaper
        than reading the matrices back (``row_min_in_tiles_pays``), otherwise they are taken
        when asked for.  The spec table is not part of it (the planner needed the local shard
        shapes before it could count flops); ``comm`` and ``transition`` are written only when a
        report asks (``fetch``).  The cost of a small table is of the host's tables as they are now (``prepare_step``), of any
        other table of those uploaded last."""
        return self.prepare_step(row_min=self.row_min_in_tiles_pays(), fused_inputs=True,
                                 outputs=self.PLANNER_OUTPUTS, spec_table=False, packed=packed, repeated=repeated)

    @_guarded
    def check_error_flag(self):
        """After a synchronisation: raises if a strategy with flops had an unsupported dtype."""
        err = getattr(self, "_step_error_flag", None)
        if err is not None:
            self._check_flag(int(err.item()))

    def _check_flag(self, flag: int):
        if flag == 2:
            raise RuntimeError("packed tiles were taken by fewer lanes than some tile has rows or columns")
        if flag != 0:
            # compute_estimation.py:198-201
            raise ValueError(f"a strategy with non-zero flops uses a dtype not supported on {self.params.device_name}")

    @_guarded
    def fetch(self, name: str) -> torch.Tensor:
        """The device array ``comm`` / ``transition`` / ``cost``; one that the pass did not write
        is computed now by a launch of the table kernel with that output alone (same values:
        the kernel evaluates an entry the same way whichever arrays it stores)."""
        have = {"comm": self.comm, "transition": self.transition, "cost": self.cost}
        if name not in have:
            raise KeyError(name)
        if have[name] is not None:
            return have[name]
        if self.tensor_bytes is None or self.compute_cost_per_arg is None:
            raise RuntimeError("no table pass has run yet")
        n = self.tables.n_entries
        out = self._empty((n,), torch.uint8 if name == "transition" else torch.float64)
        self._bind_redistribute_tables(*(out if k == name else None for k in have)).run()
        setattr(self, name, out)
        return out

    @_guarded
    def cost_objective(self, n_vars: int, group_var_begin, group_member_begin, member_entry_begin):
        """-> (objective f64[n_vars], forced_zero u8[n_vars]) on the device: the ILP objective
        summed from ``cost`` (``apc_cost_objective``).  The index arrays are host arrays."""
        n_groups = len(group_var_begin) - 1
        if n_groups < 0 or len(group_member_begin) != n_groups + 1:
            raise ValueError("group_var_begin and group_member_begin must have n_groups + 1 rows")
        if n_groups and (int(group_var_begin[0]) != 0 or int(group_var_begin[-1]) != n_vars
                         or int(group_member_begin[-1]) != len(member_entry_begin)):
            raise ValueError("group pointers do not span the variables / members")
        if n_groups and not bool((np.diff(np.asarray(group_var_begin, np.int64)) > 0).all()):
            raise ValueError("every variable group needs at least one variable (the kernel takes one workgroup per group)")
        index = self._upload(*(np.ascontiguousarray(a, np.int64) for a in (group_var_begin, group_member_begin, member_entry_begin)))
        return self.ops.cost_objective(int(n_vars), *index, self.fetch("cost"), float(self.params.inf_replacement_cost))

    @_guarded
    def capture_step_graph(self, step):
        """Records one pass (the launchers of ``prepare_step``) into a HIP graph: one launch per
        pass, and the three kernels that only read the uploaded tables (tensor, spec and
        compute-cost tables) sit on parallel branches, so they overlap on the device instead
        of queueing behind each other.  Returns the ``torch.cuda.CUDAGraph``, which holds every array
        its launches read or write; ``replay()`` enqueues the pass on the current stream.  For callers that want a single launch per
        pass; it is not the fast way to loop over passes: on the Llama-3-8B table a replay was
        measured at 61 us against 39 us for the five plain launches in stream order (the
        runtime's per-node replay cost exceeds what the overlap saves), and equal on tables
        large enough to be bandwidth-bound."""
        graph = torch.cuda.CUDAGraph()
        branches = [torch.cuda.Stream(device=self.device) for _ in range(2)]  # default priority
        with torch.cuda.graph(graph):
            main = torch.cuda.current_stream()
            for b in branches:
                b.wait_stream(main)
            one_launch = step.get("build_tables") or step.get("build_tables_packed")
            if one_launch is not None:
                one_launch(main)
            elif "input_tables" in step:
                step["input_tables"](main)
            else:
                step["spec_tables"](main)
                step["tensor_tables"](branches[0])
                step["compute_costs"](branches[1])
            for b in branches:
                main.wait_stream(b)
            if "redistribute_tables" in step:
                step["redistribute_tables"](main)
            if "segmented_min" in step:
                step["segmented_min"](main)
        graph.apcost_launches = tuple(step.values()), branches
        return graph

    # ---- segmented min ---------------------------------------------------------------------
    def _row_copies(self):
        """Device arrays of ``CostTables.row_copies()`` when reading only the distinct rows saves
        at least a quarter of the matrix bytes, else None."""
        tb = self.tables
        if tb.dup_entry_begin is None or len(tb.dup_entry_begin) == 0:
            return None
        cached = getattr(self, "_row_copies_cache", None)
        if cached is not None and cached[0] is tb.tile_records:  # (a new tiling packs new records)
            return cached[1]
        selected, copy_ptr, copy_rows, n_read = tb.row_copies()
        out = None
        if n_read <= 0.75 * tb.n_entries:
            out = (*self._upload(selected, copy_ptr, copy_rows), n_read)
        self._row_copies_cache = (tb.tile_records, out)
        return out

    @_guarded
    def row_minima(self):
        """(min, first argmin) of every matrix row of ``cost``: what the table launch already took,
        else a segmented minimum that reads every distinct row once."""
        if self.row_min is not None:
            return self.row_min, self.row_argmin
        tb = self.tables
        copies = self._row_copies()
        row_ptr = _to_device(tb.row_ptr(), self.device)
        if copies is None:
            return self.segmented_min(self.fetch("cost"), row_ptr, check=False)
        selected, copy_ptr, copy_rows, n_read = copies
        n_rows = row_ptr.numel() - 1
        mins = self._empty((n_rows,), torch.float64)
        args = self._empty((n_rows,), torch.int32)
        self.ops.bind_segmented_min(self.fetch("cost"), row_ptr, selected, copy_ptr, copy_rows, n_read, mins, args).run()
        return mins, args  # (the index arrays stay cached with the tables)

    @_guarded
    def segmented_min(self, values: torch.Tensor, seg_ptr, check: bool = True):
        if not isinstance(seg_ptr, torch.Tensor):
            seg_ptr = torch.from_numpy(np.ascontiguousarray(seg_ptr, dtype=np.int64)).to(self.device)
        if values.dtype != torch.float64 or seg_ptr.dtype != torch.int64:
            raise TypeError("segmented_min takes float64 values and an int64 segment pointer")
        if not (values.is_contiguous() and seg_ptr.is_contiguous()):
            raise ValueError("segmented_min takes contiguous arrays")
        n_seg = seg_ptr.numel() - 1
        if n_seg < 0:
            raise ValueError("seg_ptr must have at least one element")
        if check and n_seg > 0:
            # the kernel trusts the pointer array: keep it inside the value array
            ok = bool((seg_ptr[1:] >= seg_ptr[:-1]).all()) and int(seg_ptr[0]) >= 0 and int(seg_ptr[-1]) <= values.numel()
            if not ok:
                raise ValueError("seg_ptr must be non-decreasing and end within the value array")
        return self.ops.segmented_min(values, seg_ptr)

    # ---- dual ascent over the planning program's labelling form ---------------------------------
    # A wait of the resident sweeps for another workgroup's minima: microseconds when all workgroups are on the
    # chip.  One that lasts this long (100 MHz ticks: 0.2 s) means that they are not, and ends the kernel.
    SWEEP_WAIT_TICKS = 20_000_000

    # what the plan, and the copies on the device, are made of (the last one stays on the host)
    _SWEEP_INDEX = ("color_nodes", "label_begin", "inc_begin", "inc_edge", "inc_side", "edge_begin", "edge_i", "edge_j", "color_begin")

    @staticmethod
    def _sweep_plan(graph):
        """-> (plan words, first word of every workgroup, slots, bytes of LDS, threads) of the resident sweeps
        (``apc_sweep_plan_host``), None when the problem does not fit the chip's LDS."""
        most = _native.APC_SWEEP_MAX_WORKGROUPS
        labels, degree = np.diff(graph.label_begin), np.diff(graph.inc_begin)
        ends = np.concatenate([graph.edge_i, graph.edge_j])
        n_colors = len(graph.color_begin) - 1
        capacity = (n_colors + 80) * most + int((9 * labels + degree)[ends].sum())
        plan, begin, sizes = np.empty(capacity, np.int32), np.empty(most + 1, np.int64), np.empty(5, np.int64)
        index = index_arrays(graph)
        color_begin, color_nodes = np.ascontiguousarray(graph.color_begin, np.int64), np.ascontiguousarray(graph.color_nodes, np.int32)
        if n_colors < 0 or len(color_nodes) < graph.n_classes:
            raise ValueError("the colours must partition the classes")
        _native.host_call("apc_sweep_plan_host", graph.n_classes, *index[:4], graph.n_edges, *index[4:], n_colors, color_begin,
                          color_nodes, most, capacity, plan, begin, sizes)
        n, words, *rest = sizes.tolist()
        return (plan[:words], begin[:n + 1], *rest) if n else None

    @_guarded
    def diffusion_sweeps(self, graph, theta: np.ndarray, unary: np.ndarray, n_sweeps: int):
        """``n_sweeps`` sweeps of min-sum diffusion over ``graph`` (``pruning.LabelGraph``) starting
        from the host arrays ``theta`` / ``unary``; returns the updated pair as new host arrays
        (read-only: handed back to the next call unchanged, they are not uploaded again).  A problem
        that fits the chip's LDS takes one kernel for all sweeps (``apc_diffusion_sweeps_resident``), any
        other one launch per colour (``apc_diffusion_sweeps``); the same bits.  What either needs of the
        graph is worked out and uploaded once, and again when one of its index arrays was replaced."""
        cached = getattr(self, "_diffusion_graph", None)
        arrays = [getattr(graph, k) for k in self._SWEEP_INDEX]
        if cached is None or cached["graph"] is not graph or any(x is not y for x, y in zip(cached["arrays"], arrays)):
            cached = self._diffusion_graph = {"graph": graph, "arrays": arrays, "plan": self._sweep_plan(graph)}
            self._diffusion_state = None
        state = getattr(self, "_diffusion_state", None)
        if state is not None and state[0] is theta and state[1] is unary:
            th, un = state[2], state[3]  # what the last call left on the device, returned as these very arrays
        else:
            th, un = self._upload(np.ascontiguousarray(theta, np.float64), np.ascontiguousarray(unary, np.float64))
        plan = cached["plan"]
        if plan is not None and "on_device" not in cached:
            cached["on_device"] = self._upload(*plan[:2])
        out = None
        if plan is not None:
            *pair, status = self.ops.diffusion_sweeps_resident(
                int(n_sweeps), *cached["on_device"], *plan[2:], int(graph.label_begin[-1]), int(graph.edge_begin[-1]), th, un,
                self.SWEEP_WAIT_TICKS)
            theta_out, unary_out, flag = (t.numpy() for t in self.ops.download([*pair, status]))
            if int(flag[0]) == 0:
                out = pair
            else:  # (the next chunk of sweeps would wait as long again)
                cached["plan"] = None
                del cached["on_device"]
        if out is None:
            d = cached.get("index")
            if d is None:
                d = cached["index"] = self._upload(*arrays[:-1])
            out = (th, un)
            max_labels = int(np.diff(graph.label_begin).max()) if graph.n_classes else 0
            self.ops.diffusion_sweeps_(int(n_sweeps), torch.from_numpy(np.ascontiguousarray(graph.color_begin, np.int64)), *d, max_labels,
                                       int(graph.label_begin[-1]), int(graph.edge_begin[-1]), *out)
            theta_out, unary_out = (t.numpy() for t in self.ops.download(list(out)))
        theta_out.setflags(write=False)
        unary_out.setflags(write=False)
        self._diffusion_state = (theta_out, unary_out, *out)
        return theta_out, unary_out

    def _index_of_bounds(self, row_min):
        t = self.tables
        if row_min.dtype != torch.float64 or not row_min.is_contiguous():
            raise TypeError("strategy_bounds takes a contiguous float64 array of row minima")
        if row_min.numel() != t.n_rows:
            raise ValueError("row_min must hold one value per matrix row")
        if getattr(self, "_bound_index", None) is None:
            index = dict(t.strategy_bound_index(), node_strat_begin=np.ascontiguousarray(t.node_strat_begin, np.int64))
            self._bound_index = dict(zip(index, self._upload(*index.values())))
        return self._bound_index

    @_guarded
    def strategy_bounds(self, row_min: torch.Tensor) -> torch.Tensor:
        """Per-(node, strategy) sum of the row minima of the node's edges (``row_min`` in the
        order of ``CostTables.row_ptr()``)."""
        ix = self._index_of_bounds(row_min)
        return self.ops.strategy_bounds(ix["strat_node"], ix["node_strat_begin"], ix["node_edge_begin"], ix["edges_by_node"],
                                        ix["edge_row_begin"], row_min)

    @_guarded
    def greedy_strategies(self, row_min: torch.Tensor):
        """-> (bound per strategy, min per node, argmin per node): the cheapest strategy of every
        node when each of its edges is charged its row minimum."""
        ix = self._index_of_bounds(row_min)
        return self.ops.greedy_strategies(ix["node_strat_begin"], ix["node_edge_begin"], ix["edges_by_node"], ix["edge_row_begin"], row_min,
                                          ix["strat_node"].numel())

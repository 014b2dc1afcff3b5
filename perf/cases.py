"""What this package is used for, as cases that can be timed.

A planner takes a graph from strategies to a plan in five stages, and each kind of case is one of
them, or all, through the calls that a program makes:

  pass     the table pass over a graph whose tables are on the device (``planner_pass``): the cost of
           every (consumer strategy, producer strategy) pair of every edge, the compute costs, the row
           minima where the pass takes them.  What is repeated when the cost model changes, and what
           the benchmark counts.
  tables   a new graph: from the flattened arrays of the encoding on the host to what the planner reads
           back (objective coefficient and forced-to-zero flag of every variable, compute costs), with
           the upload, shard shapes, flop / byte counts, tiling and checks on the way.
  report   every table and all three per-entry arrays, the row minima and the greedy strategies: what a
           report over a graph, or a warm start from the cost table, reads.
  prune    from the objective of the variable blocks to the pruned program: labelling form, sweeps of
           the dual ascent, bound, rounding, local search, the variables that can be fixed.
  plan     a traced model to its plan: ``ShardingOptimizer``, its constraints, ``get_solution``.

Graphs are drawn by ``synthetic.stress_dag``; ``layers`` repeats the drawn graph as the layers of a
transformer repeat (same tensors, same placements, same operators: identical edges, which are
evaluated once and share their variables when ``linked``).  Sizes follow the package's own
configurations: the single block on (64,), the 32-layer decoder on (32, 8) (324 nodes and 390 edges a
layer, 12 strategies a node), the 80-layer decoder on (8, 8, 8) (50 strategies a node, up to 124), the
mixture of experts on (64, 4), the stress DAG on (16, 8, 4).
"""

from __future__ import annotations

import dataclasses

import numpy as np
import torch

from autoparallel_amd import CostModelParams, pruning
from autoparallel_amd._native import APC_MAX_RANK
from autoparallel_amd.device_tables import DeviceCostTables
from autoparallel_amd.encoding import CostTables
from autoparallel_amd.graphs import workloads
from autoparallel_amd.graphs.capture import capture_joint_graph
from autoparallel_amd.graphs.cost_inputs import StrategyRecipes
from autoparallel_amd.optimize_sharding import DeviceBackend, ShardingOptimizer
from autoparallel_amd.synthetic import OP_MATMUL, OP_VIEW, stress_dag

DEVICE = "cuda:0"
RESCALE = 2.2  # gradients reduced in fp32, parameters in bf16 (api.py)
NODE_ZERO, NODE_BYTES, NODE_MM, NODE_BMM = 0, 1, 2, 3  # include/apcost.h: APC_NODE_*
SWEEP_CHUNKS = (40, 40, 80)  # the first chunks of ShardingOptimizer.prune_sweep_chunks


def _case(kind, mesh, nodes, lo, hi, layers=1, linked=True, fanout=1.1):
    return {"kind": kind, "mesh": "x".join(str(m) for m in mesh), "nodes": nodes, "lo": lo, "hi": hi, "layers": layers,
            "linked": linked, "fanout": fanout}


def _prune_case(classes, labels, degree):
    return {"kind": "prune", "classes": classes, "labels": labels, "degree": degree}


def _plan_case(model, mesh, layers, batch, seq):
    return {"kind": "plan", "model": model, "mesh": "x".join(str(m) for m in mesh), "layers": layers, "batch": batch, "seq": seq}


def listed():
    named = {
        # the smallest graph that is planned, one transformer block on a 1-D mesh: one launch and its latency
        "pass_block_1d": _case("pass", (64,), 300, 1, 4),
        # a 32-layer decoder on a 2-D mesh, the benchmark's own size (2 M entries)
        "pass_layers_2d": _case("pass", (32, 8), 324, 1, 24, layers=32),
        # mesh sizes that are no powers of two and rows wider than a tile; no edge like another
        "pass_ragged_2d": _case("pass", (12, 6), 700, 2, 90, fanout=1.6),
        # an 80-layer decoder on a 3-D mesh: up to 100 strategies a node, 75 M entries
        "pass_layers_3d": _case("pass", (8, 8, 8), 320, 2, 100, layers=80),
        # a DAG without repetition on a 3-D mesh (21 M entries, 20 k edges)
        "pass_dag_3d": _case("pass", (16, 8, 4), 9000, 4, 64, fanout=2.0),
        # the table stage of a plan, from the encoded arrays to the planner's numbers: block, decoder, large DAG
        "tables_block_1d": _case("tables", (64,), 300, 1, 4),
        "tables_layers_2d": _case("tables", (32, 8), 324, 1, 24, layers=32),
        "tables_dag_3d": _case("tables", (16, 8, 4), 4000, 4, 64, linked=False, fanout=2.0),
        # every array of a graph of the mixture-of-experts' size, with row minima and greedy strategies
        "report_moe_2d": _case("report", (64, 4), 520, 1, 24, layers=16),
        # pruning the decoder's program on a 2-D mesh (288 classes of at most 24 labels) ...
        "prune_labels_24": _prune_case(288, 24, 1.25),
        # ... and on a 3-D mesh (124 labels), where a class's matrices no longer fit on-chip memory
        "prune_labels_124": _prune_case(288, 124, 1.25),
        # a traced two-layer decoder to its plan
        "plan_decoder_2d": _plan_case("llama3_8b", (32, 8), 2, 32, 8192),
    }
    return [dict(c, name=name) for name, c in named.items()]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


MESHES = ((64,), (6,), (32, 8), (64, 4), (12, 6), (3, 8), (8, 8, 8), (16, 8, 4), (6, 4, 2), (2, 4, 2, 2), (3, 2, 2, 2))


def draw(rng):
    kind = rng.choice(("pass", "pass", "pass", "tables", "tables", "report", "prune", "prune", "plan"))
    if kind == "prune":
        return _prune_case(_log_int(rng, 20, 1100), _log_int(rng, 3, 64), 1.0 + 0.6 * rng.random())
    if kind == "plan":
        model, mesh = rng.choice((("block_1k", (64,)), ("block_1k", (8, 4)), ("llama3_8b", (32, 8)), ("llama3_8b", (16, 4))))
        layers = 1 if model == "block_1k" else rng.randint(1, 2)
        return _plan_case(model, mesh, layers, 32, 64 * rng.randint(8, 32) if model == "block_1k" else 1024 * rng.randint(1, 8))
    mesh = rng.choice(MESHES)
    layers = rng.choice((1, 1, _log_int(rng, 2, 60)))
    hi = _log_int(rng, 4, 4 if len(mesh) == 1 else 90)
    # entries about nodes x fanout x (hi / 2)^2 x layers: at most 20 M, less where every array is made or the host
    # has a part; nodes as many as the largest graphs have
    most = {"pass": 20e6, "tables": 6e6, "report": 10e6}[kind]
    fanout = round(1.0 + rng.random(), 2)
    most_nodes = min(6000, 26000 // layers, int(most / (layers * (fanout + 0.5) * (hi / 2 + 1) ** 2)))
    nodes = _log_int(rng, 40, max(41, most_nodes))
    return _case(kind, mesh, nodes, rng.randint(1, min(4, hi)), hi, layers=layers, linked=rng.random() < 0.7, fanout=fanout)


# ---- graphs ------------------------------------------------------------------------------------------
def _mesh(case):
    return tuple(int(x) for x in case["mesh"].split("x"))


def _block(case):
    """One layer of the case's graph: its nodes, edges, strategy counts and tensor ranks, which the case alone decides."""
    mesh = _mesh(case)
    return stress_dag(seed=0, n_nodes=case["nodes"], mesh_sizes=tuple(1 << (m - 1).bit_length() for m in mesh),
                      min_strategies=case["lo"], max_strategies=case["hi"], fanout_lambda=case["fanout"], window=64,
                      max_log2_dim=13, max_log2_numel=30)


def _values(tb, mesh, seed):
    """What the seed decides in the layer ``tb``: which of its valid placements a strategy has (the placements of a
    node's outputs, and of each argument, in another order) and the sizes of the tensors.
    -> (placement codes, tensor shapes, tensor strides, factor of every node's tensor)"""
    rng = np.random.Generator(np.random.PCG64(seed))
    n_strat = np.diff(tb.node_strat_begin)
    owner = np.concatenate([np.repeat(np.arange(tb.n_nodes), n_strat), tb.n_nodes + np.repeat(np.arange(tb.n_edges), tb.edge_n_tgt)])
    codes = tb.spec_codes[np.lexsort((rng.random(tb.n_specs), owner))]
    # every dim is a multiple of the odd part of the mesh sizes (a sharded dim has to be divisible), the first 1 to 3 times larger
    odd = int(np.lcm.reduce([m // (m & -m) for m in mesh]))
    factor = rng.integers(1, 4, tb.n_tensors)
    live = np.arange(APC_MAX_RANK)[None, :] < tb.tensor_rank[:, None]
    scale = np.where(live, odd, 1)
    scale[:, 0] *= factor
    # a dim's stride spans the dims inside it (those of smaller stride)
    inside = (tb.tensor_stride[:, None, :] < tb.tensor_stride[:, :, None]) & live[:, None, :] & live[:, :, None]
    stride = tb.tensor_stride * np.where(inside, scale[:, None, :], 1).prod(axis=2)
    return codes, tb.tensor_shape * scale, stride, factor


def _arrays(case, seed, counts):
    """-> (the encoding's arrays of the case's graph, operator class of every node).  ``counts``: with the flop
    and byte counts of the strategies (a planner works them out from the shard shapes)."""
    tb = _block(case)
    codes, shape, stride, factor = _values(tb, _mesh(case), seed)
    per_strategy = np.repeat(factor, np.diff(tb.node_strat_begin))  # (one tensor per node, in node order)
    L = case["layers"]
    S, NS, NP, N, E = tb.n_strategies, tb.n_specs, len(tb.pt_values), tb.n_nodes, tb.n_entries
    layer = np.arange(L, dtype=np.int64)

    def rep(a):
        return np.tile(a, L)

    def shifted(a, by):  # the rows of layer k name rows k * by further on
        return (a[None, :].astype(np.int64) + (layer * by)[:, None]).ravel()

    zeros = np.zeros(S * L, np.int64)
    arrays = dict(
        mesh_sizes=_mesh(case), tensor_rank=tb.tensor_rank, tensor_itemsize=tb.tensor_itemsize, tensor_shape=shape,
        tensor_stride=stride, spec_codes=rep(codes), spec_tensor=rep(tb.spec_tensor),
        strat_flops=rep(tb.strat_flops * per_strategy) if counts else zeros,
        strat_rw_bytes=rep(tb.strat_rw_bytes * per_strategy) if counts else zeros,
        strat_dtype=rep(tb.strat_dtype), strat_zero_cost=rep(tb.strat_zero_cost), strat_num_args=rep(tb.strat_num_args),
        node_strat_begin=np.append(shifted(tb.node_strat_begin[:-1], S), S * L),
        edge_node=shifted(tb.edge_node, N), edge_arg=rep(tb.edge_arg), edge_src_begin=shifted(tb.edge_src_begin, NS),
        edge_n_src=rep(tb.edge_n_src), edge_tgt_begin=shifted(tb.edge_tgt_begin, NS), edge_n_tgt=rep(tb.edge_n_tgt),
        edge_flags=rep(tb.edge_flags), edge_pt_begin=np.where(rep(tb.edge_pt_begin) >= 0, shifted(tb.edge_pt_begin, NP), -1),
        edge_entry_begin=np.append(shifted(tb.edge_entry_begin[:-1], E), E * L),
        edge_strat_begin=shifted(tb.edge_strat_begin, S), pt_values=rep(tb.pt_values))
    return arrays, rep(tb.node_op)


def _recipes(arrays, node_op):
    """Per-node recipes of the flop and byte counts, as the graph front-end writes them: a product's flops from the
    local shapes of its arguments, bytes from its argument and output specs; views cost nothing."""
    n_nodes = len(arrays["node_strat_begin"]) - 1
    node = arrays["edge_node"]
    order = np.argsort(node, kind="stable")
    n_edges = np.bincount(node, minlength=n_nodes)
    first = np.cumsum(n_edges) - n_edges
    tgt = arrays["edge_tgt_begin"][order]
    r = StrategyRecipes(n_nodes)
    matmul = node_op == OP_MATMUL
    a, b = tgt[first], tgt[first + np.minimum(n_edges - 1, 1)]
    rank = np.where(arrays["spec_tensor"] >= 0, arrays["tensor_rank"][np.maximum(arrays["spec_tensor"], 0)], 0)
    batched = (rank[a] >= 3) & (rank[b] >= 3)
    real = (rank[a] >= 2) & (rank[b] >= 2)
    r.node_kind[:] = np.where(node_op == OP_VIEW, NODE_ZERO, np.where(~matmul | ~real, NODE_BYTES, np.where(batched, NODE_BMM, NODE_MM)))
    r.node_dtype[:] = arrays["strat_dtype"][arrays["node_strat_begin"][:-1]]
    r.node_flop_rows[:, 0], r.node_flop_rows[:, 1] = a, b
    np.cumsum(n_edges + 1, out=r.node_row_begin[1:])
    rows = np.empty(int(r.node_row_begin[-1]), np.int32)
    within = np.arange(len(tgt)) - first[node[order]]
    rows[r.node_row_begin[node[order]] + within] = tgt
    # the output specs of a layer's nodes stand in strategy order at the layer's first spec row
    per_layer = n_nodes // arrays["_layers"]
    k = np.arange(n_nodes) // per_layer
    begin = arrays["node_strat_begin"]
    rows[r.node_row_begin[1:] - 1] = k * (len(arrays["spec_codes"]) // arrays["_layers"]) + begin[:-1] - begin[k * per_layer]
    r.byte_rows = rows
    return r


def _groups(arrays, layers, linked):
    """Variable groups of the objective: one per edge, shared by the same edge of every layer when ``linked``."""
    begin = arrays["edge_entry_begin"]
    n = (len(begin) - 1) // layers
    shares = layers if linked else 1
    n_groups = (len(begin) - 1) // shares
    sizes = np.diff(begin)[:n_groups]
    var_begin = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    members = (np.arange(n_groups)[:, None] + np.arange(shares)[None, :] * n).ravel()
    return int(var_begin[-1]), var_begin, np.arange(n_groups + 1, dtype=np.int64) * shares, begin[:-1][members].astype(np.int64)


def _labelling(case, seed):
    """The variable blocks of a planning program: a chain of classes of nodes with side branches (three in ten
    classes read a second or a far producer, a few are read by many), one strategy a label.  A strategy is a
    placement pair; a block charges the change between its two ends' placements, the consumer's compute cost on
    its rows, and forbids what cannot be redistributed."""
    rng = np.random.Generator(np.random.PCG64(0))  # the classes and their neighbours: the case's own
    n, top = case["classes"], case["labels"]
    sizes = np.where(rng.random(n) < 0.05, 1, rng.integers(max(1, top // 5), max(2, (2 * top) // 3 + 1), n))
    sizes[rng.random(n) < 0.03] = top
    sizes[rng.integers(0, n)] = top
    pairs = [(i, i - 1) for i in range(1, n)]
    extra = int(n * (case["degree"] - 1.0))
    far = rng.integers(1, n, extra)
    hubs = rng.integers(0, max(1, n // 25), extra)
    near = np.maximum(far - rng.integers(2, 20, extra), 0)
    for i, h, m, pick in zip(far.tolist(), hubs.tolist(), near.tolist(), rng.random(extra).tolist()):
        j = h if pick < 0.3 else m
        if j != i and abs(i - j) > 1:
            pairs.append((i, j))
    pairs = sorted(set(pairs))
    rng = np.random.Generator(np.random.PCG64(seed))
    place = [rng.integers(0, 12, s) for s in sizes]
    compute = [7.0 + 100.0 * rng.random(s) * (rng.random() < 0.3) for s in sizes]
    blocks, costs, at = [], [], 0
    for i, j in pairs:
        nt, ns = int(sizes[i]), int(sizes[j])
        blocks.append((at, nt, ns, i, j))
        at += nt * ns
        move = 8.0 + 200.0 * rng.random((12, 12)) ** 3
        move[rng.random((12, 12)) < 0.08] = np.inf
        np.fill_diagonal(move, 0.0)
        costs.append(move[place[i][:, None], place[j][None, :]] + compute[i][:, None])
    return blocks, sizes.tolist(), costs


def _placements(model, ndim):
    from torch.distributed.tensor.placement_types import Replicate, Shard

    rest = (Replicate(),) * (ndim - 1)
    if model == "block_1k":  # (the batch does not divide the mesh: pin the sequence)
        return (Shard(1),) + rest, (Shard(1),) + rest
    return (Shard(0),) + rest, (Shard(0), Shard(2)) if ndim == 2 else (Shard(0),) + rest


# ---- the cases -----------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "prune":
        blocks, sizes, costs = _labelling(case, seed)
        # a device handle of a small graph, as a planner holds one when it prunes
        dev = DeviceCostTables(stress_dag(seed=seed, n_nodes=20, mesh_sizes=(4, 2)), CostModelParams.from_mesh((4, 2)), device=DEVICE)
        return {"kind": kind, "blocks": blocks, "sizes": sizes, "costs": costs, "dev": dev}
    mesh = _mesh(case)
    if kind == "plan":
        logical = workloads.logical_mesh(mesh)
        config = workloads.WORKLOADS[case["model"]][0]
        # inputs of another seed are another model: the width of its feed-forward network differs
        config = dataclasses.replace(config, multiple_of=512 * (1 + seed % 7))
        model, input_fn, _, dynamo = workloads.build_model(case["model"], logical, n_layers=case["layers"], batch=case["batch"],
                                                           seq=case["seq"], config=config)
        with capture_joint_graph(model, input_fn, param_dtype=torch.bfloat16, dynamo=dynamo) as (gm, _):
            pass
        return {"kind": kind, "gm": gm, "mesh": logical, "placements": _placements(case["model"], len(mesh)),
                "rescale": 1.0 + seed % 1009 / 500}
    params = CostModelParams.from_mesh(mesh, rescale=RESCALE)
    arrays, node_op = _arrays(case, seed, counts=kind != "tables")
    if kind == "tables":
        recipes = _recipes(dict(arrays, _layers=case["layers"]), node_op)
        return {"kind": kind, "arrays": arrays, "recipes": recipes, "params": params,
                "groups": _groups(arrays, case["layers"], case["linked"])}
    tables = CostTables(**arrays)
    tables.build_tiles(None, dedupe=True)
    dev = DeviceCostTables(tables, params, device=DEVICE)
    return {"kind": kind, "dev": dev, "step": dev.planner_pass() if kind == "pass" else None}


def run(state):
    return {"pass": _run_pass, "tables": _run_tables, "report": _run_report, "prune": _run_prune, "plan": _run_plan}[state["kind"]](state)


def _run_pass(state):
    for launch in state["step"].values():
        launch()
    dev = state["dev"]
    return (dev.cost, dev.tensor_bytes, dev.tensor_contiguous, dev.compute_cost, dev.compute_cost_per_arg, dev.row_min, dev.row_argmin)


def _run_tables(state):
    tables = CostTables(**state["arrays"])
    backend = DeviceBackend(tables, state["params"], DEVICE)
    backend.strategy_inputs(state["recipes"])
    backend.upload_strategy_inputs(tables)
    backend.launch_tables()
    out = backend.finish(*state["groups"])
    return out, tables.strat_flops, tables.strat_rw_bytes, backend.dev.cost


def _run_report(state):
    dev = state["dev"]
    dev.run_spec_tables()
    comm, transition, cost = dev.build_all()
    row_min, row_argmin = dev.row_minima()
    bound, node_min, node_arg = dev.greedy_strategies(row_min)
    return dev.spec_out, comm, transition, cost, dev.compute_cost, row_min, row_argmin, bound, node_min, node_arg


def _run_prune(state):
    costs = state["costs"]
    index = {b[0]: k for k, b in enumerate(state["blocks"])}
    graph = pruning.build_label_graph([pruning.Block(*b) for b in state["blocks"]], state["sizes"],
                                      lambda b: costs[index[b.var_begin]], {}, [])
    theta, unary = graph.theta.copy(), graph.unary.copy()
    bounds = []
    for chunk in SWEEP_CHUNKS:
        theta, unary = state["dev"].diffusion_sweeps(graph, theta, unary, chunk)
        bound = pruning.lower_bound(graph, theta, unary)[0]
        labels = pruning.refine(graph, theta, unary, pruning.decode(graph, theta, unary))
        cost = sum(float(costs[k][labels[b[3]], labels[b[4]]]) for k, b in enumerate(state["blocks"]))
        bounds += [bound, cost]
    dead_label, dead_pair = pruning.prune_masks(graph, theta, unary, min(bounds[1::2]))
    return theta, unary, bounds, labels, dead_label, dead_pair


def _run_plan(state):
    mesh = state["mesh"]
    opt = ShardingOptimizer(state["gm"], mesh, state["rescale"], repeated_subgraphs=True)
    opt.add_grad_param_constraints()
    opt.add_parameter_memory_constraint(0.0, 1.0 / mesh.size())
    given, wanted = state["placements"]
    opt.add_sharded_input_constraint([given])
    opt.add_sharded_output_constraint([wanted])
    opt.get_solution()
    return opt.objective_vector, opt.forced_zero_vars, opt.compute_cost, opt.objective_value(), opt.res_entries


# ---- what a pass cannot do without ---------------------------------------------------------------------
def _graph_bytes(tb, layers, cost=True, comm=False, minima=False, shapes=False, host=False):
    """Inputs of the encoding read once, outputs written once (``tb``: one layer)."""
    width = 4  # values of a local shape row: the drawn tensors have at most four dims
    b = 8 * tb.n_specs + 22 * tb.n_strategies + 56 * tb.n_edges + 8 * len(tb.pt_values)  # read
    b += 16 * tb.n_strategies + 8 * tb.n_entries * cost + 9 * tb.n_entries * comm  # written
    if minima:
        b += 12 * tb.n_rows + 8 * tb.n_strategies + 12 * tb.n_nodes
    if shapes:
        b += (24 + 16 * width) * tb.n_specs
    if host:
        b += 18 * tb.n_strategies
    return b * layers + 145 * tb.n_tensors


def work(case):
    kind = case["kind"]
    if kind == "prune":
        blocks, sizes, _ = _labelling(case, 0)
        elements = sum(nt * ns for _, nt, ns, _, _ in blocks)
        sweeps = sum(SWEEP_CHUNKS)
        # a sweep takes every element's minimum, difference and share once from each side; the matrices cross
        # between host and device once each way per call
        return {"bytes": 16 * (elements + sum(sizes)) * (1 + len(SWEEP_CHUNKS)), "flops": 6 * elements * sweeps}
    if kind == "plan":
        # the entries of a traced decoder layer on its mesh (356 nodes, 430 edges a layer; 12 strategies a node
        # on a 2-D mesh, 3 on a 1-D one) and its share of specs and strategies
        per_edge = 146 if case["mesh"].count("x") else 8
        return {"bytes": (8 * per_edge + 500) * 430 * case["layers"], "flops": 9 * per_edge * 430 * case["layers"]}
    tb = _block(case)
    L, M = case["layers"], len(_mesh(case))
    n_bytes = _graph_bytes(tb, L, comm=kind == "report", minima=kind == "report", shapes=kind != "pass", host=kind == "tables")
    if kind == "tables":
        n_bytes += 9 * tb.n_entries * (1 if case["linked"] else L)
    return {"bytes": n_bytes, "flops": (4 * M + 2) * tb.n_entries * L}


def tolerance(case):
    # fp64 sums of a few terms (prune: of some hundred updates); every whole number is exact
    return {"rel": 1e-9 if case["kind"] == "prune" else 1e-12, "max": 1e-9}

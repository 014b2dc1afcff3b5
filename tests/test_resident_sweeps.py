"""Sweeps of the dual ascent with the matrices resident on the chip (apc_diffusion_sweeps_resident)
against the oracle's sweeps, bit for bit, at the sizes that choose workgroups, lanes per row and exchanges;
the plan they run from; and the way out when a wait expires."""

import numpy as np
import pytest

from autoparallel_amd import CostModelParams, pruning
from autoparallel_amd.synthetic import stress_dag
from test_pruning import _sweep


def _problem(seed, sizes, pairs, p_inf=0.1):
    rng = np.random.default_rng(seed)
    blocks, costs, at = [], {}, 0
    for i, j in pairs:
        m = rng.uniform(0, 100, (sizes[i], sizes[j]))
        m[rng.random(m.shape) < p_inf] = np.inf
        blocks.append(pruning.Block(at, sizes[i], sizes[j], i, j))
        costs[at] = m
        at += m.size
    masks = {0: np.arange(sizes[0]) % 3 != 1}
    return pruning.build_label_graph(blocks, list(sizes), lambda b: costs[b.var_begin], masks, [])


CASES = {
    "one matrix of one element": ([1, 1], [(0, 1)], 0.0),
    "rows of 1 to 70 elements, one workgroup's": ([1, 70, 2, 3], [(0, 1), (1, 2), (2, 3)], 0.1),
    "a chain over many workgroups": ([5 + i % 20 for i in range(150)], [(i, i - 1) for i in range(1, 150)], 0.1),
    "a class with 70 matrices (more than the kept reciprocals)": ([6] + [4] * 70, [(0, i) for i in range(1, 71)], 0.05),
    "a class with five matrices in as many workgroups": ([60, 50, 50, 50, 50, 50], [(i, 0) for i in range(1, 6)], 0.1),
    "as many rows in a step as threads": ([256, 1, 256], [(0, 1), (2, 1)], 0.0),
    "more rows in a step than 256 threads": ([300, 3], [(0, 1)], 0.1),
    "the largest matrix that fits": ([128, 134], [(0, 1)], 0.1),
    "labels that can never be taken": ([4, 3, 2], [(0, 1), (1, 2)], 0.7),
}


def _device():
    from autoparallel_amd.device_tables import DeviceCostTables

    return DeviceCostTables(stress_dag(seed=1, n_nodes=10, mesh_sizes=(2, 2)), CostModelParams.from_mesh((2, 2)))


@pytest.mark.gpu
@pytest.mark.parametrize("name", CASES)
def test_resident_sweeps_equal_the_oracle(gpu_device, name):
    sizes, pairs, p_inf = CASES[name]
    g = _problem(len(name), sizes, pairs, p_inf)
    dev = _device()
    plan = dev._sweep_plan(g)
    assert plan is not None, "the problem was meant to be resident"
    theta, unary = g.theta, g.unary
    want = (g.theta, g.unary)
    for n in (1, 2, 7):
        theta, unary = dev.diffusion_sweeps(g, theta, unary, n)
        want = _sweep(g, *want, n)
        assert np.array_equal(theta, want[0]) and np.array_equal(unary, want[1])
    if "many workgroups" in name or "five" in name:
        assert len(plan[1]) > 3 and plan[2] > 0  # (several workgroups, with something to exchange)


@pytest.mark.gpu
def test_an_expired_wait_leaves_the_sweeps_to_the_launches(gpu_device):
    sizes, pairs, p_inf = CASES["a chain over many workgroups"]
    g = _problem(3, sizes, pairs, p_inf)
    dev = _device()
    dev.SWEEP_WAIT_TICKS = 0  # no wait is long enough: every workgroup leaves at its first one
    theta, unary = dev.diffusion_sweeps(g, g.theta, g.unary, 3)
    want = _sweep(g, g.theta, g.unary, 3)
    assert np.array_equal(theta, want[0]) and np.array_equal(unary, want[1])


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["a chain over many workgroups", "a class with 70 matrices (more than the kept reciprocals)"])
def test_an_expired_wait_ends_the_kernel_whatever_the_sweeps(gpu_device, name):
    """By teams: a million sweeps whose first unmet wait is given up.  An update takes 0.2 us and more, so that all of them would
    be 400 ms; those of a sweep after the wait are some microseconds."""
    import torch

    g = _problem(4, *CASES[name])
    dev = _device()
    plan = dev._sweep_plan(g)
    assert (plan[0][plan[1][:-1] + 5] == 2).all() and len(plan[1]) > 3
    arrays = dev._upload(*plan[:2], g.theta, g.unary)
    run = lambda n: dev.ops.diffusion_sweeps_resident(  # noqa: E731
        n, *arrays[:2], *plan[2:], int(g.label_begin[-1]), int(g.edge_begin[-1]), *arrays[2:], 0)
    run(1)
    begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    begin.record()
    *_, status = run(1_000_000)
    end.record()
    assert int(status.item()) == 1 and begin.elapsed_time(end) < 40


def test_an_expired_wait_is_paid_once_per_problem():
    """On the CPU, with operators that only keep count: after a wait that expired, the chunks that follow take the launches
    at once; another problem has a plan again."""
    import torch

    from autoparallel_amd.device_tables import DeviceCostTables

    class Ops:
        resident = launches = 0

        def upload(self, arrays, device):
            return [t.clone() for t in arrays]

        def download(self, arrays):
            return [t.clone() for t in arrays]

        def diffusion_sweeps_resident(self, n, plan, begin, slots, lds, threads, n_labels, n_elements, theta, unary, ticks):
            Ops.resident += 1
            return theta.clone(), unary.clone(), torch.ones(1, dtype=torch.int32)  # expired

        def diffusion_sweeps_(self, *args):
            Ops.launches += 1

    dev = DeviceCostTables.__new__(DeviceCostTables)
    dev.ops, dev.device = Ops(), torch.device("cpu")
    sizes, pairs, p_inf = CASES["a chain over many workgroups"]
    for i in (1, 2):
        g = _problem(i, sizes, pairs, p_inf)
        pair = g.theta, g.unary
        for chunk in range(3):
            pair = dev.diffusion_sweeps(g, *pair, 4)
        assert (Ops.resident, Ops.launches) == (i, 3 * i)


def test_a_graph_whose_arrays_were_replaced_has_a_new_plan():
    """On the CPU: an old plan would index the new problem's arrays by the old one's sizes."""
    import torch

    from autoparallel_amd.device_tables import DeviceCostTables

    seen = []

    class Ops:
        def upload(self, arrays, device):
            return [t.clone() for t in arrays]

        def download(self, arrays):
            return [t.clone() for t in arrays]

        def diffusion_sweeps_resident(self, n, plan, begin, slots, lds, threads, n_labels, n_elements, theta, unary, ticks):
            seen.append((sum(int(plan[b + 1]) for b in begin[:-1]), n_elements))  # elements of the plan, of the problem
            return theta.clone(), unary.clone(), torch.zeros(1, dtype=torch.int32)

    dev = DeviceCostTables.__new__(DeviceCostTables)
    dev.ops, dev.device = Ops(), torch.device("cpu")
    g, small = (_problem(1, *CASES[name]) for name in ("a chain over many workgroups", "rows of 1 to 70 elements, one workgroup's"))
    dev.diffusion_sweeps(g, g.theta, g.unary, 4)
    for name in ("label_begin", "unary", "edge_i", "edge_j", "edge_begin", "theta", "inc_begin", "inc_edge", "inc_side", "color_begin",
                 "color_nodes"):
        setattr(g, name, getattr(small, name))
    dev.diffusion_sweeps(g, g.theta, g.unary, 4)
    assert all(a == b for a, b in seen) and seen[0][0] > seen[1][0] == len(small.theta)


@pytest.mark.parametrize("sizes,pairs", [([140, 140], [(0, 1)]), ([1500, 2], [(0, 1)])])
def test_problems_that_do_not_fit_have_no_plan(sizes, pairs):
    from autoparallel_amd.device_tables import DeviceCostTables

    assert DeviceCostTables._sweep_plan(_problem(0, sizes, pairs)) is None


def test_a_plan_holds_every_matrix_once_and_places_every_minimum():
    """Each workgroup's words against the problem: elements covered once, every class stored once, the
    minima of an incidence read where its row, or its slot, is written."""
    from autoparallel_amd.device_tables import DeviceCostTables

    sizes, pairs, p_inf = CASES["a chain over many workgroups"]
    g = _problem(5, sizes, pairs + [(149, 3), (80, 3), (20, 3), (120, 3), (60, 3)], p_inf)
    words, begin, n_slots, lds, threads = DeviceCostTables._sweep_plan(g)
    elements, stored, written, read = np.zeros(len(g.theta), int), np.zeros(len(g.unary), int), {}, {}
    for b, e in zip(begin[:-1], begin[1:]):
        p = words[b:e].astype(np.int64) & 0xFFFFFFFF
        first, n_el, n_rows, n_inc, n_steps = p[:5].tolist()
        rows = p[8:8 + 8 * n_rows].reshape(-1, 8)
        labels = p[8 + 8 * n_rows:8 + 9 * n_rows]
        elements[first:first + n_el] += 1
        np.add.at(stored, (labels & 0x7FFFFFFF)[labels >> 31 == 1], 1)
        assert ((rows[:, 0] & 0xFFFF) + ((rows[:, 0] >> 16) - 1) * (rows[:, 1] & 0xFFFF) < n_el).all()
        for r, label in zip(rows.tolist(), (labels & 0x7FFFFFFF).tolist()):
            if r[2] != 0xFFFFFFFF:
                assert r[2] not in written
                written[r[2]] = label
            for ref in r[4:]:
                if ref & 0x40000000:
                    read.setdefault(ref & 0x3FFFFFFF, set()).add(label)
                else:
                    assert ref == n_rows or labels[ref] & 0x7FFFFFFF == label
    degree = np.diff(g.inc_begin)
    assert (elements == 1).all() and np.array_equal(stored, np.repeat(degree > 0, np.diff(g.label_begin)))
    assert sorted(written) == list(range(n_slots)) and all(labels == {written[s]} for s, labels in read.items())


def _star(centre, first_leaf, n):
    """``n`` matrices between class ``centre`` and classes ``first_leaf`` .., stored either way round."""
    return [(centre, first_leaf + i) if i % 2 else (first_leaf + i, centre) for i in range(n)]


# (sizes, pairs, threads of a workgroup, whether the plan is by teams)
TEAMS = {
    "one wavefront a matrix, rows of 1 to 64 elements": (
        [17, 15, 64, 63, 1, 5, 33, 16, 4, 3, 2, 31], [(i, i - 1) for i in range(1, 12)], 512, True),
    "teams of two, four and eight wavefronts": ([64, 65, 90, 60, 20, 129, 9, 65, 3], [(i, i - 1) for i in range(1, 9)], 512, True),
    "teams of sixteen wavefronts": ([600, 3, 70, 120, 9], [(i, i - 1) for i in range(1, 5)], 1024, True),
    "classes of 4, 5, 8, 9 and 13 matrices over several workgroups": (
        [6 + i % 9 for i in range(60)],
        _star(0, 5, 4) + _star(1, 9, 5) + _star(2, 14, 8) + _star(3, 22, 9) + _star(4, 31, 13) + [(i, i - 5) for i in range(31, 60)], 512, True),
    # (two colours: teams of sixteen wavefronts a workgroup from 48 elements a matrix on, of eight from 10)
    "one wavefront more than half the workgroups' hold": ([7, 8] * 897, [(i, i - 1) for i in range(1, 1794)], 1024, True),
    "as many with few elements": ([6, 7] * 897, [(i, i - 1) for i in range(1, 1794)], 256, False),
    "as many with few elements and three colours": ([2, 3] * 897, [(i, i - 1) for i in range(1, 1794)] + [(2, 0)], 1024, True),
    "ten elements a matrix": ([2, 5] * 40, [(i, i - 1) for i in range(1, 80)], 512, True),
    "nine elements a matrix": ([3] * 80, [(i, i - 1) for i in range(1, 80)], 256, False),
    "more matrices than wavefronts": ([1, 2] * 1800, [(i, i - 1) for i in range(1, 3600)], 256, False),
    "few elements in one workgroup": ([3] * 20, [(i, i - 1) for i in range(1, 20)], 256, False),
}


@pytest.mark.parametrize("name", TEAMS)
def test_a_plan_by_teams_gives_every_row_its_wavefronts(name):
    """On the CPU: every matrix in one team, the side of the lower colour first, a lane for every row; all rows of a side agree on
    what the kernel takes to be uniform; the words end inside the plan and the bytes inside the LDS asked for."""
    from autoparallel_amd.device_tables import DeviceCostTables

    sizes, pairs, threads_wanted, by_teams = TEAMS[name]
    g = _problem(1, sizes, pairs)
    words, begin, n_slots, lds, threads = DeviceCostTables._sweep_plan(g)
    assert threads == threads_wanted and (words[begin[:-1] + 5] == (2 if by_teams else 0)).all()
    color = np.empty(g.n_classes, int)
    for c in range(len(g.color_begin) - 1):
        color[g.color_nodes[g.color_begin[c]:g.color_begin[c + 1]]] = c
    held = np.zeros(len(g.theta), int)
    for b, e in zip(begin[:-1], begin[1:]) if by_teams else ():
        p = words[b:e].astype(np.int64) & 0xFFFFFFFF
        first, n_el, n_rows, n_inc = p[:4].tolist()
        rows, labels = p[8:8 + 8 * n_rows].reshape(-1, 8), p[8 + 8 * n_rows:8 + 9 * n_rows] & 0x7FFFFFFF
        wave = p[8 + 9 * n_rows + n_inc:][:64].reshape(16, 4)
        assert 32 * n_rows + 8 * n_el + 4 * (n_inc + 17) <= lds <= 150 * 1024 and not wave[threads // 64:].any()
        classes = np.searchsorted(g.label_begin, labels, side="right") - 1
        teams, covered = {}, np.zeros(n_rows, int)
        for w in wave.tolist():
            if w[2] >> 16:
                teams.setdefault(w[2] & 0xFF, []).append((w[2] >> 8 & 0xFF, w[2] >> 16, w[0], w[1] & 0xFFFF, w[1] >> 16))
        for t in teams.values():
            (waves, at, n, m), = {x[1:] for x in t}
            assert sorted(x[0] for x in t) == list(range(waves)) and 1 <= n <= 64 * waves and 1 <= m <= 64 * waves
            covered[at:at + n + m] += 1
            side = rows[at:at + n], rows[at + n:at + n + m]
            assert color[classes[at]] < color[classes[at + n]] and len(set(classes[at:at + n])) == len(set(classes[at + n:at + n + m])) == 1
            for s, other in ((side[0], m), (side[1], n)):
                assert (s[:, 0] >> 16 == other).all() and len({(*r[[1, 3]] & [0xFFFF, -1], r[2] == 0xFFFFFFFF, *r[4:] >> 30 & 1) for r in s}) == 1
                elements = (s[:, :1] & 0xFFFF) + np.arange(other) * (s[:, 1:2] & 0xFFFF)
                assert len(np.unique(elements)) == n * m and elements.max() < n_el
                np.add.at(held, first + elements.ravel(), 1)
        assert (covered == 1).all()
    assert (held == (2 if by_teams else 0)).all()


@pytest.mark.parametrize("n_matrices", [1, 215, 218, 224])
def test_the_plan_buffer_holds_teams_up_to_the_most_workgroups(n_matrices):
    """On the CPU: one matrix a workgroup, up to as many workgroups as can be resident."""
    from autoparallel_amd.device_tables import DeviceCostTables

    words, begin, *_ = DeviceCostTables._sweep_plan(_problem(1, [130] * (n_matrices + 1), [(i, i - 1) for i in range(1, n_matrices + 1)]))
    assert len(begin) - 1 == n_matrices and set(words[begin[:-1] + 5].tolist()) == {2}


@pytest.mark.gpu
@pytest.mark.parametrize("name", TEAMS)
def test_sweeps_by_teams_equal_the_oracle(gpu_device, name):
    sizes, pairs, _, _ = TEAMS[name]
    g = _problem(len(name), sizes, pairs)
    dev = _device()
    theta, unary = g.theta, g.unary
    want = (g.theta, g.unary)
    for n in (1, 2, 5):
        theta, unary = dev.diffusion_sweeps(g, theta, unary, n)
        want = _sweep(g, *want, n)
        assert dev._diffusion_graph["plan"] is not None  # (no wait expired)
        assert np.array_equal(theta, want[0]) and np.array_equal(unary, want[1])

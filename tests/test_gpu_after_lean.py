"""GPU: what may follow a lean iteration besides another iteration of the same search.  A lean iteration keeps rows
that repeat others once and, on few roots, leaves the ranges in a second buffer; a captured graph, a snapshot, the
launch-per-operation path and ranges written by the caller all go on from there as from a plain iteration, bit for bit."""
import numpy as np
import pytest
import torch

from tests.helpers import random_boards, random_ranges
from tests.test_gpu_lean_search import STATE

pytestmark = pytest.mark.gpu

CFR = [("discounted", False), ("linear", True)]


def build(cfr_type, cfr_avg, *, one_walk, n=3, cls=None):
    from poker2_amd.config import river_dcfr_config
    from poker2_amd.evaluator import HipSparseCFREvaluator
    from poker2_amd.fused_cfr_hip import CFRType
    from poker2_amd.tree import RootStates
    rng = np.random.default_rng(17)
    boards = random_boards(rng, n)
    beliefs = torch.from_numpy(random_ranges(rng, boards))
    roots = RootStates.at_round_start(3, np.full(n, 200), np.full((n, 2), 800), boards, bb=100)
    cfg = river_dcfr_config(n, iterations=8, depth=16)
    cfg.search.cfr_type, cfg.search.cfr_avg = CFRType[cfr_type], cfr_avg
    cfg.env.bet_bins = [0.5, 1.0]
    ev = HipSparseCFREvaluator(None, torch.device("cuda"), cfg, max_raises=3)
    ev.initialize_subgame(roots, np.arange(n), beliefs)
    ev.prepare_search(t_sample=torch.full((ev.total_nodes,), 3))
    assert ev._one_walk
    ev._one_walk = one_walk
    return ev


def assert_same(a, b, names=STATE):
    for name in names:
        assert torch.equal(getattr(a, name), getattr(b, name)), name


@pytest.mark.parametrize("alternate", [0, 1, 2])       # how many of the two lean iterations alternate reach_avg
@pytest.mark.parametrize("one_walk", [False, True])
@pytest.mark.parametrize("cfr_type,cfr_avg", CFR)
def test_replay_of_a_captured_graph(cfr_type, cfr_avg, one_walk, alternate):
    from poker2_amd.evaluator import GraphedCFRIteration
    plain, lean = (build(cfr_type, cfr_avg, one_walk=one_walk) for _ in range(2))
    graph = GraphedCFRIteration(lean)
    graph.capture(2)                                   # runs iterations 2, 3 and 2
    for t in (2, 3, 2):
        plain.cfr_iteration(t)
    for base in (3, 7):                                # twice: the second time a replay lies before
        for k in range(2):
            plain.cfr_iteration(base + k)
            lean.cfr_iteration(base + k, lean=True, alternate_reach_avg=k < alternate)
        for k in (2, 3):
            plain.cfr_iteration(base + k)
            graph.replay(base + k)
            assert_same(plain, lean)
    plain.cfr_iteration(11)
    lean.cfr_iteration(11)
    assert_same(plain, lean)


@pytest.mark.parametrize("one_walk", [False, True])
@pytest.mark.parametrize("cfr_type,cfr_avg", CFR)
def test_snapshot(cfr_type, cfr_avg, one_walk):
    """Taken after lean iterations and restored into another evaluator, into the same one, and before a replay."""
    from poker2_amd.evaluator import GraphedCFRIteration, _EvaluatorStateSnapshot
    plain, lean, other, graphed = (build(cfr_type, cfr_avg, one_walk=one_walk) for _ in range(4))
    graph = GraphedCFRIteration(graphed)
    graph.capture(0)
    for t in range(3):
        plain.cfr_iteration(t)
        lean.cfr_iteration(t, lean=True, alternate_reach_avg=True)
    kept = _EvaluatorStateSnapshot.from_evaluator(lean)
    for ev in (lean, graphed):                         # restored over a state left by another lean iteration
        ev.cfr_iteration(3, lean=True, alternate_reach_avg=True)
    for ev in (lean, other, graphed):
        kept.restore_to(ev)
    for t in (3, 4):
        plain.cfr_iteration(t)
        lean.cfr_iteration(t)
        other.cfr_iteration(t)
        graph.replay(t)
        for ev in (lean, other, graphed):
            assert_same(plain, ev)


@pytest.mark.parametrize("one_walk", [False, True])
@pytest.mark.parametrize("cfr_type,cfr_avg", CFR)
def test_root_ranges_written_between_iterations(cfr_type, cfr_avg, one_walk):
    plain, lean = (build(cfr_type, cfr_avg, one_walk=one_walk) for _ in range(2))
    for t in range(6):                                 # one lean iteration, and two, before a plain one
        plain.cfr_iteration(t)
        lean.cfr_iteration(t, lean=t in (0, 2, 3), alternate_reach_avg=True)
        if t in (1, 4, 5):
            assert_same(plain, lean)
        for ev in (plain, lean):
            for table in (ev.beliefs, ev.beliefs_avg):
                table[:ev.root_nodes] = table[:ev.root_nodes].flip(1)


@pytest.mark.parametrize("one_walk", [False, True])
@pytest.mark.parametrize("cfr_type,cfr_avg", CFR)
def test_iteration_by_single_operations(cfr_type, cfr_avg, one_walk):
    plain, lean = (build(cfr_type, cfr_avg, one_walk=one_walk) for _ in range(2))
    for t in range(4):
        plain.cfr_iteration(t)
        lean.cfr_iteration(t, lean=True, alternate_reach_avg=t > 0)
    for ev in (plain, lean):
        ev.fused_iteration = False
        ev.cfr_iteration(4)
    assert_same(plain, lean)


@pytest.mark.parametrize("one_walk", [False, True])
@pytest.mark.parametrize("cfr_type,cfr_avg", CFR)
def test_tensors_put_in_place_of_the_ranges(cfr_type, cfr_avg, one_walk):
    """A caller may bind its own tensors to ``beliefs`` and ``beliefs_avg`` before the first iteration, and they stay bound."""
    kept, bound = (build(cfr_type, cfr_avg, one_walk=one_walk) for _ in range(2))
    for ev in (kept, bound):
        for table in (ev.beliefs, ev.beliefs_avg):
            table[:] = table.flip(1)
    mine = {name: getattr(bound, name).clone() for name in ("beliefs", "beliefs_avg")}
    for name, table in mine.items():
        getattr(bound, name).fill_(float("nan"))
        setattr(bound, name, table)
    for t in range(6):
        for ev in (kept, bound):
            ev.cfr_iteration(t, lean=t in (1, 3, 4), alternate_reach_avg=True)
        if t in (0, 2, 5):
            assert_same(kept, bound)
            assert all(getattr(bound, name) is table for name, table in mine.items())
    assert torch.equal(kept._compute_exploitability().local_exploitability, bound._compute_exploitability().local_exploitability)


@pytest.mark.parametrize("one_walk", [False, True])
def test_cfr_avg_switched_off_between_iterations(one_walk):
    plain, lean = (build("linear", True, one_walk=one_walk) for _ in range(2))
    for t in range(4):
        for ev in (plain, lean):
            ev.cfr_avg = t < 1
        plain.cfr_iteration(t)
        lean.cfr_iteration(t, lean=t in (0, 2), alternate_reach_avg=True)
        if t in (1, 3):
            assert_same(plain, lean)


def captured(ev, **kw):
    """A graph of one iteration, recorded by the caller's own means; replayed for any t behind ``prepare_replay``."""
    ev.prepare_replay(2)
    ev._skip_t_scalars_update = True
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ev.cfr_iteration(2, **kw)
    ev._skip_t_scalars_update = False

    def replay(t):
        ev.prepare_replay(t)
        graph.replay()
    return replay


@pytest.mark.parametrize("lean", [False, True])        # what is recorded
@pytest.mark.parametrize("alternate", [False, True])   # the two eager lean iterations before a replay
@pytest.mark.parametrize("one_walk", [False, True])
@pytest.mark.parametrize("cfr_type,cfr_avg", CFR)
def test_graph_recorded_by_the_caller(cfr_type, cfr_avg, one_walk, alternate, lean):
    """Replays between eager iterations, which cannot know that a replay ran; recording itself runs nothing."""
    plain, ev = (build(cfr_type, cfr_avg, one_walk=one_walk) for _ in range(2))
    kw = dict(lean=True, alternate_reach_avg=alternate)
    for t in (2, 3):
        plain.cfr_iteration(t)
    ev.cfr_iteration(2)
    ev.cfr_iteration(3, lean=alternate)
    replay = captured(ev, lean=lean)                   # recorded behind a plain iteration and behind a lean one
    t = 4
    for eager in (alternate, 1, 2, 2, 1):              # a plain iteration, or a pair of lean ones, between replays
        for _ in range(eager % 2):
            plain.cfr_iteration(t)
            ev.cfr_iteration(t)
            assert_same(plain, ev)
            t += 1
        for _ in range(eager // 2 * 2):
            plain.cfr_iteration(t)
            ev.cfr_iteration(t, **kw)
            t += 1
        for _ in range(2):
            plain.cfr_iteration(t)
            replay(t)
            if not lean:
                assert_same(plain, ev)
            t += 1
    plain.cfr_iteration(t)
    ev.cfr_iteration(t)
    assert_same(plain, ev)


@pytest.mark.parametrize("cfr_type,cfr_avg", CFR)
def test_graph_recorded_while_the_ranges_lie_in_the_second_buffer(cfr_type, cfr_avg):
    plain, ev = (build(cfr_type, cfr_avg, one_walk=True) for _ in range(2))
    for t in (2, 3):
        plain.cfr_iteration(t)
        ev.cfr_iteration(t, lean=t == 3, alternate_reach_avg=True)
    replay = captured(ev)
    for t in range(4, 8):
        plain.cfr_iteration(t)
        replay(t)
        assert_same(plain, ev)
    for t in range(8, 11):
        plain.cfr_iteration(t)
        ev.cfr_iteration(t, lean=t < 10, alternate_reach_avg=t < 10)
    assert_same(plain, ev)

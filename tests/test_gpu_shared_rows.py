"""GPU: rows of the search state that repeat others (the range of the player who did not act, the values of a fold
leaf) are kept once by lean iterations.  The rows left out are overwritten with NaN between iterations: the state
at the end is that of plain iterations, bit for bit."""
import numpy as np
import pytest
import torch

from tests.test_gpu_lean_search import STATE, VARIANTS, build

pytestmark = pytest.mark.gpu


def expected_range_rows(tree) -> np.ndarray:
    """By the rule's definition, from the root downwards."""
    out = 2 * np.arange(tree.total)
    to_act = np.asarray(tree.state["to_act"])
    for c in range(tree.n_roots, tree.total):
        p = tree.parent_index[c]
        o = 1 - to_act[p]
        if p < tree.n_roots:
            out[c] = 2 * c + o
        else:
            out[c] = out[p] if out[p] % 2 == o else 2 * p + o
    return out


@pytest.mark.parametrize("seed", range(8))
def test_range_rows_and_the_rows_they_stand_for(seed):
    ev = build(seed, VARIANTS[seed % len(VARIANTS)], None, lean=False, iters=4)
    want = expected_range_rows(ev.tree)
    assert np.array_equal(ev._range_rows.cpu().numpy(), want)
    for t in range(3):
        ev.cfr_iteration(t)
    rows = torch.from_numpy(want[ev.root_nodes:]).to(ev.device)
    at = torch.arange(ev.root_nodes, ev.total_nodes, device=ev.device) * 2 + rows % 2
    for name in ("self_reach", "self_reach_avg", "beliefs", "beliefs_avg"):
        flat = getattr(ev, name).view(-1, 1326)
        assert torch.equal(flat[at], flat[rows]), name
    folds = torch.from_numpy(np.nonzero(ev.tree.fold_mask)[0]).to(ev.device)
    for name in ("latest_values", "values_avg"):
        x = getattr(ev, name)[folds]
        assert torch.equal(x, x[:, :, :1].expand_as(x)), name


@pytest.mark.parametrize("one_walk", [False, True])
@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("seed", range(8))
def test_rows_kept_elsewhere_are_never_read(seed, split, one_walk):
    variant = VARIANTS[(seed + 5) % len(VARIANTS)]
    iters = 5 + seed % 2
    plain = build(seed, variant, split, lean=False, iters=iters)
    lean = build(seed, variant, split, lean=True, iters=iters)
    lean._one_walk = lean._one_walk and one_walk
    if one_walk and not (lean._one_walk and seed % 3 and not lean.enforce_zero_sum and not lean._rows_are_watched()):
        pytest.skip("this search is not one of the one-walk kernel: the other half of the parametrisation runs it")
    tree = lean.tree
    want = expected_range_rows(tree)
    network = tree.leaf_mask & ~np.asarray(tree.state["done"]) & (lean.model is not None)
    moved = (want // 2 != np.arange(tree.total)) & ~network
    dead = torch.from_numpy(np.nonzero(moved)[0] * 2 + want[moved] % 2).to(lean.device)
    folds = torch.from_numpy(np.nonzero(tree.fold_mask)[0]).to(lean.device)
    for t in range(iters):
        plain.cfr_iteration(t)
        last = t + 1 == iters
        lean.cfr_iteration(t, lean=not last, alternate_reach_avg=bool(seed % 3))
        if not last:
            assert lean._walked == one_walk
            for name in ("self_reach", "self_reach_avg", "beliefs") + (() if lean.enforce_zero_sum else ("beliefs_avg",)):
                getattr(lean, name).view(-1, 1326)[dead] = float("nan")
            lean.values_avg[folds, :, 2:] = float("nan")
    for name in STATE:
        assert torch.equal(getattr(plain, name), getattr(lean, name)), f"seed {seed} {variant} split {split}: {name}"
    # and plain iterations go on from there
    plain.cfr_iteration(iters)
    lean.cfr_iteration(iters)
    for name in STATE:
        assert torch.equal(getattr(plain, name), getattr(lean, name)), name


@pytest.mark.parametrize("cfr_type,cfr_avg,street", [("discounted", False, 3), ("linear", True, 3), ("discounted", False, 2)])
def test_one_walk_over_long_family_lists(cfr_type, cfr_avg, street):
    """More than 64 families per work item (the window of the family list moves), one root and three, with and
    without showdown rows; the one-walk kernel against plain iterations, and against the three walks."""
    from poker2_amd.config import river_dcfr_config
    from poker2_amd.evaluator import HipSparseCFREvaluator
    from poker2_amd.fused_cfr_hip import CFRType
    from poker2_amd.tree import RootStates
    from tests.helpers import random_boards, random_ranges
    for n in (1, 3):
        rng = np.random.default_rng(77 + n)
        boards = random_boards(rng, n)
        if street == 2:
            boards[:, 4] = -1
        beliefs = torch.from_numpy(random_ranges(rng, boards))
        roots = RootStates.at_round_start(street, np.full(n, 200), np.full((n, 2), 4000), boards, bb=100)
        runs = []
        for lean, walk in ((False, False), (True, False), (True, True)):
            cfg = river_dcfr_config(n, iterations=6, depth=8)
            cfg.search.cfr_type, cfg.search.cfr_avg = CFRType[cfr_type], cfr_avg
            cfg.env.bet_bins = [0.5, 1.0]
            ev = HipSparseCFREvaluator(None, torch.device("cuda"), cfg, max_raises=4, split_small_batches=False,
                                       lean_search=lean)
            ev.initialize_subgame(roots, np.arange(n), beliefs)
            assert ((ev.tree.child_count > 0).sum() > 64 * n) and (not lean or ev._one_walk)
            ev._one_walk = walk
            ev.prepare_search(t_sample=torch.full((ev.total_nodes,), 2))
            ev.run_search_iterations()
            runs.append(ev)
        for ev in runs[1:]:
            for name in STATE:
                assert torch.equal(getattr(runs[0], name), getattr(ev, name)), f"{n} roots: {name}"


def test_entry_point_refuses_what_the_one_walk_kernel_cannot_run():
    import ctypes
    from poker2_amd import _lib
    ev = build(1, VARIANTS[0], False, lean=True, iters=4)
    lib, stream, p = _lib.load(), _lib.stream_ptr(), _lib.ptr
    args = ev._iter_bundle(True).main
    rows, a, b = p(ev._range_rows), p(ev.beliefs), p(torch.empty_like(ev.beliefs))
    walk = 64 | 32 | 16

    def refused(*call):
        return lib.p2hip_cfr_iteration_shared(*call, stream) != 0
    n = ev.root_nodes
    assert refused(ctypes.byref(args), rows, a, a, n, 4, walk | 3)             # one range buffer
    assert refused(ctypes.byref(args), rows, a, None, n, 4, walk | 3)
    assert refused(ctypes.byref(args), None, a, b, n, 4, walk | 3)             # no range rows
    assert refused(ctypes.byref(args), rows, a, b, n, 6, walk | 3)             # six children
    assert refused(ctypes.byref(args), rows, a, b, n, 4, walk | 8)             # a part of the first walk
    assert refused(ctypes.byref(args), rows, a, b, n, 4, 64 | 16 | 3)
    assert refused(ctypes.byref(ev._iter_bundle(False).main), rows, a, b, n, 4, walk | 3)   # reach_avg in place
    assert refused(ctypes.byref(args), rows, None, b, n, 4, 3)                 # a second range buffer without the walk
    torch.cuda.synchronize()


@pytest.mark.parametrize("bins", [[0.5, 1.0], [0.25, 0.5, 1.0, 2.0]])
@pytest.mark.parametrize("one_walk", [False, True])
def test_rows_of_one_number_at_any_child(bins, one_walk):
    """Rows flagged as one number per player need not be fold leaves, nor the first of their siblings: here every leaf
    at the depth limit is one too.  The closing iteration mixes a row's first pair in every wave and stores it in one."""
    from poker2_amd.config import river_dcfr_config
    from poker2_amd.evaluator import HipSparseCFREvaluator
    from poker2_amd.tree import RootStates
    from tests.helpers import random_boards, random_ranges
    n = 48
    rng = np.random.default_rng(31)
    boards = random_boards(rng, n)
    beliefs = torch.from_numpy(random_ranges(rng, boards))
    roots = RootStates.at_round_start(3, np.full(n, 200), np.full((n, 2), 4000), boards, bb=100)
    runs = []
    for lean in (False, True):
        cfg = river_dcfr_config(n, iterations=5, depth=3)
        cfg.env.bet_bins = bins
        ev = HipSparseCFREvaluator(None, torch.device("cuda"), cfg, lean_search=lean)
        ev.initialize_subgame(roots, np.arange(n), beliefs)
        ev.prepare_search(t_sample=torch.full((ev.total_nodes,), 2))
        gen = torch.Generator(device="cuda").manual_seed(5)
        for table in (ev.latest_values, ev.values_avg):
            table[ev.model_indices] = torch.rand(ev.model_indices.numel(), 2, 1, generator=gen, device="cuda") - 0.5
        if lean:
            ev._node_flags[ev.model_indices] |= 16
            ev._one_walk = ev._one_walk and one_walk
        ev.run_search_iterations()
        runs.append(ev)
    siblings = runs[1].tree.parent_index[runs[1].model_indices.cpu().numpy()]
    assert (np.diff(siblings) == 0).any() and (runs[1]._max_children > 5) == (len(bins) > 2)
    for name in STATE:
        assert torch.equal(getattr(runs[0], name), getattr(runs[1], name)), name


@pytest.mark.parametrize("split", [False, None])       # one tier of whole roots; the rule's own cut at every level
@pytest.mark.parametrize("network", [False, True])
@pytest.mark.parametrize("cfr_type,cfr_avg", [("discounted", False), ("linear", True)])
def test_one_walk_reads_only_what_it_keeps(cfr_type, cfr_avg, network, split):
    """The one-walk kernel on river trees with showdown leaves, alternating throughout: rows it leaves out, and all but
    the roots' rows of the two buffers that its next iteration writes, hold NaN between iterations."""
    from poker2_amd.config import river_dcfr_config
    from poker2_amd.evaluator import HipSparseCFREvaluator
    from poker2_amd.fused_cfr_hip import CFRType
    from poker2_amd.leaf_models import NetworkLeafModel, RangeBoardMLP
    from poker2_amd.tree import RootStates
    from tests.helpers import random_boards, random_ranges
    n, iters = 5, 6
    rng = np.random.default_rng(41)
    boards = random_boards(rng, n)
    beliefs = torch.from_numpy(random_ranges(rng, boards))
    stacks = np.full((n, 2), 4000 if network else 800)
    roots = RootStates.at_round_start(3, np.full(n, 200), stacks, boards, button=rng.integers(0, 2, n), bb=100)
    runs = []
    for lean in (False, True):
        model = (NetworkLeafModel(RangeBoardMLP(hidden=64, layers=2).cuda(), torch.device("cuda")) if network else None)
        cfg = river_dcfr_config(n, iterations=iters, depth=4 if network else 16)
        cfg.search.cfr_type, cfg.search.cfr_avg = CFRType[cfr_type], cfr_avg
        cfg.env.bet_bins = [0.5, 1.0]
        ev = HipSparseCFREvaluator(model, torch.device("cuda"), cfg, max_raises=None if network else 3,
                                    split_small_batches=split, lean_search=lean)
        ev.initialize_subgame(roots, np.arange(n), beliefs)
        ev.prepare_search(t_sample=torch.full((ev.total_nodes,), 2))
        runs.append(ev)
    plain, ev = runs
    tree = ev.tree
    assert ev._one_walk and ev._has_model_leaves == network and tree.showdown_mask.any()
    assert len(ev._iter_bundle(True).walk) == (1 if split is False else 4 if network else 5)
    want = expected_range_rows(tree)
    at_network = tree.leaf_mask & ~np.asarray(tree.state["done"])
    moved = (want // 2 != np.arange(tree.total)) & ~at_network
    passive = torch.from_numpy(np.nonzero(moved)[0] * 2 + want[moved] % 2).cuda()
    showdown = torch.from_numpy(np.nonzero(tree.showdown_mask)[0]).cuda()
    folds = torch.from_numpy(np.nonzero(tree.fold_mask)[0]).cuda()
    for t in range(iters):
        plain.cfr_iteration(t)
        ev.cfr_iteration(t, lean=t + 1 < iters, alternate_reach_avg=True)
        if t + 1 < iters:
            assert ev._walked
            for name in ("self_reach", "self_reach_avg", "beliefs", "beliefs_avg"):
                getattr(ev, name).view(-1, 1326)[passive] = float("nan")
            for name in ("beliefs", "beliefs_avg"):
                getattr(ev, name)[showdown] = float("nan")
            ev._leaf_alt[n:] = float("nan")
            ev._reach_avg_alt[n:] = float("nan")
            ev.values_avg[folds, :, 2:] = float("nan")
    for name in STATE:
        assert torch.equal(getattr(plain, name), getattr(ev, name)), name


@pytest.mark.parametrize("lean", [False, True])
@pytest.mark.parametrize("alternate", [False, True])
@pytest.mark.parametrize("seed", [1, 2, 6])
def test_the_entry_point_without_shared_rows(seed, alternate, lean):
    """p2hip_cfr_iteration called directly, in place and between two reach_avg buffers, against the evaluator."""
    import ctypes
    from poker2_amd import _lib
    lib = _lib.load()
    iters = 6
    want, got = (build(seed, VARIANTS[0], False, lean=False, iters=iters) for _ in range(2))
    other = got.self_reach_avg.clone()
    for t in range(iters):
        want.cfr_iteration(t)
        got.prepare_replay(t)
        args = (got._build_iter_args(reach_avg=other, reach_avg_prev=got.self_reach_avg) if alternate
                else got._build_iter_args())
        code = lib.p2hip_cfr_iteration(ctypes.byref(args), got.root_nodes, got._max_children,
                                       3 | (16 if lean and t + 1 < iters else 0), _lib.stream_ptr())
        assert code == 0
        if alternate:
            got.self_reach_avg, other = other, got.self_reach_avg
    for name in STATE:
        assert torch.equal(getattr(want, name), getattr(got, name)), name

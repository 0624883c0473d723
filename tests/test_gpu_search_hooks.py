"""GPU: code from outside the package that runs between the parts of a search's iterations (a leaf model with the
node table or the evaluator in hand, an overridden method) finds the rows there that a lean iteration has always
stored, whole, and the node table at one address."""
import numpy as np
import pytest
import torch

from tests.helpers import random_boards, random_ranges
from tests.test_gpu_lean_search import STATE

pytestmark = pytest.mark.gpu


def build(make_model, lean, cfr_type, cfr_avg, cls=None):
    from poker2_amd.config import river_dcfr_config
    from poker2_amd.evaluator import HipSparseCFREvaluator
    from poker2_amd.fused_cfr_hip import CFRType
    from poker2_amd.tree import RootStates
    n = 3
    rng = np.random.default_rng(23)
    boards = random_boards(rng, n)
    roots = RootStates.at_round_start(3, np.full(n, 200), np.full((n, 2), 4000), boards, bb=100)
    cfg = river_dcfr_config(n, iterations=6, depth=3)
    cfg.search.cfr_type, cfg.search.cfr_avg = CFRType[cfr_type], cfr_avg
    cfg.env.bet_bins = [0.5, 1.0]
    ev = (cls or HipSparseCFREvaluator)(make_model(), torch.device("cuda"), cfg, lean_search=lean)
    ev.initialize_subgame(roots, np.arange(n), torch.from_numpy(random_ranges(rng, boards)))
    ev.prepare_search(t_sample=torch.full((ev.total_nodes,), 2))
    return ev


def seen(ev, ranges=None) -> dict:
    """What a lean iteration stores whatever else it leaves out."""
    tree = ev.tree
    parents = torch.from_numpy(np.nonzero(tree.child_count > 0)[0]).cuda()
    leaves = torch.from_numpy(np.nonzero(tree.showdown_mask)[0]).cuda()
    rows = torch.cat([parents, leaves, ev.model_indices])
    ranges = (ev.beliefs_avg if ev.cfr_avg else ev.beliefs) if ranges is None else ranges
    return {"ranges": ranges[rows].clone(), "beliefs": ev.beliefs[parents].clone(),
            "reach": ev.self_reach[parents].clone(), "reach_avg": ev.self_reach_avg[parents].clone(),
            "values": ev.latest_values.clone(), "average values": ev.values_avg.clone(),
            "policy": ev.policy_probs.clone(), "average policy": ev.policy_probs_avg.clone()}


class GatheredRows:
    enforce_zero_sum = False

    def __init__(self):
        self.log, self.addresses = [], set()

    def leaf_values(self, beliefs, rows, ev):
        self.log.append(seen(ev))
        self.addresses.add((ev.beliefs_avg if ev.cfr_avg else ev.beliefs).data_ptr())
        return 0.3 * torch.flip(beliefs, dims=[1]) * 50.0 - 0.01


class NodeTable(GatheredRows):
    def leaf_values_from_nodes(self, table, rows, ev):
        self.log.append(seen(ev, table))
        self.addresses.add(table.data_ptr())
        return 0.3 * torch.flip(table[rows], dims=[1]) * 50.0 - 0.01


def assert_same_logs(want, got):
    assert len(want) == len(got) >= 5
    for k, (a, b) in enumerate(zip(want, got)):
        for name in a:
            assert torch.equal(a[name], b[name]), f"call {k}: {name}"


@pytest.mark.parametrize("cfr_type,cfr_avg", [("discounted", False), ("linear", True)])
@pytest.mark.parametrize("kind", [GatheredRows, NodeTable])
def test_leaf_model_that_looks_around(kind, cfr_type, cfr_avg):
    runs = []
    for lean in (False, True):
        ev = build(kind, lean, cfr_type, cfr_avg)
        ev.run_search_iterations()
        runs.append(ev)
    assert_same_logs(runs[0].model.log, runs[1].model.log)
    assert len(runs[1].model.addresses) == 1
    for name in STATE:
        assert torch.equal(getattr(runs[0], name), getattr(runs[1], name)), name


@pytest.mark.parametrize("hook", ["cfr_iteration", "set_leaf_values", "prepare_replay"])
@pytest.mark.parametrize("bound", ["subclass", "instance"])
def test_overridden_method_that_looks_around(hook, bound):
    from poker2_amd.evaluator import HipSparseCFREvaluator
    from poker2_amd.leaf_models import NetworkLeafModel, RangeBoardMLP

    def wrapped(log, inner):
        def call(self, *args, **kw):
            out = inner(self, *args, **kw)
            if getattr(self, "recording", False):
                log.append(seen(self))
            return out
        return call
    runs = []
    for lean in (False, True):
        log = []
        method = wrapped(log, getattr(HipSparseCFREvaluator, hook))
        cls = type("Recording", (HipSparseCFREvaluator,), {hook: method}) if bound == "subclass" else None
        ev = build(lambda: NetworkLeafModel(RangeBoardMLP(hidden=64, layers=2).cuda(), torch.device("cuda")), lean,
                   "discounted", False, cls)
        if cls is None:
            setattr(ev, hook, method.__get__(ev))
        ev.recording = True
        ev.run_search_iterations()
        runs.append((ev, log))
    assert_same_logs(runs[0][1], runs[1][1])


def test_the_packages_own_models_share_rows():
    """The models of this package look at the rows they are asked about only: their searches take the short way."""
    from poker2_amd.leaf_models import ChanceLeafModel, NetworkLeafModel, RangeBoardMLP
    net = RangeBoardMLP(hidden=64, layers=2).cuda()
    for make in (lambda: NetworkLeafModel(net, torch.device("cuda")), lambda: ChanceLeafModel(net, torch.device("cuda")),
                 lambda: None, lambda: net):
        ev = build(make, True, "discounted", False)
        assert ev._one_walk
        ev.cfr_iteration(0, lean=True, alternate_reach_avg=True)
        assert ev._walked and ev._rows_short
    ev = build(GatheredRows, True, "discounted", False)
    ev.cfr_iteration(0, lean=True, alternate_reach_avg=True)
    assert not ev._walked

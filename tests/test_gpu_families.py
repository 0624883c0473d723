"""The evaluator's methods as one launch per family or level (csrc/cfr_families.hip) against the same methods as the
reference composes them of single operations: bit for bit, on trees with up to five and up to eight children per
parent, roots of mixed streets and single ones, ranges and reaches with zeros, and rows without any mass."""
import numpy as np
import pytest
import torch

from tests.helpers import random_boards, random_ranges

pytestmark = pytest.mark.gpu
H = 1326


def make(n, bins, depth, streets, seed):
    from poker2_amd.config import Config, EnvConfig, SearchConfig
    from poker2_amd.evaluator import HipSparseCFREvaluator
    from poker2_amd.tree import RootStates
    rng = np.random.default_rng(seed)
    at = rng.choice(streets, n)
    boards = random_boards(rng, n, 5)
    for k, street in enumerate(at):
        boards[k, street + 2:] = -1
    roots = RootStates.at_round_start(at, rng.integers(1, 9, n) * 100, rng.integers(4, 41, (n, 2)) * 100, boards,
                                      button=rng.integers(0, 2, n))
    cfg = Config(num_envs=n, env=EnvConfig(bet_bins=bins, bb=100), search=SearchConfig(depth=depth, iterations=8))
    ev = HipSparseCFREvaluator(None, torch.device("cuda"), cfg, fused_iteration=False)
    ev.initialize_subgame(roots, np.arange(n), torch.from_numpy(random_ranges(rng, boards)))
    ev.prepare_search(t_sample=torch.full((ev.total_nodes,), -1, dtype=torch.long))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    # a state no search would leave: zeros, whole families without positive regret, rows without reach
    ev.cumulative_regrets.normal_(generator=gen)
    ev.cumulative_regrets[::3] = -1.0
    for t in (ev.self_reach, ev.self_reach_avg):
        t[n:] = torch.rand(t[n:].shape, generator=gen, device="cuda") ** 4
        t[n + 1::7] = 0
    ev.policy_probs_avg.uniform_(generator=gen)
    ev.policy_probs_avg[n::5] = 0
    ev.latest_values.normal_(generator=gen)
    return ev


CASES = [(1, [0.5, 1.0], 16, [3], 0), (7, [0.5, 1.0], 5, [1, 2, 3], 1), (5, [0.3, 0.5, 0.8, 1.0, 1.5], 3, [2, 3], 2)]


@pytest.fixture(params=CASES, ids=["one root", "mixed streets", "eight actions"])
def ev(request):
    ev = make(*request.param)
    assert (ev._max_children > 5) == (len(ev.bet_bins) == 5)
    ev.prepare_replay(3)
    return ev


def test_regrets(ev):
    from poker2_amd import fused_cfr_hip as F
    bottom, top = ev.depth_offsets[1], ev.depth_offsets[-2]
    achieved, expected = ev.latest_values, ev.latest_values.roll(1, dims=0).contiguous()
    want = torch.zeros_like(ev.policy_probs)
    rows = torch.arange(top, device="cuda")
    F.fused_regret_tail_(regrets=want, values_achieved=achieved,
                         actor_values=expected[:top][rows, ev.env.to_act[:top]].contiguous(),
                         src_weights=F.unblocked_mass_opp_at_parents_triton(ev.beliefs_avg if ev.cfr_avg else ev.beliefs,
                                                                             ev.env.to_act, top),
                         parent_index=ev.parent_index, prev_actor=ev.prev_actor, bottom=bottom)
    junk = torch.full_like(want, float("nan"))
    del junk                                             # the result may get its memory: every row has to be written
    assert torch.equal(ev.compute_instantaneous_regrets(achieved, expected), want)
    # what is read at parents may end behind the last of them
    assert torch.equal(ev.compute_instantaneous_regrets(achieved, expected[:top]), want)
    with pytest.raises(AssertionError):
        ev.compute_instantaneous_regrets(achieved, expected[:top - 1])


@pytest.mark.parametrize("cfr", ["standard", "discounted", "discounted_plus"])
@pytest.mark.parametrize("plus", [False, True])
def test_regret_update(ev, cfr, plus):
    from poker2_amd import fused_cfr_hip as F
    ev.cfr_type, ev.cfr_plus = F.CFRType[cfr], plus
    ev.dcfr_beta_initial = -1.0
    start = {k: getattr(ev, k).clone() for k in ("cumulative_regrets", "regret_weight_sums")}
    start["regret_weight_sums"].uniform_()
    runs = []
    for own in (False, True):
        for k, v in start.items():
            getattr(ev, k).copy_(v)
        ev.prepare_replay(3)
        if own:                                          # an override takes the two operations one after the other
            inner = ev.compute_instantaneous_regrets
            ev.compute_instantaneous_regrets = lambda values: inner(values)
        saved = ev.update_policy, ev.set_leaf_values, ev.compute_expected_values, ev.update_average_values
        ev.update_policy = ev.set_leaf_values = ev.compute_expected_values = ev.update_average_values = lambda *a: None
        ev.cfr_iteration(3)
        ev.update_policy, ev.set_leaf_values, ev.compute_expected_values, ev.update_average_values = saved
        runs.append({k: getattr(ev, k).clone() for k in start})
    for k in start:
        assert torch.equal(runs[0][k], runs[1][k]) and not torch.equal(runs[0][k], start[k]), k


def test_policies_reach_and_ranges(ev, monkeypatch):
    from poker2_amd import fused_cfr_hip as F
    n, bottom, top = ev.root_nodes, ev.depth_offsets[1], ev.depth_offsets[-2]

    def normalise(pos, fallback, out, eps):
        total = F.fused_parent_sum(pos, ev.child_offsets[:top].contiguous(), ev.child_count[:top].contiguous(),
                                   max_children=ev.num_actions)
        F.fused_divide_by_parent_sum_(pos=pos[bottom:], fallback=fallback[bottom:], parent_sum=total,
                                      parent_index=ev.parent_index[bottom:].contiguous(), out=out[bottom:], eps=eps)

    def push(reach, policy, beliefs):
        ev._calculate_reach_weights(reach, policy)
        ev._propagate_all_beliefs(beliefs, reach)
    names = ("policy_probs", "policy_probs_avg", "self_reach", "self_reach_avg", "beliefs", "beliefs_avg")
    start = {k: getattr(ev, k).clone() for k in names}
    normalise(ev.cumulative_regrets.clamp(min=0.0), ev.uniform_policy, ev.policy_probs, 1e-8)
    push(ev.self_reach, ev.policy_probs, ev.beliefs)
    F.fused_average_policy_mix_with_tensors_(
        policy_probs_avg=ev.policy_probs_avg, policy_probs=ev.policy_probs, self_reach=ev.self_reach,
        self_reach_avg=ev.self_reach_avg, to_act=ev.env.to_act, parent_index=ev.parent_index, old=ev._t_scalars.mix_old,
        new=ev._t_scalars.mix_new, total_weight=ev._t_scalars.mix_total, bottom=n)
    normalise(ev.policy_probs_avg, ev.policy_probs_avg, ev.policy_probs_avg, 1e-5)
    ev.policy_probs_avg[:n] = 0.0
    push(ev.self_reach_avg, ev.policy_probs_avg, ev.beliefs_avg)
    want = {k: getattr(ev, k).clone() for k in names}
    for k in names:
        getattr(ev, k).copy_(start[k])
    ev.update_policy(3)
    for k in names:
        assert torch.equal(getattr(ev, k), want[k]), k
    # a tree too large for the walk down from the roots: an operation per level
    for k in names:
        getattr(ev, k).copy_(start[k])
    monkeypatch.setattr(F, "TREE_ONE_LAUNCH_ROWS", ev.total_nodes - 1)
    monkeypatch.setattr(F, "tree_reach_beliefs_", None)
    ev.update_policy(3)
    for k in names:
        assert torch.equal(getattr(ev, k), want[k]), k
    monkeypatch.undo()
    # an override of one of the two steps is not passed by
    calls = []
    ev._calculate_reach_weights = lambda *a: calls.append("reach")
    ev.update_policy(3)
    assert calls == ["reach", "reach"]


def test_expected_values(ev):
    from poker2_amd import fused_cfr_hip as F
    bottom, top = ev.depth_offsets[1], ev.depth_offsets[-2]
    want = ev.latest_values.clone()
    rows = torch.arange(top, device="cuda")
    ranges = ev.beliefs[:top][rows, ev.env.to_act[:top]].contiguous()
    other = torch.zeros_like(ev.policy_probs)
    other[bottom:] = F.unblocked_mass_ratio_indirect_triton(
        numer_target=ranges.index_select(0, ev.parent_index[bottom:]) * ev.policy_probs[bottom:], denom_target=ranges,
        parent_index=ev.parent_index[bottom:].contiguous())
    for depth in range(ev.tree_depth - 1, -1, -1):
        base, end = ev.depth_offsets[depth], ev.depth_offsets[depth + 1]
        F.fused_weighted_parent_sum(values=want, prev_actor=ev.prev_actor, policy_hero=ev.policy_probs, policy_opp=other,
                                    child_offsets=ev.child_offsets[base:end].contiguous(),
                                    child_count=ev.child_count[base:end].contiguous(), parent_base=base,
                                    max_children=ev.num_actions)
    start = ev.latest_values.clone()
    ev.compute_expected_values(beliefs=ev.beliefs[:top], values=start, leaf_values=start)
    assert torch.equal(start, want)
    ev.compute_expected_values()
    assert torch.equal(ev.latest_values, want)
    # one value for a row, or for all
    leaf = ev.leaf_mask[:, None, None]
    for values in (ev.latest_values[:, :, :1], torch.tensor(0.5, device="cuda")):
        a, b = torch.empty_like(want), torch.where(leaf, values, torch.zeros_like(want))
        ev.compute_expected_values(leaf_values=values, values=a)
        ev.compute_expected_values(leaf_values=b, values=b)
        assert torch.equal(a, b)


def test_showdown_rows(ev):
    if ev.showdown_indices.numel() == 0:
        pytest.skip("no showdown leaf at this depth")
    want = ev.latest_values.clone()
    beliefs = ev.beliefs_avg if ev.cfr_avg else ev.beliefs
    want[ev.showdown_indices] = ev._showdown_value_both(beliefs[ev.showdown_indices])
    ev.set_leaf_values(3)
    keep = torch.ones(ev.total_nodes, dtype=torch.bool, device="cuda")
    keep[ev.model_indices] = False                       # (zeros here: there is no model)
    assert torch.equal(ev.latest_values[keep], want[keep])
    ev._showdown_value_both = lambda beliefs: torch.full_like(beliefs, 2.5)
    ev.set_leaf_values(3)
    assert bool((ev.latest_values[ev.showdown_indices] == 2.5).all())


def test_wrappers_refuse_what_would_index_out_of_bounds(ev):
    from poker2_amd import fused_cfr_hip as F
    total = ev.total_nodes
    with pytest.raises(AssertionError):
        F.family_regret_matching_(ev.policy_probs, ev.cumulative_regrets, ev.uniform_policy, ev.child_offsets,
                                  ev.child_count, total + 1, 5)
    with pytest.raises(AssertionError):
        F.level_expected_values_(ev.latest_values, ev.policy_probs, ev.beliefs, ev.env.to_act.int(), ev.child_offsets,
                                 ev.child_count, 0, 1, 5)
    with pytest.raises(AssertionError):
        F.tree_reach_beliefs_(ev.self_reach, ev.beliefs, ev.policy_probs, ev.allowed_hands, ev.allowed_hands_prob,
                              ev.parent_index, ev.prev_actor, ev._root_index, ev.root_nodes, 65)
    with pytest.raises(AssertionError):
        F.family_regrets(ev.latest_values[:-1], ev.latest_values, ev.beliefs, ev.env.to_act, ev.prev_actor,
                         ev.child_offsets, ev.child_count, 1, 1)


def test_a_family_larger_than_claimed_is_left_alone():
    from poker2_amd import fused_cfr_hip as F
    ev = make(*CASES[2])
    ev.prepare_replay(3)
    n, top, base = ev.root_nodes, ev.depth_offsets[-2], ev.depth_offsets[-3]
    large = ev.child_count[:top] > 5
    assert bool(large.any()) and bool((ev.child_count[:top] == 5).any())
    of_large = torch.zeros(ev.total_nodes, dtype=torch.bool, device="cuda")
    of_large[n:] = large[ev.parent_index[n:]]

    def run(names, call):
        start, ends = {k: getattr(ev, k).clone() for k in names}, []
        for claim in (5, 8):
            for k in names:
                getattr(ev, k).copy_(start[k])
            call(claim)
            ends.append({k: getattr(ev, k).clone() for k in names})
        return start, *ends
    tree = (ev.child_offsets, ev.child_count)
    s = ev._t_scalars
    for name, call in (
            ("policy_probs", lambda claim: F.family_regret_matching_(ev.policy_probs, ev.cumulative_regrets,
                                                                     ev.uniform_policy, *tree, top, claim)),
            ("policy_probs_avg", lambda claim: F.family_average_policy_(
                ev.policy_probs_avg, ev.policy_probs, ev.self_reach, ev.self_reach_avg, ev.env.to_act, *tree, s.mix_old,
                s.mix_new, s.mix_total, n, top, claim))):
        start, small, whole = run((name,), call)
        assert torch.equal(small[name][of_large], start[name][of_large])
        assert torch.equal(small[name][~of_large], whole[name][~of_large])
    start, small, whole = run(("latest_values",), lambda claim: F.level_expected_values_(
        ev.latest_values, ev.policy_probs, ev.beliefs, ev.env.to_act, *tree, base, top, claim))
    want = torch.where(large[base:, None, None], start["latest_values"][base:top], whole["latest_values"][base:top])
    assert torch.equal(small["latest_values"][base:top], want)

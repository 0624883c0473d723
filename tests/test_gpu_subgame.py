"""What a search writes before its first iteration and reads after its last (csrc/subgame.hip) against the same steps in
torch, bit for bit: constant rows, allowed hands, the uniform start (against the program that goes down level by level),
leaf rows, and the check for numbers that are not finite."""
import numpy as np
import pytest
import torch

from tests.helpers import random_boards, random_ranges

pytestmark = pytest.mark.gpu
H = 1326
STATE = ("policy_probs", "policy_probs_avg", "self_reach", "self_reach_avg", "beliefs", "beliefs_avg")


def make(n, bins, depth, streets, seed, model=None):
    from poker2_amd.config import Config, EnvConfig, SearchConfig
    from poker2_amd.evaluator import HipSparseCFREvaluator
    from poker2_amd.tree import RootStates
    rng = np.random.default_rng(seed)
    at = rng.choice(streets, n)
    boards = random_boards(rng, n, 5)
    for k, street in enumerate(at):
        boards[k, street + 2 if street else 0:] = -1
    roots = RootStates.at_round_start(at, rng.integers(1, 9, n) * 100, rng.integers(4, 41, (n, 2)) * 100, boards,
                                      button=rng.integers(0, 2, n))
    cfg = Config(num_envs=n, env=EnvConfig(bet_bins=bins, bb=100), search=SearchConfig(depth=depth, iterations=8))
    ev = HipSparseCFREvaluator(model, torch.device("cuda"), cfg)
    ranges = random_ranges(rng, boards).astype(np.float32)
    ranges[::3, 1] *= (rng.random(H) < 0.01)              # hardly any mass, not normalised
    ranges[1::4, 0] = 0                                   # none: the allowed hands take its place
    junk = torch.full((64 << 20,), float("nan"), device="cuda")
    del junk                                              # new tensors may get its memory
    ev.initialize_subgame(roots, np.arange(n), torch.from_numpy(ranges))
    return ev


CASES = [(1, [0.5, 1.0], 16, [3], 0), (9, [0.5, 1.0], 5, [0, 1, 2, 3], 1), (6, [0.3, 0.5, 0.8, 1.0, 1.5], 3, [2, 3], 2),
         (4, [1.0], 0, [3], 3)]


@pytest.fixture(params=CASES, ids=["one root", "all streets", "eight actions", "no level"])
def ev(request):
    return make(*request.param)


def test_constant_rows_and_allowed_hands(ev):
    from poker2_amd.card_utils import hand_combos_tensor
    n, t = ev.root_nodes, ev.tree
    share = np.zeros(ev.total_nodes, dtype=np.float32)
    share[n:] = np.float32(1.0) / t.child_count[t.parent_index[n:]].astype(np.float32)
    assert torch.equal(ev.uniform_policy, torch.from_numpy(share).cuda()[:, None].expand(-1, H))
    for reach in (ev.self_reach, ev.self_reach_avg):
        assert bool((reach[:n] == 1).all()) and not bool(reach[n:].any())
    won = np.where(t.fold_mask, t.reward, 0).astype(np.float32)
    want = torch.from_numpy(np.stack([won, -won], axis=1)).cuda()[:, :, None].expand(-1, -1, H)
    assert torch.equal(ev.latest_values, want) and torch.equal(ev.values_avg, want)
    cards = hand_combos_tensor().numpy()
    board = t.board[t.root_index]
    allowed = ~(cards[None, :, :, None] == board[:, None, None, :]).any(axis=(2, 3))
    assert np.array_equal(ev.allowed_hands.cpu().numpy(), allowed)
    prob = allowed.astype(np.float32) / np.maximum(allowed.sum(axis=1, keepdims=True), 1).astype(np.float32)
    assert np.array_equal(ev.allowed_hands_prob.cpu().numpy(), prob)


def test_uniform_start_is_the_level_by_level_program(ev):
    assert ev._starts_uniform()
    start = {k: getattr(ev, k).clone() for k in STATE}
    inner = ev._normalize_beliefs
    ev._normalize_beliefs = lambda *a: inner(*a)           # an override: every level calls it
    assert not ev._starts_uniform()
    ev.initialize_policy_and_beliefs()
    want = {k: getattr(ev, k).clone() for k in STATE}
    for k in STATE:
        getattr(ev, k).copy_(start[k])
    del ev._normalize_beliefs
    for k in ("policy_probs", "policy_probs_avg"):
        getattr(ev, k).fill_(float("nan"))                 # every row is written
    ev.initialize_policy_and_beliefs()
    for k in STATE:
        assert torch.equal(getattr(ev, k), want[k]), k


def test_a_model_with_a_policy_is_asked():
    from types import SimpleNamespace
    calls = []

    class Model:
        enforce_zero_sum = False

        def leaf_values(self, beliefs, rows, ev):
            return torch.zeros_like(beliefs)

        def policy_logits(self, beliefs, rows, ev):
            calls.append(rows.numel())
            return torch.zeros(rows.numel(), H, ev.num_actions, device="cuda")
    ev = make(3, [0.5, 1.0], 2, [3], 4, Model())
    ev.initialize_policy_and_beliefs()
    assert len(calls) == ev.tree_depth
    asked = {k: getattr(ev, k).clone() for k in STATE}
    other = make(3, [0.5, 1.0], 2, [3], 4)                 # zeros: the same policy
    other.initialize_policy_and_beliefs()
    for k in STATE:
        assert torch.equal(asked[k], getattr(other, k)), k

    def answer(features):
        return SimpleNamespace(hand_values=torch.zeros(len(features), 2, H, device="cuda"))

    class Net:                                             # a bare network: wrapped, and asked if it takes the keyword
        def __call__(self, features):
            calls.append("values")
            return answer(features)

    class PolicyNet:
        def __call__(self, features, include_policy=False):
            calls.append("policy")
            return answer(features)
    for net, asks in ((Net(), 0), (PolicyNet(), ev.tree_depth)):
        calls.clear()
        e = make(3, [0.5, 1.0], 2, [3], 4, net)
        e.initialize_policy_and_beliefs()
        assert len(calls) == asks


def test_leaf_rows_and_finite_check(ev):
    gen = torch.Generator(device="cuda").manual_seed(1)
    values = torch.randn(ev.total_nodes, 2, H, generator=gen, device="cuda") * 2
    values[0, 0, 5] = float("nan")
    keep = ev.leaf_mask[:, None, None]
    zero = torch.zeros_like(values)
    for clamp, src in ((False, values), (True, values.clamp(-1, 1))):
        got, want = ev._leaf_rows(values, clamp), torch.where(keep, src, zero)
        assert torch.equal(got.nan_to_num(9.0), want.nan_to_num(9.0))
    ev.latest_values.uniform_(-1, 1).mul_(3e38)
    ev._require_finite_values("here")
    for bad, at in ((float("nan"), 0), (float("inf"), -1), (-float("inf"), 777)):
        old = ev.latest_values.view(-1)[at].clone()
        ev.latest_values.view(-1)[at] = bad
        with pytest.raises(ValueError, match="after here"):
            ev._require_finite_values("here")
        ev.latest_values.view(-1)[at] = old


def test_exploitability_asks_overrides_as_the_reference_does():
    """An overridden ``_best_response_values`` gets four arguments and the clamped values of every row, an overridden
    ``compute_expected_values`` two tensors."""
    ev = make(5, [0.5, 1.0], 5, [3], 4)
    ev.initialize_policy_and_beliefs()
    ev.values_avg.normal_(generator=torch.Generator(device="cuda").manual_seed(1))
    want = ev._compute_exploitability()
    seen = []
    best, expected = ev._best_response_values, ev.compute_expected_values

    def best_response(policy, beliefs, base_values, deviating_player=None):
        seen.append(base_values.clone())
        return best(policy, beliefs, base_values, deviating_player)

    def expected_values(policy=None, beliefs=None, leaf_values=None, values=None):
        assert leaf_values is not values and not bool(values.any())
        expected(policy=policy, beliefs=beliefs, leaf_values=leaf_values, values=values)
    for name, method in (("_best_response_values", best_response), ("compute_expected_values", expected_values)):
        setattr(ev, name, method)
        got = ev._compute_exploitability()
        assert torch.equal(got.local_exploitability, want.local_exploitability)
        assert torch.equal(got.local_best_response_values, want.local_best_response_values)
    assert len(seen) == 4 and all(torch.equal(x, ev.values_avg.clamp(-1.0, 1.0)) for x in seen)

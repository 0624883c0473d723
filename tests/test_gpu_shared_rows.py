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


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("seed", range(8))
def test_rows_kept_elsewhere_are_never_read(seed, split):
    variant = VARIANTS[(seed + 5) % len(VARIANTS)]
    iters = 5 + seed % 2
    plain = build(seed, variant, split, lean=False, iters=iters)
    lean = build(seed, variant, split, lean=True, iters=iters)
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

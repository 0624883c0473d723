"""GPU: roots of unequal size are cut into work items while their largest tree would outlast the launch; the state is
that of whole roots, bit for bit."""
import numpy as np
import pytest
import torch

from tests.helpers import random_boards, random_ranges
from tests.test_gpu_lean_search import STATE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("large,cut", [(1, True), (499, False)])
def test_unequal_roots(large, cut):
    """500 river roots: all of them behind short stacks but one, or all behind deep stacks but one."""
    from poker2_amd.config import river_dcfr_config
    from poker2_amd.evaluator import HipSparseCFREvaluator
    from poker2_amd.tree import RootStates
    n = 500
    rng = np.random.default_rng(5)
    boards = random_boards(rng, n)
    beliefs = torch.from_numpy(random_ranges(rng, boards))
    stacks = np.full((n, 2), 60)
    stacks[rng.permutation(n)[:large]] = 800
    roots = RootStates.at_round_start(3, np.full(n, 200), stacks, boards, bb=100)
    runs = []
    for split in (None, False):
        cfg = river_dcfr_config(n, iterations=5, depth=16)
        cfg.env.bet_bins = [0.5, 1.0]
        ev = HipSparseCFREvaluator(None, torch.device("cuda"), cfg, max_raises=1, split_small_batches=split)
        ev.initialize_subgame(roots, np.arange(n), beliefs)
        ev.prepare_search(t_sample=torch.full((ev.total_nodes,), 2))
        ev.run_search_iterations()
        runs.append(ev)
    assert (runs[0]._items is not None) == cut and runs[1]._items is None
    for name in STATE:
        assert torch.equal(getattr(runs[0], name), getattr(runs[1], name)), name

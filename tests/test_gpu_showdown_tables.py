"""The per-board strength tables byte for byte: every section rebuilt with numpy from the oracle's order and ranks, on
boards that tie all hands, pair, flush, straighten, repeat a card or are not fully dealt."""
import numpy as np
import pytest
import torch

from oracle import cards as OC
from oracle import ranker as ORK

pytestmark = pytest.mark.gpu

BOARDS = [[0, 1, 2, 3, 4],            # straight flush on the board: most hands tie
          [8, 9, 10, 11, 12],         # royal flush: all hands tie
          [12, 25, 38, 51, 0],        # quads
          [0, 13, 1, 14, 27],         # full house
          [3, 17, 31, 45, 7], [51, 50, 38, 20, 2], [0, 2, 4, 6, 8],
          [7, 7, 20, 33, 50], [12, 12, 11, 10, 9], [12, 12, 12, 12, 25], [51, 51, 51, 51, 51],   # a card repeated: the suit
          [0, 0, 1, 1, 2],            # masks of the card ranker carry, up to two bits past the ace
          [5, 18, 30, -1, -1], [-1, -1, -1, -1, -1]]   # flop only, nothing dealt


def expected_table(board: np.ndarray, order: np.ndarray, rank: np.ndarray) -> np.ndarray:
    combos = OC.hand_combos()
    r = rank[order]
    first, behind = np.searchsorted(r, r, "left"), np.searchsorted(r, r, "right")
    on_board = np.isin(np.arange(52), board[board >= 0])
    c = combos[order]                                       # cards by sorted position
    blocked = on_board[c].any(axis=1)
    lists = np.stack([np.nonzero((c == card).any(axis=1))[0] for card in range(52)])        # [52, 51] ascending
    below = lambda card, bound: (lists[card] < bound[:, None]).sum(axis=1)
    cidx = np.stack([below(c[:, 0], first), below(c[:, 0], behind), below(c[:, 1], first), below(c[:, 1], behind)], 1)
    lists = np.where(on_board[:, None], 0xFFFF, lists)
    parts = [(order | np.where(blocked, 0x8000, 0)).astype("<u2"), np.stack([first, behind], 1).astype("<u2"),
             cidx.astype("u1"), lists.astype("<u2")]
    return np.concatenate([p.reshape(-1).view(np.uint8) for p in parts])


@pytest.mark.parametrize("triton_order", [True, False])
@pytest.mark.parametrize("extra", [0, 1, 40])
def test_tables_match_numpy(triton_order, extra):
    from poker2_amd import rules_hip as K
    drawn = np.argsort(np.random.default_rng(extra).random((extra, 52)), axis=1)[:, :5]
    boards = np.concatenate([np.array(BOARDS), drawn]).astype(np.int64)
    device = torch.from_numpy(boards).cuda()
    tables = K.build_showdown_tables(device, triton_order=triton_order).cpu().numpy()
    ranks, order = (x.cpu().numpy() for x in (K.rank_hands_triton(device) if triton_order else K.rank_hands(device)))
    want_ranks, want_order = (ORK.rank_hands_cards if triton_order else ORK.rank_hands)(boards)
    dealt = (boards >= 0).all(axis=1)                       # the oracle ranks dealt boards
    assert np.array_equal(ranks[dealt], want_ranks[dealt]) and np.array_equal(order[dealt], want_order[dealt])
    for k, board in enumerate(boards):
        assert np.array_equal(order[k], np.argsort(ranks[k], kind="stable"))
        want = expected_table(board, order[k], ranks[k])
        assert np.array_equal(tables[k, :want.size], want), board


@pytest.mark.parametrize("triton_order", [True, False])
@pytest.mark.parametrize("suited", [1, 2, 3, 4, 5])
def test_scores_by_ranks_and_one_by_one_agree_with_the_oracle(triton_order, suited):
    """Boards with every number of cards of one suit, paired or not: which hands take the score of their two ranks and
    which are scored one by one depends on these."""
    from poker2_amd import rules_hip as K
    rng = np.random.default_rng(suited)
    boards = []
    for k in range(12):
        suit, ranks = int(rng.integers(0, 4)), rng.permutation(13)
        cards = [13 * suit + r for r in ranks[:suited]]
        others = [13 * s + r for s in range(4) if s != suit for r in (ranks[:3] if k % 2 else range(13))]   # odd: pairs
        cards += [int(c) for c in rng.permutation(others)][:5 - suited]
        boards.append(rng.permutation(cards))
    boards = np.array(boards, dtype=np.int64)
    device = torch.from_numpy(boards).cuda()
    ranks, order = (x.cpu().numpy() for x in (K.rank_hands_triton(device) if triton_order else K.rank_hands(device)))
    want_ranks, want_order = (ORK.rank_hands_cards if triton_order else ORK.rank_hands)(boards)
    assert np.array_equal(ranks, want_ranks) and np.array_equal(order, want_order)
    alone = K.rank_hands_triton(device[5:6])[0] if triton_order else K.rank_hands(device[5:6])[0]
    assert np.array_equal(alone.cpu().numpy()[0], want_ranks[5])        # the dealing of work changes with the board's place

"""Workloads of the search framework, as data: what is prepared, what one pass runs, what it cannot do without.

``listed()`` are fixed cases, ``draw(rng)`` gives more of the same ranges.  Seven kinds of work, each through the
package's public entry points:

* ``search``    a slice of a search on a subgame that stands ready: its next iterations, as a search runs them, as a
                caller runs them one by one (``cfr_iteration``), replayed from a captured graph
                (``GraphedCFRIteration``) or with one launch per operation (``fused_iteration=False``);
* ``solve``     a whole river search from public states to exploitability;
* ``datagen``   one data-generation step: mixed-street roots, value network at the leaves, training batches;
* ``turn``      the next iterations of turn subgames whose leaves are chance nodes in front of a network;
* ``showdown``  the river showdown of many public states, from boards to values;
* ``unblocked`` the card-compatible mass of many ranges;
* ``ranker``    comparisons of 7-card hands.
"""
from __future__ import annotations

import functools

import numpy as np
import torch

from poker2_amd import fused_cfr_hip as F
from poker2_amd import rules_hip as R
from poker2_amd.card_utils import hand_combos_tensor
from poker2_amd.config import Config, EnvConfig, SearchConfig
from poker2_amd.evaluator import GraphedCFRIteration, HipSparseCFREvaluator
from poker2_amd.fused_cfr_hip import CFRType
from poker2_amd.leaf_models import ChanceLeafModel, NetworkLeafModel, RangeBoardMLP
from poker2_amd.tree import CARDS_ON_STREET, RootStates

H = 1326
ROW = 4 * H

_SEARCH = {"kind": "search", "mode": "search", "street": "river", "cfr": "discounted", "mixed": False, "warm_start": 0}


def listed() -> list[dict]:
    return [
        # one subgame solved while a player waits: nothing fills the chip, every launch and every chain of
        # dependent steps shows
        dict(_SEARCH, name="river_1_root", roots=1, depth=16, max_raises=3, iterations=32),
        # the batch of the reference's own settings (192 hands), its discounted_plus schedules, unequal stacks
        dict(_SEARCH, name="river_192_schedules", roots=192, depth=16, max_raises=3, iterations=16,
             cfr="rebel", mixed=True),
        # the same batch replayed from a captured graph, every tensor written in every iteration
        dict(_SEARCH, name="river_192_graph", roots=192, depth=16, max_raises=3, iterations=8, mode="graph"),
        # the benchmark workload of bench.py: 4096 subgames of the three-raise tree
        dict(_SEARCH, name="river_4096", roots=4096, depth=16, max_raises=3, iterations=4),
        # an odd number of depth-2 trees under the reference's default algorithm (linear CFR+ with CFR-AVG)
        dict(_SEARCH, name="river_1003_default_cfr", roots=1003, depth=2, max_raises=0, iterations=12, cfr="default"),
        # the reference benchmark's iteration: 192 roots of mixed streets to depth 5, one launch per operation
        dict(_SEARCH, name="mixed_192_per_operation", roots=192, depth=5, max_raises=0, iterations=4,
             mode="per_op", street="mixed", mixed=True),
        # a whole search: tree, state, warm start, 64 iterations, sampled leaves, exploitability
        {"kind": "solve", "name": "solve_192", "roots": 192, "depth": 16, "max_raises": 3, "iterations": 64,
         "cfr": "discounted", "mixed": False, "warm_start": 4, "street": "river"},
        # self-play data: flop / turn / river roots searched to the end of the street, bf16 network at the leaves
        {"kind": "datagen", "name": "datagen_1024_bf16", "roots": 1024, "depth": 64, "max_raises": 3, "iterations": 16,
         "cfr": "discounted", "mixed": True, "warm_start": 0, "street": "mixed", "net": "bfloat16", "zero_sum": False},
        # turn subgames, 48 river cards behind every street-end leaf, network in float32
        {"kind": "turn", "name": "turn_64_chance", "roots": 64, "depth": 16, "max_raises": 3, "iterations": 2,
         "net": "float32"},
        # the showdown benchmark: 4096 public states, boards ranked anew
        {"kind": "showdown", "name": "showdown_4096", "states": 4096, "boards": True},
        # the reference benchmark's unblocked mass on the GPU
        {"kind": "unblocked", "name": "unblocked_400000", "rows": 400_000},
        # the reference benchmark's smallest batch of hand comparisons
        {"kind": "ranker", "name": "compare_1024_planes", "hands": 1024, "form": "planes"},
    ]


def _log(rng, lo: float, hi: float) -> int:
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return max(int(lo), min(int(hi), int(round(float(lo) * (float(hi) / float(lo)) ** rng.random()))))


# nodes per root of the trees that are searched (bins half pot and pot, stacks of four pots)
_TREES = {(16, 3): 105, (16, 2): 57, (16, 1): 21, (2, 0): 21, (5, 0): 117}
# the most that one of them grows to behind unequal stacks
_TREES_MOST = {(16, 3): 129, (16, 2): 57, (16, 1): 21, (2, 0): 21, (5, 0): 267}


def draw(rng) -> dict:
    kind = rng.choice(["search", "search", "search", "search", "solve", "datagen", "turn", "showdown", "unblocked",
                       "ranker"])
    if kind == "search":
        depth, max_raises = rng.choice(sorted(_TREES))
        nodes = _TREES_MOST[depth, max_raises]
        mode = rng.choice(["search", "search", "search", "plain", "graph", "per_op"])
        cfr = rng.choice(["discounted", "discounted", "rebel", "default", "standard"])
        # a launch per operation is for the batches of the reference's settings
        most = min(4096, (40_000 if mode == "per_op" else 430_080) // nodes)
        roots = _log(rng, 1, most)
        iterations = max(1, min(32, _log(rng, 2, 48), 2_500_000 // (nodes * roots)))
        return dict(_SEARCH, roots=roots, depth=depth, max_raises=max_raises, iterations=iterations, mode=mode, cfr=cfr,
                    mixed=rng.random() < 0.5, street=rng.choice(["river", "river", "mixed"]))
    if kind == "solve":
        depth, max_raises = rng.choice(sorted(_TREES))
        return {"kind": kind, "roots": _log(rng, 1, 40_000 // _TREES_MOST[depth, max_raises]), "depth": depth,
                "max_raises": max_raises, "iterations": _log(rng, 16, 64), "cfr": rng.choice(["discounted", "rebel"]),
                "mixed": rng.random() < 0.5, "warm_start": rng.choice([0, 4]), "street": "river"}
    if kind == "datagen":
        return {"kind": kind, "roots": _log(rng, 32, 1024), "depth": rng.choice([5, 64]), "max_raises": rng.choice([2, 3]),
                "iterations": _log(rng, 4, 16), "cfr": "discounted", "mixed": True, "warm_start": 0, "street": "mixed",
                "net": rng.choice(["bfloat16", "float16", "float32"]), "zero_sum": rng.random() < 0.3}
    if kind == "turn":
        return {"kind": kind, "roots": _log(rng, 1, 64), "depth": 16, "max_raises": rng.choice([1, 2, 3]), "iterations": 2,
                "net": rng.choice(["float32", "bfloat16"])}
    if kind == "showdown":
        return {"kind": kind, "states": _log(rng, 16, 8192), "boards": rng.random() < 0.5}
    if kind == "unblocked":
        return {"kind": kind, "rows": _log(rng, 64, 400_000)}
    return {"kind": kind, "hands": _log(rng, 1024, 1 << 20),
            "form": rng.choice(["planes", "cards_int8", "cards_int16", "cards_int64"])}


# ----------------------------------------------------------------------------------------------- inputs
def _config(case: dict) -> Config:
    presets = {
        "discounted": dict(dcfr_alpha=1.5, dcfr_beta=0.0, dcfr_gamma=2.0, dcfr_plus_delay=0,
                           cfr_type=CFRType.discounted, cfr_plus=False, cfr_avg=False),
        # the shipped settings of the reference's trainer, delay scaled to the number of iterations
        "rebel": dict(dcfr_alpha=2.0, dcfr_beta=-1.0, dcfr_gamma=5.0, dcfr_alpha_final=4.0, dcfr_beta_final=-2.0,
                      dcfr_gamma_final=0.0, dcfr_plus_delay=case["iterations"] // 4,
                      cfr_type=CFRType.discounted_plus, cfr_plus=False, cfr_avg=False),
        "default": dict(cfr_type=CFRType.linear, cfr_plus=True, cfr_avg=True),
        "standard": dict(cfr_type=CFRType.standard, cfr_plus=False, cfr_avg=False),
    }
    warm = case.get("warm_start", 0)
    return Config(num_envs=case["roots"], env=EnvConfig(bet_bins=[0.5, 1.0], bb=100),
                  search=SearchConfig(depth=case["depth"], iterations=case["iterations"] + warm,
                                      warm_start_iterations=warm, **presets[case.get("cfr", "discounted")]))


def _roots(n: int, street: str, mixed: bool, deal: np.random.Generator) -> RootStates:
    """Public states at the start of a betting round: pot 200 and stacks 800, or, mixed, pots of 1 to 200 big blinds
    (a river search: 2 to 8) in front of equal or unequal stacks.  The chips are a matter of the case, so that every
    seed searches trees of the same shape; the cards are dealt from ``deal``."""
    rng = np.random.default_rng(n)
    at = {"river": np.full(n, 3), "turn": np.full(n, 2), "mixed": rng.integers(1, 4, n)}[street]
    runout = np.argsort(deal.random((n, 52)), axis=1)[:, :5].astype(np.int64)
    board = np.where(np.arange(5)[None, :] < CARDS_ON_STREET[at][:, None], runout, -1)
    if not mixed:
        pot, stacks = np.full(n, 200), np.full((n, 2), 800)
    elif street == "mixed":
        pot, stacks = rng.integers(1, 201, n) * 100, np.full((n, 2), 10000)
    else:
        pot, stacks = rng.integers(2, 9, n) * 100, rng.integers(4, 41, (n, 2)) * 100
    roots = RootStates.at_round_start(at, pot, stacks, board, button=rng.integers(0, 2, n))
    roots.runout = runout
    return roots


def _ranges(board: np.ndarray, gen: torch.Generator) -> torch.Tensor:
    """Normalised ranges of both players, [n, 2, 1326]: Gamma(1/2) weights, no hand that touches the board."""
    dev = torch.device("cuda")
    b = torch.from_numpy(np.where(board >= 0, board, 52)).to(dev)
    on = torch.zeros(b.shape[0], 53, dtype=torch.bool, device=dev).scatter_(1, b, True)
    cards = hand_combos_tensor(dev)
    allowed = ~(on[:, cards[:, 0]] | on[:, cards[:, 1]])
    x = torch.randn(b.shape[0], 2, H, generator=gen, device=dev).square_() * allowed[:, None, :]
    return x / x.sum(-1, keepdim=True)


@functools.lru_cache(maxsize=1)
def _network() -> RangeBoardMLP:
    """The value network of the turn configuration; a program has one for all of its searches."""
    return RangeBoardMLP().to("cuda")


def _autocast(case: dict):
    return None if case["net"] == "float32" else getattr(torch, case["net"])


def _hands(n: int, rng: np.random.Generator) -> np.ndarray:
    return np.argsort(rng.random((n, 52), dtype=np.float32), axis=1)[:, :7]


def prepare(case: dict, seed: int) -> dict:
    rng, dev = np.random.default_rng(seed), torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    torch.manual_seed(seed)          # the sampling schedule of a search draws from the default generator
    kind = case["kind"]
    if kind in ("search", "solve", "datagen", "turn"):
        n = case["roots"]
        roots = _roots(n, case.get("street", "turn"), case.get("mixed", False), rng)
        ranges = _ranges(roots.board, gen)
        model = None
        if kind == "datagen":
            model = NetworkLeafModel(_network(), dev, autocast_dtype=_autocast(case), enforce_zero_sum=case["zero_sum"])
        elif kind == "turn":
            model = ChanceLeafModel(_network(), dev, autocast_dtype=_autocast(case))
        ev = HipSparseCFREvaluator(model, dev, _config(case), generator=gen, max_raises=case["max_raises"] or None,
                                   fused_iteration=case.get("mode") != "per_op")
        state = {"case": case, "ev": ev, "roots": roots, "index": np.arange(n), "ranges": ranges}
        if kind == "datagen":
            ev.chance_helper.autocast_dtype = _autocast(case)
        if kind in ("search", "turn"):
            ev.initialize_subgame(roots, state["index"], ranges)
            ev.prepare_search()
            state["t"] = ev.warm_start_iterations
        if case.get("mode") == "graph":
            state["graph"] = GraphedCFRIteration(ev)
            state["graph"].capture(0)
        return state
    if kind == "showdown":
        m = case["states"]
        boards = np.argsort(rng.random((m, 52)), axis=1)[:, :5].astype(np.int64)
        state = {"case": case, "boards": torch.from_numpy(boards).to(dev), "ranges": _ranges(boards, gen),
                 "potential": torch.rand(m, 2, generator=gen, device=dev) * 1000, "scale": torch.full((m,), 1000.0, device=dev)}
        if not case["boards"]:
            state["tables"] = R.build_showdown_tables(state["boards"])
        return state
    if kind == "unblocked":
        x = torch.rand(case["rows"], H, generator=gen, device=dev)
        return {"case": case, "target": x / x.sum(-1, keepdim=True)}
    n = case["hands"]
    cards = np.stack([_hands(n, rng), _hands(n, rng)], axis=1)
    if case["form"] != "planes":
        return {"case": case, "cards": torch.from_numpy(cards).to(dev).to(getattr(torch, case["form"][6:]))}
    planes = torch.zeros(n, 2, 52, dtype=torch.bool, device=dev)
    planes.scatter_(2, torch.from_numpy(cards).to(dev), True)
    return {"case": case, "planes": planes.view(n, 2, 4, 13)}


# ----------------------------------------------------------------------------------------------- one pass
def _batch(batch) -> dict:
    f = batch.features
    out = {"context": f.context, "street": f.street, "to_act": f.to_act, "board": f.board, "beliefs": f.beliefs,
           "legal": batch.legal_masks, "value": batch.value_targets, "policy": batch.policy_targets}
    out.update({k: v for k, v in batch.statistics.items() if v is not None})
    return {k: v for k, v in out.items() if v is not None}


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind in ("search", "turn"):
        ev, mode, first = state["ev"], case.get("mode", "search"), state["t"]
        state["t"] = last = first + case["iterations"]
        for t in range(first, last):
            if mode == "graph":
                state["graph"].replay(t)
            elif mode == "search":
                # every iteration but the last as a search runs it; the last leaves the whole state behind
                ev.cfr_iteration(t, lean=t + 1 < last, alternate_reach_avg=True)
            else:
                ev.cfr_iteration(t)
        return ev.state_dict()
    if kind == "solve":
        ev = state["ev"]
        ev.initialize_subgame(state["roots"], state["index"], state["ranges"])
        leaves = ev.evaluate_cfr()
        stats = ev._compute_exploitability()
        return {**ev.state_dict(), "leaves": leaves.nodes, "exploitability": stats.local_exploitability,
                "best_response": stats.local_best_response_values}
    if kind == "datagen":
        ev = state["ev"]
        ev.initialize_subgame(state["roots"], state["index"], state["ranges"])
        leaves = ev.evaluate_cfr()
        value, pre_value, policy = ev.training_data()
        return {"leaves": leaves.nodes, "next_beliefs": leaves.beliefs, "value": _batch(value),
                "pre_value": _batch(pre_value), "policy": _batch(policy)}
    if kind == "showdown":
        tables = R.build_showdown_tables(state["boards"]) if case["boards"] else state["tables"]
        return R.showdown_value_both(state["ranges"], tables, state["potential"], state["scale"])
    if kind == "unblocked":
        return F.unblocked_mass_triton(state["target"])
    if case["form"] == "planes":
        return R.compare_7_single_batch_triton(state["planes"])
    return R.compare_7_cards_single_batch_triton(state["cards"])


# ----------------------------------------------------------------------------------------------- what a pass is
# multiply-adds of one sample through the value network
_NET_MACS = (2 * H + 52) * 1536 + 2 * 1536 * 1536 + 1536 * 2 * H


def work(case: dict) -> dict:
    """Bytes and operations one pass cannot do without.  An iteration carries five vectors of 1326 floats per node
    from one iteration to the next (regrets, their weights, the average policy, the average values of both players):
    each is read once and written once per iteration, everything else follows from them; a pass that returns the
    state writes its seventeen vectors once.  The network: its multiply-adds, its samples' values."""
    kind = case["kind"]
    if kind in ("search", "solve", "datagen", "turn"):
        per_root = _TREES.get((case["depth"], case["max_raises"]), 105)
        if case.get("street") == "mixed":
            per_root = {5: 40, 64: 38}.get(case["depth"], 0.4 * per_root)
        elif case.get("mixed"):
            per_root *= 0.8
        nodes = case["roots"] * per_root
        iterations = case["iterations"]
        out = {"bytes": nodes * ROW * (10.0 * iterations + 17), "flops": nodes * H * 60.0 * iterations}
        if kind == "datagen":
            # 10 leaves per root and iteration; a third of the roots stand on a flop (256 flops before it),
            # two thirds on a turn or river (about 48 cards)
            out["flops"] += 2.0 * _NET_MACS * case["roots"] * (10 * iterations + 256 / 3 + 32)
        elif kind == "turn":
            # a third of the nodes are leaves with 48 river cards behind them; the last layer is linear, so the
            # mean over the cards may be taken in front of it
            hidden = _NET_MACS - 1536 * 2 * H
            out["flops"] += 2.0 * hidden * nodes / 3 * 48 * iterations
        return out
    if kind == "showdown":
        m = case["states"]
        return {"bytes": m * (4.0 * ROW + 40), "flops": m * H * 40.0}
    if kind == "unblocked":
        return {"bytes": case["rows"] * 2.0 * ROW, "flops": case["rows"] * H * 5.0}
    size = {"planes": 52, "cards_int8": 7, "cards_int16": 14, "cards_int64": 56}[case["form"]]
    return {"bytes": case["hands"] * (2.0 * size + 4), "flops": case["hands"] * 400.0}


def tolerance(case: dict):
    """What two correct programs may differ by, measured: the same case with every range moved by one rounding
    (1e-7), and with the sums of the launch-per-operation path; about four times that is stated.

    A search amplifies roundings (regret matching divides differences of nearly equal values, and a showdown value
    over next to no compatible mass is a quotient of roundings): 64 iterations 5e-3, discounted_plus from its first
    iteration on 1e-1, single entries more than their own size.  A network in 16 bits adds its own rounding."""
    kind = case["kind"]
    if kind == "ranker":
        return "exact"
    if kind == "unblocked":
        return {"rel": 3e-7, "max": 1e-5}
    if kind == "showdown":
        return {"rel": 1e-6, "max": 1e-4}
    if kind == "turn":
        return {"rel": 1e-5, "max": 1e-3} if case["net"] == "float32" else {"rel": 2e-2, "max": 0.9}
    if kind == "search" and case["cfr"] != "rebel":
        return {"rel": 2e-2, "max": 0.9}
    if kind == "solve":
        return {"rel": 2e-2, "max": 0.9, "differ": 0.005}
    return {"rel": 0.03, "max": 0.9, "differ": 0.01}

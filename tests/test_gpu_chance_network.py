"""A ReLU network behind single-card chance nodes (``chance_node_helper.chance_network``): its answers against the
network in float64 on every sample, at the edges of what the kernels cut up - widths that are no whole tile, one state
and many, states of unequal sample counts, networks of 3 to 6 layers - and for ranges that lose most of their mass to a
card.  Which networks take this path is tested without a GPU at the end."""
import numpy as np
import pytest
import torch

from poker2_amd import chance_node_helper as K
from poker2_amd.card_utils import hand_combos_tensor
from poker2_amd.leaf_models import RangeBoardMLP

H = 1326


def make_net(hidden, layers, bias=True, seed=3, device="cuda"):
    net = RangeBoardMLP(hidden=hidden, layers=layers, seed=seed)
    gen = torch.Generator().manual_seed(seed)
    with torch.no_grad():
        for lin in net.linears:
            lin.bias.copy_(torch.randn(lin.bias.shape, generator=gen) * 0.02)
            if not bias:
                lin.bias = None
    return net.to(device)


def make_inputs(n, kind, seed, on_board=None):
    rng = np.random.default_rng(seed)
    boards = np.full((n, 5), -1, dtype=np.int64)
    for i in range(n):
        m = on_board if on_board is not None else int(rng.integers(0, 5))
        boards[i, :m] = rng.permutation(52)[:m]
    x = rng.gamma(0.5, size=(n, 2, H))
    if kind == "peaked":                       # a few hands hold nearly everything: their cards take the samples whole
        x = x ** 8
    elif kind == "one hand":
        x[:] = 0
        x[np.arange(n), 0, rng.integers(0, H, n)] = 1.0
        x[np.arange(n), 1, rng.integers(0, H, n)] = 0.25
    elif kind == "three hands":                # six cards of a player hold a third of his range each
        x[:] = 0
        for _ in range(3):
            x[np.arange(n), 0, rng.integers(0, H, n)] = 1.0
            x[np.arange(n), 1, rng.integers(0, H, n)] = 1.0
    elif kind == "one hand against none":
        x[:] = 0
        x[np.arange(n), np.arange(n) % 2, rng.integers(0, H, n)] = 1.0
    elif kind == "some empty":
        x[::2, 0] = 0
        x[1::3, 1] = 0
    x = x / np.maximum(x.sum(-1, keepdims=True), 1e-300)
    return torch.from_numpy(x.astype(np.float32)).cuda(), torch.from_numpy(boards).cuda()


def reference(net, pre, boards):
    """(mean over the samples in float64, bound on what float32 sums of split products may differ by)."""
    cards = hand_combos_tensor().cuda()
    layers = [(lin.weight.double(), lin.bias.double() if lin.bias is not None else 0.0) for lin in net.linears]
    out, tol = [], []
    for x0, board in zip(pre.double(), boards):
        dealt = [int(c) for c in board if c >= 0]
        rows = []
        for c in range(52):
            if c in dealt:
                continue
            allowed = torch.ones(H, dtype=torch.bool, device="cuda")
            for d in dealt + [c]:
                allowed &= (cards != d).all(dim=1)
            x = x0 * allowed
            total = x.sum(-1, keepdim=True)
            x = torch.where(total > 1e-12, x / total.clamp(min=1e-12), allowed.double() / allowed.sum())
            onehot = torch.zeros(52, dtype=torch.float64, device="cuda")
            onehot[dealt + [c]] = 1
            rows.append(torch.cat([x.reshape(-1), onehot]))
        h = torch.stack(rows)
        # per layer: three products of 22-bit numbers for one (what is dropped and rounded: 3 x 2^-22 of it), sums of 32
        # at a time (40 roundings) and one more rounding for every 32 columns; errors of the layer before pass through
        # |W|.  The first layer subtracts at most a quarter of what it subtracts from: twice that bound covers it.
        err = torch.zeros_like(h) + h.abs() * 2.0 ** -22
        for k, (w, b) in enumerate(layers):
            c = 3 * 2.0 ** -22 + (40 + w.shape[1] / 32) * 2.0 ** -24
            err = (err + (2 if k == 0 else 1) * c * h.abs()) @ w.abs().T
            h = h @ w.T + b
            err = err + h.abs() * 2.0 ** -23
            if k + 1 < len(layers):
                h = h.relu()
        out.append(h.mean(0).view(2, H))
        tol.append(err.mean(0).view(2, H))
    return torch.stack(out), torch.stack(tol)


@pytest.mark.gpu
@pytest.mark.parametrize("hidden,layers,n,kind,on_board,bias", [
    (256, 2, 1, "gamma", 4, True),             # one state, the smallest network and tile
    (288, 2, 5, "gamma", None, True),          # a width of no whole tile; 48 to 52 samples per state
    (256, 3, 40, "peaked", 3, False),
    (320, 5, 3, "one hand", None, True),       # maxima of rows carried through two buffers
    (256, 4, 7, "some empty", None, True),
    (1536, 3, 6, "gamma", 4, True),
    (512, 2, 180, "gamma", 4, True),           # states across tiles of 128 rows
    (288, 2, 40, "three hands", None, True),   # several tiles of samples taken whole, the last of both kinds no full one
    (256, 2, 9, "one hand against none", 4, True),
])
def test_matches_float64(hidden, layers, n, kind, on_board, bias):
    net = make_net(hidden, layers, bias)
    pre, boards = make_inputs(n, kind, seed=n + layers, on_board=on_board)
    stack = K.network_layers(net, pre.device)
    assert stack is not None
    with torch.no_grad():
        got = K.chance_network(pre, torch.arange(n).cuda(), boards, stack, on_board)
        want, tol = reference(net, pre, boards)
    assert bool(((got.double() - want).abs() <= tol).all())
    # and not only within the worst case: as close as a float32 product that adds its columns one after the other
    assert float((got.double() - want).norm() / want.norm()) < 2.0 ** -22 * len(stack)


def rescale_units(net, kind):
    """The same function with hidden units that answer in other sizes: what they are multiplied by is taken out of the
    columns that read them."""
    gen = torch.Generator().manual_seed(11)
    with torch.no_grad():
        for lin, reader in zip(net.linears[:-1], net.linears[1:]):
            power = torch.zeros(lin.weight.shape[0])
            if kind == "all":
                power = (torch.randn(power.shape, generator=gen) * 6).round()
            elif kind == "dead":                        # a unit that is always 0, with outgoing weights out of proportion
                lin.weight[3], lin.bias[3] = 0.0, 0.0
                reader.weight[:, 3] *= 2.0 ** 30
            else:
                power[5] = kind
            up = torch.exp2(power).to(lin.weight)
            lin.weight.mul_(up[:, None])
            lin.bias.mul_(up)
            reader.weight.div_(up)


@pytest.mark.gpu
@pytest.mark.parametrize("ranges", ["gamma", "one hand"])
@pytest.mark.parametrize("kind", [8, 12, 16, 20, 24, 40, -30, "all", "dead"])
def test_units_of_unequal_size(kind, ranges):
    """As close as with units of one size (``test_matches_float64``), which is as close as float32 products are."""
    net = make_net(320, 4)
    rescale_units(net, kind)
    pre, boards = make_inputs(3, ranges, seed=21, on_board=4)
    with torch.no_grad():
        got = K.chance_network(pre, torch.arange(3).cuda(), boards, K.network_layers(net, pre.device), 4)
        want, tol = reference(net, pre, boards)
    assert bool(((got.double() - want).abs() <= tol).all())
    assert float((got.double() - want).norm() / want.norm()) < 2.0 ** -22 * len(net.linears)


@pytest.mark.gpu
@pytest.mark.parametrize("bias", [-1e4, -3e38, -float("inf")])
def test_units_switched_off_by_their_bias(bias):
    """As if nothing read them."""
    net, without = make_net(320, 4), make_net(320, 4)
    with torch.no_grad():
        for k in range(4):
            net.linears[k].bias[k::50] = bias
            without.linears[k + 1].weight[:, k::50] = 0
        pre, boards = make_inputs(3, "three hands", seed=22, on_board=4)
        got = K.chance_network(pre, torch.arange(3).cuda(), boards, K.network_layers(net, pre.device), 4)
        want, tol = reference(without, pre, boards)
    assert bool(((got.double() - want).abs() <= tol).all())
    assert float((got.double() - want).norm() / want.norm()) < 2.0 ** -22 * len(net.linears)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["gamma", "three hands"])
def test_256_row_tiles_and_a_selection_of_rows(kind):
    """Enough samples for the largest tiles (4 per CU), taken from a table through ``root_indices``, and enough of them
    taken whole for several tiles per workgroup; a few states against float64, all against the network sample by sample
    in float32."""
    n = 1400
    net = make_net(1024, 2)
    pre, boards = make_inputs(n + 3, kind, seed=1, on_board=4)
    roots = torch.randperm(n + 3, generator=torch.Generator().manual_seed(2))[:n].cuda()
    with torch.no_grad():
        got = K.chance_network(pre, roots, boards, K.network_layers(net, pre.device), 4, check_rows=False)
        some = torch.tensor([0, 5, 6, 700, n - 1]).cuda()
        want, tol = reference(net, pre[roots[some]], boards[roots[some]])
        assert bool(((got[some].double() - want).abs() <= tol).all())
        rows, _, _, offsets = K.chance_expand(pre, roots, boards, 4, input_dtype=torch.float32)
        whole = K.chance_mean(net.forward_input(rows).hand_values, offsets)
    assert float((got - whole).norm() / whole.norm()) < 2e-6


@pytest.mark.gpu
@pytest.mark.parametrize("row_tiles", [1, 4, 5, 9, 10, 11, 21, 22])
def test_tiles_of_whole_samples_in_parts(row_tiles):
    """Tiles are 64 samples by 128 of 1024 columns; their steps are cut into 14, 14, 7, 7, 6, 3, 3 and 1 parts, as many as
    512 workgroups take."""
    net = make_net(1024, 2)
    pre, boards = make_inputs(240, "three hands", seed=31, on_board=4)
    cards = hand_combos_tensor().cuda()
    on = torch.zeros(240, 52, device="cuda").scatter_(1, boards[:, :4], 1.0)
    left = pre * (1 - on[:, cards].amax(2))[:, None]
    held = torch.stack([(left * (cards == c).any(1)).sum(2) for c in range(52)], dim=2)
    whole = ((held > 0.25 * left.sum(2, keepdim=True)).any(1) & (on == 0)).sum(1).cumsum(0)
    n = int((whole <= 64 * (row_tiles - 1)).sum()) + 1   # the first state that needs the last tile
    assert -(-int(whole[n - 1]) // 64) == row_tiles
    roots = torch.arange(n).cuda()
    with torch.no_grad():
        got = K.chance_network(pre, roots, boards, K.network_layers(net, pre.device), 4)
        rows, _, _, offsets = K.chance_expand(pre, roots, boards, 4, input_dtype=torch.float32)
        want = K.chance_mean(net.forward_input(rows).hand_values, offsets)
    assert float((got - want).norm() / want.norm()) < 2e-6


@pytest.mark.gpu
def test_a_wrong_card_count_claim_and_a_row_outside_the_table():
    """The rest of a state's share is samples with an input of zeros, as the expansion writes them."""
    net = make_net(256, 2)
    pre, boards = make_inputs(5, "gamma", seed=8, on_board=3)
    boards[1, 3] = 40 if 40 not in boards[1].tolist() else 41
    boards[2] = torch.arange(5).cuda()
    roots = torch.tensor([0, 1, 2, 7, 4]).cuda()
    with torch.no_grad():
        got = K.chance_network(pre, roots, boards, K.network_layers(net, pre.device), 3, check_rows=False)
        rows, _, _, offsets = K.chance_expand(pre, roots, boards, 3, check_rows=False, input_dtype=torch.float32)
        want = K.chance_mean(net.forward_input(rows).hand_values, offsets)
    assert float((got - want).abs().max() / want.abs().max()) < 1e-5
    with pytest.raises(IndexError):
        K.chance_network(pre, roots, boards, K.network_layers(net, pre.device), 3)


@pytest.mark.gpu
def test_weights_are_read_anew_and_every_replay_of_a_graph_agrees():
    net = make_net(256, 3)
    pre, boards = make_inputs(9, "gamma", seed=4, on_board=4)
    roots = torch.arange(9).cuda()
    helper = K.ChanceNodeHelper(torch.device("cuda"), torch.float32, 2, net, autocast_dtype=None)
    feats = K.MLPFeatures(context=torch.zeros(9, 1).cuda(), street=torch.full((9,), 2).cuda(),
                          to_act=torch.zeros(9, dtype=torch.long).cuda(), board=boards, beliefs=pre.view(9, -1))

    def run():
        return helper.single_card_chance_values(roots, feats, pre, boards, cards_on_board=4, check_rows=False)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run()
    for step in range(3):
        with torch.no_grad():
            net.linears[1].weight.mul_(-1.5)
            pre.copy_(pre.roll(1, dims=0))
        graph.replay()
        eager = run()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        with torch.no_grad():
            want, tol = reference(net, pre, boards)
        assert bool(((out.double() - want).abs() <= tol).all())


def test_which_networks_take_this_path():
    cpu = torch.device("cpu")
    net = make_net(256, 2, device="cpu")
    stack = K.network_layers(net, cpu)
    assert stack is not None and [lin.weight.shape[0] for lin in stack] == [256, 256, 2 * H]
    assert K.network_layers(net, torch.device("cuda", 0)) is None
    for bad in (make_net(64, 2, device="cpu"), make_net(272, 2, device="cpu"), make_net(256, 1, device="cpu"),
                make_net(256, 2, device="cpu").double(), make_net(256, 2, device="cpu").bfloat16(), torch.nn.Identity()):
        assert K.network_layers(bad, cpu) is None

    class Other(RangeBoardMLP):
        def forward_input(self, x):
            return super().forward_input(x * 2)
    assert K.network_layers(Other(hidden=256, layers=2), cpu) is None
    patched = make_net(256, 2, device="cpu")
    patched.forward_input = lambda x: None
    assert K.network_layers(patched, cpu) is None
    hooked = make_net(256, 2, device="cpu")
    handle = hooked.linears[1].register_forward_hook(lambda *a: None)
    assert K.network_layers(hooked, cpu) is None
    handle.remove()
    assert K.network_layers(hooked, cpu) is not None
    handle = torch.nn.modules.module.register_module_forward_hook(lambda *a: None)
    assert K.network_layers(hooked, cpu) is None
    handle.remove()
    normed = make_net(256, 2, device="cpu")
    torch.nn.utils.parametrizations.weight_norm(normed.linears[0])
    assert K.network_layers(normed, cpu) is None
    strided = make_net(256, 2, device="cpu")
    strided.linears[1].weight = torch.nn.Parameter(strided.linears[1].weight.t())
    assert K.network_layers(strided, cpu) is None
    torch.set_autocast_enabled("cuda", True)
    try:
        assert K.network_layers(net, cpu) is None
    finally:
        torch.set_autocast_enabled("cuda", False)


@pytest.mark.parametrize("hidden,layers,states,cards_on_board,one_call", [
    (256, 2, 1, 4, True), (288, 2, 1, 4, False), (512, 3, 1, None, True), (544, 3, 1, 4, False), (1536, 3, 19, 4, False),
    (1536, 3, 20, 4, True), (1536, 3, 1, None, False), (256, 2, 174762, 4, True),
    (256, 2, 174763, 4, False),                # more samples than the library's limit, 8388607
    (1536, 3, 170000, None, False),            # the same if every board is empty
])
def test_which_calls_take_this_path(monkeypatch, hidden, layers, states, cards_on_board, one_call):
    taken = []

    def note(name):
        def stop(*args, **kw):
            taken.append(name)
            raise StopIteration
        return stop
    monkeypatch.setattr(K, "chance_network", note("one call"))
    monkeypatch.setattr(K, "chance_expand", note("layer by layer"))
    cpu = torch.device("cpu")
    helper = K.ChanceNodeHelper(cpu, torch.float32, 2, make_net(hidden, layers, device="cpu"), autocast_dtype=None)
    with pytest.raises(StopIteration):
        helper.single_card_chance_values(torch.zeros(states, dtype=torch.int64), None, torch.zeros(1, 2, H),
                                         torch.full((1, 5), -1), cards_on_board=cards_on_board)
    assert taken == ["one call" if one_call else "layer by layer"]


def test_library_refuses_what_it_does_not_take():
    import ctypes
    from poker2_amd import _lib
    lib = _lib.load()

    def size(n, samples, *widths):
        return lib.p2hip_chance_network_workspace(n, samples, (ctypes.c_int32 * len(widths))(*widths), len(widths))
    assert size(1, 48, 256, 256, 2 * H) > 0
    assert size(1, 48, 256, 2 * H) == -1 and size(1, 48, 256, 250, 2 * H) == -1 and size(1, 48, 256, 256, 100) == -1
    assert size(-1, 48, 256, 256, 2 * H) == -1 and size(1, 1 << 23, 256, 256, 2 * H) == -1
    assert size(1, 48, *([256] * 16), 2 * H) == -1
    widths = (ctypes.c_int32 * 3)(256, 256, 2 * H)
    assert lib.p2hip_chance_network(None, None, None, 1, None, 1, 48, None, None, widths, 3, None, 0, None, None) == 1
    assert lib.p2hip_chance_network(None, None, None, 0, None, 1, 0, None, None, widths, 3, None, 0, None, None) == 0

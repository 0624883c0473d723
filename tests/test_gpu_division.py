"""The iteration kernels' quotient (p2_div in csrc/common.h) against IEEE division: regret matching's policy is the
quotient of the regrets that the same iteration leaves, bit for bit, from sums at the threshold to sums whose
reciprocal is subnormal.  A dividend below 2^-102 has a remainder that can be subnormal and is rounded to a multiple of
2^-149: its quotient may be off by half of that over the divisor and by the rounding of the product.  The quotients of
the discounts and of the average policy's mix, which share their reciprocals, against the launch-per-operation path,
which divides as IEEE does.  (What of this needs no GPU: tests/test_oracle_quotient.py.)"""
import pytest
import torch

from tests.test_gpu_families import CASES, make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", CASES, ids=["one root", "five", "eight"])
@pytest.mark.parametrize("cfr", ["standard", "discounted", "discounted_plus", "linear"])
@pytest.mark.parametrize("t", [1, 7, 300])
def test_discounts_and_mixes_are_those_of_ieee_division(shape, cfr, t):
    from poker2_amd.evaluator import STATE_NAMES
    from poker2_amd.fused_cfr_hip import CFRType
    print(shape, cfr, t, flush=True)
    ev = make(*shape)
    ev.cfr_type = CFRType[cfr]
    ev.dcfr_beta_initial = -1.0
    gen = torch.Generator(device="cuda").manual_seed(5)
    ev.regret_weight_sums.uniform_(generator=gen)
    start = {k: getattr(ev, k).clone() for k in STATE_NAMES}
    ends = []
    for fused in (False, True):
        for k, v in start.items():
            getattr(ev, k).copy_(v)
        ev.fused_iteration = fused
        ev.prepare_replay(t)
        ev.cfr_iteration(t)
        ends.append({k: getattr(ev, k).clone() for k in STATE_NAMES})
    n = ev.root_nodes                                    # (make() leaves root rows that no search would)
    for k in ("cumulative_regrets", "regret_weight_sums", "policy_probs", "policy_probs_avg", "self_reach", "self_reach_avg"):
        assert torch.equal(ends[0][k][n:], ends[1][k][n:]) and not torch.equal(ends[1][k], start[k]), k


@pytest.mark.parametrize("scale", [2e-8, 1.0, 1e30, 1.2e38])
@pytest.mark.parametrize("shape", [(1, [0.5, 1.0], 16, [3], 0), (7, [0.5, 1.0], 5, [1, 2, 3], 1),
                                   (5, [0.3, 0.5, 0.8, 1.0, 1.5], 3, [2, 3], 2)], ids=["one root", "five", "eight"])
@pytest.mark.parametrize("lean", [False, True])
def test_policy_is_the_quotient_of_the_regrets(shape, scale, lean):
    print(shape, scale, lean, flush=True)
    ev = make(*shape)
    ev.fused_iteration = True
    gen = torch.Generator(device="cuda").manual_seed(7)
    # magnitudes over forty binary orders, so that quotients of every size occur
    ev.cumulative_regrets.uniform_(-1, 1, generator=gen)
    ev.cumulative_regrets.mul_(torch.exp2(-40 * torch.rand(ev.cumulative_regrets.shape, generator=gen, device="cuda")))
    ev.cumulative_regrets.mul_(scale)
    ev.latest_values.mul_(min(scale, 1.0))
    ev.cfr_iteration(2, lean=lean)
    torch.cuda.synchronize()
    bottom, top = ev.depth_offsets[1], ev.depth_offsets[-2]
    pos = ev.cumulative_regrets.clamp(min=0)
    first, count = ev.child_offsets[:top], ev.child_count[:top]
    total = torch.zeros_like(pos[:top])
    for k in range(int(count.max())):
        has = count > k
        total[has] += pos[(first + k)[has]]
    total = total[ev.parent_index[bottom:]]
    uniform = 1.0 / count[ev.parent_index[bottom:]].float()[:, None]
    want = torch.where(total > 1e-8, pos[bottom:] / total.clamp(min=1e-8), uniform)
    got = ev.policy_probs[bottom:]
    if scale > 1e38:
        assert bool((total > 2.0 ** 126).any())
    same = got == want
    bound = 2.0 ** -150 / total.double() + 2.0 ** -23 * want.double() + 2.0 ** -149
    assert bool((same | ((got.double() - want.double()).abs() <= bound) & (pos[bottom:] < 2.0 ** -102)).all())
    assert float(same.float().mean()) > 0.999

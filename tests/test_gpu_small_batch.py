"""The forward of small batches (T <= 64: k_small_front, k_small_route, k_skinny_fwd)
at its edges, and the top-k on special values at every routing width."""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as mo
from oxidizr_amd.moe import MoeConfig, Plan
from tests.gpu_helpers import Case, gpu_run, oracle_run
from tests.test_gpu_parity import _check, _routing_equal

pytestmark = pytest.mark.gpu

SMALL_CASES = [
    # one chunk of token rows (T <= 16) and four (17 .. 64); ragged rows (N % 16 = 8),
    # ragged k-chunks (K % 256 != 0), fewer chunks than waves
    dict(T=1, H=8, E=1, k=1, I=8, S=8),
    dict(T=1, H=2056, E=64, k=6, I=1400, S=2824),
    dict(T=16, H=264, E=16, k=2, I=520, S=0),
    dict(T=17, H=520, E=4, k=3, I=264, S=88),
    dict(T=64, H=256, E=3, k=2, I=40, S=4104),    # more rows than 32 in most experts
    dict(T=5, H=4360, E=20, k=4, I=24, S=16),     # router partials of two chunks (H > 4096)
    dict(T=64, H=64, E=1024, k=16, I=16, S=16),   # as many experts as threads; probabilities
    dict(T=63, H=72, E=200, k=3, I=16, S=0),      #   re-read from memory (T E > 8192)
]


@pytest.mark.parametrize("spec", SMALL_CASES)
def test_small_batch_edges(spec):
    # 1e-2: the bf16 bar; the oracle is fp64 on the same bf16 inputs.  One token: the
    # forward alone.  Its d logits are p (dp - sum p dp) with nothing to average over,
    # and with a peaked softmax the two terms cancel: at H = 2056, |p dp| is four times
    # |d logits|, so bf16's 3e-3 in dp is 1.2e-2 of d_router, whatever the kernels.
    case = Case(**spec, dtype="bf16", w_std=0.05)
    back = case.T > 1
    g = gpu_run(case, d_aux=0.01, d_z=0.001, backward=back)
    o = oracle_run(case, g["logits"], d_aux=0.01, d_z=0.001, backward=back)
    _routing_equal(g, o)
    _check(case, g, o, 1e-2, backward=back)


@pytest.mark.parametrize("T", [48, 100])
@pytest.mark.parametrize("E,k", [(7, 7), (64, 9), (100, 16), (256, 8), (500, 4), (1000, 16)])
def test_topk_of_special_values(T, E, k):
    # -0 equals +0, NaN selects as -inf, ties go to the lower index
    rng = np.random.default_rng(E)
    values = np.array([0.0, -0.0, 1e-45, -1e-45, np.nan, -np.inf, 3e38, -3e38, 1.0, -1.0],
                      np.float32)
    logits = values[rng.integers(0, len(values), size=(T, E))]
    logits[0] = np.nan
    logits[1] = -0.0
    order = np.where(np.isnan(logits), -np.inf, logits + 0.0)
    want = np.argsort(-order, axis=1, kind="stable")[:, :k].astype(np.int32)
    cfg = MoeConfig(hidden_size=8, num_experts=E, experts_per_tok=k, intermediate_size=8,
                    shared_expert_enabled=False)
    dev = torch.device("cuda:0")
    plan = Plan(cfg, torch.bfloat16, dev)
    saved = plan.route_from_logits(torch.tensor(logits, device=dev))
    torch.cuda.synchronize()
    f = lambda n: plan.saved_field(saved, T, n).cpu().numpy()
    np.testing.assert_array_equal(f("topk_idx"), want)
    counts, offsets, perm, inv = mo.dispatch(want, E)
    np.testing.assert_array_equal(f("counts"), counts)
    np.testing.assert_array_equal(f("perm"), perm)
    np.testing.assert_array_equal(f("inv_perm"), inv)


@pytest.mark.parametrize("T,E,k", [(65, 1, 1), (64, 70, 3), (1000, 3, 2), (2500, 1000, 4),
                                   (18000, 1000, 2), (5000, 300, 16)])
def test_dispatch_and_mean_probabilities_of_given_logits(T, E, k):
    # k_scan's three chunk sizes (at most 8 and 64 histogram blocks to a thread, more) with
    # the column sums that ride it; P within 32-bit sums of T terms in rows of 64
    rng = np.random.default_rng(T + E)
    logits = rng.normal(size=(T, E)).astype(np.float32)
    cfg = MoeConfig(hidden_size=8, num_experts=E, experts_per_tok=k, intermediate_size=8,
                    shared_expert_enabled=False)
    dev = torch.device("cuda:0")
    plan = Plan(cfg, torch.float32, dev)
    saved = plan.route_from_logits(torch.tensor(logits, device=dev))
    torch.cuda.synchronize()
    f = lambda n: plan.saved_field(saved, T, n).cpu().numpy()
    want = np.argsort(-logits, axis=1, kind="stable")[:, :k].astype(np.int32)
    np.testing.assert_array_equal(f("topk_idx"), want)
    counts, offsets, perm, inv = mo.dispatch(want, E)
    np.testing.assert_array_equal(f("counts"), counts)
    np.testing.assert_array_equal(f("offsets"), offsets)
    np.testing.assert_array_equal(f("perm"), perm)
    np.testing.assert_array_equal(f("inv_perm"), inv)
    p = np.exp(logits.astype(np.float64))
    p /= p.sum(1, keepdims=True)
    np.testing.assert_allclose(f("mean_prob"), p.mean(0), rtol=2e-5)


def test_small_batches_of_one_plan_share_no_scratch():
    # the list of touched experts lies in the call's own workspace: calls of two batches
    # whose workspaces differ (one per stream) leave each other's lists alone
    torch.manual_seed(5)
    dev = torch.device("cuda:0")
    H, I, E, k = 256, 136, 32, 2
    cfg = MoeConfig(hidden_size=H, num_experts=E, experts_per_tok=k, intermediate_size=I,
                    shared_expert_enabled=False)
    t = lambda *shape: (torch.randn(*shape, device=dev) * 0.05).to(torch.bfloat16)
    plan = Plan(cfg, torch.bfloat16, dev)
    router, tabs = t(E, H), [list(t(E, I, H)), list(t(E, I, H)), list(t(E, H, I))]
    w, keep = plan.weights_struct(router, *tabs)
    xs = [torch.randn(T, H, device=dev).to(torch.bfloat16) for T in (3, 61)]
    want = [plan.forward(x, w, need_grad=False)[0].clone() for x in xs]
    streams = [torch.cuda.Stream(dev) for _ in xs]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(20):
        for i, (x, s) in enumerate(zip(xs, streams)):
            with torch.cuda.stream(s):
                got[i].append(plan.forward(x, w, need_grad=False)[0])
    torch.cuda.synchronize()
    for i in range(2):
        assert all(torch.equal(g, want[i]) for g in got[i])

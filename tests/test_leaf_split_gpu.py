"""Leaf lists and active flags shared between the two-position kernel and its one-position form: live counts
at the edges of a round, against the whole batch evaluated at once, bit for bit."""
import pytest
import torch

from brokefish_amd import encoder_impl, positions
from brokefish_amd.hip_impl import compact_leaves
from brokefish_amd.net import BrokefishNet

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def made():
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2).eval().randomise_layers_(seed=6)
    batch = [t.cuda() for t in positions.random_positions(1300, plies=80, seed=6)]
    model = encoder_impl("hip")(net, int8=True)
    want = [t.clone() for t in model.forward_full(*batch[:3])]
    return model, batch, want


@pytest.mark.parametrize("live", [0, 1, 2, 255, 256, 257, 511, 512, 513, 768, 769, 1024, 1025, 1300])
def test_live_counts_at_the_edges_of_a_round(made, live):
    model, (b, c, r, _), want = made
    n = b.shape[0]
    flags = torch.zeros(n, dtype=torch.uint8, device="cuda")
    flags[torch.randperm(n, generator=torch.Generator().manual_seed(live))[:live].cuda()] = 3
    on = flags != 0
    for how in ("list", "flags"):
        model.forward_full(b, c, r)                            # the buffers exist
        for t in (model.policy_out, model.promo_out, model.value_out):
            t.fill_(7.0)
        got = model.forward_full(b, c, r, leaves=compact_leaves(flags)) if how == "list" else model.forward_full(b, c, r, active=flags)
        for g, w in zip(got, want):
            assert torch.equal(g[on], w[on]), how
            assert bool((g[~on] == 7.0).all()), how            # rows of the others are left as they were


@pytest.mark.parametrize("n,kernel", [(1300, "auto"), (1201, "auto"), (601, "duo"), (257, "auto"), (90, "auto"), (33, "auto"), (90, "twin"), (90, "board"), (90, "quad")])
def test_of_a_count_above_n_the_first_n_entries_are_taken(n, kernel):
    # a list longer than the launch, and a count that says so: what lies behind the n-th entry is no business of this launch
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=1).eval().randomise_layers_(seed=7)
    model = encoder_impl("hip")(net, int8=True, kernel=kernel)
    b, c, r, _ = [t.cuda() for t in positions.random_positions(n, plies=80, seed=7)]
    want = [t.clone() for t in model.forward_full(b, c, r)]
    order = torch.randperm(n, generator=torch.Generator().manual_seed(n)).int()
    index = torch.cat([order, torch.zeros(700, dtype=torch.int32)]).cuda()
    for count in (n, n + 1, n + 300, n + 600):
        for t in (model.policy_out, model.promo_out, model.value_out):
            t.fill_(7.0)
        got = model.forward_full(b, c, r, leaves=(index, torch.tensor([count], dtype=torch.int32, device="cuda")))
        for g, w in zip(got, want):
            assert torch.equal(g, w), count

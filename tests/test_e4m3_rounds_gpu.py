"""e4m3 launches of more than 256 positions: the two-position kernel and, for a last round of at most 256, its one-position
form, by size and by leaf list and flags.  The reference is the kernel with one position per
workgroup of four wavefronts, which none of these launches run."""
import pytest
import torch

from brokefish_amd import encoder_impl, positions
from brokefish_amd.hip_impl import compact_leaves
from brokefish_amd.net import BrokefishNet

pytestmark = pytest.mark.gpu
N = 1300


@pytest.fixture(scope="module")
def made():
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2).eval().randomise_layers_(seed=3)
    auto, board = (encoder_impl("hip")(net, fp8=True, out_dtype=torch.float32, kernel=k) for k in ("auto", "board"))
    batch = [t.cuda() for t in positions.random_positions(N, plies=100, seed=3)]
    return auto, board, batch, [t.clone() for t in board.forward_masked(*batch)]


@pytest.mark.parametrize("n", [257, 258, 511, 512, 513, 576, 577, 768, 769, 1024, 1025, N])
def test_every_size_of_a_last_round(made, n):
    auto, _, batch, want = made
    assert auto.launch_form(n) == "duo"
    for g, w in zip(auto.forward_masked(*[t[:n] for t in batch]), want):
        assert torch.equal(g, w[:n])


@pytest.mark.parametrize("live", [0, 1, 2, 255, 256, 257, 511, 512, 513, 768, 769, N])
def test_live_counts_at_the_edges_of_a_round(made, live):
    auto, _, (b, c, r, m), want = made
    flags = torch.zeros(N, dtype=torch.uint8, device="cuda")
    flags[torch.randperm(N, generator=torch.Generator().manual_seed(live))[:live].cuda()] = 1
    on = flags != 0
    for how in ("list", "flags"):
        auto.forward_full(b, c, r, m)
        for t in (auto.policy_out, auto.promo_out, auto.value_out):
            t.fill_(7.0)
        got = auto.forward_full(b, c, r, m, leaves=compact_leaves(flags)) if how == "list" else auto.forward_full(b, c, r, m, active=flags)
        for g, w in zip(got, want):
            assert torch.equal(g[on], w[on]) and bool((g[~on] == 7.0).all()), how

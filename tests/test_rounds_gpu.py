"""Launches of more than 256 positions in rounds of 512: the two-position kernel and, for a last round of at most 256, the
one-position form, by size, by leaf list and flags, and for the pooled value heads.  e4m3 and the 512-wide network; int8 of
the 256-wide one is in test_leaf_split_gpu.py.  The reference is the kernel with one position per workgroup of four
wavefronts, which none of these launches run."""
import pytest
import torch

from brokefish_amd import encoder_impl, positions
from brokefish_amd.hip_impl import compact_leaves
from brokefish_amd.net import BrokefishNet

pytestmark = pytest.mark.gpu
N = 1300
WIDE = dict(d_model=512, n_heads=16, d_ff=2048)


def _models(shape, quant, **kw):
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2, **shape, **kw).eval().randomise_layers_(seed=3)
    return [encoder_impl("hip")(net, out_dtype=torch.float32, kernel=k, **{quant: True}) for k in ("auto", "board")]


@pytest.fixture(scope="module", params=["e4m3", "wide"])
def made(request):
    auto, board = _models({}, "fp8") if request.param == "e4m3" else _models(WIDE, "int8")
    batch = [t.cuda() for t in positions.random_positions(N, plies=100, seed=3)]
    return auto, batch, [t.clone() for t in board.forward_masked(*batch)]


@pytest.mark.parametrize("n", [257, 258, 511, 512, 513, 544, 576, 577, 768, 769, 1024, 1025, N])
def test_every_size_of_a_last_round(made, n):
    auto, batch, want = made
    for g, w in zip(auto.forward_masked(*[t[:n] for t in batch]), want):
        assert torch.equal(g, w[:n])


@pytest.mark.parametrize("live", [0, 1, 2, 255, 256, 257, 511, 512, 513, 768, 769, N])
def test_live_counts_at_the_edges_of_a_round(made, live):
    auto, (b, c, r, m), want = made
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


@pytest.mark.parametrize("profile", [False, True])
@pytest.mark.parametrize("n,live", [(600, 0), (600, 1), (600, 200), (N, 430), (N, N)])
def test_flags_passed_to_the_library_as_they_are(made, n, live, profile):
    # FusedEncoder compacts flags above 256 positions; a C caller need not, and the profile does not
    auto, batch, want = made
    b, c, r, m = [t[:n] for t in batch]
    flags = torch.zeros(n, dtype=torch.uint8, device="cuda")
    flags[torch.randperm(n, generator=torch.Generator().manual_seed(live))[:live].cuda()] = 3
    on = flags != 0
    auto.forward_masked(b, c, r, m)                            # the buffers exist
    outs = (auto.policy_out, auto.promo_out, auto.value_out, auto.best_out)
    for t in outs:
        t.fill_(7)
    if profile:
        auto.set_profile(True)
        try:
            auto.forward_full(b, c, r, m, active=flags)
        finally:
            cycles, waves = auto.read_profile()
            auto.set_profile(False)
            auto.reset_profile()
        assert waves == (4 if auto.fp8 else 8) * n and (int(cycles[-1]) > 0) == (live > 0)
    else:
        auto._call(auto._args(b, c, r, m, *outs, active=flags))
    for g, w in zip(outs, want):
        assert torch.equal(g[on], w[:n][on]) and bool((g[~on] == 7).all())


@pytest.mark.parametrize("head,n_value", [("pooled", 1), ("prenorm", 1), ("pooled", 3), ("king", 3)])
def test_value_heads_of_the_wide_network(head, n_value):
    auto, board = _models(WIDE, "int8", value_head=head, n_value=n_value)
    batch = [t.cuda() for t in positions.random_positions(601, plies=100, seed=5)]
    want = [t.clone() for t in board.forward_masked(*batch)]
    for g, w in zip(auto.forward_masked(*batch), want):
        assert torch.equal(g, w)

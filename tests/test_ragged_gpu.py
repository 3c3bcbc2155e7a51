"""Sizes whose last round of 512 positions goes to workgroups of one position, in the same launch as the pairs: outputs (every value
head, both formats of the logits) and the encoder alone against the kernel of one position per workgroup of four
wavefronts, bit for bit.  (Leaf lists: test_leaf_split_gpu.py, test_rounds_gpu.py.)"""
import pytest
import torch

from brokefish_amd import encoder_impl, positions
from brokefish_amd.net import BrokefishNet

pytestmark = pytest.mark.gpu
N = 1281


@pytest.fixture(scope="module", params=["int8", "fp8"])
def made(request):
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2).eval().randomise_layers_(seed=9)
    auto, board = (encoder_impl("hip")(net, out_dtype=torch.float32, kernel=k, **{request.param: True}) for k in ("auto", "board"))
    batch = [t.cuda() for t in positions.random_positions(N, plies=100, seed=9)]
    x = torch.randn(N, 32, 256, device="cuda", generator=torch.Generator("cuda").manual_seed(9)) * 0.14
    alive = ((batch[0].to(torch.int32) >> 11) & 1) == 0
    return auto, batch, [t.clone() for t in board.forward_masked(*batch)], x, alive, board.forward(x, alive).clone()


# the smallest and largest last round that pairs leave (65 to 256), its neighbours on either side, behind one round and two
@pytest.mark.parametrize("n", [576, 577, 600, 767, 768, 769, 1088, 1089, 1280, N])
def test_a_last_round_in_the_same_launch(made, n):
    auto, batch, want, x, alive, stream = made
    for g, w in zip(auto.forward_masked(*[t[:n] for t in batch]), want):
        assert torch.equal(g, w[:n])
    assert torch.equal(auto.forward(x[:n].contiguous(), alive[:n].contiguous()), stream[:n])


@pytest.mark.parametrize("quant", ["int8", "fp8"])
@pytest.mark.parametrize("head,n_value,dtype", [("king", 3, torch.float16), ("pooled", 1, torch.float16), ("pooled", 3, torch.float32),
                                                ("prenorm", 1, torch.float32), ("prenorm", 3, torch.float16)])
def test_value_heads_and_halves(quant, head, n_value, dtype):
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2, value_head=head, n_value=n_value).eval().randomise_layers_(seed=10)
    auto, board = (encoder_impl("hip")(net, out_dtype=dtype, kernel=k, **{quant: True}) for k in ("auto", "board"))
    batch = [t.cuda() for t in positions.random_positions(577, plies=100, seed=10)]      # a round of pairs and 65 alone
    want = [t.clone() for t in board.forward_masked(*batch)]
    got = auto.forward_masked(*batch)
    assert got[0].dtype == dtype
    for g, w in zip(got, want):
        assert torch.equal(g, w)


@pytest.mark.parametrize("n,live", [(577, 0), (577, 1), (600, 200), (768, 700), (1281, 1281)])
def test_flags_passed_to_the_library_as_they_are(n, live):
    # FusedEncoder compacts flags above 256 positions; a C caller need not (e4m3 and 512 wide: test_rounds_gpu.py)
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2).eval().randomise_layers_(seed=9)
    auto, board = (encoder_impl("hip")(net, int8=True, out_dtype=torch.float32, kernel=k) for k in ("auto", "board"))
    batch = [t.cuda() for t in positions.random_positions(n, plies=100, seed=9)]
    want = [t.clone() for t in board.forward_masked(*batch)]
    flags = torch.zeros(n, dtype=torch.uint8, device="cuda")
    flags[torch.randperm(n, generator=torch.Generator().manual_seed(live))[:live].cuda()] = 1
    on = flags != 0
    auto.forward_masked(*batch)                                # the buffers exist
    outs = (auto.policy_out, auto.promo_out, auto.value_out, auto.best_out)
    for t in outs:
        t.fill_(7)
    auto._call(auto._args(*batch, *outs, active=flags))
    for g, w in zip(outs, want):
        assert torch.equal(g[on], w[on]) and bool((g[~on] == 7).all())

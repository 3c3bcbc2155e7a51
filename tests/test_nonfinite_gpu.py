"""Infinities and NaN in the tokens, in the attention scores and behind dead keys: the forms AUTO runs mask keys by adding 0 or
-inf inside a fused operation and take row maxima without quieting, and have to return what the four-wavefront kernel, which
selects and compares, returns (NaN for NaN; every other value bit for bit)."""
import pytest
import torch

from brokefish_amd import encoder_impl, positions
from brokefish_amd.net import BrokefishNet

pytestmark = pytest.mark.gpu
INF, NAN = float("inf"), float("nan")
WIDE = dict(d_model=512, n_heads=16, d_ff=2048)


def _models(wide, quant, scores):
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2, **(WIDE if wide else {})).eval().randomise_layers_(seed=8)
    d = 512 if wide else 256
    with torch.no_grad():
        for layer in net.encoder.layers:      # queries and keys: with 2^64 most of their products leave the range of a float
            layer.self_attn.in_proj_weight[:2 * d] *= scores
            layer.self_attn.in_proj_bias[:2 * d] *= scores
    return [encoder_impl("hip")(net, kernel=k, out_dtype=torch.float32, **{quant: True}) for k in ("auto", "board")]


@pytest.fixture(scope="module", params=[(w, q, s) for w, q in ((False, "int8"), (False, "fp8"), (True, "int8")) for s in (1.0, 2.0 ** 64)],
                ids=lambda p: f"{'wide' if p[0] else 'base'}-{p[1]}-{'scores' if p[2] > 1 else 'tokens'}")
def models(request):
    return request.param, _models(*request.param)


def _same(got, want):
    assert bool(((got == want) | (got.isnan() & want.isnan())).all())


# the team form, the one-position form, two positions per workgroup
@pytest.mark.parametrize("n", [3, 100, 301])
def test_the_stack_alone(models, n):
    (wide, _, _), (auto, board) = models
    d = 512 if wide else 256
    x = 0.2 * torch.randn(n, 32, d, generator=torch.Generator().manual_seed(n))
    alive = torch.rand(n, 32, generator=torch.Generator().manual_seed(n)) < 0.8
    alive[:, 15] = alive[:, 31] = True
    alive[0] = False                                       # no key at all
    for i in range(n):                                     # live and dead tokens alike: one element, a few, a whole row
        t = i % 32
        for value in ((INF,), (-INF,), (NAN,), (INF, -INF), (3e38,), ())[i % 6]:
            x[i, t, (37 * i) % d] = value
            x[i, (t + 7) % 32, i % 5::5] = value
            x[i, (t + 19) % 32] = value
    x, alive = x.cuda(), alive.cuda()
    want = board.forward(x, alive)
    _same(auto.forward(x, alive), want)
    assert bool(want.isnan().any())


@pytest.mark.parametrize("n", [3, 100, 301])
def test_the_whole_network(models, n):
    (_, quant, scores), (auto, board) = models
    batch = [t.cuda() for t in positions.random_positions(n, plies=100, seed=8)]
    want = [t.clone() for t in board.forward_masked(*batch)]
    got = auto.forward_masked(*batch)
    for g, w in zip(got[:3], want):
        _same(g, w)
    nan = want[0].isnan().any(2).any(1)                    # the int8 quantisers make 0 of a NaN, e4m3 has a code for it
    assert bool(nan.any()) == (scores > 1 and quant == "fp8")
    assert torch.equal(got[3][~nan], want[3][~nan])        # among NaN logits no move is the largest: a legal one comes back
    best, words = got[3].cpu().tolist(), batch[3].cpu().tolist()
    assert all(words[i][m // 64] >> (m % 64) & 1 for i, m in enumerate(best) if m >= 0)      # -1: no legal move

"""How the two-position kernel and its one-position form take an accumulator's scale apart (significand and exponent), at
scales far from 1: LayerNorm gains and values of one power of two, the weights that read them of its inverse.  The
reference is the four-wavefront kernel, which converts and multiplies."""
import pytest
import torch

from brokefish_amd import encoder_impl, positions
from brokefish_amd.net import BrokefishNet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [100, 258])
@pytest.mark.parametrize("power", [-100, -60, -1, 1, 60, 100])
def test_scales_of_any_exponent(power, n):
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2).eval().randomise_layers_(seed=5)
    g = 2.0 ** power
    with torch.no_grad():
        for layer in net.encoder.layers:
            for norm, reader in ((layer.norm1, layer.self_attn.in_proj_weight), (layer.norm2, layer.linear1.weight)):
                norm.weight.mul_(g)
                norm.bias.mul_(g)
                reader.div_(g)
            v = slice(2 * 256, 3 * 256)                      # values, and what reads the heads' outputs
            layer.self_attn.in_proj_weight[v].mul_(2.0 ** (power // 4))
            layer.self_attn.in_proj_bias[v].mul_(2.0 ** (power // 4))
            layer.self_attn.out_proj.weight.div_(2.0 ** (power // 4))
    batch = [t.cuda() for t in positions.random_positions(n, plies=100, seed=5)]
    got, want = ([t.clone() for t in encoder_impl("hip")(net, int8=True, out_dtype=torch.float32, kernel=k).forward_masked(*batch)]
                 for k in ("duo" if n > 256 else "octo", "board"))
    assert all(bool(torch.isfinite(t[t > -float("inf")]).all()) for t in want[:3])
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("quant", ["int8", "fp8"])
@pytest.mark.parametrize("n", [100, 258])
@pytest.mark.parametrize("power", [-100, 96])
def test_results_near_the_ends_of_the_quantisers_range(quant, power, n):
    # values and hidden rows of magnitude 2^power, and inverse weights behind them: within what the header states, where the
    # scales' product, the folded exponent and the e4m3 quotient at an eighth are farthest from 1
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2).eval().randomise_layers_(seed=5)
    g = 2.0 ** power
    with torch.no_grad():
        for layer in net.encoder.layers:
            v = slice(2 * 256, 3 * 256)
            for p in (layer.self_attn.in_proj_weight[v], layer.self_attn.in_proj_bias[v], layer.linear1.weight, layer.linear1.bias):
                p.mul_(g)
            for p in (layer.self_attn.out_proj.weight, layer.linear2.weight):
                p.div_(g)
    batch = [t.cuda() for t in positions.random_positions(n, plies=100, seed=5)]
    got, want = ([t.clone() for t in encoder_impl("hip")(net, out_dtype=torch.float32, kernel=k, **{quant: True}).forward_masked(*batch)]
                 for k in ("duo" if n > 256 else "octo", "board"))
    assert all(bool(torch.isfinite(t[t > -float("inf")]).all()) for t in want[:3])
    for a, b in zip(got, want):
        assert torch.equal(a, b)

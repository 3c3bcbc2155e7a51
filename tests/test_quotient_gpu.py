"""The kernels' reciprocal and reciprocal square root on the device, every float of their range, and rows at the ends of
the range: squares that overflow, magnitudes too small for a scale."""
import numpy as np
import pytest
import torch

from brokefish_amd import encoder_impl, positions
from brokefish_amd.hip_impl import recip_probe
from brokefish_amd.net import BrokefishNet
from oracle import c_oracle

pytestmark = pytest.mark.gpu


def every_float(exponent):
    """All 2^23 positive floats of one binade."""
    return (torch.arange(1 << 23, dtype=torch.int32, device="cuda") + ((exponent + 127) << 23)).view(torch.float32)


def test_reciprocal_is_correctly_rounded_for_every_float_of_its_range():
    for e in range(-126, 126):
        x = every_float(e)
        want = (1.0 / x.double()).float()        # a quotient of two 24-bit significands, rounded to 53 bits first, rounds the same
        assert torch.equal(recip_probe(x), want), e
        assert torch.equal(recip_probe(-x[:4096]), -want[:4096]), e
    assert recip_probe(torch.tensor([2.0 ** 126], device="cuda")).item() == 2.0 ** -126


def test_reciprocal_root_is_two_correctly_rounded_steps_for_every_float_of_its_range():
    for e in range(-102, 128):
        x = every_float(e)
        want = (1.0 / x.double().sqrt().float().double()).float()
        assert torch.equal(recip_probe(x, root=True), want), e
    assert recip_probe(torch.tensor([float("inf")], device="cuda"), root=True).item() == 0.0
    assert recip_probe(torch.tensor([float("nan")], device="cuda"), root=True).isnan().item()


@pytest.mark.parametrize("kernel", ["auto", "octo", "duo", "twin", "board", "quad"])
def test_rows_whose_squares_overflow_normalise_as_in_the_checker(kernel):
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2).eval().randomise_layers_(seed=4)
    b, c, r, m = positions.random_positions(6, plies=60, seed=4)
    x = torch.randn(6, 32, 256, generator=torch.Generator().manual_seed(0)) * 0.2
    x[1, 3] *= 1e20          # squares overflow: the row becomes beta
    x[2, 5] *= 1e15          # they do not
    x[4, 7, 0] = 3e38
    want = c_oracle.COracle({k: v.detach() for k, v in net.state_dict().items()}).forward(b.numpy(), c.numpy(), r.numpy(), mask=m.numpy(), x_in=x)
    model = encoder_impl("hip")(net, int8=True, kernel=kernel)
    got = model.forward_taps(b.cuda(), c.cuda(), r.cuda(), mask=m.cuda(), x_in=x.cuda(), want=[])
    for name in ("policy", "promo", "value"):
        assert np.array_equal(got[name].cpu().numpy().view(np.int32), want[name].view(np.int32)), name
    if kernel == "auto":     # and the form that spreads a position over several compute units, through the encoder alone
        octo = encoder_impl("hip")(net, int8=True, kernel="octo")
        assert torch.equal(model.forward(x.cuda()).nan_to_num(7.0), octo.forward(x.cuda()).nan_to_num(7.0))


@pytest.mark.parametrize("quant,kernel", [("int8", k) for k in ("auto", "octo", "duo", "twin", "board", "quad")] + [("fp8", k) for k in ("auto", "octo", "duo", "twin", "board", "quad")])
@pytest.mark.parametrize("tiny", [1e-37, 1e-39, 1e-42])
def test_rows_too_small_for_a_scale_count_as_zero(quant, kernel, tiny):
    b, c, r, _ = (t.cuda() for t in positions.random_positions(5, plies=60, seed=4))
    outs = []
    for gamma in (tiny, 0.0):
        torch.manual_seed(0)
        net = BrokefishNet(n_layers=2).eval().randomise_layers_(seed=4)
        with torch.no_grad():
            for layer in net.encoder.layers:
                layer.norm1.weight.fill_(gamma), layer.norm1.bias.zero_()
        model = encoder_impl("hip")(net, kernel=kernel, out_dtype=torch.float32, **{quant: True})
        outs.append([t.clone() for t in model.forward_full(b, c, r)])
    for got, want in zip(*outs):
        assert bool(got.isfinite().all()) and torch.equal(got, want)

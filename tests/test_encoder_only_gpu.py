"""The encoder-only builds (half-precision stream in and out, split last round) against the taps builds of the
other kernels, bit for bit."""
import pytest
import torch

from brokefish_amd import encoder_impl
from brokefish_amd.net import BrokefishNet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide,fmt,other", [(False, "int8", "twin"), (False, "fp8", "board"), (True, "int8", "board")])
def test_encoder_only_builds_return_the_bits_of_the_taps_builds(wide, fmt, other):
    torch.manual_seed(0)
    shape = dict(d_model=512, n_heads=16, d_ff=2048, n_layers=3) if wide else dict(n_layers=3)
    net = BrokefishNet(**shape).eval().randomise_layers_(seed=4)
    hip = encoder_impl("hip")
    model, ref = hip(net, **{fmt: True}), hip(net, kernel=other, **{fmt: True})
    d = 512 if wide else 256
    for n in (1, 3, 256, 257, 512, 600, 769, 1100):      # one round, odd pairs, rounds with short and long rests
        x = 0.2 * torch.randn(n, 32, d, device="cuda")
        alive = torch.rand(n, 32, device="cuda") < 0.8
        alive[:, 15] = alive[:, 31] = True
        want = ref.forward(x, alive)
        assert torch.equal(model.forward(x, alive), want), n
        assert torch.equal(model.forward(x, alive, out=torch.empty_like(x, dtype=torch.float16)), want.half()), n
        xh = x.half()
        want = ref.forward(xh.float(), alive)
        got = model.forward(xh, alive)
        assert got.dtype is torch.float16 and torch.equal(got, want.half()), n
        assert torch.equal(model.forward(xh, alive, out=torch.empty_like(x)), want), n
        assert model.forward(xh, alive, out=xh) is xh and torch.equal(xh, want.half()), n     # in place
    xb = (0.2 * torch.randn(5, 32, d, device="cuda")).bfloat16()
    assert torch.equal(model.forward(xb), ref.forward(xb.float()).bfloat16())                 # a type with passes of its own

"""The encoder-only builds (half-precision stream in and out, split last round) against the taps builds of the
other kernels, bit for bit."""
import ctypes

import pytest
import torch

from brokefish_amd import encoder_impl, hip_impl
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


@pytest.mark.parametrize("kernel", ["twin", "octo", "duo"])
def test_a_kernel_asked_for_by_name_takes_a_half_precision_stream_in_e4m3(kernel):
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=3).eval().randomise_layers_(seed=4)
    model, ref = encoder_impl("hip")(net, fp8=True, kernel=kernel), encoder_impl("hip")(net, fp8=True, kernel="board")
    assert hasattr(model._lib, f"_ZN2bf{len('launch_twin256_fp8_enc')}launch_twin256_fp8_encERKNS_5KArgsEP12ihipStream_t")
    for n in (1, 2, 300, 513):
        x = 0.2 * torch.randn(n, 32, 256, device="cuda").half()
        alive = (torch.rand(n, 32, device="cuda") < 0.8).to(torch.int8)
        want = ref.forward(x.float(), alive).half()
        taps, a, got = hip_impl._Taps(), model._choice_args(n), torch.empty_like(x)
        taps.alive, taps.x_in_h, taps.resid_last_h = alive.data_ptr(), x.data_ptr(), got.data_ptr()
        a.board_wstream, a.board_fparams, a.taps = model.board_wstream.data_ptr(), model.board_fparams.data_ptr(), ctypes.pointer(taps)
        model._call(a)
        assert torch.equal(got, want), n

"""The start of the two-position kernel and its one-position form.  The first layer's parameters go straight to LDS and the weights
asked for behind them may still be under way when they are waited for, so the wait may count only loads that every
wavefront of every launch has issued: on the CPU, by a host program over the functions the kernel is compiled with.  On the GPU the
launches with the fewest such loads (up to 24 workgroups of one position, as a launch of their own and as a last round) against the kernel of
four wavefronts, bit for bit."""
import os
import subprocess

import pytest
import torch

from brokefish_amd import _build, encoder_impl, positions
from brokefish_amd.net import BrokefishNet

HERE = os.path.dirname(os.path.abspath(__file__))


def test_the_wait_counts_loads_that_every_wavefront_issues(tmp_path):
    exe = str(tmp_path / "duo_start_check")
    subprocess.run([_build.hipcc_path(), "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-Wno-unused-command-line-argument",
                    "-I", _build.INCLUDE, "-I", _build.CSRC, os.path.join(HERE, "abi", "duo_start_check.hip"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.count(" 0 faults") == 4, out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("quant", ["int8", "fp8"])
def test_launches_of_few_workgroups(quant):
    torch.manual_seed(0)
    net = BrokefishNet(n_layers=2).eval().randomise_layers_(seed=12)
    solo, auto, board = (encoder_impl("hip")(net, out_dtype=torch.float32, kernel=k, **{quant: True}) for k in ("octo", "auto", "board"))
    batch = [t.cuda() for t in positions.random_positions(536, plies=100, seed=12)]
    want = [t.clone() for t in board.forward_masked(*batch)]
    x = torch.randn(26, 32, 256, device="cuda", generator=torch.Generator("cuda").manual_seed(12)) * 0.14
    stream = board.forward(x).clone()
    for n in range(1, 27):
        for g, w in zip(solo.forward_masked(*[t[:n] for t in batch]), want):
            assert torch.equal(g, w[:n]), n
        assert torch.equal(solo.forward(x[:n].contiguous()), stream[:n]), n
    auto._team_bytes = 0                                       # without a workspace a last round of up to 64 goes to workgroups of one position
    for n in (513, 520, 536):
        for g, w in zip(auto.forward_masked(*[t[:n] for t in batch]), want):
            assert torch.equal(g, w[:n]), n

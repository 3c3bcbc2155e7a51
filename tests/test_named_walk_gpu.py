"""The native walk over a module's parameters (fingerprint, packing): shared parameters and modules count as
torch.nn.Module.named_parameters counts them, and a module that walks in its own way is left to Python."""
import copy

import pytest
import torch

from brokefish_amd import sync
from brokefish_amd.net import BrokefishNet

pytestmark = pytest.mark.gpu


def network():
    torch.manual_seed(0)
    return BrokefishNet(n_layers=3).eval().randomise_layers_(seed=4)


def tied_parameter(net):
    net.encoder.layers[2].norm1.weight = net.encoder.layers[0].norm1.weight
    return net


def tied_module(net):
    net.encoder.layers[2].linear1 = net.encoder.layers[1].linear1
    return net


class OwnWalk(BrokefishNet):
    def named_parameters(self, *args, **kwargs):
        return iter([(n, p) for n, p in super().named_parameters(*args, **kwargs) if "norm" not in n])


def own_walk(net):
    other = OwnWalk(n_layers=3).eval()
    other.load_state_dict(net.state_dict())
    return other


@pytest.mark.parametrize("change", [lambda net: net, tied_parameter, tied_module, own_walk])
def test_fingerprint_and_blobs_of_unusual_modules(change):
    net = change(network())
    plain = network()
    plain.load_state_dict(copy.deepcopy(net.state_dict()))
    want = sync.weight_fingerprint(net)             # on the CPU, over named_parameters
    net, plain = net.cuda(), plain.cuda()
    assert abs(sync.weight_fingerprint(net) - want) <= 1e-9 * abs(want)
    got, ref = (sync.PackedWeights.pack(n, 1, int8=True) for n in (net, plain))
    assert torch.equal(got.encoder.board_wstream, ref.encoder.board_wstream)
    assert torch.equal(got.encoder.board_fparams.view(torch.int32), ref.encoder.board_fparams.view(torch.int32))   # holds integers too
    got.assert_current(net, 1)

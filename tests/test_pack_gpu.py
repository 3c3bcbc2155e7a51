"""The device packer (bf_pack_board) against the numpy packer, byte for byte, and the device fingerprint
against the CPU's: both widths and formats, more layers than one launch carries, all-zero weight blocks,
unaligned and half-precision parameters."""
import ctypes as C

import numpy as np
import pytest
import torch

from brokefish_amd import hip_impl, sync
from brokefish_amd.net import BrokefishNet

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,layers,nv,fmt,where", [(256, 8, 1, "int8", "cuda"), (256, 1, 3, "e4m3", "cuda"), (256, 17, 3, "int8", "cpu"),
                                                   (512, 2, 3, "int8", "cuda"), (512, 16, 1, "int8", "cuda")])
def test_device_packing_equals_the_numpy_packing(d, layers, nv, fmt, where):
    torch.manual_seed(3)
    net = BrokefishNet(d_model=d, n_heads=d // 32, d_ff=4 * d, n_layers=layers, n_value=nv).eval().randomise_layers_(seed=layers)
    with torch.no_grad():
        net.encoder.layers[0].linear1.weight[128:256] = 0.0                     # a block without a maximum
        net.encoder.layers[0].linear2.weight[:, :256] *= 1e-3                   # e4m3: k-chunks of different scales
    sd = {k: v.detach() for k, v in net.state_dict().items()}
    ws, fp = hip_impl.pack_network_board(sd, layers, d, 4 * d, nv, fmt=fmt)
    f_cpu = sync.weight_fingerprint(net)
    net = net.to(where)
    if where == "cuda":
        assert abs(sync.weight_fingerprint(net) - f_cpu) <= 1e-9 * abs(f_cpu)
        assert sync.weight_fingerprint(net) == sync.weight_fingerprint(net)
    shape = hip_impl._Shape(d, layers, d // 32, 4 * d, nv, 1e-5)
    got_ws, got_fp = hip_impl.pack_board_on_device(net, net.encoder, shape, fmt == "e4m3", torch.device("cuda", 0))
    assert got_ws.numel() == ws.size == hip_impl.load_library().bf_board_wstream_bytes(C.byref(shape))
    assert np.array_equal(got_ws.cpu().numpy(), ws)
    assert np.array_equal(got_fp.cpu().numpy().view(np.uint32), fp.view(np.uint32))


def test_parameters_that_are_unaligned_or_of_another_type_are_taken_as_fp32():
    torch.manual_seed(5)
    net = BrokefishNet(n_layers=1).eval().randomise_layers_(seed=2).cuda()
    lin = net.encoder.layers[0].linear1
    flat = torch.empty(lin.weight.numel() + 1, device="cuda")
    flat[1:] = lin.weight.detach().reshape(-1)
    lin.weight = torch.nn.Parameter(flat[1:].view_as(lin.weight))               # 4 bytes past an aligned address
    net.policy.half()
    shape = hip_impl._Shape(256, 1, 8, 1024, 1, 1e-5)
    got_ws, got_fp = hip_impl.pack_board_on_device(net, net.encoder, shape, False, torch.device("cuda", 0))
    ws, fp = hip_impl.pack_network_board({k: v.detach() for k, v in net.state_dict().items()}, 1, 256, 1024, 1)
    assert np.array_equal(got_ws.cpu().numpy(), ws) and np.array_equal(got_fp.cpu().numpy().view(np.uint32), fp.view(np.uint32))
    with pytest.raises(ValueError, match="wants"):
        hip_impl.pack_board_on_device(net, net.encoder, hip_impl._Shape(256, 1, 8, 1024, 3, 1e-5), False, torch.device("cuda", 0))


def test_a_fingerprint_that_nobody_reads_keeps_its_host_memory_until_it_is_written(monkeypatch):
    # the value is written to pinned memory by a kernel; here the stream is busy with something else when the
    # fingerprint is dropped, as it is where packing the same network raises
    net = BrokefishNet(n_layers=1).eval().randomise_layers_(seed=2).cuda()
    want = sync.weight_fingerprint(net)
    monkeypatch.setattr(sync, "encoder_impl", lambda impl: (_ for _ in ()).throw(RuntimeError("no evaluator today")))
    for how in ("dropped", "raised"):
        torch.cuda._sleep(100_000_000)
        if how == "dropped":
            hip_impl.fingerprint_on_device(net)
        else:
            with pytest.raises(RuntimeError, match="no evaluator today"):
                sync.PackedWeights.pack(net, 1, int8=True)
        held = [torch.full((1,), 1.0, dtype=torch.float64).pin_memory() for _ in range(64)]
        torch.cuda.synchronize()
        assert all(t.item() == 1.0 for t in held), how
    assert sync.weight_fingerprint(net) == want

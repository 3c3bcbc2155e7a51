"""The device fingerprint at the edges of its workgroups (8192 elements), of its launches (192 parameters) and of
the second launch's batches, against the definition in float64 (reference brokefish/train/sync.py:34-49)."""
import pytest
import torch

from brokefish_amd import sync

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1], [255], [256], [257], [8191], [8192], [8193, 1, 16384], [5] * 192, [3] * 191 + [9000, 7, 8192],
                                   [8192 * 2047 + 1], [8192 * 2048 + 8191, 2]],
                         ids=lambda s: f"{len(s)}x{max(s)}")
def test_fingerprint_at_the_edges_of_its_chunks(sizes):
    g = torch.Generator().manual_seed(sum(sizes))
    net = torch.nn.Module()
    for i, n in enumerate(sizes):
        net.register_parameter(f"p{i:04d}", torch.nn.Parameter(torch.randn(n, generator=g)))
    want = all_ = 0.0
    for i, (_, p) in enumerate(sorted(net.named_parameters())):
        term = (i + 1) * p.detach().double() * (torch.arange(1, p.numel() + 1, dtype=torch.float64) % 9973.0 + 1.0)
        want, all_ = want + float(term.sum()), all_ + float(term.abs().sum())
    got = sync.weight_fingerprint(net.cuda())
    # a sum of n terms in any order, each of two roundings: at most n + 2 roundings' worth of the terms' magnitudes
    assert abs(got - want) <= (sum(sizes) + 2) * 2.0 ** -53 * all_
    assert got == sync.weight_fingerprint(net)

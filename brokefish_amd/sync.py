"""Weight synchronisation between a trainer's torch module and the packed evaluator.

The evaluator object is a snapshot: construction copies the weights into device blobs in kernel
order.  ``PackedWeights`` carries the two facts that say whether a snapshot is still the right
one -- the generation it was packed at and a fingerprint of the master weights -- and refuses to
hand out a stale evaluator.  Mirrors the reference's brokefish/train/sync.py:34-106 for
``impl="hip"`` (same names, same arguments, same errors), so a training loop written against
that module works unchanged.
"""
from __future__ import annotations

import math
from dataclasses import dataclass

import torch

from . import encoder_impl


def _fingerprint_on_device(net):
    """The fingerprint queued on the GPU that holds the parameters, or None."""
    if not torch.cuda.is_available():
        return None
    from .hip_impl import fingerprint_on_device
    return fingerprint_on_device(net)


@torch.no_grad()
def weight_fingerprint(net) -> float:
    """One float that changes if any parameter does, or if the same values are permuted: an
    index-weighted float64 sum over the parameters in name order (brokefish/train/sync.py:34-49).
    Parameters on a GPU (fp32, as a trainer holds them) are summed there, two launches and one wait
    for the whole network; the order of the sum differs from the CPU's, so a value is compared with
    one taken on the same device."""
    got = _fingerprint_on_device(net)
    if got is not None:
        return got.value()
    acc = 0.0
    for i, (_, p) in enumerate(sorted(net.named_parameters(), key=lambda kv: kv[0])):
        f = p.detach().reshape(-1).double()
        idx = torch.arange(1, f.numel() + 1, device=f.device, dtype=torch.float64)
        acc += float(((i + 1) * f * (idx % 9973.0 + 1.0)).sum())
    return acc


@dataclass
class PackedWeights:
    """A packed evaluator plus the generation and fingerprint it was built from."""

    encoder: object
    weight_gen: int
    fingerprint: float

    @classmethod
    def pack(cls, net, weight_gen: int, impl: str = "hip", fp8: bool = False, int8: bool = False,
             **kwargs) -> "PackedWeights":
        """Snapshot ``net`` into the evaluator's device blobs (brokefish/train/sync.py:60-90).
        ``int8`` / ``fp8`` select the format as in the reference; with neither, int8 (this
        library carries no unquantised evaluator)."""
        if fp8 and int8:
            raise ValueError("fp8 and int8 quantise the same matmuls; pick one")
        if impl != "hip":
            raise ValueError(f"this library provides impl 'hip'; impl is {impl!r}")
        kw = {"fp8": True} if fp8 else {"int8": True}
        kw.update(kwargs)
        queued = _fingerprint_on_device(net)      # runs in front of the packing: one wait for both
        encoder = encoder_impl(impl)(net, **kw)
        return cls(encoder=encoder, weight_gen=int(weight_gen),
                   fingerprint=queued.value() if queued is not None else weight_fingerprint(net))

    def evaluate(self):
        """The evaluator the search wants: ``(boards, control, rep) -> fp16 logits, fp32 value``."""
        return self.encoder.forward_full

    def assert_current(self, net, weight_gen: int) -> None:
        """Raises rather than silently self-playing a stale network (brokefish/train/sync.py:92-106)."""
        if self.weight_gen != int(weight_gen):
            raise AssertionError(
                f"self-play is about to run weights packed at generation {self.weight_gen} while the "
                f"loop is at generation {weight_gen}: the packed evaluator is a snapshot and has to "
                f"be rebuilt after every gradient phase")
        got = weight_fingerprint(net)
        if got != self.fingerprint:
            raise AssertionError(
                f"the master weights changed since they were packed (fingerprint "
                f"{self.fingerprint!r} at pack time, {got!r} now) without the generation moving")


@torch.no_grad()
def check_weights_propagate(net, packed: PackedWeights, tol: float = 3e-2, n_probe: int = 8, **pack_kwargs) -> dict:
    """Start-up consistency check of a packed evaluator against the master network: perturb the
    weights, repack, and require that the evaluator's output moved and that the repacked
    evaluator agrees with the master network's own forward on a fixed probe batch -- the check a
    training loop runs before its first self-play game (reference brokefish/train/loop.py:1109-1166;
    quantised formats are held to 8 % of the largest logit, :1158-1159).  The perturbation is undone
    before returning.  Raises ``AssertionError`` on a stale snapshot, a non-finite output or a
    disagreement; returns ``{"moved", "agree", "tol"}``."""
    from . import positions
    dev = packed.encoder.device
    boards, control, rep, _ = (t.to(dev) for t in positions.random_positions(n_probe, plies=0, seed=0))
    before = packed.encoder.forward_full(boards, control, rep)[0].float().clone()
    saved = {k: v.detach().clone() for k, v in net.state_dict().items()}
    fmt = {"fp8": True} if packed.encoder.fp8 else {"int8": True}
    fmt.update(pack_kwargs)
    try:
        g = torch.Generator().manual_seed(0)
        for p in net.parameters():
            p.add_((torch.randn(p.shape, generator=g) * 0.02).to(p.device, p.dtype))
        repacked = PackedWeights.pack(net, packed.weight_gen + 1, device=dev, **fmt)
        after = repacked.encoder.forward_full(boards, control, rep)[0].float().clone()
        where = next(net.parameters()).device
        ref = net(boards.to(where), control.to(where), rep.to(where))[0].float().to(dev)
    finally:
        net.load_state_dict(saved)
    moved = float((after - before).abs().max())
    agree = float((after - ref).abs().max())
    scale = float(ref.abs().max())
    if moved == 0.0:
        raise AssertionError("the evaluator's output did not change after a weight update: self-play would run a "
                             "stale snapshot")
    if not (math.isfinite(moved) and math.isfinite(agree)):      # explicitly: nan > tol is False
        raise AssertionError(f"the evaluator produced a non-finite output (moved={moved}, agree={agree})")
    tol = max(tol, 0.08 * scale)                                  # int8 and e4m3 are quantised paths
    if agree > tol:
        raise AssertionError(f"the repacked evaluator disagrees with the updated master network by {agree:.4g} "
                             f"(tolerance {tol:.4g}): a stale snapshot or a wrong weight slab")
    return {"moved": moved, "agree": agree, "tol": tol}

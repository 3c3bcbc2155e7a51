"""What the performance of this framework is measured on: the calls that a search, a self-play loop
or an analysis tool makes, over the sizes they make them at.

A case is a dict of plain values.  ``what`` names the call:

``eval``      ``FusedEncoder.forward_full`` / ``forward_masked``: boards to logits
``step``      ``FusedEncoder.forward_expand``: move generation, evaluation and edge expansion of one search step
``staged``    the same over a flat leaf buffer of which a share is live (compacted list or flags)
``backbone``  ``FusedEncoder.forward``: the encoder stack alone on a caller's tokens
``movegen``   ``movegen``: legal-move words of a batch of games
``expand``    ``expand_edges``: edges of search nodes from logits that are already there
``repack``    ``PackedWeights.pack`` / ``assert_current`` / first evaluation: a new weight generation

Positions are seeded uniformly random legal playouts of 0 to 120 plies, as in the benchmark; the
weights of the evaluating cases are one fixed random network per shape, packed once and kept, as a
program keeps its evaluator between calls.
"""
import functools
import math

import torch

from brokefish_amd import encoder_impl, positions
from brokefish_amd.hip_impl import compact_leaves, expand_edges, movegen
from brokefish_amd.net import BrokefishNet
from brokefish_amd.sync import PackedWeights

SHAPES = {"base": dict(d_model=256, n_heads=8, d_ff=1024, n_layers=8),
          "wide": dict(d_model=512, n_heads=16, d_ff=2048, n_layers=16)}
POOL = 2048          # different games a batch is drawn from


def listed():
    return [
        # an analysis board or an engine's root: one position, the masked best move wanted at once
        {"name": "position_1", "what": "eval", "net": "base", "format": "int8", "n": 1, "masked": True, "head": "king", "wdl": False, "fp32": False},
        # one simulation step of a small search: 64 leaves, everything on the device
        {"name": "step_64", "what": "step", "format": "int8", "n": 64, "edges": 96},
        # a flat leaf buffer of an odd size of which about a third needs evaluating
        {"name": "staged_1000", "what": "staged", "format": "int8", "n": 1000, "live": 0.37, "list": True},
        # the benchmark's own batch
        {"name": "batch_4096", "what": "eval", "net": "base", "format": "int8", "n": 4096, "masked": True, "head": "king", "wdl": False, "fp32": False},
        # re-evaluating a replay buffer: large, ragged, raw fp32 logits, pooled win/draw/loss value
        {"name": "batch_50021", "what": "eval", "net": "base", "format": "int8", "n": 50021, "masked": False, "head": "pooled", "wdl": True, "fp32": True},
        # the fp8 format at the benchmark's batch
        {"name": "e4m3_4096", "what": "eval", "net": "base", "format": "e4m3", "n": 4096, "masked": True, "head": "king", "wdl": False, "fp32": False},
        # the 16-layer, 512-wide network at a serving batch
        {"name": "wide_1500", "what": "eval", "net": "wide", "format": "int8", "n": 1500, "masked": True, "head": "king", "wdl": False, "fp32": False},
        # the encoder inside another model: half-precision tokens in and out
        {"name": "backbone_600", "what": "backbone", "format": "int8", "n": 600, "fp32": False, "alive": True},
        # the moves of the games a self-play loop runs side by side, once per ply
        {"name": "movegen_250", "what": "movegen", "n": 250},
        # the moves of a whole replay buffer
        {"name": "movegen_65536", "what": "movegen", "n": 65536},
        # the expansion of a wide search step, logits from elsewhere
        {"name": "expand_5000", "what": "expand", "n": 5000, "edges": 96, "fp32": False},
        # the trainer hands a new generation to self-play
        {"name": "repack_8", "what": "repack", "format": "int8", "layers": 8, "wdl": False},
    ]


def _size(rng, lo, hi):
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    u = rng.random()
    fmt = "e4m3" if rng.random() < 0.25 else "int8"
    if u < 0.35:
        net = "wide" if rng.random() < 0.25 else "base"
        if net == "wide":
            fmt = "int8"        # the wide network runs in int8 only
        hi = 2500 if net == "wide" else 12000 if fmt == "e4m3" else 40000
        head = rng.choice(["king", "king", "pooled", "prenorm"])
        return {"what": "eval", "net": net, "format": fmt, "n": _size(rng, 1, hi), "masked": rng.random() < 0.5,
                "head": head, "wdl": rng.random() < 0.5, "fp32": rng.random() < 0.25}
    if u < 0.52:
        return {"what": "step", "format": fmt, "n": _size(rng, 4, 12000), "edges": rng.choice([96, 96, 32])}
    if u < 0.64:
        return {"what": "staged", "format": fmt, "n": _size(rng, 64, 12000), "live": round(math.exp(rng.uniform(math.log(0.05), 0.0)), 3),
                "list": rng.random() < 0.5}
    if u < 0.74:
        return {"what": "backbone", "format": fmt, "n": _size(rng, 1, 8000), "fp32": rng.random() < 0.5, "alive": rng.random() < 0.8}
    if u < 0.83:
        return {"what": "movegen", "n": _size(rng, 1, 200000)}
    if u < 0.92:
        return {"what": "expand", "n": _size(rng, 1, 100000), "edges": rng.choice([96, 96, 32]), "fp32": rng.random() < 0.25}
    return {"what": "repack", "format": fmt, "layers": rng.randint(4, 12), "wdl": rng.random() < 0.5}


# --------------------------------------------------------------------------- #

@functools.lru_cache(maxsize=None)
def _evaluator(net, fmt, head, wdl, fp32):
    """The evaluator a program holds: one network per shape, packed once."""
    torch.manual_seed(0)
    master = BrokefishNet(n_value=3 if wdl else 1, value_head=head, **SHAPES[net]).eval().randomise_layers_(seed=1)
    quant = {"fp8": True} if fmt == "e4m3" else {"int8": True}
    return encoder_impl("hip")(master, out_dtype=torch.float32 if fp32 else torch.float16, **quant)


def _batch(n, seed):
    """(boards, control, rep, mask) of ``n`` positions on the GPU; beyond the pool's size the same
    games come up again in another order, as they do in a replay buffer."""
    parts = positions.random_positions(min(n, POOL), plies=120, seed=seed)
    parts = [t.cuda() for t in parts]
    if n <= POOL:
        return parts
    at = torch.randint(POOL, (n,), generator=torch.Generator().manual_seed(seed)).cuda()
    return [t[at].contiguous() for t in parts]


def prepare(case, seed):
    what = case["what"]
    s = {"what": what}
    if what == "repack":
        torch.manual_seed(seed)
        net = BrokefishNet(n_layers=case["layers"], n_value=3 if case["wdl"] else 1).eval().randomise_layers_(seed=seed)
        s.update(net=net.cuda(), generation=seed, quant={"fp8": True} if case["format"] == "e4m3" else {"int8": True})
        s["probe"] = _batch(64, seed)[:3]
        return s
    n = case["n"]
    boards, control, rep, mask = _batch(n, seed)
    s.update(boards=boards, control=control, rep=rep, mask=mask)
    g = torch.Generator(device="cuda").manual_seed(seed)
    if what == "eval":
        s.update(model=_evaluator(case["net"], case["format"], case["head"], case["wdl"], case["fp32"]), masked=case["masked"])
    elif what == "step":
        s.update(model=_evaluator("base", case["format"], "king", False, False), edges=case["edges"])
    elif what == "staged":
        flags = (torch.rand(n, generator=g, device="cuda") < case["live"]).to(torch.uint8)
        flags[seed % n] = 1
        # the search's own node storage and list, made once and written by every step
        out = {k: torch.zeros(shape, dtype=dtype, device="cuda") for k, shape, dtype in (
            ("edge_move", (n, 96), torch.int16), ("edge_prior", (n, 96), torch.float16), ("n_edges", (n,), torch.int32),
            ("count", (n,), torch.int32), ("dropped", (n,), torch.float32), ("node_value", (n,), torch.float16))}
        leaves = (torch.zeros(n, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda"))
        s.update(model=_evaluator("base", case["format"], "king", False, False), flags=flags, out=out,
                 leaves=leaves if case["list"] else None)
    elif what == "backbone":
        x = torch.randn(n, 32, 256, generator=g, device="cuda") * 0.14      # the scale of the embedding sums
        alive = ((boards.to(torch.int32) >> 11) & 1) == 0
        s.update(model=_evaluator("base", case["format"], "king", False, False), x=x if case["fp32"] else x.half(),
                 alive=alive if case["alive"] else None)
    elif what == "expand":
        dt = torch.float32 if case["fp32"] else torch.float16
        s.update(policy=(1.3 * torch.randn(n, 32, 64, generator=g, device="cuda")).to(dt),
                 promo=(1.3 * torch.randn(n, 32, 4, generator=g, device="cuda")).to(dt),
                 value=torch.tanh(torch.randn(n, generator=g, device="cuda")), edges=case["edges"])
    return s


def run(s):
    what = s["what"]
    if what == "eval":
        if s["masked"]:
            return s["model"].forward_masked(s["boards"], s["control"], s["rep"], s["mask"])
        return s["model"].forward_full(s["boards"], s["control"], s["rep"])
    if what == "step":
        return s["model"].forward_expand(s["boards"], s["control"], s["rep"], max_edges=s["edges"])
    if what == "staged":
        if s["leaves"] is None:
            return s["model"].forward_expand(s["boards"], s["control"], s["rep"], active=s["flags"], out=s["out"])
        leaves = compact_leaves(s["flags"], out=s["leaves"])
        edges = s["model"].forward_expand(s["boards"], s["control"], s["rep"], out=s["out"], leaves=leaves)
        return edges, leaves
    if what == "backbone":
        return s["model"].forward(s["x"], s["alive"])
    if what == "movegen":
        return movegen(s["boards"], s["control"])
    if what == "expand":
        return expand_edges(s["policy"], s["promo"], s["value"], s["mask"], s["boards"], s["control"], max_edges=s["edges"])
    packed = PackedWeights.pack(s["net"], s["generation"], **s["quant"])
    packed.assert_current(s["net"], s["generation"])
    policy, promo, value = packed.evaluate()(*s["probe"])
    return policy, promo, value, packed.fingerprint


# --------------------------------------------------------------------------- #

POSITION_BYTES = 64 + 2 + 1          # words, control, repetition
MASK_BYTES = 256


def _network(net, n_value=1, layers=None):
    """(parameter bytes as packed, operations of the encoder stack, operations of the heads) per position."""
    d, nl = SHAPES[net]["d_model"], layers or SHAPES[net]["n_layers"]
    packed = nl * (12 * d * d + 4 * 13 * d) + 4 * d * (64 + 12 + 4 + 101 + 3 + 2 + 68 + n_value)
    return packed, 2 * 32 * nl * (12 * d * d + 2 * 32 * d), 2 * (32 * 68 + n_value) * d


def _edge_bytes(n, edges):
    # about 31 legal moves per position of these playouts, in some 18 half-rows of logits
    return n * (4 * edges + 4 + 4 + 4 + 2)


def work(case):
    what = case["what"]
    if what == "repack":
        packed, stack, heads = _network("base", 3 if case["wdl"] else 1, case["layers"])
        master = 4 * (case["layers"] * (12 * 256 * 256 + 13 * 256) + 256 * (64 + 12 + 4 + 101 + 3 + 2 + 69))
        return {"bytes": master + packed + 64 * (POSITION_BYTES + 4364), "flops": 64 * (stack + heads)}
    n = case["n"]
    if what == "eval":
        packed, stack, heads = _network(case["net"], 3 if case["wdl"] else 1)
        out = 32 * 68 * (4 if case["fp32"] else 2) + 4 + (4 if case["masked"] else 0)
        return {"bytes": packed + n * (POSITION_BYTES + out + (MASK_BYTES if case["masked"] else 0)), "flops": n * (stack + heads)}
    packed, stack, heads = _network("base")
    if what == "step":
        return {"bytes": packed + n * (POSITION_BYTES + MASK_BYTES + 1) + _edge_bytes(n, case["edges"]), "flops": n * (stack + heads)}
    if what == "staged":
        live = max(1, int(n * case["live"]))
        return {"bytes": packed + n * (66 + MASK_BYTES + 2) + live + _edge_bytes(live, 96), "flops": live * (stack + heads)}
    if what == "backbone":
        return {"bytes": packed + n * 32 * 256 * 2 * (4 if case["fp32"] else 2) + (32 * n if case["alive"] else 0), "flops": n * stack}
    if what == "movegen":
        return {"bytes": n * (64 + 2 + MASK_BYTES + 1), "flops": 0}
    logit = 4 if case["fp32"] else 2
    return {"bytes": n * (66 + 4 + MASK_BYTES + 18 * 32 * logit) + _edge_bytes(n, case["edges"]), "flops": 0}


def tolerance(case):
    what = case["what"]
    if what == "movegen":
        return "exact"
    if what == "expand":
        return {"rel": 1e-3, "max": 1e-2, "differ": 1e-4}      # fp16 priors; moves may swap at a tie of the cut
    # A quantised forward: an operand byte that lies at a rounding tie may fall either way under another
    # order of the fp32 sums, and the later layers carry it to about a percent of that position's logits.
    return {"rel": 1e-2, "max": 0.5, "differ": 1e-3}

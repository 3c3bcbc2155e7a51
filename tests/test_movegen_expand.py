"""bf_movegen_expand, move generation and edge expansion in one launch, against the two calls: every output equal, at the edges of its
workgroups of eight positions, for positions of ordinary and of very many moves; and what it refuses."""
import collections
import ctypes

import pytest
import torch

from brokefish_amd import encoder_impl, hip_impl, positions
from brokefish_amd.hip_impl import expand_edges, movegen
from brokefish_amd.net import BrokefishNet

PAWN, QUEEN, KING, BLACK, CAPTURED = 0, 4 << 6, 5 << 6, 0x400, 0x800


def crowded(n, seed):
    """``n`` boards of eight white queens and seven pawns about to promote, most with more than 128 edges (a second build of the expansion)."""
    g = torch.Generator().manual_seed(seed)
    boards = torch.full((n, 32), CAPTURED, dtype=torch.int32)
    for i in range(n):
        pawns, victims, rest = (torch.randperm(k, generator=g) for k in (8, 8, 40))
        for k in range(8):
            boards[i, k] = int(rest[k]) | QUEEN
        for k in range(7):
            boards[i, 8 + k] = 48 + int(pawns[k]) | PAWN
        boards[i, 15] = int(rest[8]) | KING
        for k in range(4):
            boards[i, 16 + k] = 56 + int(victims[k]) | PAWN | BLACK
        boards[i, 31] = int(rest[9]) | KING | BLACK
    return boards.to(torch.int16), torch.ones(n, dtype=torch.int16)


def both(policy, promo, value, boards, control, edges):
    mask, check = movegen(boards, control)
    want = expand_edges(policy, promo, value, mask, boards, control, edges)
    got = hip_impl._native().movegen_expand(policy, promo, value, boards, control, edges, None)
    assert torch.equal(got["mask"], mask) and torch.equal(got["in_check"], check)
    for k, v in want.items():
        assert torch.equal(got[k], v), k
    return want


@pytest.mark.gpu
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("n,edges", [(1, 96), (2, 1), (7, 96), (8, 32), (9, 255), (250, 96), (1001, 40)])
def test_one_launch_is_the_two_calls(n, edges, fp32):
    boards, control, _, _ = [t.cuda() for t in positions.random_positions(n, plies=120, seed=n)]
    g = torch.Generator("cuda").manual_seed(n)
    dt = torch.float32 if fp32 else torch.float16
    policy, promo = (torch.randn(n, 32, k, generator=g, device="cuda").to(dt) for k in (64, 4))
    both(policy, promo, torch.tanh(torch.randn(n, generator=g, device="cuda")), boards, control, edges)


@pytest.mark.gpu
def test_positions_of_very_many_moves():
    n = 61
    boards, control = [t.cuda() for t in crowded(n, 3)]
    g = torch.Generator("cuda").manual_seed(3)
    policy, promo = (torch.randn(n, 32, k, generator=g, device="cuda") for k in (64, 4))
    count = both(policy, promo, torch.zeros(n, device="cuda"), boards, control, 96)["count"]
    assert int((count > 128).sum()) > 0 and int((count <= 128).sum()) > 0


@pytest.mark.gpu
def test_positions_of_more_moves_than_the_layout_holds():
    # more than 256 edges (fifteen queens on one square): the words just generated are read back, beside positions of the ordinary kind
    n = 21
    boards, control = [t[:n].clone() for t in positions.random_positions(n, plies=80, seed=7)[:2]]
    for i in (0, 3, 4, 8, 15, 20):
        boards[i] = CAPTURED
        boards[i, :15] = (27 + i) | QUEEN
        boards[i, 15], boards[i, 31] = KING, 63 | KING | BLACK
        control[i] = 1
    g = torch.Generator("cuda").manual_seed(7)
    policy, promo = (torch.randn(n, 32, k, generator=g, device="cuda").half() for k in (64, 4))
    count = both(policy, promo, torch.zeros(n, device="cuda"), boards.cuda(), control.cuda(), 96)["count"]
    assert int((count > 256).sum()) == 6 and int((count <= 128).sum()) == 15


@pytest.mark.gpu
def test_forward_expand_on_either_side_of_the_line(monkeypatch):
    torch.manual_seed(0)
    model = encoder_impl("hip")(BrokefishNet(n_layers=1).eval().randomise_layers_(seed=4), int8=True)
    batch = [t.cuda() for t in positions.random_positions(70, plies=100, seed=4)][:3]
    got = {k: v.clone() for k, v in model.forward_expand(*batch).items()}
    monkeypatch.setattr(hip_impl, "MOVEGEN_EXPAND_MOST", 69)
    want = model.forward_expand(*batch)
    assert got.keys() == want.keys() and all(torch.equal(got[k], v) for k, v in want.items())


@pytest.mark.gpu
def test_the_callers_dict_is_the_one_that_comes_back():
    # an OrderedDict lists what was put into it by its own methods only
    n = 9
    torch.manual_seed(0)
    model = encoder_impl("hip")(BrokefishNet(n_layers=1).eval().randomise_layers_(seed=4), int8=True)
    batch = [t.cuda() for t in positions.random_positions(n, plies=100, seed=4)][:3]
    for kind in (dict, collections.OrderedDict):
        out = kind((k, v.clone()) for k, v in model.forward_expand(*batch).items() if k not in ("mask", "in_check"))
        got = model.forward_expand(*batch, out=out)
        assert got is out and list(got)[6:] == ["mask", "in_check"] and len(got.values()) == 8


@pytest.mark.parametrize("boards,control", [([[0] * 32], torch.ones(1)), (None, torch.ones(1)), (torch.zeros(1, 32).numpy(), torch.ones(1)),
                                            (torch.zeros(1, 32, dtype=torch.int16), None), (torch.zeros(1, 32, dtype=torch.int16), [1])])
def test_what_is_no_tensor_is_refused_as_by_movegen(boards, control):
    with pytest.raises(Exception) as want:
        movegen(boards, control)
    with pytest.raises(want.type, match=str(want.value)):
        hip_impl.FusedEncoder.forward_expand(None, boards, control, None)


@pytest.mark.gpu
def test_into_the_callers_buffers():
    # node storage that earlier steps have written: every row is this step's, in the caller's memory
    n = 21
    torch.manual_seed(0)
    model = encoder_impl("hip")(BrokefishNet(n_layers=1).eval().randomise_layers_(seed=4), int8=True)
    steps = [[t.cuda() for t in positions.random_positions(n, plies=100, seed=s)][:3] for s in (5, 6)]
    want = [{k: v.clone() for k, v in model.forward_expand(*b).items()} for b in steps]
    out = {k: torch.full_like(v, 7) for k, v in want[0].items() if k not in ("mask", "in_check")}
    at = {k: v.data_ptr() for k, v in out.items()}
    for batch, w in zip(steps, want):
        got = model.forward_expand(*batch, out=out)
        assert got is out and all(got[k].data_ptr() == p for k, p in at.items())
        assert got.keys() == w.keys() and all(torch.equal(got[k], w[k]) for k in w)
    for other, edges in (([t[:20] for t in steps[0]], 96), (steps[0], 40)):
        with pytest.raises(ValueError, match="another n or max_edges"):
            model.forward_expand(*other, max_edges=edges, out=out)


def test_refused_arguments():
    lib = hip_impl.load_library()
    a = hip_impl._ExpandArgs()
    a.n, a.max_edges = 4, 96
    for name in ("policy", "promo", "value", "boards", "control", "edge_move", "edge_prior", "n_edges"):
        setattr(a, name, 16)
    call = lambda mask=16, check=16: lib.bf_movegen_expand(ctypes.byref(a), ctypes.c_void_p(mask), ctypes.c_void_p(check), None)
    assert call(mask=None) == -1 and call(check=None) == -1
    for names in (("mask",), ("active",), ("leaf_index", "leaf_count"), ("leaf_index",), ("leaf_count",)):
        for name in names:
            setattr(a, name, 16)
        assert call() == -1 and b"no mask, flags or leaf list" in lib.bf_last_error()
        for name in names:
            setattr(a, name, None)
    a.max_edges = 256
    assert call() == -1 and b"max_edges" in lib.bf_last_error()

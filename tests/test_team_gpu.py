"""Launches small enough for several workgroups per position (kernel="auto") return the bits of the
one-workgroup-per-position kernel: the edges of the launch sizes, skipped positions, leaf lists, the
encoder alone, replays of a graph between eager calls, and two streams at once."""
import pytest
import torch

from brokefish_amd import encoder_impl, positions
from brokefish_amd.hip_impl import compact_leaves
from brokefish_amd.net import BrokefishNet

pytestmark = pytest.mark.gpu
SHAPES = {"base": dict(n_layers=2), "wide": dict(d_model=512, n_heads=16, d_ff=2048, n_layers=2)}


def pair(shape="base", fp8=False, head="king", wdl=False):
    torch.manual_seed(3)
    net = BrokefishNet(n_value=3 if wdl else 1, value_head=head, **SHAPES[shape]).eval().randomise_layers_(seed=3)
    make = lambda kernel: encoder_impl("hip")(net, kernel=kernel, out_dtype=torch.float32, **({"fp8": True} if fp8 else {"int8": True}))
    team, single = make("auto"), make("octo")
    assert team._team_bytes > 0
    return team, single


def batch(n, seed=0):
    return [t.cuda() for t in positions.random_positions(n, plies=120, seed=seed)]


def assert_same(got, want):
    for g, w in zip(got, want):
        assert torch.equal(g, w)


@pytest.mark.parametrize("shape,fp8,n", [("base", False, 1), ("base", False, 7), ("base", False, 64), ("base", True, 9), ("wide", False, 1),
                                         ("wide", False, 32), ("wide", False, 50), ("wide", False, 256 + 5), ("base", False, 512 + 17)])
@pytest.mark.parametrize("head,wdl", [("king", False), ("pooled", True), ("prenorm", False)])
def test_team_launches_return_the_bits_of_the_single_workgroup_kernel(shape, fp8, n, head, wdl):
    team, single = pair(shape, fp8, head, wdl)
    x = batch(n)
    for seed in (0, 1):     # a second launch finds the first one's counts in the workspace
        assert_same(team.forward_masked(*x), single.forward_masked(*x))
        x = batch(n, seed + 1)
    assert_same(team.forward_full(*x[:3]), single.forward_full(*x[:3]))
    if n <= 64:
        tokens = torch.randn(n, 32, team.d_model, device="cuda") * 0.14
        alive = torch.rand(n, 32, device="cuda") < 0.8
        alive[:, 15] = True
        assert torch.equal(team.forward(tokens, alive), single.forward(tokens, alive))


def test_team_launches_skip_positions_and_take_leaf_lists():
    team, single = pair()
    x = batch(40)[:3]
    flags = (torch.arange(40, device="cuda") % 3 == 1).to(torch.uint8)
    want = [t.clone() for t in single.forward_full(*x)]
    live = flags.bool()
    for kwargs in ({"active": flags}, {"leaves": compact_leaves(flags)}):
        team._ensure_full_buffers(40)
        for t in (team.policy_out, team.promo_out, team.value_out):
            t.fill_(7.0)
        for g, w in zip(team.forward_full(*x, **kwargs), want):
            assert torch.equal(g[live], w[live]) and bool((g[~live] == 7.0).all())


def test_team_launches_in_a_graph_and_on_two_streams():
    team, single = pair()
    x, y = batch(20), batch(64, 5)
    want_x, want_y = ([t.clone() for t in single.forward_masked(*b)] for b in (x, y))
    team.forward_masked(*x)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = team.forward_masked(*x)
    for _ in range(3):
        g.replay()
        torch.cuda.synchronize()
        assert_same(out, want_x)
        assert_same([t.clone() for t in team.forward_masked(*x)], want_x)
    other, _ = pair()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    for _ in range(20):
        with torch.cuda.stream(s):
            a = other.forward_masked(*y)
        b = team.forward_masked(*x)
    torch.cuda.synchronize()
    assert_same(a, want_y)
    assert_same(b, want_x)


@pytest.mark.parametrize("shape,n,parts", [("base", 3, 3), ("base", 512 + 9, 9), ("wide", 20, 20), ("wide", 50, 32)])
def test_a_captured_launch_has_exchange_memory_of_its_size_and_clears_its_flags(shape, n, parts):
    team, single = pair(shape)
    x = batch(n)
    want = [t.clone() for t in single.forward_masked(*x)]
    team.forward_masked(*x)
    taken = []
    make = team._captured_team_workspace
    team._captured_team_workspace = lambda k: taken.append(make(k)) or taken[-1]
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = team.forward_masked(*x)
    ws, = taken
    assert ws.numel() == parts * (team._team_bytes // (64 if shape == "base" else 32))
    ws = ws.view(parts, -1)
    for junk in (0, 0x55, 0xff):          # what a replay finds there does not matter, and it clears no more than the flags
        ws.fill_(junk)
        g.replay()
        torch.cuda.synchronize()
        assert_same(out, want)
        # the counts start anew (two layers; the wide network's fifty positions are two launches), and nothing else was cleared
        assert bool((ws.view(torch.int32)[:, 0] <= 4).all()) and bool((ws[:, 2048:3072] == 0).all()) and bool((ws[:, -256:] == junk).all())


@pytest.mark.parametrize("shape,head,wdl", [("base", "king", False), ("base", "prenorm", True), ("wide", "king", True)])
def test_a_launch_that_gives_up_marks_its_outputs_and_is_reported(shape, head, wdl):
    # member 0 of every position counts ahead of the others: it waits for flags they do not raise in this launch, gives
    # up at the limit of its waiting, and the others, who need its pieces, do so too: the launch ends
    team, single = pair(shape, head=head, wdl=wdl)
    x = batch(3)
    want = [t.clone() for t in single.forward_masked(*x)]
    assert_same(team.forward_masked(*x), want)
    ws, = team._team.values()
    saved = ws.clone()
    ws.view(torch.int32).view(64 if shape == "base" else 32, -1)[:, 0] += 1000
    policy, promo, value, best = team.forward_masked(*x)
    torch.cuda.synchronize()
    legal = ((x[3].unsqueeze(-1) >> torch.arange(64, device="cuda")) & 1).bool()
    assert bool((best == -1).all()) and bool(value.isnan().all()) and bool(promo.isnan().all())
    assert bool(policy[legal].isnan().all()) and bool((policy[~legal] == float("-inf")).all())
    ws.copy_(saved)
    with pytest.raises(RuntimeError, match="gave up"):
        team.forward_masked(*x)
    assert_same(team.forward_masked(*x), want)                                 # reported once
    assert team._lib.bf_team_gave_up() == 0


@pytest.mark.parametrize("shape,start", [("base", 2 ** 31 - 5), ("base", 2 ** 32 - 5), ("wide", 2 ** 31 - 5)])
def test_the_count_of_layers_wraps(shape, start):
    team, single = pair(shape)
    x = batch(9)
    team.forward_masked(*x)
    ws, = team._team.values()
    flags = ws.view(torch.int32).view(64 if shape == "base" else 32, -1)[:, :768]     # the counts and the flags of every position
    flags.fill_(start if start < 2 ** 31 else start - 2 ** 32)
    want = [t.clone() for t in single.forward_masked(*x)]
    for i in range(6):           # two layers each: before, over and behind the wrap
        if i == 3:               # a launch that raises no flag of the heads
            assert_same(team.forward_full(*x[:3]), single.forward_full(*x[:3]))
        else:
            assert_same(team.forward_masked(*x), want)


def test_launch_form_names_the_form_that_runs():
    team, single = pair()
    assert [team.launch_form(n) for n in (1, 64, 65, 256, 257)] == ["team", "team", "octo", "octo", "duo"]
    assert single.launch_form(1) == "octo" and [team.kernel_choice(n) for n in (1, 65)] == ["octo", "octo"]
    wide, _ = pair("wide")
    assert [wide.launch_form(n) for n in (1, 32, 64, 65)] == ["team", "team", "team", "octo"]

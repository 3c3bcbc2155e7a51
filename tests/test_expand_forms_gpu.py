"""Edge rows in their different forms (whole 16-byte pieces, odd lengths, longer than the LDS row) and the
leaf compaction at the edges of its workgroups."""
import ctypes as C

import pytest
import torch

from brokefish_amd import positions
from brokefish_amd.hip_impl import compact_leaves, expand_edges, load_library, movegen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 7, 515])
@pytest.mark.parametrize("edges", [1, 8, 31, 32, 95, 128, 136, 255])
def test_edge_rows_do_not_depend_on_their_form(n, edges):
    b, c, r, m = (t.cuda() for t in positions.random_positions(n, plies=150, seed=n, stamp_queen=True))
    g = torch.Generator(device="cuda").manual_seed(n)
    logits = [torch.randn(n, 32, k, generator=g, device="cuda").half() for k in (64, 4)]
    value = torch.rand(n, generator=g, device="cuda")
    got = expand_edges(*logits, value, m, b, c, edges)
    full = expand_edges(*logits, value, m, b, c, 254)            # nothing truncated, rows stored edge by edge
    assert torch.equal(got["count"], full["count"]) and torch.equal(got["n_edges"], full["count"].clamp(max=edges))
    assert torch.equal(got["node_value"], full["node_value"])
    logp = full["edge_prior"].float()
    for i in range(min(n, 64)):
        k = int(full["count"][i])
        mine, prior = got["edge_move"][i].tolist(), got["edge_prior"][i].float()
        if k <= edges:
            assert mine[:k] == full["edge_move"][i, :k].tolist() and torch.equal(got["edge_prior"][i, :k], full["edge_prior"][i, :k])
            assert float(got["dropped"][i]) == 0.0 and not any(mine[k:]) and not prior[k:].any()
        else:
            at = [full["edge_move"][i, :k].tolist().index(x) for x in mine]
            assert at == sorted(at)                              # survivors in canonical order
            cut = logp[i, :k].sort(descending=True).values[edges - 1]
            assert float(logp[i, at].min()) >= float(cut) * (1 - 2e-3)
            assert abs(float(prior.sum()) - 1) < 5e-3
            assert abs(float(got["dropped"][i]) - (1 - float(logp[i, at].sum()) / float(logp[i, :k].sum()))) < 5e-3


def with_candidates(counts, seed):
    """Positions with legal-move words of so many set bits (arbitrary ones beyond chess), and logits with ties."""
    n = len(counts)
    b, c, _, _ = positions.random_positions(n, plies=150, seed=seed, stamp_queen=True)
    g = torch.Generator().manual_seed(seed)
    bits = torch.zeros(n, 2048, dtype=torch.int64)
    for i, k in enumerate(counts):
        bits[i, torch.randperm(2048, generator=g)[:k]] = 1
    m = (bits.view(n, 32, 64) << torch.arange(64)).sum(-1)
    logits = [(torch.randint(-24, 25, (n, 32, k), generator=g) / 8).half() for k in (64, 4)]
    return [t.cuda() for t in (*logits, torch.rand(n, generator=g), m, b, c)]


@pytest.mark.parametrize("edges", [32, 96, 100, 136])
@pytest.mark.parametrize("fp32", [False, True])
def test_edges_of_a_position_do_not_depend_on_its_neighbour(edges, fp32):
    counts = [0, 1, 31, 33, 90, 110, 128, 129, 160, 218, 230, 256, 257, 400]      # promotions add to some of them
    p, q, v, m, b, c = with_candidates(counts, 3)
    if fp32:
        p, q = p.float(), q.float()
    k = len(counts)
    alone = [expand_edges(p[i:i + 1], q[i:i + 1], v[i:i + 1], m[i:i + 1], b[i:i + 1], c[i:i + 1], edges) for i in range(k)]
    at = torch.cartesian_prod(torch.arange(k), torch.arange(k)).flatten().cuda()   # every position beside every other, on either side
    pairs = expand_edges(p[at], q[at], v[at], m[at], b[at], c[at], edges)
    for name, got in pairs.items():
        want = torch.cat([a[name] for a in alone])[at]
        assert torch.equal(got.view(torch.int16) if got.dtype is torch.float16 else got, want.view(torch.int16) if want.dtype is torch.float16 else want), name


@pytest.mark.parametrize("count", [40, 120, 200, 300])
def test_the_two_zeros_are_one_value_at_the_cut(count):
    # every log-prior is a zero of either sign: the cut falls among ties, which canonical order decides
    p, q, v, m, b, c = with_candidates([count] * 8, 5)
    b |= 0x40                                                   # no pawns (a promotion would split its move's mass)
    p = torch.where(torch.rand(p.shape, generator=torch.Generator().manual_seed(1)) < 0.5, -0.0, 0.0).half().cuda()
    got = expand_edges(p, q, v, m, b, c, 32)
    for i in range(8):
        bits = ((m[i].unsqueeze(-1) >> torch.arange(64, device="cuda")) & 1).flatten().nonzero().flatten()
        assert torch.equal(got["edge_move"][i].int(), bits[:32].int()) and torch.equal(got["edge_prior"][i].float(), torch.full((32,), 1 / 32, device="cuda"))


@pytest.mark.parametrize("n", [1, 15, 16, 17, 16383, 16384, 16385, 49999])
@pytest.mark.parametrize("shift", [0, 1])
def test_compaction_at_the_edges_of_its_workgroups(n, shift):
    g = torch.Generator(device="cuda").manual_seed(n)
    for share in (0.0, 0.4, 1.0):
        raw = torch.randint(1, 256, (n + shift,), generator=g, device="cuda").to(torch.uint8)
        raw[torch.rand(n + shift, generator=g, device="cuda") >= share] = 0
        flags = raw[shift:]                                      # shift 1: not aligned to sixteen bytes
        index, count = compact_leaves(flags)
        want = flags.nonzero().flatten().int()
        assert int(count) == want.numel() and torch.equal(index[:want.numel()], want) and not index[want.numel():].any()


@pytest.mark.parametrize("n", [1, 7, 1000])
def test_outputs_of_a_call_have_memory_of_their_own(n):
    b, c, _, m = (t.cuda() for t in positions.random_positions(n, plies=60, seed=1))
    logits = [torch.randn(n, 32, k, device="cuda").half() for k in (64, 4)]
    on = (torch.arange(n, device="cuda") % 2 == 0)
    outs = [dict(zip("mk", movegen(b, c)))]
    outs += [expand_edges(*logits, torch.rand(n, device="cuda"), m, b, c, 96, **kw) for kw in ({}, {"active": on}, {"leaves": compact_leaves(on)})]
    for out in outs:
        stores = [t.untyped_storage() for t in out.values()]
        assert len({s.data_ptr() for s in stores}) == len(stores)
        assert all(s.nbytes() == t.numel() * t.element_size() and t.storage_offset() == 0 for s, t in zip(stores, out.values()))
        if len(out) > 2 and out is not outs[1]:      # rows of skipped positions start at zero, the others' are the call's
            for name, t in out.items():
                assert not t[~on].any()
                if name != "node_value":             # (each call had values of its own)
                    assert torch.equal(t[on], outs[1][name][on])


@pytest.mark.parametrize("sizes", [(0, 1, 15, 16, 17), (16383, 16384, 16385), (4096 * 16 + 5, 3, 1 << 22)])
def test_clear_writes_its_buffers_and_no_more(sizes):
    room = [torch.full((s + 64,), 7, dtype=torch.uint8, device="cuda") for s in sizes]
    lib = load_library()
    at = (C.c_void_p * len(sizes))(*[t.data_ptr() for t in room])
    assert lib.bf_clear(at, (C.c_size_t * len(sizes))(*sizes), len(sizes), C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    for t, s in zip(room, sizes):
        assert not t[:s].any() and bool((t[s:] == 7).all())
    assert lib.bf_clear(at, (C.c_size_t * 9)(), 9, None) != 0


@pytest.mark.parametrize("n", [256 * 16384, 256 * 16384 + 1, 257 * 16384 - 5, 512 * 16384 + 40000])
def test_compaction_of_more_flags_than_its_workgroups_take_in_one_run(n):
    flags = (torch.rand(n, generator=torch.Generator(device="cuda").manual_seed(n), device="cuda") < 0.3).to(torch.uint8)
    flags[n // 3:n // 2] = 0                                     # workgroups without a live flag
    index, count = compact_leaves(flags)
    want = flags.nonzero().flatten().int()
    assert int(count) == want.numel() and torch.equal(index[:want.numel()], want) and not index[want.numel():].any()

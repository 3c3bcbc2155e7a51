"""bf_launch_form: what runs for given arguments, where the answer of bf_kernel_choice names the kernel whose launches those
are.  The library answers without a device; the forms' outputs are held against one another in the GPU tests."""
import ctypes
import importlib.util
import os
import re

import pytest

from brokefish_amd import hip_impl

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
QUAD, BOARD, TWIN, OCTO, DUO, TEAM, WIDE = range(1, 8)
BASE, BIG = (256, 8, 8, 1024), (512, 16, 16, 2048)


def args(shape, n, quant=0, kernel=0):
    a = hip_impl._Args()
    d, layers, heads, f = shape
    a.shape = hip_impl._Shape(d, layers, heads, f, 1, 1e-5)
    a.board_wstream = a.board_fparams = 16                     # only tested for NULL
    a.n, a.quant, a.kernel = n, quant, kernel
    return a


def form(a):
    return hip_impl.load_library().bf_launch_form(ctypes.byref(a))


@pytest.mark.parametrize("shape,quant,small,large", [(BASE, 0, OCTO, DUO), (BASE, 1, OCTO, DUO), (BIG, 0, OCTO, WIDE)])
def test_auto_by_size(shape, quant, small, large):
    for n, want in ((1, small), (256, small), (257, large), (512, large), (513, large), (16384, large)):
        assert form(args(shape, n, quant)) == want


@pytest.mark.parametrize("shape,quant,kernels", [(BASE, 0, (BOARD, TWIN, OCTO, DUO)), (BASE, 1, (BOARD, TWIN, OCTO, DUO)), (BIG, 0, (BOARD, OCTO))])
def test_a_kernel_asked_for_by_name_runs(shape, quant, kernels):
    for kernel in kernels:
        for n in (1, 300, 4096):
            assert form(args(shape, n, quant, kernel)) == kernel


def test_the_taps_of_the_wide_network_are_the_one_position_forms():
    a = args(BIG, 4096)
    taps = hip_impl._Taps()
    taps.resid = 16
    a.taps = ctypes.pointer(taps)
    assert form(a) == OCTO
    taps.resid, taps.alive = None, 16                          # the stack alone: a build of every form AUTO takes
    assert form(a) == WIDE


@pytest.mark.parametrize("shape,quant,want", [(BASE, 0, DUO), (BASE, 1, TWIN), (BIG, 0, OCTO)])
def test_flags_without_a_list_are_not_paired_where_a_pair_costs_more(shape, quant, want):
    for n in (257, 512, 4096):
        a = args(shape, n, quant)
        a.active = 16
        assert form(a) == want
        a.active, a.leaf_index, a.leaf_count = None, 16, 16        # a list: pairs of live ones
        assert form(a) in (DUO, WIDE)


def deep(shape, layers):
    return shape[:1] + (layers,) + shape[2:]


@pytest.mark.parametrize("shape,quant,most,small,large,deep_small,deep_large", [
    (BASE, 0, 10922, OCTO, DUO, BOARD, TWIN), (BASE, 1, 10922, OCTO, DUO, BOARD, TWIN), (BIG, 0, 2730, OCTO, WIDE, OCTO, OCTO)])
def test_networks_too_deep_for_32_bit_offsets(shape, quant, most, small, large, deep_small, deep_large):
    lib = hip_impl.load_library()
    for layers in (most, most + 1, 2 ** 28, 2 ** 31 - 1):
        fits = layers == most
        s = args(deep(shape, layers), 1).shape
        assert (lib.bf_board_wstream_bytes(ctypes.byref(s)) // 4 < 2 ** 31) == fits      # a quarter's stream
        for n in (1, 256, 257, 4096):
            want = (small if n <= 256 else large) if fits else (deep_small if n <= 256 else deep_large)
            assert form(args(deep(shape, layers), n, quant)) == want
        if shape is BASE:
            for kernel in (OCTO, DUO):
                assert form(args(deep(shape, layers), 300, quant, kernel)) == (kernel if fits else -2)
            for kernel in (BOARD, TWIN):
                assert form(args(deep(shape, layers), 300, quant, kernel)) == kernel


@pytest.mark.gpu
@pytest.mark.parametrize("shape,most,other", [(BASE, 2730, OCTO), (BIG, 682, OCTO)])
def test_teams_reach_all_four_quarters_by_32_bit_offsets(shape, most, other):
    lib = hip_impl.load_library()
    for layers, want in ((most, TEAM), (most + 1, other)):
        a = args(deep(shape, layers), 8)
        a.team_workspace, a.team_workspace_bytes = 256, lib.bf_team_workspace_bytes(ctypes.byref(a.shape))
        assert a.team_workspace_bytes and form(a) == want


def test_refused_arguments():
    assert form(args((384, 8, 12, 1536), 4)) == -2
    assert form(args(BIG, 4, quant=1)) < 0 and form(args(BASE, 4, kernel=7)) == -1
    assert hip_impl.load_library().bf_launch_form(None) == -1


def test_the_traffic_of_the_two_position_forms_is_quoted_from_their_profiles():
    spec = importlib.util.spec_from_file_location("bench_module", os.path.join(ROOT, "bench.py"))
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    where = {("base", "duo", 4096, "e4m3"): "duo_kernel_e4m3_batch4096.md", ("stress", "wide", 16384, "int8"): "wide_kernel_512_int8_batch16384.md"}
    assert set(where) == set(bench.MEASURED_TRAFFIC_BYTES_PAIRS)
    for key, name in where.items():
        text = open(os.path.join(ROOT, "profiles", name)).read()
        assert bench.MEASURED_TRAFFIC_BYTES_PAIRS[key] in {float(x) for x in re.findall(r"\d+(?:\.\d+)?e\d+", text)}, key

"""The rules that choose a call's kernel form (csrc/dispatch.hpp, built here
for the host exactly as the launchers include it)."""
import ctypes
import shutil
import subprocess
from collections import namedtuple
from pathlib import Path

import pytest
from scipy import stats

from test_gpu_grouped import WIDE_PLANS

ROOT = Path(__file__).resolve().parent
Plan = namedtuple("Plan", "tile_rows gate_up_shape down_shape glu chunk blocks stream")


def build_rules(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    so = tmp_path_factory.mktemp("dispatch") / "libdispatch.so"
    subprocess.run([gxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-o", str(so),
                    str(ROOT / "native" / "dispatch_host.cpp")], check=True)
    lib = ctypes.CDLL(str(so))
    lib.expected_tiles.argtypes = [ctypes.c_int64, ctypes.c_int32, ctypes.c_int]
    lib.expected_tiles.restype = ctypes.c_double
    lib.grouped_plan.argtypes = [ctypes.c_int64] + [ctypes.c_int32] * 4 + [ctypes.c_void_p]
    lib.gateup_four_in_flight.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int]
    return lib


def grouped_plan(rules, tokens, E, top_k, hidden, inter, tiled=True):
    out = (ctypes.c_int32 * 7)()
    rules.grouped_plan(tokens * top_k, E, hidden, inter, int(tiled), out)
    return Plan(*out)


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    return build_rules(tmp_path_factory)


@pytest.mark.parametrize("P,E", [(1, 256), (232, 256), (8168, 256), (32768, 256), (90, 4),
                                 (5000, 6), (900, 1)])
@pytest.mark.parametrize("rows", [16, 32, 64])
def test_expected_tiles_is_the_poisson_expectation(rules, P, E, rows):
    lam = P / E
    n = int(lam + 12 * lam ** 0.5 + 40)
    want = E * sum(stats.poisson.pmf(k, lam) * -(-k // rows) for k in range(n))
    assert rules.expected_tiles(P, E, rows) == pytest.approx(want, rel=1e-6)


# (hidden, inter, experts, rows of each) timed on MI355X, weights not in the
# caches: the streamed form by 3 % or more, or the wide one by 8 % or more
FEW_EXPERTS_STREAMED = [
    (2048, 512, 1, 64), (2048, 512, 1, 128), (2048, 512, 2, 48), (2048, 512, 2, 96),
    (2048, 512, 4, 48), (2048, 512, 6, 64), (2048, 512, 8, 18), (2048, 512, 8, 48),
    (4096, 384, 1, 256), (4096, 384, 4, 128), (4096, 384, 8, 64), (4096, 384, 12, 64),
    (4096, 384, 16, 18), (1024, 1024, 1, 64), (1024, 1024, 2, 64), (2560, 256, 1, 192),
    (2560, 256, 2, 64), (2560, 256, 12, 48), (8192, 2048, 1, 64), (8192, 2048, 1, 192),
    (8192, 2048, 4, 24), (1024, 1024, 2, 96), (1024, 1024, 8, 24), (2048, 512, 12, 24),
    (4096, 1024, 8, 24), (256, 128, 24, 64),
]
MANY_ITEMS_WIDE = [
    (2048, 512, 2, 512), (2048, 512, 4, 128), (2048, 512, 6, 96), (2048, 512, 8, 64),
    (2048, 512, 12, 32), (2048, 512, 16, 24), (2048, 512, 64, 32), (4096, 384, 8, 256), (4096, 384, 24, 48),
    (1024, 1024, 4, 64), (1024, 1024, 8, 128), (2560, 256, 16, 64), (8192, 2048, 2, 128),
    (8192, 2048, 6, 32), (2048, 512, 256, 40), (4096, 384, 256, 40),
]


@pytest.mark.parametrize("case", FEW_EXPERTS_STREAMED)
def test_few_experts_take_the_streamed_tiles(rules, case):
    H, I, E, rows = case
    assert grouped_plan(rules, rows * E, E, 1, H, I).tile_rows == 32


@pytest.mark.parametrize("case", MANY_ITEMS_WIDE)
def test_enough_items_take_the_wide_tiles(rules, case):
    H, I, E, rows = case
    assert grouped_plan(rules, rows * E, E, 1, H, I).tile_rows == 64


# (hidden, inter, experts, rows of each, tile order): timed slower on the wide
# tiles, evenly routed or by popularity, and faster
FEW_ROWS_STREAMED = [
    (2048, 512, 256, 18, True), (4096, 384, 192, 18, True), (1024, 512, 192, 18, True),
    (1024, 1024, 256, 18, True), (1024, 1024, 256, 24, True), (1024, 1024, 192, 24, True),
    (2048, 512, 256, 16, False), (1024, 1024, 256, 28, True), (1024, 512, 512, 24, True),
    (256, 512, 1000, 28, True), (768, 384, 512, 22, True), (512, 256, 1000, 24, True),
    (3072, 128, 128, 24, False), (4096, 128, 256, 31, True),
]
ENOUGH_ROWS_WIDE = [
    (2048, 512, 256, 20, True), (2048, 512, 64, 18, True), (512, 512, 256, 18, True),
    (2048, 512, 64, 22, True), (2048, 1024, 64, 22, True),
    (1024, 1024, 256, 32, True), (1024, 1024, 64, 24, True), (2048, 512, 256, 18, False),
    (1024, 512, 256, 22, True), (512, 512, 256, 22, True), (1024, 512, 1000, 22, False),
    (2560, 256, 64, 18, False), (1024, 1024, 256, 20, False), (2048, 512, 256, 31, False),
    (4096, 128, 128, 32, False), (3072, 128, 256, 21, True),
    (2304, 128, 128, 18, False),
]


@pytest.mark.parametrize("case", FEW_ROWS_STREAMED)
def test_few_rows_take_the_streamed_tiles(rules, case):
    H, I, E, rows, tiled = case
    assert grouped_plan(rules, rows * E, E, 1, H, I, tiled).tile_rows == 32


@pytest.mark.parametrize("case", ENOUGH_ROWS_WIDE)
def test_enough_rows_take_the_wide_tiles(rules, case):
    H, I, E, rows, tiled = case
    assert grouped_plan(rules, rows * E, E, 1, H, I, tiled).tile_rows == 64


@pytest.mark.parametrize("tiled", [False, True])
def test_wide_plans_of_the_gpu_cases(rules, tiled):
    for (T, E, K, H, I), want in WIDE_PLANS.items():
        p = grouped_plan(rules, T, E, K, H, I, tiled)
        assert (p.tile_rows, p.chunk, p.blocks) == (64, *want), (T, E, K, H, I)


# (hidden, inter, experts, tokens) of top-8 calls timed on MI355X: on 16-row
# tiles slower when a few experts take most picks (the first also when none
# do), and faster
FEW_ROWS_NOT_SMALL = [(4096, 384, 256, 96), (3072, 512, 256, 80), (2048, 1024, 256, 80),
                      (8192, 512, 128, 80), (2048, 512, 256, 188), (2048, 512, 128, 92),
                      (2048, 128, 1000, 500), (4096, 128, 1000, 250), (1024, 256, 1000, 730)]
FEW_ROWS_SMALL = [(2048, 512, 256, 29), (2048, 512, 256, 128), (2048, 512, 256, 160),
                  (1024, 1024, 256, 128), (2560, 512, 256, 58), (2560, 256, 256, 96),
                  (512, 128, 1000, 250), (2048, 256, 256, 96), (512, 512, 256, 188),
                  (256, 128, 1500, 1024)]


def test_sixteen_row_tiles(rules):
    rows = {c: grouped_plan(rules, c[3], c[2], 8, *c[:2]).tile_rows
            for c in FEW_ROWS_NOT_SMALL + FEW_ROWS_SMALL}
    assert [rows[c] for c in FEW_ROWS_NOT_SMALL] == [32] * len(FEW_ROWS_NOT_SMALL)
    assert [rows[c] for c in FEW_ROWS_SMALL] == [16] * len(FEW_ROWS_SMALL)


# the same in row order: uneven picks slower from 2.5 Mi of rows x hidden x inter
@pytest.mark.parametrize("case, want", [((2048, 512, 256, 90), 32), ((1536, 512, 128, 74), 32),
                                        ((2560, 512, 256, 91), 32), ((2048, 512, 256, 128), 32),
                                        ((2048, 512, 256, 64), 16), ((2048, 256, 256, 96), 16),
                                        ((1024, 512, 256, 128), 16)])
def test_sixteen_row_tiles_in_row_order(rules, case, want):
    H, I, E, T = case
    assert grouped_plan(rules, T, E, 8, H, I, False).tile_rows == want


def test_router_tiles(rules):
    """(experts, tokens) timed on MI355X, H 2048: slower with four tiles per
    workgroup (padded experts, CUs left idle at the end), and faster."""
    one = [(8, 16384), (16, 16384), (16, 65535), (33, 8192), (48, 8192), (48, 20000), (144, 4096),
           (256, 1500), (256, 64)]
    four = [(256, 2048), (256, 3000), (256, 4096), (128, 4096), (64, 8192), (32, 16384),
            (17, 65535), (96, 8192), (144, 8192), (512, 1500)]
    assert [rules.router_four_tiles(T, E) for E, T in one] == [0] * len(one)
    assert [rules.router_four_tiles(T, E) for E, T in four] == [1] * len(four)


def test_block_carries_the_shared_expert(rules):
    """(hidden, shared inter, tokens) timed on MI355X: carried by the decode
    launches where that is faster than the two shared-expert kernels after
    them, and always for one or two tokens."""
    carried = [(2048, 512, 3), (2048, 512, 16), (2048, 1024, 8), (2048, 2048, 4), (4096, 512, 11),
               (4096, 384, 12), (4096, 1024, 4), (8192, 128, 16), (8192, 8192, 2), (128, 128, 16)]
    after = [(2048, 1024, 16), (2048, 2048, 6), (2048, 4096, 4), (2048, 8192, 3), (4096, 512, 16),
             (4096, 1024, 6), (4096, 2048, 3), (8192, 2048, 3), (8192, 8192, 3), (2048, 512, 17)]
    assert [rules.block_carries_shared(T, H, Is) for H, Is, T in carried] == [1] * len(carried)
    assert [rules.block_carries_shared(T, H, Is) for H, Is, T in after] == [0] * len(after)


def test_gate_up_loads_in_flight(rules):
    """(hidden, inter, tokens, top-k inside) of top-8 calls timed on MI355X:
    faster with 8 K-blocks of weights in flight, and with 4."""
    eight = [(2048, 512, 8, 0), (2048, 512, 16, 0), (1920, 512, 12, 0), (2048, 512, 4, 1),
             (2560, 256, 4, 0), (8192, 512, 2, 1)]
    four = [(2048, 512, 8, 1), (2048, 512, 16, 1), (2560, 256, 12, 0), (4096, 384, 8, 0),
            (8192, 512, 16, 0), (1024, 512, 1, 0), (1024, 1024, 16, 1), (1280, 512, 12, 0),
            (1536, 512, 8, 0)]

    def rule(H, I, T, topk):
        return rules.gateup_four_in_flight((H // 128 + 1) // 2, I // 16 * T * 8, topk)

    assert [rule(*c) for c in eight] == [0] * len(eight)
    assert [rule(*c) for c in four] == [1] * len(four)

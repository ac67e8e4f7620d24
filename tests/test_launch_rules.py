"""The launch rules (csrc/launch_rules.hpp) against launches measured on MI355X, on the CPU: the header is compiled
with the host compiler.

Each row holds the microseconds of every shape a call could take; the rule's choice may not be slower than the narrow
kernel's launch by more than 4 % (the margin over what repeated runs differ by), nor than the best shape by 25 %."""
import ctypes
import os
import subprocess

import pytest

import test_gpu_moe_grouped as grouped
import test_gpu_prefill_wide as wide

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kriya-rt_amd", "csrc")
SOURCE = """
#include "launch_rules.hpp"
extern "C" int choice(uint32_t m, const uint32_t *ns, int np, uint32_t k, uint32_t max_split, int converted, uint32_t *split) {
    const kr::PrefillChoice c = kr::prefill_choice(m, ns, np, k, max_split, converted, 256);
    *split = c.ksplit;
    return c.shape;
}
extern "C" int loop_pays(uint32_t m, uint32_t n, uint32_t k) { return kr::slab_loop_pays(m, &n, 1, k, false, 256); }
extern "C" uint32_t loop_groups(uint32_t m, uint32_t n, uint32_t k, uint32_t option, uint32_t blocks) {
    return kr::slab_loop_groups(m, (n + 15) / 16, k, option, blocks);
}
extern "C" int grouped_pays(uint32_t assign, uint32_t experts, uint32_t hidden, uint32_t inter) {
    return kr::moe_grouped_pays(assign, experts, hidden, inter);
}
extern "C" int wide_tiles(uint32_t assign, uint32_t experts, uint32_t ntiles, int gate_up) {
    return kr::moe_wide_tiles(assign, experts, ntiles, gate_up, 256);
}
extern "C" int route_parts(uint32_t assign, uint32_t experts) { return kr::moe_route_parts(assign, experts); }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "r.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}", str(d / "r.cpp"), "-o",
                    str(d / "r.so")], check=True)
    return ctypes.CDLL(str(d / "r.so"))


def choose(rules, m, ns, k, max_split=1, converted=0):
    split = ctypes.c_uint32()
    shape = rules.choice(m, (ctypes.c_uint32 * len(ns))(*ns), len(ns), k, max_split, converted, ctypes.byref(split))
    return shape, split.value


NARROW, WIDE = 1, {42: 0, 22: 1, 21: 2}

# m, n, k: narrow; 128 x 256, 64 x 256, 64 x 128 tiles (us)
UNSPLIT = [
    ((63, 49152, 4096), 52.0, (69.7, 46.2, 46.5)),
    ((24, 49152, 11008), 128.1, (163.8, 126.2, 129.0)),
    ((64, 49152, 1024), 17.3, (21.7, 15.7, 15.6)),
    ((33, 49152, 2816), 36.6, (44.3, 31.6, 31.6)),
    ((64, 151936, 1024), 44.9, (52.5, 36.8, 36.1)),
    ((64, 151936, 3584), 142.9, (164.0, 123.0, 120.2)),
    ((100, 12288, 4096), 32.2, (60.6, 42.9, 34.6)),
    ((384, 4096, 4096), 32.0, (61.4, 43.1, 34.6)),
    ((640, 2048, 4096), 32.6, (62.2, 43.6, 35.3)),
    ((160, 2048, 2048), 11.8, (33.4, 22.1, 16.2)),
    ((128, 256, 11008), 46.6, (145.7, 95.5, 67.3)),
    ((63, 24576, 11008), 80.5, (153.1, 111.4, 94.2)),
    ((256, 1024, 8192), 36.2, (111.7, 75.5, 65.2)),
    ((320, 512, 2048), 11.5, (33.5, 22.2, 16.0)),
    ((1500, 8192, 8192), 379.5, (216.4, 225.9, 261.1)),
    ((1500, 4096, 3584), 87.9, (62.1, 65.3, 65.3)),
    ((448, 16384, 1536), 44.3, (33.1, 32.0, 35.8)),
    ((2048, 1024, 4096), 41.4, (64.0, 44.3, 36.5)),
    ((100, 2048, 256), 6.4, (10.7, 7.5, 5.6)),
    ((193, 512, 768), 7.4, (17.5, 11.5, 8.4)),
    ((640, 32000, 512), 73.7, (35.7, 33.4, 36.4)),
    ((100, 16384, 128), 9.0, (9.9, 7.3, 5.6)),
    ((256, 65536, 256), 57.4, (20.5, 20.5, 21.2)),
    ((256, 1024, 768), 8.1, (17.9, 12.1, 9.8)),
]


@pytest.mark.parametrize("shape,narrow,others", UNSPLIT)
def test_unsplit(rules, shape, narrow, others):
    m, n, k = shape
    s, split = choose(rules, m, [n], k)
    assert split == 1
    t = narrow if s == NARROW else others[WIDE[s]]
    assert t <= 1.04 * narrow and t <= 1.25 * min(narrow, *others), (s, t)


# m, n, k: narrow (its own split); the three wide shapes unsplit; 128 x 256 tiles in 2, 4, 8 K parts (us; 0: too short)
SPLIT = [
    ((192, 16384, 2048), 26.7, (35.3, 24.2, 25.1), (33.3, 39.1, 0)),
    ((64, 49152, 2816), 37.8, (45.1, 32.8, 32.8), (51.8, 59.2, 0)),
    ((128, 16384, 4096), 38.1, (61.5, 43.4, 35.6), (42.3, 38.3, 50.3)),
    ((320, 12288, 2816), 44.8, (44.4, 32.3, 34.1), (51.2, 57.2, 0)),
    ((127, 12288, 4096), 34.6, (61.2, 42.8, 34.4), (40.0, 33.2, 42.3)),
    ((65, 16384, 4096), 33.6, (59.9, 43.1, 34.8), (38.2, 32.2, 40.4)),
    ((193, 8192, 4096), 35.1, (60.7, 42.5, 33.7), (40.2, 33.8, 40.5)),
    ((2048, 512, 4096), 26.9, (61.7, 43.4, 35.0), (38.8, 32.0, 28.5)),
    ((2048, 1024, 8192), 62.3, (114.4, 79.9, 66.5), (70.7, 52.6, 58.3)),
    ((100, 1536, 18944), 39.6, (256.2, 181.4, 144.1), (135.1, 71.4, 44.2)),
    ((448, 49152, 2816), 214.5, (136.0, 151.0, 164.1), (182.1, 260.0, 0)),
    ((448, 8192, 4096), 61.3, (64.8, 46.8, 47.7), (51.9, 57.4, 78.5)),
    ((640, 3000, 18944), 107.9, (254.3, 180.1, 147.9), (137.8, 93.2, 95.2)),
    ((257, 512, 8192), 22.9, (111.6, 75.6, 53.2), (61.5, 36.8, 26.1)),
]


@pytest.mark.parametrize("shape,narrow,others,parts", SPLIT)
def test_with_room_for_partials(rules, shape, narrow, others, parts):
    m, n, k = shape
    s, split = choose(rules, m, [n], k, max_split=8)
    t = narrow if s == NARROW else others[WIDE[s]] if split == 1 else parts[{2: 0, 4: 1, 8: 2}[split]]
    best = min(v for v in (narrow, *others, *parts) if v)
    assert 0 < t <= 1.04 * narrow and t <= 1.25 * best, (s, split, t)


def test_converted_operand_takes_128_token_tiles(rules):
    """Of the wide shapes only 128 x 256 reads x as the fp16 operand; every K part keeps eight groups."""
    for m in (64, 100, 129, 640, 1024, 3907):
        for n, k in ((1024, 2816), (2048, 11008), (3584, 18944)):
            s, split = choose(rules, m, [n], k, max_split=8, converted=1)
            assert s in (NARROW, 42) and k // 64 // split >= 8


def test_gpu_tests_reach_the_wide_launches(rules):
    for (m, n, k), launch in wide.PLAIN_42:
        assert choose(rules, m, [n], k) == launch
    for (m, n, k), launch in wide.SPLIT_42:
        assert choose(rules, m, [n], k, max_split=8) == launch
    for (m, hidden, inter), launch in wide.MLP_DOWN:
        assert choose(rules, m, [hidden], inter, max_split=8, converted=1) == launch


def test_problems_add_up(rules):
    """Three projections of one x count as one launch: the tiles of all of them."""
    assert choose(rules, 512, [2048, 256, 256], 2048) == choose(rules, 512, [2560], 2048)


# m, n, k: the slab loop, the prefill launch these sizes take otherwise (us)
LOOP = [
    ((17, 65536, 3072), 61.9, 37.2), ((24, 65536, 3072), 51.2, 37.4), ((32, 49152, 3072), 41.3, 34.9), ((17, 49152, 3072), 48.6, 34.7),
    ((27, 2048, 11008), 20.5, 46.0), ((63, 2048, 11008), 27.7, 46.0), ((17, 8192, 18944), 66.2, 81.0), ((20, 32768, 8192), 59.0, 77.4),
    ((63, 32768, 8192), 95.9, 76.9), ((48, 49152, 8192), 167.4, 99.8), ((17, 3072, 2304), 10.3, 14.7), ((49, 2048, 2304), 10.6, 14.7),
]


@pytest.mark.parametrize("shape,loop,prefill", LOOP)
def test_slab_loop_where_it_pays(rules, shape, loop, prefill):
    assert bool(rules.loop_pays(*shape)) == (loop < prefill)


def test_slab_loop_groups_follow_the_options(rules):
    """KR_OPT_SKINNY_GROUPS = 1 keeps 16-row groups, and the choice is made for KR_OPT_SKINNY_MAX_BLOCKS' grid."""
    assert rules.loop_groups(32, 65536, 3072, 2, 256) == 2 and rules.loop_groups(32, 65536, 3072, 1, 256) == 1
    assert rules.loop_groups(16, 65536, 3072, 2, 256) == 1
    assert rules.loop_groups(27, 2048, 11008, 2, 256) == 1 and rules.loop_groups(27, 2048, 11008, 2, 64) == 2


# experts, tokens per expert, hidden, inter: the few-token kernel's time over the grouped products' (the routed stage)
GROUPED = [
    ((8, 10, 2048, 1408), 0.82), ((8, 12, 2048, 1408), 0.86), ((8, 20, 2048, 1408), 1.18), ((4, 16, 2048, 1408), 0.85),
    ((4, 20, 2048, 1408), 0.94), ((4, 32, 2048, 1408), 1.11), ((2, 32, 2048, 1408), 0.92), ((16, 10, 2048, 1408), 0.81),
    ((16, 16, 2048, 1408), 1.2), ((60, 8, 2048, 1408), 0.80), ((60, 12, 2048, 1408), 1.08), ((32, 10, 2048, 1408), 0.82),
    ((128, 8, 2048, 768), 0.95), ((128, 12, 2048, 768), 1.27), ((64, 10, 2048, 768), 1.24), ((16, 12, 1024, 512), 1.25),
    ((32, 10, 1024, 512), 1.3), ((8, 16, 1024, 2048), 1.15), ((8, 10, 1024, 2048), 0.9), ((60, 10, 1152, 640), 1.45),
]


@pytest.mark.parametrize("routing,ratio", GROUPED)
def test_grouped_products_where_they_pay(rules, routing, ratio):
    experts, per, hidden, inter = routing
    assert bool(rules.grouped_pays(experts * per, experts, hidden, inter)) == (ratio > 1)


# experts, tokens per expert, tiles side by side, gate/up: the 96-token tiles' time over the 32-token tiles'
TILES = [
    ((4, 64, 22, 1), 1.15), ((8, 40, 22, 1), 0.89), ((8, 96, 8, 1), 1.18), ((32, 28, 8, 1), 0.93), ((16, 128, 8, 1), 0.92),
    ((32, 20, 22, 1), 1.07), ((60, 40, 22, 1), 0.79), ((4, 256, 12, 1), 0.98), ((1, 160, 32, 1), 1.18), ((16, 28, 16, 0), 0.91),
    ((8, 40, 16, 0), 1.04), ((4, 80, 16, 0), 1.11), ((60, 32, 16, 0), 0.93), ((8, 128, 16, 0), 0.91), ((2, 160, 16, 0), 1.10),
    ((8, 28, 32, 1), 0.9), ((8, 64, 16, 0), 0.93), ((8, 25, 32, 1), 0.95),
]


@pytest.mark.parametrize("launch,ratio", TILES)
def test_wide_tiles_where_they_pay(rules, launch, ratio):
    experts, per, ntiles, gate_up = launch
    wide = bool(rules.wide_tiles(experts * per, experts, ntiles, gate_up))
    assert (ratio if wide else 1 / ratio) <= 1.04


def test_gpu_tests_reach_the_wide_tiles(rules):
    down = []
    for pattern, times, hidden, inter in grouped.WIDE_TILES:
        experts, assign = len(pattern) * times, sum(pattern) * times
        assert rules.grouped_pays(assign, experts, hidden, inter)
        assert rules.wide_tiles(assign, experts, inter // 64, 1)
        down.append(bool(rules.wide_tiles(assign, experts, -(-hidden // 128), 0)))
    assert down == [True, True, False]


@pytest.mark.parametrize("experts,assign,passes,parts", [
    (8, 256, 3.35, 3.65), (8, 320, 3.48, 3.71), (4, 384, 3.67, 3.77), (8, 1024, 4.92, 4.15), (16, 768, 4.52, 3.93), (32, 512, 5.03, 3.74),
    (60, 256, 4.92, 3.63), (128, 128, 4.87, 3.63), (256, 65, 5.75, 3.72), (16, 128, 3.09, 3.62)])
def test_route_parts_where_they_pay(rules, experts, assign, passes, parts):
    assert bool(rules.route_parts(assign, experts)) == (parts < passes)

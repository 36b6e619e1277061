"""CPU: which kernel and tile a dense product takes (csrc/dense_plan.h, which the library asks, compiled for the host)."""
import os
import random
import shutil
import subprocess

import pytest

import test_gpu_dense_once as steps

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
UNITS = 256
BF16, F32 = 2, 4
# tokens, weight rows of a tile; the fifth has k divided in four
TILES = [(64, 64), (128, 64), (128, 128), (256, 256), (32, 64), (256, 192), (128, 192), (128, 128)]
K4 = 4


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    exe = str(tmp_path_factory.mktemp("plan") / "plan")
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "skainet_amd", "csrc"), "-o", exe,
                    os.path.join(ROOT, "tests", "c", "dense_plan.cpp")], check=True)

    def ask(what, questions):
        text = "".join(" ".join(map(str, (what, *q))) + "\n" for q in questions)
        lines = subprocess.run([exe], input=text, capture_output=True, text=True, timeout=100, check=True).stdout.split("\n")[:-1]
        assert len(lines) == len(questions)
        return [tuple(map(int, line.split())) for line in lines]

    return ask


def _tiles(plan, shapes):
    return [t for t, in plan("tile", [(*s, UNITS) for s in shapes])]


def _busiest(tile, m, rows):
    """outputs of the compute unit that has the most"""
    a, w = TILES[tile]
    return -(-(-(-m // a) * -(-rows // w)) // UNITS) * a * w


# fp32, whose loop is all of a product's time, and bf16 rows of less than 512 elements, which the costs in us were not fitted to
@pytest.mark.parametrize("size,longest", [(F32, 10240), (BF16, 448)])
def test_where_the_loop_is_all_no_compute_unit_has_much_more_than_it_must(plan, size, longest):
    rng = random.Random(size)
    shapes = [(size, rng.randint(1, 4096), 32 * rng.randint(1, 800), 64 * rng.randint(1, longest // 64)) for _ in range(3000)]
    for (_, m, rows, k), tile in zip(shapes, _tiles(plan, shapes)):
        if tile != K4:
            assert _busiest(tile, m, rows) <= 1.5 * min(_busiest(t, m, rows) for t in range(len(TILES)) if t != K4), (m, rows, k, tile)


# (measured, us: 1000 x 8512 x 2048 in fp32 339 on 64 x 64 and 515 on 256 x 256, see csrc/dense_plan.h)
@pytest.mark.parametrize("shape,tile", [((F32, 1000, 8512, 2048), 0), ((F32, 954, 8512, 2048), 0), ((F32, 512, 18496, 2048), 1), ((F32, 1700, 10752, 2048), 2),
                                        ((F32, 2048, 10752, 2048), 2), ((BF16, 1000, 8512, 256), 0), ((BF16, 954, 8512, 448), 0), ((BF16, 1700, 10752, 256), 2)])
def test_fp32_and_short_rows(plan, shape, tile):
    assert _tiles(plan, [shape]) == [tile]


# one measured shape for each tile that is the fastest of all there (profiles/dense_gemm_tiles.md), and those of test_gpu_dense_split.py
@pytest.mark.parametrize("m,rows,k,tile", [(333, 5120, 512, 0), (200, 5120, 4096, 1), (2048, 4096, 8192, 2), (1500, 8192, 4096, 3), (512, 18496, 4096, 5),
                                           (512, 10752, 4096, 6), (512, 8192, 8192, 7), (2048, 2048, 4160, 7), (1000, 2048, 4160, 1), (100, 2048, 4160, K4),
                                           (2048, 4224, 2048, 5), (1000, 4224, 2048, 2), (100, 4224, 2048, 0),
                                           (2048, 4096, 10240, 2), (2048, 4096, 18432, 2), (4096, 2048, 10240, 2), (8192, 4096, 8192, 3), (4096, 6432, 8192, 3),
                                           (1000, 10752, 10240, 6), (512, 18496, 14336, 5), (2048, 2048, 10240, 7)])
def test_bf16_by_the_fitted_costs(plan, m, rows, k, tile):
    assert _tiles(plan, [(BF16, m, rows, k)]) == [tile]


# 32 x 64 tiles with k divided in four: up to half of the compute units with rows of eight slices of 128 bytes, all of them with sixteen
@pytest.mark.parametrize("size", [BF16, F32])
@pytest.mark.parametrize("slices,rows", [(8, 8192), (15, 8192), (16, 16384), (64, 16384)])
def test_few_outputs(plan, size, slices, rows):
    k = slices * 128 // size
    at, past, wide = _tiles(plan, [(size, 32, rows, k), (size, 32, rows + 32, k), (size, 33, rows, k)])
    assert at == K4 and past != K4 and wide != K4
    assert _tiles(plan, [(size, 32, 64, 7 * 128 // size)]) != [K4]


def test_pitches_whose_tiles_need_more_than_32_bit_offsets_are_refused(plan):
    """(the kernel's offsets from a tile's first row: 255 rows and the row's own bytes)"""
    for size in (BF16, F32):
        most = (2**31 - 1) // (256 * size)
        assert plan("pitch", [(size, 64), (size, 40064), (size, most), (size, most + 1)]) == [(1,), (1,), (1,), (0,)]


PLAIN, NORM, MERGE, ADD_NORM = range(4)
STAGED = (0, 0, 0)


def _once(plan, mode=PLAIN, size=BF16, rows=2048, k=2048, ld=None, groups=1, dim=128, splits=8, second=False, segments=(0,)):
    return plan("once", [(mode, size, rows, k, ld or k, k, groups, dim, splits, int(second), UNITS, len(segments), *segments)])[0]


# a workgroup of the kernel that asks for everything at once has whole rows of one segment, and the segments cover the rows from the first on
@pytest.mark.parametrize("mode", [PLAIN, NORM, MERGE, ADD_NORM])
@pytest.mark.parametrize("rows,segments", [(2048 + 16, (0,)), (2048 + 1, ()), (2048, (32,)), (2048, (0, 1000)), (2048, (16, 1024)), (2048, (0, 1024, 512)), (2048, (0, 0))])
def test_rows_that_are_not_stacked_as_projections_are_staged(plan, mode, rows, segments):
    assert _once(plan, mode, rows=2048, segments=(0, 32, 1024)) != STAGED and _once(plan, mode, rows=2048, segments=()) != STAGED
    assert _once(plan, mode, rows=rows, segments=segments) == STAGED


@pytest.mark.parametrize("size", [BF16, F32])
def test_rows_of_a_workgroup_divide_the_padding(plan, size):
    calls = [(mode, size, rows, k, k, k, 1, 128, 8, 0, UNITS, 1, 0) for mode in (PLAIN, NORM, MERGE, ADD_NORM) for rows in (32, 512, 2624, 8192, 32000)
             for k in range(64, 40000, 192)]
    for call, (parts, pieces, r) in zip(calls, plan("once", calls)):
        if (parts, pieces, r) != STAGED:
            assert 32 % r == 0 and parts <= (16 if call[0] == PLAIN else 8) and parts * pieces * 1024 >= call[3] * size


# Rows of a workgroup at the rules' edges, each side the faster one of what was measured (profiles/dense_matvec_once.md).
@pytest.mark.parametrize("mode,size,rows,k,splits,r", [
    (PLAIN, BF16, 512, 4096, 1, 2), (PLAIN, BF16, 544, 4096, 1, 4), (PLAIN, BF16, 4096, 512, 1, 8), (PLAIN, BF16, 4096, 8192 + 64, 1, 4), (PLAIN, BF16, 32, 32768 + 64, 1, 0),
    (NORM, BF16, 64, 2048, 1, 2), (NORM, BF16, 2048, 2048, 1, 8), (NORM, BF16, 4096, 2048, 1, 16), (NORM, BF16, 4096, 4096, 1, 16), (NORM, BF16, 4096, 4096 + 64, 1, 0),
    (NORM, BF16, 12000, 3072, 1, 16), (NORM, F32, 8192, 1536, 1, 16), (NORM, F32, 12000, 1536, 1, 8), (NORM, F32, 4096, 2048 + 64, 1, 0),
    (ADD_NORM, BF16, 8192, 2048, 1, 16), (ADD_NORM, BF16, 9600, 2048, 1, 0), (ADD_NORM, BF16, 13312, 1536, 1, 0), (ADD_NORM, BF16, 16384, 1024, 1, 16),
    (ADD_NORM, BF16, 5632, 4096, 1, 8), (ADD_NORM, BF16, 5664, 4096, 1, 0), (ADD_NORM, F32, 9600, 1024, 1, 8), (ADD_NORM, F32, 12000, 1024, 1, 0),
    (MERGE, BF16, 1024, 2048, 8, 4), (MERGE, BF16, 5120, 2048, 8, 8), (MERGE, BF16, 5152, 2048, 8, 0), (MERGE, BF16, 5120, 2048, 9, 0), (MERGE, BF16, 5120, 1536, 16, 8),
    (MERGE, BF16, 2624, 3072, 16, 0), (MERGE, BF16, 8192, 1024, 16, 8), (MERGE, BF16, 2048, 4096 + 128, 8, 0)])
def test_rows_of_a_workgroup(plan, mode, size, rows, k, splits, r):
    assert _once(plan, mode, size, rows, k, splits=splits)[2] == r


def test_what_only_the_staged_kernel_takes(plan):
    assert _once(plan, PLAIN, second=True) == STAGED
    assert _once(plan, NORM, groups=8)[2] and _once(plan, NORM, k=2304, groups=9) == STAGED
    assert _once(plan, NORM, k=2064, groups=4) == STAGED and _once(plan, NORM, F32, k=2064 - 16, groups=4)[2]  # (516 elements: no whole requests of eight)
    assert _once(plan, MERGE, dim=20, k=640) == STAGED and _once(plan, MERGE, F32, dim=20, k=640)[2]
    assert _once(plan, PLAIN, ld=1 << 29) == STAGED


def _pad(n, to):
    return -(-n // to) * to


@pytest.mark.parametrize("size", [BF16, F32])
def test_what_the_decode_steps_of_the_gpu_tests_reach(plan, size):
    """The lists of test_gpu_dense_once.py have every form of the kernel that asks for everything at once, and the staged one for each input."""
    def forms(mode, products, **how):
        out = set()
        for n, k, groups, dim, splits in products:
            parts, pieces, r = _once(plan, mode, size, _pad(n, 32), _pad(k, 64), groups=groups, dim=dim, splits=splits)
            out.add((pieces, r) if mode == PLAIN else (min(s for s in (2, 4, 8, 16) if splits <= s), r) if mode == MERGE and r else r)
        return out

    rows = {0, 2, 4, 8, 16}
    assert forms(PLAIN, [(w, ff, 1, 1, 1) for w, ff, _ in steps.WIDTHS] + [(min(w, 100), w, 1, 1, 1) for w, _, _ in steps.WIDTHS]) >= {(1, 2), (1, 4), (1, 8), (2, 4), (4, 4)}
    assert forms(ADD_NORM, [(v, w, 1, 1, 1) for w, _, v in steps.WIDTHS]) >= rows
    assert forms(NORM, [(ff, w, 1, 1, 1) for w, ff, _ in steps.WIDTHS]) >= rows
    assert forms(NORM, [(v, w, g, 1, 1) for w, g, v in steps.GROUPS]) >= rows
    merged = [(w, h * d, 1, d, s) for h, _, d, w, _, s in steps.MERGES if s > 1]
    assert forms(MERGE, merged) >= {0, (2, 4), (4, 4), (4, 8), (8, 4), (16, 4), (16, 8)}

"""Which blocks and k splits the large-M projections take (csrc/mm_choice.hpp), on the CPU: the header is host code,
compiled with g++ and run for given widths."""

from __future__ import annotations

import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
OPROJ, GATE_UP, DOWN = 1, 2, 3
# MmId
LDS_64x128, LDS_64x256, LDS_128x256, LDS_128x192, WR_128x256, WR_64x128, WR_128x128, WR_64x64, WR_128x192 = 0, 2, 3, 4, 5, 6, 7, 8, 9
LDS_128x192_8W, LDS_256x192, WK_64, WK_96, WK_128 = 10, 11, 12, 13, 14

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ is not available")


@pytest.fixture(scope="module")
def runs(tmp_path_factory):
    """runs(cfg, rows of the weight, its columns): [(first row count, last, kernel, k splits), ...] of 33 to 8192."""
    exe = tmp_path_factory.mktemp("mm") / "mm_choice_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", str(ROOT / "fast-dllm-relax_amd" / "csrc"),
                    str(ROOT / "tests" / "mm_choice_check.cpp"), "-o", str(exe)], check=True)

    def get(cfg, n, k, cus=256):
        tiles = -(-n // 16 // 12) * 12 if cfg == GATE_UP else n // 16  # (packed in whole workgroups of 12 tiles)
        out = subprocess.run([str(exe), str(cfg), str(tiles), str(k // 32), str(cus)], capture_output=True, text=True, check=True)
        return [tuple(int(x) for x in line.split()) for line in out.stdout.splitlines()]

    return get


def at(table, rows):
    return next((kernel, splits) for first, last, kernel, splits in table if first <= rows <= last)


def test_1p5b_choices(runs):
    """The choices at the 1.5B widths, whose times stand beside them in mm_choice.hpp."""
    assert runs(OPROJ, 1536, 1536) == [
        (33, 64, WR_64x64, 2), (65, 512, WR_64x64, 1), (513, 1344, WR_64x128, 1), (1345, 2688, LDS_64x128, 1),
        (2689, 8192, WR_128x192, 1)]
    assert runs(GATE_UP, 17920, 1536) == [
        (33, 64, WK_64, 1), (65, 96, WK_96, 1), (97, 128, WK_128, 1), (129, 224, WR_64x128, 1), (225, 384, WR_128x128, 1),
        (385, 512, LDS_256x192, 1), (513, 640, LDS_128x192_8W, 1), (641, 896, WR_128x256, 1), (897, 2047, LDS_128x192_8W, 1),
        (2048, 8192, WR_128x256, 1)]
    assert runs(DOWN, 1536, 8960) == [
        (33, 128, WR_64x128, 7), (129, 256, WR_64x128, 5), (257, 320, WR_64x128, 4), (321, 384, LDS_128x192, 8),
        (385, 416, LDS_128x192, 7), (417, 512, WR_128x128, 5), (513, 640, WR_128x128, 4), (641, 768, WR_128x192, 5),
        (769, 1024, WR_128x192, 4), (1025, 1280, WR_128x256, 4), (1281, 1536, LDS_128x192, 4), (1537, 1664, WR_128x192, 4),
        (1665, 2048, WR_128x192, 2), (2049, 2688, WR_128x256, 2), (2689, 3200, LDS_128x192, 2), (3201, 3456, WR_128x192, 2),
        (3457, 8192, WR_128x192, 1)]


def test_gate_up_blocks_follow_their_count(runs):
    """gate_up takes register-weight 128 x 256 blocks below 2048 rows where they fill one round of two workgroups per
    compute unit, whatever the width and the device."""
    for n, k, rows in [(9728, 896, (641, 700, 896, 1200)), (5632, 1024, (641, 800, 896)), (11264, 2048, (641, 700, 800, 896)),
                       (22016, 2048, (641, 700, 896)), (2304, 640, (641, 700, 896))]:
        for r in rows:
            assert at(runs(GATE_UP, n, k), r)[0] == LDS_128x192_8W, (n, k, r)
    for n, k, rows in [(9728, 896, (1281, 1600)), (11264, 2048, (1100, 1400)), (22016, 2048, (513, 640))]:
        for r in rows:
            assert at(runs(GATE_UP, n, k), r)[0] == WR_128x256, (n, k, r)
    assert at(runs(GATE_UP, 22016, 2048), 300)[0] == LDS_256x192  # 519 blocks of 128 x 128
    assert at(runs(GATE_UP, 17920, 1536, cus=128), 700)[0] == LDS_128x192_8W


def test_o_proj_blocks_follow_their_count(runs):
    """o_proj keeps the register-weight 64 x 128 blocks while they are one round, at any width, and leaves the LDS-
    staged ones only when those pass two workgroups per compute unit."""
    for n, last in [(640, 3264), (896, 2304), (1024, 2048), (1536, 1344), (2048, 1024)]:
        table = runs(OPROJ, n, n)
        assert at(table, last)[0] == WR_64x128 and at(table, last + 1)[0] == LDS_64x128, n


def test_down_blocks_follow_their_count(runs):
    """down's large blocks and their one-round splits where the splits fill the round (or take over half of it against the
    LDS-staged 64 x 256 blocks), with at least 16 stages each; past that the splits of the other kernels."""
    # short weights: no round to fill, or only with splits of 9 or 11 stages
    for r in (450, 660, 1100, 1400):
        assert at(runs(DOWN, 640, 1152), r)[0] in (LDS_64x128, LDS_64x256), r
    for r in (450, 660, 800, 1024):
        assert at(runs(DOWN, 1024, 2816), r)[0] in (LDS_64x128, LDS_64x256), r
    assert at(runs(DOWN, 1024, 2816), 1100) == (WR_128x256, 4)
    # from 2048 rows on, widths without 192-column blocks keep the splits that more than one round takes
    assert at(runs(DOWN, 896, 4864), 2300) == (WR_128x256, 4) and at(runs(DOWN, 2048, 11008), 2300) == (WR_128x256, 2)
    for n, k in [(896, 4864), (2048, 5632), (2048, 11008)]:
        assert at(runs(DOWN, n, k), 700)[0] == WR_128x256 and at(runs(DOWN, n, k), 1500)[0] == WR_128x256, (n, k)


def test_down_splits_of_short_calls(runs):
    """down's 64 x 128 blocks take up to seven splits; eight where none of five to seven divides the k stages and four
    leave units idle or splits long."""
    for k, rows, splits in [(8960, 64, 7), (11008, 64, 8), (11008, 128, 8), (5632, 64, 8), (5632, 128, 4), (11008, 160, 4)]:
        n = 1536 if k == 8960 else 2048
        assert at(runs(DOWN, n, k), rows) == (WR_64x128, splits), (k, rows)
    assert at(runs(DOWN, 896, 4864), 40) == (WR_64x128, 8)

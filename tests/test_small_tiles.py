"""The rules that pick a W4A16, fp8 or plain-product tile (tilebench_amd/csrc/small_plan.h): the sizes
of the GPU parity tests run the tile they are listed under."""
import os
import shutil
import subprocess

import pytest

from small_tile_cases import DECODE_PLANS, DENSE_TILE_IDS, DENSE_TILES, EXPERT_TILE_IDS, EXPERT_TILES, FP8_TILE_IDS, FP8_TILES, NT_TILE_IDS, NT_TILES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _build(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "small_plan_pick")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "tilebench_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "small_plan_pick.cpp"), "-o", exe], check=True)
    return exe


def test_expert_tiles_picked(tmp_path):
    exe = _build(tmp_path)
    cases = [(tile, sum(rows), len(rows), N) for tile, cs in EXPERT_TILES.items() for rows, N, _, _ in cs]
    args = [str(x) for _, *c in cases for x in c]
    got = subprocess.run([exe, *args], check=True, capture_output=True, text=True).stdout.split()
    assert [int(g) for g in got] == [EXPERT_TILE_IDS[c[0]] for c in cases]


def test_dense_tiles_picked(tmp_path):
    exe = _build(tmp_path)
    cases = [(tile, M, 0, N) for tile, cs in DENSE_TILES.items() for M, _, N, _ in cs]
    args = [str(x) for _, *c in cases for x in c]
    got = subprocess.run([exe, *args], check=True, capture_output=True, text=True).stdout.split()
    assert [int(g) for g in got] == [DENSE_TILE_IDS[c[0]] for c in cases]


def test_fp8_tiles_picked(tmp_path):
    exe = _build(tmp_path)
    cases = [(tile, M, -K - blk, N) for tile, cs in FP8_TILES.items() for M, N, K in cs for blk in (0, 1)]
    args = [str(x) for _, *c in cases for x in c]
    got = subprocess.run([exe, *args], check=True, capture_output=True, text=True).stdout.split()
    assert [int(g) for g in got] == [FP8_TILE_IDS[c[0]] for c in cases]


def test_plain_product_tiles_picked(tmp_path):
    exe = _build(tmp_path)
    cases = [(tile, M, -10 ** 9 - Kb, N) for tile, cs in NT_TILES.items() for M, N, Kb in cs]
    args = [str(x) for _, *c in cases for x in c]
    got = subprocess.run([exe, *args], check=True, capture_output=True, text=True).stdout.split()
    assert [int(g) for g in got] == [NT_TILE_IDS[c[0]] for c in cases]


def test_decode_plans_picked(tmp_path):
    """The listed plans, and for other sizes and CU counts the bounds that the
    kernel and its scratch rely on."""
    exe = _build(tmp_path)

    def picks(cases):
        args = [str(x) for cus, K, N in cases for x in (cus, -2 * 10 ** 9 - K, N)]
        out = subprocess.run([exe, *args], check=True, capture_output=True, text=True).stdout.split()
        return [(int(g) // 1000, int(g) % 1000) for g in out]

    listed = [(plan, 256, K, N) for plan, cs in DECODE_PLANS.items() for N, K in cs]
    assert picks([c[1:] for c in listed]) == [c[0] for c in listed]
    cases = [(cus, K, N) for cus in (1, 64, 256, 304) for K in (64, 192, 256, 1024, 7168, 32768)
             for N in (8, 128, 1000, 4096, 32768, 32776, 65536)]
    for (cus, K, N), (cols, splits) in zip(cases, picks(cases)):
        slabs = -(-N // cols)
        assert cols in (128, 256) and 1 <= splits <= 16
        assert splits == 1 or (slabs * splits <= cus and splits * 8 <= K // 32)

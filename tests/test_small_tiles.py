"""The rules that pick a W4A16, fp8 or plain-product tile (tilebench_amd/csrc/small_plan.h): the sizes
of the GPU parity tests run the tile they are listed under."""
import os
import shutil
import subprocess

import pytest

from small_tile_cases import (DECODE_PLANS, DENSE_TILE_IDS, DENSE_TILES, DOWN_TILES, EXPERT_TILE_IDS, EXPERT_TILES,
                              FP8_TILE_IDS, FP8_TILES, GATE_UP_TILES, NT_TILE_IDS, NT_TILES)

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _build(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path / "small_plan_pick")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "tilebench_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "small_plan_pick.cpp"), "-o", exe], check=True)
    return exe


def _picks(exe, groups):
    """The numbers that each (rule, a, b, c) prints."""
    args = [str(x) for g in groups for x in g]
    out = subprocess.run([exe, *args], check=True, capture_output=True, text=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


def test_expert_tiles_picked(tmp_path):
    cases = [(tile, sum(rows), len(rows), N) for tile, cs in EXPERT_TILES.items() for rows, N, _, _ in cs]
    got = _picks(_build(tmp_path), [("expert", *c) for _, *c in cases])
    assert [g for g, in got] == [EXPERT_TILE_IDS[c[0]] for c in cases]


def test_gate_up_and_down_tiles_picked(tmp_path):
    """Each tile once with 16-byte and once with 4-byte weight loads."""
    exe = _build(tmp_path)
    for cases, columns in ((GATE_UP_TILES, 2), (DOWN_TILES, 1)):
        assert set(cases) == {(t, w) for t in EXPERT_TILE_IDS for w in (True, False)}
        got = _picks(exe, [("expert", T * k, E, columns * n) for T, E, k, _, n, _ in cases.values()])
        assert [g for g, in got] == [EXPERT_TILE_IDS[t] for t, _ in cases]
        assert [n % 32 == 0 for *_, n, _ in cases.values()] == [w for _, w in cases]


def test_dense_tiles_picked(tmp_path):
    cases = [(tile, M, N) for tile, cs in DENSE_TILES.items() for M, _, N, _ in cs]
    got = _picks(_build(tmp_path), [("dense", M, N, 0) for _, M, N in cases])
    assert [g for g, in got] == [DENSE_TILE_IDS[c[0]] for c in cases]


def test_fp8_tiles_picked(tmp_path):
    cases = [(tile, rule, *c) for tile, cs in FP8_TILES.items() for c in cs for rule in ("fp8", "fp8b")]
    got = _picks(_build(tmp_path), [c for _, *c in cases])
    assert [g for g, in got] == [FP8_TILE_IDS[c[0]] for c in cases]


def test_plain_product_tiles_picked(tmp_path):
    cases = [(tile, *c) for tile, cs in NT_TILES.items() for c in cs]
    got = _picks(_build(tmp_path), [("nt", *c) for _, *c in cases])
    assert [g for g, in got] == [NT_TILE_IDS[c[0]] for c in cases]


def test_decode_plans_picked(tmp_path):
    """The listed plans, and for other sizes and CU counts the bounds that the
    kernel and its scratch rely on."""
    exe = _build(tmp_path)
    listed = [(plan, N, K) for plan, cs in DECODE_PLANS.items() for N, K in cs]
    assert [g[:2] for g in _picks(exe, [("decode", 256, N, K) for _, N, K in listed])] == [c[0] for c in listed]
    cases = [(cus, N, K) for cus in (1, 64, 256, 304) for K in (64, 192, 256, 1024, 7168, 32768)
             for N in (8, 128, 1000, 4096, 32768, 32776, 65536)]
    # pairs of 128-column slabs that do not divide over the 8 XCDs: five splits of 26 pairs
    # would be 34 blocks on some XCDs of 32 CUs, three of 43 likewise
    cases += [(256, 6528, 9920), (256, 10880, 4096), (256, 6448, 7744), (256, 10816, 2560), (256, 3136, 12672)]
    for (cus, N, K), (cols, splits, blocks) in zip(cases, _picks(exe, [("decode", *c) for c in cases])):
        slabs = -(-N // cols)
        assert cols in (128, 256) and 1 <= splits <= 16
        assert splits == 1 or (slabs * splits <= cus and splits * 8 <= K // 32)
        assert blocks == (2 * 8 * -(-(-(-slabs // 2) * splits) // 8) if cols == 128 else slabs * splits)
        assert splits == 1 or blocks <= cus  # the launched grid, and with it every XCD's share


def test_reported_tiles_are_the_picked_ones():
    """tb_gemm_tile, and with it every get_last_config(), names the kernel and
    tile of each listed size (no GPU: 256 CUs)."""
    from tilebench_amd import runtime as rt

    if not rt.LIB_PATH.exists():
        pytest.skip("libtbhip.so is not built (run __graft_entry__.build())")
    big = {rt.OP_W4A16: "w4a16_prefill", rt.OP_W4A16_GROUPED: "w4a16_grouped", rt.OP_MOE_GATE_UP: "moe_gate_up",
           rt.OP_MOE_DOWN: "moe_down", rt.OP_FP8_SCALED: "fp8_gemm_kernel", rt.OP_FP8_BLOCK: "fp8_block_gemm",
           rt.OP_MATMUL_F16: "nt_gemm", rt.OP_MATMUL_FP8: "nt_gemm"}

    def check(op, tile, small, got):
        bm, bn = (256, 256) if tile == "256" else map(int, tile.split("x"))
        assert (got["kernel"], got["BM"], got["BN"]) == (big[op] if tile == "256" else small, bm, bn)

    for tile, cases in DENSE_TILES.items():
        for M, K, N, _ in cases:
            got = rt.gemm_tile(rt.OP_W4A16, M, N, K)
            check(rt.OP_W4A16, "32x64" if tile == "64x64" and M <= 32 else tile, "w4a16_dense", got)
            assert got["k_groups"] == (4 if tile == "64x64" else 1)
    for op in (rt.OP_W4A16_GROUPED, rt.OP_MOE_GATE_UP, rt.OP_MOE_DOWN):
        for tile, cases in EXPERT_TILES.items():
            for rows, N, K, _ in cases:
                check(op, tile, "w4a16_experts", rt.gemm_tile(op, sum(rows), N, K, len(rows)))
    for op in (rt.OP_FP8_SCALED, rt.OP_FP8_BLOCK):
        for tile, cases in FP8_TILES.items():
            for M, N, K in cases:
                check(op, tile, "fp8_skinny" if tile == "32x32" else "fp8_tile", rt.gemm_tile(op, M, N, K))
    for op, size in ((rt.OP_MATMUL_FP8, 1), (rt.OP_MATMUL_F16, 2)):
        for tile, cases in NT_TILES.items():
            for M, N, Kb in cases:
                check(op, tile, "nt_gemm", rt.gemm_tile(op, M, N, Kb // size))
    for (cols, splits), cases in DECODE_PLANS.items():
        for N, K in cases:
            got = rt.gemm_tile(rt.OP_W4A16, 16, N, K)
            assert (got["kernel"], got["BN"], got["k_splits"]) == ("w4a16_decode", cols, splits)
    with pytest.raises(ValueError, match="sizes must be positive"):
        rt.gemm_tile(rt.OP_W4A16_GROUPED, 64, 128, 64)
    with pytest.raises(ValueError, match="unknown operator"):
        rt.gemm_tile(10, 64, 128, 64)


def test_configs_hold_numbers():
    """get_last_config() of a call: the keys of each operator, its tile in numbers."""
    import importlib

    from tilebench_amd import runtime as rt

    if not rt.LIB_PATH.exists():
        pytest.skip("libtbhip.so is not built (run __graft_entry__.build())")
    want = [
        ("w4a16_gemm", ("rows", 48, 11008, 4096, 0),
         {"kernel": "w4a16_dense", "layout": "rows", "BM": 64, "BN": 64, "BK": 64, "waves": 8}),
        ("w4a16_gemm", ("rows", 16, 4096, 4096, 5), {"kernel": "w4a16_decode", "cols_per_block": 128, "workspace_bytes": 5}),
        ("fp8_scaled_gemm", (8192, 8192, 8192), {"kernel": "fp8_gemm_kernel", "BM": 256, "BN": 256, "BK": 128, "waves": 4}),
        ("fp8_block_scaled_gemm", (8192, 8192, 8192),
         {"kernel": "fp8_block_gemm", "BM": 256, "BN": 256, "BK": 128, "waves": 8}),
        ("moe_w4a16_grouped_gemm", (131072, 1408, 4096, 64),
         {"kernel": "w4a16_grouped", "BM": 256, "BN": 256, "BK": 64, "waves": 4,
          "last_tiles": "256 x 128 for <= 128 columns"}),
        ("fused_moe_w4a16", (32768, 64, 4096, 704, 7),
         {"kernels": ["gating", "moe_align", "moe_gate_up", "moe_down", "moe_combine"], "BM": 256, "BN_gate_up": 128,
          "BN_down": 256, "workspace_bytes": 7}),
        ("fused_moe_w4a16", (192, 64, 4096, 704, 7),
         {"kernels": ["gating", "moe_align", "w4a16_experts", "w4a16_experts", "moe_combine"], "BM": 32,
          "BN_gate_up": 128, "BN_down": 256}),
        ("matmul_fp32_fp16_fp8", (rt.OP_MATMUL_F16, 4096, 4096, 4096), {"kernel": "nt_gemm", "tile": "256x256"}),
        ("matmul_int8", (2048, 2048, 20480), {"kernel": "nt_gemm<i8>", "tile": "256x256", "k_splits": 4}),
        ("matmul_int8", (512, 512, 1024), {"kernel": "nt_gemm<i8>", "tile": "64x64", "k_splits": 1}),
    ]
    for op, last, keys in want:
        impl = importlib.import_module(f"tilebench_amd.benchmarks.operators.{op}.impl_hip")
        before, impl._last_call = impl._last_call, last
        try:
            cfg = impl.get_last_config()
        finally:
            impl._last_call = before
        assert {k: cfg.get(k) for k in keys} == keys, (op, cfg)

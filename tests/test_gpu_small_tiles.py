"""GPU parity of the small W4A16 tiles (w4a16_small.hip): every tile of the
dense, grouped, gate/up and down products against the CPU oracle, and bit for bit
against the 256-row tiles on the same rows; of the decode's slab widths and splits; and of the small-tile scaled
fp8 (fp8_small.hip) and plain products (nt_gemm.hip) against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from small_tile_cases import (DECODE_PLANS, DENSE_TILES, DOWN_TILES, EXPERT_TILES, FP8_TILES, GATE_UP_TILES,
                              NT_TILES)
from tilebench_amd import runtime as rt
from tilebench_amd.data import tensors as T

pytestmark = pytest.mark.gpu


def _say(*a):
    print("[gpu case]", *a, flush=True)


def _grouped(rows, N, K, G, seed):
    g = T._gen(seed)
    off = torch.zeros(len(rows) + 1, dtype=torch.int32)
    off[1:] = torch.cumsum(torch.tensor(rows), 0)
    A = torch.randn(int(off[-1]), K, generator=g).to(torch.float16)
    return (A, *T.random_int4_weights(K, N, G, g, experts=len(rows)), off)


@pytest.mark.parametrize("tile", list(EXPERT_TILES))
def test_grouped_tiles_match_oracle(gpu, tile):
    from tilebench_amd.benchmarks.operators.moe_w4a16_grouped_gemm import impl_hip

    for rows, N, K, G in EXPERT_TILES[tile]:
        _say("grouped", tile, sum(rows), len(rows), N, K, G)
        A, p, s, z, off = _grouped(rows, N, K, G, seed=N + K)
        Y = impl_hip.run(*(t.to(gpu) for t in (A, p, s, z, off)), G)
        torch.cuda.synchronize()
        ref = oracle.moe_w4a16_grouped_gemm(A.numpy(), p.numpy(), s.numpy(), z.numpy(), off.numpy(), G)
        np.testing.assert_allclose(Y.cpu().numpy().astype(np.float32), ref.astype(np.float32), atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("per_expert,experts,tile", [(1, 8, (32, 128)), (20, 64, (32, 256)), (60, 64, (64, 256))])
def test_grouped_rows_do_not_depend_on_the_tile(gpu, per_expert, experts, tile):
    """The first rows of the first experts alone give the bits they have in a call
    whose experts fill 256-row tiles."""
    from tilebench_amd.benchmarks.operators.moe_w4a16_grouped_gemm import impl_hip

    rows, N, K, G = EXPERT_TILES["256"][0]
    _say("grouped rows", per_expert)
    A, p, s, z, off = _grouped(rows, N, K, G, seed=5)
    d = [t.to(gpu) for t in (A, p, s, z)]
    big = impl_hip.run(*d, off.to(gpu), G)
    take = [min(r, per_expert) if e < experts else 0 for e, r in enumerate(rows)]
    for n, t in ((sum(take), tile), (sum(rows), (256, 256))):
        picked = rt.gemm_tile(rt.OP_W4A16_GROUPED, n, N, K, len(rows))
        assert (picked["BM"], picked["BN"]) == t
    o2 = torch.zeros(len(rows) + 1, dtype=torch.int32)
    o2[1:] = torch.cumsum(torch.tensor(take), 0)
    idx = torch.cat([torch.arange(int(off[e]), int(off[e]) + n) for e, n in enumerate(take)]).to(gpu)
    small = impl_hip.run(d[0][idx].contiguous(), *d[1:], o2.to(gpu), G)
    torch.cuda.synchronize()
    assert torch.equal(small.view(torch.int16), big[idx].view(torch.int16))


@pytest.mark.parametrize("Tk,E,k,H,I,g", [(1, 8, 4, 256, 128, 64), (33, 5, 3, 320, 72, 64), (70, 70, 2, 192, 704, 64),
                                          (500, 16, 8, 128, 704, 64), (700, 16, 8, 192, 1032, 64)])
def test_gate_up_and_down_tiles_match_oracle(gpu, Tk, E, k, H, I, g):
    """Token gather, SiLU epilogue, routing weights and the scatter, the down
    product on the gate/up product's rows, where the two take different tiles
    too.  Pairs routed nowhere stay unwritten."""
    _say("gate_up + down", Tk, E, k, H, I, g)
    gen = T._gen(Tk + I)
    X = torch.randn(Tk, H, generator=gen).to(torch.float16)
    ids = T.zipf_routing(Tk, k, E, 1.1, seed=7).to(torch.int32)
    if Tk > 1:
        ids[::5, 0] = E + 2
    w = torch.rand(Tk, k, generator=gen)
    sid, off = oracle.moe_align(ids.numpy(), E)
    P = Tk * k
    sorted_ids = np.full(P, -1, np.int32)
    sorted_ids[:len(sid)] = sid
    dev = {n: t.to(gpu) for n, t in dict(X=X, sid=torch.from_numpy(sorted_ids), off=torch.from_numpy(off), w=w).items()}
    W13 = T.random_int4_weights(H, 2 * I, g, gen, experts=E)
    d13 = [t.to(gpu) for t in W13]
    act = torch.empty((P, I), dtype=torch.float16, device=gpu)
    rt.call("tb_moe_w4a16_gate_up", rt.ptr(dev["X"]), rt.ptr(dev["sid"]), rt.ptr(dev["off"]), *map(rt.ptr, d13),
            rt.ptr(act), Tk, k, E, H, I, g, rt.stream_handle(gpu))
    torch.cuda.synchronize()
    want = oracle.moe_gate_up(X.numpy(), sid, off, k, *(t.numpy() for t in W13), g)
    got = act.cpu().numpy()[:len(sid)]
    np.testing.assert_allclose(got.astype(np.float32), want[:len(sid)].astype(np.float32), atol=1e-2, rtol=1e-2)
    if I % 64 or g > I:
        return  # down needs K = I in whole groups
    W2 = T.random_int4_weights(I, H, 64, gen, experts=E)
    d2 = [t.to(gpu) for t in W2]
    y = torch.full((P, H), float("nan"), dtype=torch.float16, device=gpu)
    rt.call("tb_moe_w4a16_down", rt.ptr(act), rt.ptr(dev["sid"]), rt.ptr(dev["off"]), rt.ptr(dev["w"]),
            *map(rt.ptr, d2), rt.ptr(y), P, E, I, H, 64, rt.stream_handle(gpu))
    torch.cuda.synchronize()
    want, written = oracle.moe_down(got, sid, off, w.numpy(), P, *(t.numpy() for t in W2), 64)
    y = y.cpu().numpy()
    np.testing.assert_allclose(y[written].astype(np.float32), want[written].astype(np.float32), atol=1e-2, rtol=1e-2)
    assert np.isnan(y[~written].astype(np.float32)).all()


def _routed(T_, E, k, gen, gpu):
    """(ids by expert, offsets, routing weights) on the host and on the GPU; every fifth token's first pair goes nowhere."""
    ids = T.zipf_routing(T_, k, E, 1.1, seed=7).to(torch.int32)
    ids[::5, 0] = E + 2
    w = torch.rand(T_, k, generator=gen)
    sid, off = oracle.moe_align(ids.numpy(), E)
    sorted_ids = np.full(T_ * k, -1, np.int32)
    sorted_ids[:len(sid)] = sid
    return sid, off, w, [t.to(gpu) for t in (torch.from_numpy(sorted_ids), torch.from_numpy(off), w)]


@pytest.mark.parametrize("tile,wide", list(GATE_UP_TILES))
def test_gate_up_tiles_match_oracle(gpu, tile, wide):
    Tk, E, k, H, I, g = GATE_UP_TILES[tile, wide]
    _say("gate_up", tile, wide, Tk, E, k, H, I, g)
    gen = T._gen(Tk + I)
    X = torch.randn(Tk, H, generator=gen).to(torch.float16)
    sid, off, _, (dsid, doff, _) = _routed(Tk, E, k, gen, gpu)
    W = T.random_int4_weights(H, 2 * I, g, gen, experts=E)
    dX, dW = X.to(gpu), [t.to(gpu) for t in W]
    act = torch.empty((Tk * k, I), dtype=torch.float16, device=gpu)
    rt.call("tb_moe_w4a16_gate_up", rt.ptr(dX), rt.ptr(dsid), rt.ptr(doff), *map(rt.ptr, dW), rt.ptr(act), Tk, k, E, H, I,
            g, rt.stream_handle(gpu))
    torch.cuda.synchronize()
    want = oracle.moe_gate_up(X.numpy(), sid, off, k, *(t.numpy() for t in W), g)[:len(sid)]
    np.testing.assert_allclose(act.cpu().numpy()[:len(sid)].astype(np.float32), want.astype(np.float32), atol=1e-2,
                               rtol=1e-2)


@pytest.mark.parametrize("tile,wide", list(DOWN_TILES))
def test_down_tiles_match_oracle(gpu, tile, wide):
    Tk, E, k, I, H, g = DOWN_TILES[tile, wide]
    _say("down", tile, wide, Tk, E, k, I, H, g)
    gen = T._gen(Tk + H)
    act = torch.randn(Tk * k, I, generator=gen).to(torch.float16)
    sid, off, w, (dsid, doff, dw) = _routed(Tk, E, k, gen, gpu)
    W = T.random_int4_weights(I, H, g, gen, experts=E)
    dact, dW = act.to(gpu), [t.to(gpu) for t in W]
    y = torch.full((Tk * k, H), float("nan"), dtype=torch.float16, device=gpu)
    rt.call("tb_moe_w4a16_down", rt.ptr(dact), rt.ptr(dsid), rt.ptr(doff), rt.ptr(dw), *map(rt.ptr, dW), rt.ptr(y), Tk * k,
            E, I, H, g, rt.stream_handle(gpu))
    torch.cuda.synchronize()
    want, written = oracle.moe_down(act.numpy(), sid, off, w.numpy(), Tk * k, *(t.numpy() for t in W), g)
    y = y.cpu().numpy()
    np.testing.assert_allclose(y[written].astype(np.float32), want[written].astype(np.float32), atol=1e-2, rtol=1e-2)
    assert np.isnan(y[~written].astype(np.float32)).all()


@pytest.mark.parametrize("tile", list(DENSE_TILES))
def test_dense_tiles_match_oracle(gpu, tile):
    from tilebench_amd.benchmarks.operators.w4a16_gemm import impl_hip

    for M, K, N, G in DENSE_TILES[tile]:
        _say("dense", tile, M, K, N, G)
        A, p, s, z, G = T.generate_w4a16_gemm_inputs(M, K, N, G, seed=M + N, device="cpu")
        Y = impl_hip.run(A.to(gpu), p.to(gpu), s.to(gpu), z.to(gpu), G)
        torch.cuda.synchronize()
        rows = np.unique(np.r_[np.arange(min(M, 96)), np.arange(max(0, M - 96), M)])
        ref = oracle.w4a16_gemm(A.numpy()[rows], p.numpy(), s.numpy(), z.numpy(), G)
        np.testing.assert_allclose(Y.cpu().numpy()[rows].astype(np.float32), ref.astype(np.float32), atol=1e-2,
                                   rtol=1e-2)


@pytest.mark.parametrize("M,N,tile", [(65, 11008, (64, 128)), (500, 11008, (128, 256)), (300, 22040, (64, 256)),
                                      (64, 32768, (64, 128))])
def test_dense_rows_do_not_depend_on_the_tile(gpu, M, N, tile):
    """Tiles that do not split K: the first M rows alone give the bits they have in a
    product of 256 x 256 tiles, at 64 rows too where N is wide.  64 rows are reproducible."""
    from tilebench_amd.benchmarks.operators.w4a16_gemm import impl_hip

    A, p, s, z, G = T.generate_w4a16_gemm_inputs(1024, 448, N, 64, seed=3, device="cpu")
    _say("dense rows", M, N)
    for m, t in ((M, tile), (1024, (256, 256))):
        picked = rt.gemm_tile(rt.OP_W4A16, m, N, 448)
        assert (picked["BM"], picked["BN"]) == t
    A, p, s, z = (t.to(gpu) for t in (A, p, s, z))
    big = impl_hip.run(A, p, s, z, G)
    small = impl_hip.run(A[:M].contiguous(), p, s, z, G)
    a, b = (impl_hip.run(A[:64].contiguous(), p, s, z, G) for _ in range(2))
    torch.cuda.synchronize()
    assert torch.equal(small.view(torch.int16), big[:M].view(torch.int16))
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("M", [17, 31, 32])
@pytest.mark.parametrize("K,N", [(64, 8), (704, 1000), (2048, 4096)])  # N % 32 != 0 and == 0
def test_dense_32_row_tile(gpu, M, K, N):
    """Up to 32 rows: the oracle's values, and the bits of the same rows on a 64-row tile."""
    from tilebench_amd.benchmarks.operators.w4a16_gemm import impl_hip

    _say("dense 32 rows", M, K, N)
    A, p, s, z, G = T.generate_w4a16_gemm_inputs(33, K, N, 64, seed=M + N, device="cpu")
    d = [t.to(gpu) for t in (A, p, s, z)]
    big = impl_hip.run(*d, G)
    small = impl_hip.run(d[0][:M].contiguous(), *d[1:], G)
    torch.cuda.synchronize()
    assert torch.equal(small.view(torch.int16), big[:M].view(torch.int16))
    ref = oracle.w4a16_gemm(A.numpy()[:M], p.numpy(), s.numpy(), z.numpy(), G)
    np.testing.assert_allclose(small.cpu().numpy().astype(np.float32), ref.astype(np.float32), atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("cols,splits", list(DECODE_PLANS))
def test_decode_plans_match_oracle(gpu, cols, splits):
    """Each slab width and split of the decode at 1, 5 and 16 rows, twice in a row
    (the arrival counters are back at zero) with equal bits."""
    from tilebench_amd.benchmarks.operators.w4a16_gemm import impl_hip

    for N, K in DECODE_PLANS[cols, splits]:
        for M in (1, 5, 16):
            _say("decode", cols, splits, M, N, K)
            A, p, s, z, G = T.generate_w4a16_gemm_inputs(M, K, N, 64, seed=N + K + M, device="cpu")
            d = [t.to(gpu) for t in (A, p, s, z)]
            Y, Y2 = impl_hip.run(*d, G), impl_hip.run(*d, G)
            torch.cuda.synchronize()
            assert torch.equal(Y.view(torch.int16), Y2.view(torch.int16))
            ref = oracle.w4a16_gemm(A.numpy(), p.numpy(), s.numpy(), z.numpy(), G)
            np.testing.assert_allclose(Y.cpu().numpy().astype(np.float32), ref.astype(np.float32), atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("tile", list(FP8_TILES))
@pytest.mark.parametrize("scaling", ["row", "block"])
def test_fp8_tiles_match_oracle(gpu, tile, scaling):
    """bf16 within the operators' 1e-2, and reproducible bit for bit."""
    if scaling == "row":
        from tilebench_amd.benchmarks.operators.fp8_scaled_gemm import impl_hip
        gen, ref_gemm = T.generate_fp8_scaled_gemm_inputs, oracle.fp8_scaled_gemm
    else:
        from tilebench_amd.benchmarks.operators.fp8_block_scaled_gemm import impl_hip
        gen, ref_gemm = T.generate_fp8_block_scaled_gemm_inputs, oracle.fp8_block_gemm
    for M, N, K in FP8_TILES[tile]:
        _say("fp8", scaling, tile, M, N, K)
        Aq, W, sa, sw = gen(M, N, K, seed=M + N, device="cpu")
        d = [t.to(gpu) for t in (Aq, W, sa, sw)]
        Y, again = impl_hip.run(*d), impl_hip.run(*d)
        torch.cuda.synchronize()
        r = np.unique(np.r_[np.arange(min(M, 70)), np.arange(max(0, M - 70), M)])
        s = sa.numpy()[r] if scaling == "row" else sa.numpy()[:, r]
        ref = ref_gemm(Aq.view(torch.uint8).numpy()[r], W.contiguous().view(torch.uint8).numpy(), s, sw.numpy())
        np.testing.assert_allclose(Y.float().cpu().numpy()[r], oracle.bf16_bits_to_f32(ref), atol=1e-2, rtol=1e-2)
        assert torch.equal(Y.view(torch.int16), again.view(torch.int16))


@pytest.mark.parametrize("scaling", ["row", "block"])
def test_fp8_rows_across_tiles(gpu, scaling):
    """The first M rows of a call alone, against the same rows on 256 x 256 tiles:
    equal bits wherever one wavefront group adds all of K, and otherwise a bf16 step
    of rounding beside the fp32 sums' own error (9 blocks, each sum at most 9 max |y|)."""
    N, K = 8200, 1152
    if scaling == "row":
        from tilebench_amd.benchmarks.operators.fp8_scaled_gemm import impl_hip
        gen, op = T.generate_fp8_scaled_gemm_inputs, rt.OP_FP8_SCALED
    else:
        from tilebench_amd.benchmarks.operators.fp8_block_scaled_gemm import impl_hip
        gen, op = T.generate_fp8_block_scaled_gemm_inputs, rt.OP_FP8_BLOCK
    Aq, W, sa, sw = (t.to(gpu) for t in gen(1024, N, K, seed=11, device="cpu"))
    WT = W.t().contiguous() if scaling == "row" else W
    big = impl_hip.run(Aq, W, sa, sw)
    assert rt.gemm_tile(op, 1024, N, K)["BM"] == 256
    groups = set()
    for M, n in [(16, 2112), (64, N), (192, N), (300, N), (448, N), (512, N)]:
        t = rt.gemm_tile(op, M, n, K)
        _say("fp8 rows", scaling, M, n, K, t)
        w = WT[:n].contiguous()
        s = sa[:M].contiguous() if scaling == "row" else sa[:, :M].contiguous()
        got = impl_hip.run(Aq[:M].contiguous(), w.t() if scaling == "row" else w, s,
                           sw[:n].contiguous() if scaling == "row" else sw[:-(-n // 128)].contiguous())
        want = big[:M, :n]
        torch.cuda.synchronize()
        groups.add((t["kernel"], t["k_groups"]))
        if t["k_groups"] == 1:
            assert torch.equal(got.view(torch.int16), want.contiguous().view(torch.int16))
        else:
            d, y = (got.double() - want.double()).abs(), want.double().abs()
            assert bool((d <= 2.0 ** -7 * y + 9 * 9 * 2.0 ** -24 * y.max()).all())
    assert groups == {("fp8_skinny", 4), ("fp8_tile", 1)} | ({("fp8_tile", 2)} if scaling == "block" else set())


@pytest.mark.parametrize("tile", list(NT_TILES))
@pytest.mark.parametrize("dt", ["fp16", "fp32", "fp8", "int8"])
def test_plain_product_tiles_match_oracle(gpu, tile, dt):
    """Every type on every tile, at the tolerances of the products' own tests
    (fp32 within 1e-4 of the float64 product, int8 exact, e4m3 codes equal on
    99.5 % and never more than a step apart)."""
    from tilebench_amd.benchmarks.operators.matmul_fp32_fp16_fp8 import impl_hip as mm
    from tilebench_amd.benchmarks.operators.matmul_int8 import impl_hip as mi

    for M, N, Kb in NT_TILES[tile]:
        # elements of K whose GEMM row has Kb bytes (fp32: three bf16 terms, K % 64 == 0)
        K = {"fp16": Kb // 2, "fp32": max(64, Kb // 6 // 64 * 64), "fp8": Kb, "int8": Kb}[dt]
        _say("plain", dt, tile, M, N, K)
        r = np.unique(np.r_[np.arange(min(M, 40)), np.arange(max(0, M - 40), M)])
        if dt == "int8":
            a, b = T.generate_matmul_int8_inputs(M, N, K, seed=M, device="cpu")
            out = mi.run(a.to(gpu), b.to(gpu))
            np.testing.assert_array_equal(out.cpu().numpy()[r], oracle.matmul_int8(a.numpy()[r], b.numpy()))
            continue
        tdt = {"fp16": torch.float16, "fp32": torch.float32, "fp8": torch.float8_e4m3fn}[dt]
        a, b = T.generate_matmul_fp32_fp16_fp8_inputs(M, N, K, dtype=tdt, seed=M, device="cpu")
        out = mm.run(a.to(gpu), b.to(gpu)).cpu()
        if dt == "fp8":
            got = out.view(torch.uint8).numpy()[r]
            ref = oracle.matmul_fp8(a.view(torch.uint8).numpy()[r], b.view(torch.uint8).numpy())
            assert (got == ref).mean() > 0.995
            g, f = oracle.e4m3_to_f32(got), oracle.e4m3_to_f32(ref)
            step = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(f), 2.0 ** -6))) - 3)
            assert (np.abs(g - f) <= step + 1e-12).all()
        elif dt == "fp16":
            ref = oracle.matmul_f16(a.numpy()[r], b.numpy()).astype(np.float32)
            np.testing.assert_allclose(out.numpy()[r].astype(np.float32), ref, atol=2e-3, rtol=2e-3)
        else:
            np.testing.assert_allclose(out.numpy()[r], oracle.matmul_f32(a.numpy()[r], b.numpy()), atol=1e-4, rtol=1e-4)


def test_plain_fp8_product_to_a_4_byte_aligned_output(gpu):
    """tb_matmul_fp8_bt takes an output on 4 bytes: the small tiles store 8-byte
    granules, so such an output takes the 256 x 256 tiles."""
    M, N, K = 65, 200, 256
    _say("plain fp8, output on 4 bytes", M, N, K)
    a, b = T.generate_matmul_fp32_fp16_fp8_inputs(M, N, K, dtype=torch.float8_e4m3fn, seed=1, device="cpu")
    ag, bt = a.to(gpu), b.t().contiguous().to(gpu)
    buf = torch.zeros(M * N + 16, dtype=torch.uint8, device=gpu)
    out = torch.zeros(M * N, dtype=torch.uint8, device=gpu)
    for dst in (buf.data_ptr() + 4, out.data_ptr()):
        rt.call("tb_matmul_fp8_bt", ag.data_ptr(), bt.data_ptr(), dst, M, N, K, rt.stream_handle())
    torch.cuda.synchronize()
    assert torch.equal(buf[4:4 + M * N], out) and int(buf[:4].sum()) == 0 and int(buf[4 + M * N:].sum()) == 0


@pytest.mark.parametrize("form", ["none", "cuda", "cuda:0", "index", "device"])
def test_stream_handle_takes_every_form_of_a_device(gpu, form):
    device = {"none": None, "index": 0, "device": torch.device("cuda", 0)}.get(form, form)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        assert rt.stream_handle(device) == side.cuda_stream
    assert rt.stream_handle(device) == torch.cuda.current_stream().cuda_stream
    with pytest.raises(ValueError):
        rt.stream_handle(torch.device("cpu", 0))


@pytest.mark.parametrize("op,case", [
    ("w4a16_gemm", dict(M=16, K=4096, N=4096)), ("w4a16_gemm", dict(M=20, K=256, N=1024)),
    ("w4a16_gemm", dict(M=48, K=256, N=1024)), ("w4a16_gemm", dict(M=300, K=512, N=512)),
    ("w4a16_gemm", dict(M=1024, K=128, N=11008)),
    ("fp8_scaled_gemm", dict(M=16, N=8192, K=896)), ("fp8_scaled_gemm", dict(M=300, N=5000, K=384)),
    ("fp8_block_scaled_gemm", dict(M=200, N=2112, K=1152)), ("fp8_block_scaled_gemm", dict(M=1024, N=8200, K=1152)),
    ("moe_w4a16_grouped_gemm", dict(tokens=64, topk=2, experts=8, K=256, N=264)),
    ("fused_moe_w4a16", dict(tokens=24, experts=8, topk=2, H=256, I=128)),
    ("matmul_fp32_fp16_fp8", dict(M=513, N=2056, K=320, dtype="fp16")),
    ("matmul_int8", dict(M=100, N=1000, K=640, dtype="int8")),
], ids=lambda x: x if isinstance(x, str) else None)
def test_config_names_what_was_launched(gpu, op, case):
    """get_last_config() after a call against the kernels the profiler saw: the
    name, and the tile from the template arguments."""
    import importlib
    import re

    from tilebench_amd.profiling import probe

    _say("config", op, case)
    impl = importlib.import_module(f"tilebench_amd.benchmarks.operators.{op}.impl_hip")
    names = probe.probe_case(impl, op, case)["names"]
    cfg = impl.get_last_config()
    moe = op == "fused_moe_w4a16"
    products = [n for n in names if re.search(r"w4a16|fp8|moe_gate_up|moe_down|nt_gemm", n)]
    kernels = cfg["kernels"][2:4] if moe else [cfg["kernel"].split("<")[0]]
    assert [n.split("<")[0].split("::")[-1] for n in products] == kernels, (names, cfg)
    for i, name in enumerate(products):
        if "<" not in name:  # a 256-row kernel
            assert (cfg["BM"], cfg["BN"]) == (256, 256)
            continue
        args = [int({"true": 1, "false": 0}.get(x, x)) for x in re.findall(r"\b(\d+|true|false)\b", name)]
        kernel = kernels[i]
        if kernel == "w4a16_decode":
            assert cfg["cols_per_block"] == 128 * (1 + args[0])
        elif kernel in ("w4a16_dense", "w4a16_experts"):
            bn = (cfg["BN_down"] if i else 2 * cfg["BN_gate_up"]) if moe else cfg["BN"]
            assert (cfg["BM_down"] if moe and i else cfg["BM"], bn) == (32 * args[0], 64 * args[1])
        elif kernel == "fp8_tile":
            assert (cfg["BM"], cfg["BN"], cfg["k_groups"]) == (64 * args[0], 64 * args[1], args[4])
        elif kernel == "fp8_block_gemm":
            assert (cfg["BM"], cfg["BN"], cfg["waves"]) == (256, args[0], args[1])
        elif kernel == "nt_gemm":
            assert cfg["tile"] == f"{args[2]}x{args[3]}"
        else:
            assert kernel == "fp8_skinny" and (cfg["BM"], cfg["BN"], cfg["waves"]) == (32, 32, args[0])


def _same_specials(got, want):
    """NaN and infinities (with their signs) of `got` where `want` has them."""
    got, want = got.double().cpu(), want.double().cpu()
    assert torch.equal(got.isnan(), want.isnan())
    inf = want.isinf()
    assert torch.equal(got.isinf(), inf) and torch.equal(got[inf], want[inf])


@pytest.mark.parametrize("tile", ["32x32", "64x64", "64x128", "128x128"])
@pytest.mark.parametrize("scaling", ["row", "block"])
def test_fp8_special_rows(gpu, tile, scaling):
    """Row 0 as the quantiser leaves a row of zeros (scale 0, NaN codes), row 2 of
    infinite scale, row 5 with one NaN code: their own outputs as IEEE has them, and
    every other row's bits as without them."""
    if scaling == "row":
        from tilebench_amd.benchmarks.operators.fp8_scaled_gemm import impl_hip
        gen = T.generate_fp8_scaled_gemm_inputs
    else:
        from tilebench_amd.benchmarks.operators.fp8_block_scaled_gemm import impl_hip
        gen = T.generate_fp8_block_scaled_gemm_inputs
    M, N, K = next(c for c in FP8_TILES[tile] if c[0] > 8)
    _say("fp8 special rows", scaling, tile, M, N, K)
    Aq, W, sa, sw = (t.to(gpu) for t in gen(M, N, K, seed=M, device="cpu"))
    plain = impl_hip.run(Aq, W, sa, sw)
    codes, scale = Aq.view(torch.uint8).clone(), sa.clone()
    rows = scale if scaling == "row" else scale.t()  # [M] or [M, K / 128], views
    codes[0], codes[5, K - 1] = 0xFF, 0x7F
    rows[0], rows[2] = 0.0, float("inf")
    Y = impl_hip.run(codes.view(torch.float8_e4m3fn), W, scale, sw)
    torch.cuda.synchronize()
    others = [m for m in range(M) if m not in (0, 2, 5)]
    assert torch.equal(Y[others].view(torch.int16), plain[others].view(torch.int16))
    assert bool(Y[[0, 5]].isnan().all())
    if scaling == "row":  # one product, then the scale: +-inf, as the plain row's signs
        _same_specials(Y[2], plain[2].float() * float("inf"))
    else:  # infinite terms of either sign: NaN unless K has one block
        assert not bool(Y[2].isfinite().any())


@pytest.mark.parametrize("tile", ["64x64", "64x128", "64x256", "128x256"])
def test_dense_special_rows(gpu, tile):
    """A row of NaN, one infinity and a row of the largest values: their own outputs
    as the oracle has them, and every other row's bits as without them."""
    from tilebench_amd.benchmarks.operators.w4a16_gemm import impl_hip

    M, K, N, G = DENSE_TILES[tile][1]
    _say("dense special rows", tile, M, K, N, G)
    A, p, s, z, G = T.generate_w4a16_gemm_inputs(M, K, N, G, seed=M, device="cpu")
    d = [t.to(gpu) for t in (p, s, z)]
    plain = impl_hip.run(A.to(gpu), *d, G)
    B = A.clone()
    B[1], B[3, K - 1], B[M - 1] = float("nan"), float("-inf"), 65504.0
    Y = impl_hip.run(B.to(gpu), *d, G)
    torch.cuda.synchronize()
    others = [m for m in range(M) if m not in (1, 3, M - 1)]
    assert torch.equal(Y[others].view(torch.int16), plain[others].view(torch.int16))
    rows = [1, 3, M - 1]
    with np.errstate(all="ignore"):
        want = torch.from_numpy(oracle.w4a16_gemm(B.numpy()[rows], p.numpy(), s.numpy(), z.numpy(), G))
    _same_specials(Y[rows[:2]], want[:2])
    # sums of 65504 w near fp16's own largest value may round to infinity in one order and not in another
    clear = (want[2].float().abs() < 6e4) | want[2].isinf()
    got = Y[M - 1].cpu()
    big = want[2].isinf() & got.isinf()
    assert torch.equal(got[big], want[2][big]) and not bool(got.isnan().any())
    assert bool((got[clear & ~want[2].isinf()].isfinite()).all())


@pytest.mark.parametrize("tile", ["64x64", "64x128", "128x128"])
@pytest.mark.parametrize("dt", ["fp16", "fp8"])
def test_plain_product_special_rows(gpu, tile, dt):
    from tilebench_amd.benchmarks.operators.matmul_fp32_fp16_fp8 import impl_hip

    M, N, Kb = NT_TILES[tile][-1] if tile != "128x128" else NT_TILES[tile][0]
    K = Kb // 2 if dt == "fp16" else Kb
    _say("plain special rows", dt, tile, M, N, K)
    tdt = torch.float16 if dt == "fp16" else torch.float8_e4m3fn
    a, b = (t.to(gpu) for t in T.generate_matmul_fp32_fp16_fp8_inputs(M, N, K, dtype=tdt, seed=M, device="cpu"))
    plain = impl_hip.run(a, b)
    c = a.clone()
    raw = c.view(torch.uint8 if dt == "fp8" else torch.int16)
    nan, other = (0x7F, 0xFF) if dt == "fp8" else (0x7E00, 0x7C00)  # fp8 has no infinity: the other NaN code
    raw[1], raw[4, K - 1] = nan, other
    Y = impl_hip.run(c, b)
    torch.cuda.synchronize()
    others = [m for m in range(M) if m not in (1, 4)]
    bits = torch.uint8 if dt == "fp8" else torch.int16
    assert torch.equal(Y[others].view(bits), plain[others].view(bits))
    assert bool(Y[1].float().isnan().all())
    if dt == "fp8":
        assert bool(Y[4].float().isnan().all())
    else:
        _same_specials(Y[4], float("inf") * b[K - 1].float())  # inf times 0 is NaN


@pytest.mark.parametrize("M,N,tile", [(64, 136, (64, 64)), (320, 4104, (64, 128)), (640, 4104, (128, 128))])
def test_fp8_block_scales_at_the_largest_k(gpu, M, N, tile):
    """K = 65536: 512 scale blocks fill the tiles' scale table.  The last rows and
    columns against 64-bit sums; fp32 sums of 512 blocks, then bf16 (half a step, 2^-9)."""
    from tilebench_amd.benchmarks.operators.fp8_block_scaled_gemm import impl_hip

    K = 65536
    t = rt.gemm_tile(rt.OP_FP8_BLOCK, M, N, K)
    assert (t["BM"], t["BN"]) == tile
    _say("fp8 block, largest K", M, N, t)
    g = torch.Generator(device=gpu).manual_seed(M)
    Aq, W = ((torch.randint(0, 112, (n, K), generator=g, device=gpu, dtype=torch.uint8)
              | torch.randint(0, 2, (n, K), generator=g, device=gpu, dtype=torch.uint8) << 7).view(torch.float8_e4m3fn)
             for n in (M, N))  # both signs, at most 120
    sa = torch.rand(K // 128, M, generator=g, device=gpu) + 0.5
    sw = torch.rand(-(-N // 128), K // 128, generator=g, device=gpu) + 0.5
    Y = impl_hip.run(Aq, W, sa, sw)
    r, c = slice(max(0, M - 32), M), slice(max(0, N - 64), N)
    a = Aq[r].float().double().view(-1, K // 128, 128) * sa[:, r].t().double()[:, :, None]
    scale = sw.double().repeat_interleave(128, dim=0)[:N][c]
    w = W[c].float().double().view(-1, K // 128, 128) * scale[:, :, None]
    want, size = torch.zeros_like(Y[r, c], dtype=torch.float64), torch.zeros_like(Y[r, c], dtype=torch.float64)
    for kb in range(K // 128):
        want += a[:, kb] @ w[:, kb].t()
        size += a[:, kb].abs() @ w[:, kb].abs().t()
    torch.cuda.synchronize()
    # 128-term and 512-term fp32 sums: (128 + 512) roundings of 2^-24 of the sum of magnitudes at most
    bound = 2.0 ** -8 * want.abs() + 640 * 2.0 ** -24 * size
    assert bool(((Y[r, c].double() - want).abs() <= bound).all())


@pytest.mark.parametrize("dt,op", [("fp16", "OP_MATMUL_F16"), ("fp32", "OP_MATMUL_F32"), ("fp8", "OP_MATMUL_FP8")])
def test_plain_product_rows_do_not_depend_on_the_tile(gpu, dt, op):
    """The first M rows alone give the bits they have in a product of 256 x 256 tiles."""
    from tilebench_amd.benchmarks.operators.matmul_fp32_fp16_fp8 import impl_hip

    N, K, tdt = {"fp16": (4104, 576, torch.float16), "fp32": (4104, 384, torch.float32),
                 "fp8": (4104, 1152, torch.float8_e4m3fn)}[dt]
    tile = lambda m: tuple(rt.gemm_tile(getattr(rt, op), m, N, K)[k] for k in ("BM", "BN"))
    a, b = (t.to(gpu) for t in T.generate_matmul_fp32_fp16_fp8_inputs(4096, N, K, dtype=tdt, seed=5, device="cpu"))
    big, seen = impl_hip.run(a, b), set()
    assert tile(4096) == (256, 256)
    for M in (100, 400, 1000):
        _say("plain rows", dt, M, N, K, tile(M))
        seen.add(tile(M))
        small = impl_hip.run(a[:M].contiguous(), b)
        torch.cuda.synchronize()
        assert torch.equal(small.view(torch.uint8), big[:M].contiguous().view(torch.uint8))
    assert seen == {(64, 64), (64, 128), (128, 128)}

"""Performance cases: the quantized-inference work a program gives this package.

Every case is one pass through the operators' public ``run`` functions, on
inputs that already are on the GPU, over the sizes a serving program meets:
one token, a decode batch, a ragged chunk of a prompt, a whole prompt.

kind        one pass
router      moe_topk_gating on a batch of router logits
w4a16       w4a16_gemm on packed ("rows") or decode-layout ("slabs") weights
fp8         a dynamically quantised linear layer: fp8_act_quant, fp8_scaled_gemm
fp8_block   the same with 128-channel activation and 128 x 128 weight scales
moe         the fused W4A16 mixture-of-experts feed-forward layer
matmul      the plain matrix products (fp16, fp32, fp8, int8 x 2-bit)
"""
import math

import torch

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # the smallest call: the router of one decode batch (latency and launches)
        {"name": "router_m64", "kind": "router", "M": 64, "E": 256, "k": 8, "dtype": "fp32"},
        # one token through an MLP up projection, weights stored in the decode layout
        {"name": "w4a16_slabs_m1", "kind": "w4a16", "M": 1, "K": 4096, "N": 11008, "group": 128, "layout": "slabs"},
        # a small decode batch on weights as a checkpoint packs them
        {"name": "w4a16_decode_m16", "kind": "w4a16", "M": 16, "K": 4096, "N": 11008, "group": 128, "layout": "rows"},
        # a decode batch of a busy server
        {"name": "w4a16_batch_m48", "kind": "w4a16", "M": 48, "K": 4096, "N": 11008, "group": 128, "layout": "rows"},
        # a ragged chunk of a prompt through the down projection
        {"name": "w4a16_chunk_m500", "kind": "w4a16", "M": 500, "K": 11008, "N": 4096, "group": 128, "layout": "rows"},
        # a whole prompt
        {"name": "w4a16_prefill_m4096", "kind": "w4a16", "M": 4096, "K": 4096, "N": 11008, "group": 128,
         "layout": "rows"},
        # an fp8 linear layer in decode and on a large prefill batch
        {"name": "fp8_linear_m32", "kind": "fp8", "M": 32, "K": 8192, "N": 8192},
        {"name": "fp8_linear_m8192", "kind": "fp8", "M": 8192, "K": 8192, "N": 8192},
        # block-scaled fp8: a ragged mid-size batch on a narrow projection
        {"name": "fp8_block_m200", "kind": "fp8_block", "M": 200, "K": 7168, "N": 2112},
        # the mixture-of-experts layer: a decode batch and a prompt
        {"name": "moe_t24", "kind": "moe", "tokens": 24, "experts": 64, "topk": 8, "H": 4096, "I": 704,
         "group13": 128, "group2": 64},
        {"name": "moe_t4096", "kind": "moe", "tokens": 4096, "experts": 64, "topk": 8, "H": 4096, "I": 704,
         "group13": 128, "group2": 64},
        # the plain product of unquantised layers
        {"name": "matmul_fp16", "kind": "matmul", "dtype": "fp16", "M": 4096, "N": 4096, "K": 4096},
    ]


# ----------------------------------------------------------------------------- drawn cases

#: the largest drawn product, in multiply-adds (the largest listed prefill and fp8 layers)
_MOST_W4A16 = 4096 * 4096 * 11008
_MOST_FP8 = 8192 ** 3
_MOST_MATMUL = {"fp16": 4096 ** 3, "fp8": 4096 ** 3, "int8": 4096 ** 3, "fp32": 4096 * 4096 * 2048}


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["router", "w4a16", "w4a16", "w4a16", "fp8", "fp8_block", "moe", "moe", "matmul"])
    if kind == "router":
        E = rng.choice([8, 60, 64, 96, 128, 160, 256, 384])
        return {"kind": kind, "M": _log_int(rng, 1, 20480), "E": E, "k": rng.randint(1, 8),
                "dtype": rng.choice(["fp32", "fp16", "bf16"])}
    if kind == "w4a16":
        M = _log_int(rng, 1, 4096)
        if M <= 16 and rng.random() < 0.4:
            K = rng.choice([1024, 2048, 4096])
            group = 64 if K == 1024 else rng.choice([64, 128])
            return {"kind": kind, "M": M, "K": K, "N": 64 * rng.randint(16, 192), "group": group, "layout": "slabs"}
        if rng.random() < 0.5:
            K, N = rng.choice([(4096, 11008), (11008, 4096), (4096, 4096), (4096, 12288), (4096, 1408)])
        else:
            K, N = 64 * rng.randint(16, 172), 8 * rng.randint(128, 1536)
        group = rng.choice([64, 128]) if K % 128 == 0 else 64
        M = max(1, min(M, _MOST_W4A16 // (K * N)))
        return {"kind": kind, "M": M, "K": K, "N": N, "group": group, "layout": "rows"}
    if kind == "fp8":
        K, N = 128 * rng.randint(8, 64), 8 * rng.randint(128, 1024)
        return {"kind": kind, "M": _log_int(rng, 1, 8192), "K": K, "N": N}
    if kind == "fp8_block":
        K = rng.choice([7168, 128 * rng.randint(8, 56)])
        N = rng.choice([2112, 7168, 8 * rng.randint(128, 1024)])
        return {"kind": kind, "M": _log_int(rng, 1, 4096), "K": K, "N": N}
    if kind == "moe":
        E = rng.choice([8, 16, 32, 64])
        H, I = 64 * rng.randint(16, 64), 64 * rng.randint(4, 11)
        return {"kind": kind, "tokens": _log_int(rng, 1, 4096), "experts": E, "topk": rng.randint(1, 8), "H": H,
                "I": I, "group13": 128 if H % 128 == 0 else 64, "group2": 128 if I % 128 == 0 else 64}
    dtype = rng.choice(["fp16", "fp32", "fp8", "int8"])
    M, N, K = _log_int(rng, 16, 4096), 8 * rng.randint(32, 512), 128 * rng.randint(2, 48)
    M = max(16, min(M, _MOST_MATMUL[dtype] // (N * K)))
    return {"kind": kind, "dtype": dtype, "M": M, "N": N, "K": K}


# ----------------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _int4(K, N, group, g, experts=()):
    """Codes and zero-points uniform on 0..15, scales uniform on [1e-3, 1e-2]."""
    packed = torch.randint(0, 256, experts + (K, N // 2), generator=g, device="cuda", dtype=torch.uint8)
    scales = (torch.rand(experts + (K // group, N), generator=g, device="cuda") * 9e-3 + 1e-3).half()
    zeros = torch.randint(0, 256, experts + (K // group, N // 2), generator=g, device="cuda", dtype=torch.uint8)
    return packed, scales, zeros


def _activations(M, K, g, outliers=False):
    """N(0, 1); with outliers, one value in a thousand times 20."""
    A = torch.randn(M, K, generator=g, device="cuda")
    if outliers:
        A = torch.where(torch.rand(M, K, generator=g, device="cuda") < 1e-3, A * 20.0, A)
    return A.half()


def _router_logits(tokens, experts, g, device="cuda"):
    """Top-k of these is a draw of experts with popularity rank^-1.1."""
    rank = torch.randperm(experts, generator=g, device=device)
    u = torch.rand(tokens, experts, generator=g, device=device).clamp_(1e-7, 1.0 - 1e-7)
    return -1.1 * torch.log(rank.float() + 1.0) - torch.log(-torch.log(u))


def _inputs(case, seed):
    """The values of a case, before any layout the package prepares."""
    g, kind = _gen(seed), case["kind"]
    if kind == "router":
        return (torch.randn(case["M"], case["E"], generator=g, device="cuda").to(DTYPES[case["dtype"]]),)
    if kind == "w4a16":
        return (_activations(case["M"], case["K"], g), *_int4(case["K"], case["N"], case["group"], g))
    if kind == "fp8":
        A = _activations(case["M"], case["K"], g, outliers=True)
        W = torch.randn(case["N"], case["K"], generator=g, device="cuda") * 0.02
        sw = W.abs().amax(dim=1) / 448.0
        return A, (W / sw[:, None]).to(torch.float8_e4m3fn), sw
    if kind == "fp8_block":
        K, N = case["K"], case["N"]
        A = _activations(case["M"], K, g, outliers=True)
        nb = -(-N // 128)
        W = torch.randn(nb * 128, K, generator=g, device="cuda") * 0.02
        W[N:] = 0
        tiles = W.view(nb, 128, K // 128, 128)
        sw = tiles.abs().amax(dim=(1, 3)) / 448.0
        return A, (tiles / sw[:, None, :, None]).view(nb * 128, K)[:N].to(torch.float8_e4m3fn).contiguous(), sw
    if kind == "moe":
        E, H, I = case["experts"], case["H"], case["I"]
        X = _activations(case["tokens"], H, g)
        logits = _router_logits(case["tokens"], E, g)
        return (X, logits, *_int4(H, 2 * I, case["group13"], g, (E,)), *_int4(I, H, case["group2"], g, (E,)))
    M, N, K = case["M"], case["N"], case["K"]
    if case["dtype"] == "int8":
        return (torch.randint(-64, 65, (M, K), generator=g, device="cuda", dtype=torch.int8),
                torch.randint(0, 256, (K // 4, N), generator=g, device="cuda", dtype=torch.uint8))
    to = torch.float8_e4m3fn if case["dtype"] == "fp8" else DTYPES[case["dtype"]]
    # products of unit variance; fp8 operands of equal size, so that few e4m3 codes are subnormal
    scale = K ** (-0.25 if case["dtype"] == "fp8" else -0.5)
    a = torch.randn(M, K, generator=g, device="cuda") * (scale if case["dtype"] == "fp8" else 1.0)
    b = torch.randn(K, N, generator=g, device="cuda") * scale
    return a.to(to), b.to(to)


def prepare(case, seed):
    state = dict(case, inputs=_inputs(case, seed))
    if case["kind"] == "w4a16" and case["layout"] == "slabs":
        from tilebench_amd.formats import w4a16_to_slabs

        A, packed, scales, zeros = state["inputs"]
        state["inputs"] = (A, w4a16_to_slabs(packed), scales, zeros)  # once, when the weights are loaded
    return state


# ----------------------------------------------------------------------------- one pass


def run(state):
    kind, x = state["kind"], state["inputs"]
    if kind == "router":
        from tilebench_amd.benchmarks.operators.moe_topk_gating import impl_hip

        return impl_hip.run(x[0], state["M"], state["E"], state["k"])
    if kind == "w4a16":
        from tilebench_amd.benchmarks.operators.w4a16_gemm import impl_hip

        return impl_hip.run(*x, state["group"])
    if kind == "fp8":
        from tilebench_amd.benchmarks.operators.fp8_act_quant import impl_hip as quant
        from tilebench_amd.benchmarks.operators.fp8_scaled_gemm import impl_hip as gemm

        A, WqT, sw = x
        Aq, sa = quant.run(A)
        return gemm.run(Aq, WqT.t(), sa, sw)
    if kind == "fp8_block":
        from tilebench_amd.benchmarks.operators.fp8_act_quant_blocks import impl_hip as quant
        from tilebench_amd.benchmarks.operators.fp8_block_scaled_gemm import impl_hip as gemm

        A, WqT, sw = x
        Aq, sa = quant.run(A)
        return gemm.run(Aq, WqT, sa, sw)
    if kind == "moe":
        from tilebench_amd.benchmarks.operators.fused_moe_w4a16 import impl_hip

        return impl_hip.run(*x, state["topk"], state["group13"], state["group2"])
    if state["dtype"] == "int8":
        from tilebench_amd.benchmarks.operators.matmul_int8 import impl_hip

        return impl_hip.run(*x)
    from tilebench_amd.benchmarks.operators.matmul_fp32_fp16_fp8 import impl_hip

    out = impl_hip.run(*x)
    return out.view(torch.uint8) if state["dtype"] == "fp8" else out  # the e4m3 codes


# ----------------------------------------------------------------------------- work


def _int4_bytes(K, N, group):
    return K * N // 2 + (K // group) * N * 2 + (K // group) * N // 2


def work(case):
    kind = case["kind"]
    if kind == "router":
        size = 4 if case["dtype"] == "fp32" else 2
        M, E, k = case["M"], case["E"], case["k"]
        return {"bytes": M * E * size + M * k * (size + 4), "flops": 0}
    if kind == "moe":
        T, k, E, H, I = case["tokens"], case["topk"], case["experts"], case["H"], case["I"]
        # an expert's weights are read if a token is routed to it
        logits = _router_logits(T, E, torch.Generator().manual_seed(0), device="cpu")
        used = torch.topk(logits, k, dim=1).indices.unique().numel()
        weights = used * (_int4_bytes(H, 2 * I, case["group13"]) + _int4_bytes(I, H, case["group2"]))
        return {"bytes": weights + 4 * T * H + 4 * T * E, "flops": 6 * T * k * H * I}
    M, N, K = case["M"], case["N"], case["K"]
    flops = 2 * M * N * K
    if kind == "w4a16":
        return {"bytes": 2 * M * K + _int4_bytes(K, N, case["group"]) + 2 * M * N, "flops": flops}
    if kind == "fp8":
        return {"bytes": 2 * M * K + N * K + 4 * N + 2 * M * N, "flops": flops}
    if kind == "fp8_block":
        return {"bytes": 2 * M * K + N * K + 4 * (-(-N // 128)) * (K // 128) + 2 * M * N, "flops": flops}
    if case["dtype"] == "int8":
        return {"bytes": M * K + K * N // 4 + 4 * M * N, "flops": flops}
    size = {"fp32": 4, "fp16": 2, "fp8": 1}[case["dtype"]]
    return {"bytes": (M * K + K * N + M * N) * size, "flops": flops}


# ----------------------------------------------------------------------------- results


def tolerance(case):
    kind = case["kind"]
    if kind == "router":
        # indices are exact; the weights are a softmax in fp32 rounded to the logits' type
        return {"rel": {"fp32": 1e-6, "fp16": 1e-3, "bf16": 8e-3}[case["dtype"]]}
    if kind == "w4a16":
        return {"rel": 1.2e-3}  # fp16 output and fp16 weights
    if kind in ("fp8", "fp8_block"):
        return {"rel": 7e-3}  # bf16 output of the same e4m3 codes
    if kind == "moe":
        return {"rel": 2e-3}  # fp16 gate/up, activation, per-slot and final values
    if case["dtype"] == "int8":
        return "exact"
    if case["dtype"] == "fp8":
        return {"rel": 0.0, "differ": 1e-3}  # bf16 and e4m3 roundings of sums in another order
    return {"rel": {"fp16": 1e-3, "fp32": 2e-5}[case["dtype"]]}


def _unpack(packed):
    """uint8 [.., N/2] -> codes [.., N], low nibble first."""
    return torch.stack((packed & 15, packed >> 4), dim=-1).flatten(-2).double()


def _dequant(packed, scales, zeros, group):
    """The fp16 weights the int4 format stands for, as fp64."""
    K, N = packed.shape[0], packed.shape[1] * 2
    q = _unpack(packed).view(K // group, group, N) - _unpack(zeros)[:, None, :]
    return (q * scales.double()[:, None, :]).half().double().view(K, N)


def _quantise(A):
    """e4m3 codes (as fp64) and fp32 scales (as fp64) of rows of 64-bit values of fp16 A."""
    s = (A.abs().amax(dim=-1, keepdim=True) / 448.0).float().double()
    return (A / s).float().to(torch.float8_e4m3fn).float().double(), s


def _bytes(v):
    return v.to(torch.bfloat16).float().to(torch.float8_e4m3fn).view(torch.uint8)


def exact(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    if kind == "router":
        v, i = torch.sort(x[0].double(), dim=1, descending=True, stable=True)
        return torch.softmax(v[:, :case["k"]], dim=1), i[:, :case["k"]].int()
    if kind == "w4a16":
        return x[0].double() @ _dequant(*x[1:], case["group"])
    if kind == "fp8":
        q, s = _quantise(x[0].double())
        return (q @ x[1].float().double().t()) * s * x[2].double()
    if kind == "fp8_block":
        A, WqT, sw = x
        M, K = A.shape
        q, s = _quantise(A.double().view(M, K // 128, 128))
        N = WqT.shape[0]
        sw = sw.double().repeat_interleave(128, dim=0)[:N].repeat_interleave(128, dim=1)
        return (q * s).view(M, K) @ (WqT.float().double() * sw).t()
    if kind == "moe":
        X, logits, W13, S13, Z13, W2, S2, Z2 = x
        v, ids = torch.topk(logits.double(), case["topk"], dim=1)
        w = torch.softmax(v, dim=1)
        out = torch.zeros(X.shape, dtype=torch.float64, device=X.device)
        for e in range(case["experts"]):
            tok, slot = torch.nonzero(ids == e, as_tuple=True)
            if tok.numel() == 0:
                continue
            h = X[tok].double() @ _dequant(W13[e], S13[e], Z13[e], case["group13"])
            gate, up = h.chunk(2, dim=1)
            y = (torch.nn.functional.silu(gate) * up) @ _dequant(W2[e], S2[e], Z2[e], case["group2"])
            out.index_add_(0, tok, y * w[tok, slot][:, None])
        return out
    a, b = x
    if case["dtype"] == "int8":
        B = torch.cat([((b >> (2 * i)) & 3) for i in range(4)], dim=0).double() - 1.0
        return (a.double() @ B).to(torch.int32)
    if case["dtype"] == "fp8":
        return _bytes(a.float().double() @ b.float().double())
    return a.double() @ b.double()

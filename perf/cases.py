"""What a program does with this library, as cases that can be timed: the five kernel entries of ``tiledcuda_amd``
(GEMM, back-to-back GEMM, attention, LSTM, scatter_nd) over the range of sizes that they accept, called the way a
program calls them - defaults wherever the entry has one, outputs and workspaces left to the call.

A case is a dict of plain values: ``op`` names the entry, the rest are its sizes and options.
"""
import math

import torch

import tiledcuda_amd as tcu

_DTYPES = {"f16": torch.float16, "f32": torch.float32}
# (N, K, P) of the fused two-GEMM example's driver that have a whole row block at M % 64 == 0
_B2B_WEIGHTS = ((64, 64, 64), (128, 64, 64), (256, 128, 128), (512, 128, 128), (1024, 128, 128), (2048, 128, 128))


def listed():
    return [
        # the README's product: one small tile, all latency and launch
        {"name": "gemm_128x64x256_f32", "op": "gemm", "M": 128, "N": 64, "K": 256, "out": "f32"},
        # a few rows against a full weight matrix (a decoding step, a small batch of requests): bound by the weights
        {"name": "gemm_32x4096x4096", "op": "gemm", "M": 32, "N": 4096, "K": 4096, "out": "f16"},
        # sizes that are whole 16 x 16 tiles and nothing more: edges in M, N and K at once
        {"name": "gemm_2064x1040x1072", "op": "gemm", "M": 2064, "N": 1040, "K": 1072, "out": "f16"},
        # the benchmark's product
        {"name": "gemm_4096x4096x4096", "op": "gemm", "M": 4096, "N": 4096, "K": 4096, "out": "f16"},
        # the benchmark's fused pair of products
        {"name": "b2b_8192x256x128x128", "op": "b2b", "M": 8192, "N": 256, "K": 128, "P": 128, "batch": 1, "out": "f16"},
        # prefill of a long prompt, 32 heads (the benchmark's longer sequence)
        {"name": "attn_h32_s8192_d128", "op": "attn", "batch": 32, "M": 8192, "N": 8192, "D": 128, "v": "row"},
        # a short block of new queries against a long cache of keys: the decoding direction
        {"name": "attn_h32_m64_n8192_d128", "op": "attn", "batch": 32, "M": 64, "N": 8192, "D": 128, "v": "row"},
        # 8 short sequences of 12 heads with the smaller head size, lengths that are not powers of two
        {"name": "attn_h96_s576_d64", "op": "attn", "batch": 96, "M": 576, "N": 576, "D": 64, "v": "row"},
        # the reference op's own call: one head, 64 queries, V column-major, flattened tensors
        {"name": "attn_op_m64_n256_d128", "op": "attn", "batch": 1, "M": 64, "N": 256, "D": 128, "v": "col"},
        # the benchmark's LSTM layer
        {"name": "lstm_t16_b256_i1024_h1024", "op": "lstm", "T": 16, "B": 256, "I": 1024, "H": 1024, "algo": "auto"},
        # a layer whose batch, input and hidden sizes are odd multiples of 16
        {"name": "lstm_t24_b80_i336_h656", "op": "lstm", "T": 24, "B": 80, "I": 336, "H": 656, "algo": "auto"},
        # gradients of 8192 looked-up rows added into a table: duplicate rows, f32
        {"name": "scatter_add_8192x1024_f32", "op": "scatter", "rows": 32768, "inner": 1, "slice": 1024, "n": 8192,
         "dtype": "f32", "mode": "add"},
    ]


def _log_uniform(rng, low, high, step):
    """A multiple of ``step`` in [low, high], spread evenly over the logarithm."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    return min(max(int(round(v / step)) * step, low), high)


def draw(rng):
    op = rng.choice(("gemm", "gemm", "b2b", "attn", "attn", "lstm", "scatter"))
    if op == "gemm":
        while True:
            M, N, K = (_log_uniform(rng, 16, 8192, 16) for _ in range(3))
            if rng.random() < 0.5:  # a layer's sizes are usually rounder than its batch
                N, K = max(64, N // 64 * 64), max(64, K // 64 * 64)
            if M * N * K <= 4096 ** 3 * 2:
                return {"op": op, "M": M, "N": N, "K": K, "out": rng.choice(("f16", "f16", "f32"))}
    if op == "b2b":
        N, K, P = rng.choice(_B2B_WEIGHTS)
        batch = rng.choice((1, 1, 2, 5, 16))
        M = _log_uniform(rng, 64, 65536 // batch // 64 * 64, 64)
        return {"op": op, "M": M, "N": N, "K": K, "P": P, "batch": batch, "out": rng.choice(("f16", "f32"))}
    if op == "attn":
        while True:
            v = rng.choice(("row", "row", "col"))
            D = 128 if v == "col" else rng.choice((64, 128))
            batch = _log_uniform(rng, 1, 128, 1)
            N = _log_uniform(rng, 64, 16384, 64)
            M = N if rng.random() < 0.5 else _log_uniform(rng, 64, 2048, 64)
            if batch * M * N * D <= 32 * 4096 * 4096 * 128 and batch * (M + N) * D <= 1 << 28:
                return {"op": op, "batch": batch, "M": M, "N": N, "D": D, "v": v}
    if op == "lstm":
        if rng.random() < 0.25:  # the single-launch layer, which a caller asks for by name
            H = rng.choice((256, 512, 768, 1024))
            B = 32 * rng.randint(1, 8)
            T = 8 * rng.randint(1, 3)
            return {"op": op, "T": T, "B": B, "I": _log_uniform(rng, 64, 1024, 64), "H": H, "algo": "persistent"}
        step = rng.choice((16, 16, 128))
        B = _log_uniform(rng, 16, 256, 16) if step == 16 else 64 * rng.randint(1, 4)
        I, H = (_log_uniform(rng, max(step, 64), 1024, step) for _ in range(2))
        return {"op": op, "T": _log_uniform(rng, 1, 24, 1), "B": B, "I": I, "H": H, "algo": "auto"}
    size = _log_uniform(rng, 16, 4096, 1)
    if rng.random() < 0.7:
        size = max(16, size // 8 * 8)
    n = _log_uniform(rng, 64, min(65536, (1 << 26) // size), 1)
    inner = rng.choice((1, 1, 7))
    rows = max(1, n * rng.choice((1, 2, 4)) // inner)
    return {"op": op, "rows": rows, "inner": inner, "slice": size, "n": min(n, rows * inner), "dtype": rng.choice(("f32", "f16")),
            "mode": rng.choice(("assign", "add"))}


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)

    def uniform(*shape):
        return torch.rand(*shape, generator=gen, device="cuda").mul_(2).sub_(1).half()

    def normal(*shape, std=1.0, dtype=torch.float16):
        return torch.randn(*shape, generator=gen, device="cuda").mul_(std).to(dtype)

    state = {"case": case}
    if case["op"] == "gemm":
        state["a"] = uniform(case["M"], case["K"])
        state["b_t"] = uniform(case["N"], case["K"])
    elif case["op"] == "b2b":
        b, M, N, K, P = (case[k] for k in ("batch", "M", "N", "K", "P"))
        state["a"] = normal(b, M, K, std=0.1)
        state["b_t"] = normal(b, N, K, std=0.1)
        state["c_t"] = normal(b, P, N, std=0.1)
    elif case["op"] == "attn":
        b, M, N, D = (case[k] for k in ("batch", "M", "N", "D"))
        state["q"], state["k"], state["v"] = normal(b, M, D), normal(b, N, D), normal(b, N, D)
        if case["v"] == "col":  # the op's convention: flattened, V stored [d, n], the output given by the caller
            state["v"] = state["v"].transpose(1, 2).contiguous()
            for name in ("q", "k", "v"):
                state[name] = state[name].flatten()
            state["o"] = torch.empty(b * M * D, dtype=torch.float16, device="cuda")
    elif case["op"] == "lstm":
        T, B, I, H = (case[k] for k in ("T", "B", "I", "H"))
        state["x"] = normal(T, B, I, std=0.5)
        state["W"] = normal(4 * H, I + H, std=0.05)
        state["bias"] = normal(4 * H, std=0.1)
        state["h0"] = normal(B, H, std=0.5)
        state["c0"] = normal(B, H, std=0.5, dtype=torch.float32)
    else:
        rows, inner, size, n = (case[k] for k in ("rows", "inner", "slice", "n"))
        dtype = _DTYPES[case["dtype"]]
        lead = (rows,) if inner == 1 else (rows, inner)
        state["data"] = normal(*lead, size, dtype=dtype)
        state["updates"] = normal(n, size, std=0.01, dtype=dtype)
        if case["mode"] == "assign":  # distinct rows: with duplicates any of their updates may stay
            flat = torch.randperm(rows * inner, generator=gen, device="cuda")[:n]
        else:
            flat = torch.randint(rows * inner, (n,), generator=gen, device="cuda")
        state["indices"] = (flat.view(n, 1) if inner == 1 else torch.stack((flat // inner, flat % inner), 1)).contiguous()
    return state


def run(state):
    case = state["case"]
    if case["op"] == "gemm":
        return tcu.gemm(state["a"], state["b_t"], out_dtype=_DTYPES[case["out"]])
    if case["op"] == "b2b":
        return tcu.b2b_gemm(state["a"], state["b_t"], state["c_t"], out_dtype=_DTYPES[case["out"]])
    if case["op"] == "attn":
        if case["v"] == "row":
            return tcu.flash_attention(state["q"], state["k"], state["v"])
        D = case["D"]
        tcu.flash_attention_fwd(state["q"], state["k"], state["v"], state["o"], case["M"], case["N"], D, D,
                                scale=1.0 / math.sqrt(D), batch=case["batch"])
        return state["o"]
    if case["op"] == "lstm":
        return tcu.lstm(state["x"], state["W"], state["bias"], state["h0"], state["c0"], algo=case["algo"])
    tcu.scatter_nd(state["data"], state["indices"], state["updates"], mode=case["mode"])
    return state["data"]


def work(case):
    if case["op"] == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * (M + N) * K + (2 if case["out"] == "f16" else 4) * M * N, "flops": 2 * M * N * K}
    if case["op"] == "b2b":
        b, M, N, K, P = (case[k] for k in ("batch", "M", "N", "K", "P"))
        return {"bytes": b * (2 * (M * K + N * K + P * N) + (2 if case["out"] == "f16" else 4) * M * P),
                "flops": 2 * b * M * N * (K + P)}
    if case["op"] == "attn":
        b, M, N, D = (case[k] for k in ("batch", "M", "N", "D"))
        return {"bytes": 2 * b * D * (2 * M + 2 * N), "flops": 4 * b * M * N * D}
    if case["op"] == "lstm":
        T, B, I, H = (case[k] for k in ("T", "B", "I", "H"))
        return {"bytes": 2 * (T * B * (I + H) + 4 * H * (I + H) + 4 * H + B * H) + 8 * B * H,
                "flops": 8 * T * B * H * (I + H)}
    size, n, elem = case["slice"], case["n"], 4 if case["dtype"] == "f32" else 2
    cells = case["rows"] * case["inner"]
    index = 8 * n * (1 if case["inner"] == 1 else 2)
    if case["mode"] == "assign":
        return {"bytes": 2 * n * size * elem + index, "flops": 0}
    distinct = int(cells * (1.0 - (1.0 - 1.0 / cells) ** n)) if cells > 1 else 1  # rows that n uniform indices touch
    return {"bytes": (n + 2 * distinct) * size * elem + index, "flops": n * size}


def tolerance(case):
    # Four times the relative error (2-norm) measured against the same path in 64 bits, over the listed and two dozen drawn
    # cases: rounding to f16 2.1e-4, with an f16 intermediate before it 2.9e-4, the attention path 3.7e-4, the LSTM layers
    # 2.6e-4; f32 outputs of products 1e-7 here and 1.6e-6 for the vendor library's f32 product in another order of the
    # sum; f32 additions into a table 1.3e-8 to 4e-8, in another order where rows are hit more than once.
    if case["op"] == "scatter":
        if case["mode"] == "assign":
            return "exact"
        return {"rel": 2e-7} if case["dtype"] == "f32" else {"rel": 8e-4}
    if case["op"] == "gemm":
        return {"rel": 6e-6} if case["out"] == "f32" else {"rel": 8e-4}
    if case["op"] == "b2b":
        return {"rel": 8e-4} if case["out"] == "f32" else {"rel": 1.2e-3}
    if case["op"] == "attn":
        return {"rel": 1.5e-3}
    return {"rel": 1e-3}

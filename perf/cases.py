"""The calls whose speed this library is judged by: C[M,N] = A[M,K] . B[N,K]^T on one GPU.

``listed()`` names a dozen calls, ``draw(rng)`` makes more of the same ranges.  Every case goes
through the package's public entry points on torch tensors that are already on the GPU, as a
program that keeps its weights and activations there calls them:

    "run"       runKernel            bf16, the library's own choice of kernel
    "gemm"      gpu_gemm             bf16 or fp16
    "epilogue"  gemm_epilogue        alpha / beta, row-major or column-major C
    "ws"        gemm_epilogue        with a caller-owned workspace (a loop that must not allocate)
    "golden"    reference_gpu_gemm   the order-preserving GEMM every run of the test program checks with

Operands: U[-1, 1) where both are generic matrices, A ~ N(0, 1) with B ~ N(0, 0.02^2) where A
stands for activations and B for weights.
"""
import math

import torch

import h100_gemm_amd as mi


def _case(entry, M, N, K, dtype="bf16", fill="uniform", col_major=False, alpha=1.0, beta=0.0):
    return {"entry": entry, "M": M, "N": N, "K": K, "dtype": dtype, "fill": fill, "col_major": col_major,
            "alpha": alpha, "beta": beta}


def listed():
    return [
        # one token of one sequence through a square projection: a matrix-vector product
        dict(_case("run", 1, 4096, 4096, fill="normal"), name="decode_1"),
        # the benchmark's decode shapes: a small and a full batch of tokens through 8192 x 8192 weights,
        # the latter from a serving loop that brings its own workspace
        dict(_case("run", 16, 8192, 8192, fill="normal"), name="decode_16"),
        dict(_case("ws", 128, 8192, 8192, fill="normal"), name="decode_128"),
        # the benchmark's smallest square: launch latency
        dict(_case("run", 512, 512, 512), name="square_512"),
        # small, odd in every extent, fp16 as the test program uses it
        dict(_case("gemm", 257, 515, 77, dtype="fp16"), name="ragged_small"),
        # few output tiles under a long K (a weight gradient: hidden x hidden over the tokens)
        dict(_case("run", 1024, 1024, 4096), name="few_tiles"),
        # mid-sized, with the golden's epilogue and the column-major C of the bf16 benchmark kernel
        dict(_case("epilogue", 1536, 1536, 1536, dtype="fp16", col_major=True, alpha=0.5, beta=0.25), name="mid_1536"),
        # a chunk of a prompt through a square projection
        dict(_case("run", 2048, 8192, 8192, fill="normal"), name="prefill_2048"),
        # the benchmark's ragged shape: no extent a multiple of anything, rows of A and B at odd offsets
        dict(_case("run", 4095, 6143, 3073), name="unaligned"),
        # the benchmark's headline
        dict(_case("run", 8192, 8192, 8192), name="square_8192"),
        # the benchmark's widest MLP projection
        dict(_case("run", 8192, 28672, 8192, fill="normal"), name="mlp_up"),
        # the golden of the test program at its default size
        dict(_case("golden", 4096, 4096, 4096), name="golden_4096"),
    ]


def _log_int(rng, lo, hi, step=1):
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(n / step)) * step))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "small", "small", "mid", "mid", "mid", "large", "large", "golden"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "decode":                      # 1 .. 128 tokens, weights of 1024 .. 28672 (whole 64s)
        while True:
            N, K = _log_int(rng, 1024, 28672, 64), _log_int(rng, 1024, 28672, 64)
            if N * K <= 28672 * 8192:
                break
        entry = rng.choice(["gemm", "gemm", "ws"])
        return _case(entry, _log_int(rng, 1, 128), N, K, dtype=dtype, fill="normal")
    if kind == "golden":
        M, N, K = (_log_int(rng, 256, 4096) for _ in range(3))
        return _case("golden", M, N, K, dtype=dtype)
    lo, hi_mn, hi_k = {"small": (32, 1024, 1024), "mid": (512, 4096, 16384), "large": (2048, 28672, 28672)}[kind]
    step = rng.choice([1, 8, 64, 128])        # half of the shapes aligned to a K slab, a quarter odd
    while True:
        M, N, K = _log_int(rng, lo, hi_mn, step), _log_int(rng, lo, hi_mn, step), _log_int(rng, lo, hi_k, step)
        if M * N * K <= 8192 * 28672 * 8192 and max(M * N, M * K, N * K) <= 28672 * 28672:
            break
    if rng.random() < 0.25:
        return _case("epilogue", M, N, K, dtype=dtype, col_major=rng.random() < 0.5, alpha=0.5, beta=0.25)
    return _case("gemm", M, N, K, dtype=dtype, fill=rng.choice(["uniform", "normal"]))


_TORCH = {"bf16": torch.bfloat16, "fp16": torch.float16}
_MI = {"bf16": mi.MI_DTYPE_BF16, "fp16": mi.MI_DTYPE_FP16}


def prepare(case, seed):
    M, N, K, dt = case["M"], case["N"], case["K"], _TORCH[case["dtype"]]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    if case["fill"] == "uniform":
        A = torch.empty(M, K, dtype=dt, device="cuda").uniform_(-1.0, 1.0, generator=gen)
        B = torch.empty(N, K, dtype=dt, device="cuda").uniform_(-1.0, 1.0, generator=gen)
    else:
        A = torch.empty(M, K, dtype=dt, device="cuda").normal_(0.0, 1.0, generator=gen)
        B = torch.empty(N, K, dtype=dt, device="cuda").normal_(0.0, 0.02, generator=gen)
    C = torch.empty((N, M) if case["col_major"] else (M, N), dtype=dt, device="cuda")
    state = {"case": dict(case), "A": A, "B": B, "C": C, "dtype": _MI[case["dtype"]],
             "params": mi.GemmParams(M, N, K, A, B, C, case["alpha"], case["beta"]),
             "layout": mi.MI_C_COL_MAJOR if case["col_major"] else mi.MI_C_ROW_MAJOR, "workspace": None}
    if case["entry"] == "ws":
        state["workspace"] = mi.DeviceBuffer(mi.workspace_bytes(M, N, K, dtype=state["dtype"]))
    return state


def run(state):
    c, entry = state["case"], state["case"]["entry"]
    if entry == "run":
        mi.runKernel(c["M"], c["N"], c["K"], state["A"], state["B"], state["C"])
    elif entry == "gemm":
        mi.gpu_gemm(state["params"], dtype=state["dtype"])
    elif entry == "golden":
        mi.reference_gpu_gemm(state["params"], dtype=state["dtype"])
    else:
        mi.gemm_epilogue(state["params"], dtype=state["dtype"], c_layout=state["layout"], workspace=state["workspace"])
    return state["C"]


def work(case):
    M, N, K = case["M"], case["N"], case["K"]
    return {"bytes": 2.0 * (M * K + N * K + M * N), "flops": 2.0 * M * N * K}


def tolerance(case):
    # The golden has one result: a single fp32 accumulator per element fed in ascending k.
    if case["entry"] == "golden":
        return "exact"
    # Four times the distance of the result from the product in float64 (the rounding of C to the
    # storage type: 1.65e-3 for bf16, 2.07e-4 for fp16, whatever the shape); `max` is two units in
    # the last place of the storage type.
    return {"rel": 6.6e-3, "max": 1.6e-2} if case["dtype"] == "bf16" else {"rel": 8.3e-4, "max": 2.0e-3}

"""The workloads whose speed this framework is judged by.

Every case is one call of a public entry point of ridge_amd.gemm on buffers that
the caller owns, at the sizes the framework's own benchmark, sweeps and checks
use, each GEMM with the table row that the committed sweeps (or the rows timed
against each other on that shape) found fastest, as a program that tuned its
shape would call it. Inputs are FP16, U[-1, 1), the benchmark's distribution;
C is FP16 and the sums are FP32. A case names its row by the seven fields of the
kernel table:

    listed()             the standing cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program holds before the call
    run(state)           one pass
    work(case)           the bytes and operations a pass cannot do without
    tolerance(case)      how far two correct results may lie apart
    exact(case, seed)    the result in 64 bits, without this package's code
"""

import math

import numpy as np
import torch

from ridge_amd import gemm as G

DEVICE = "cuda:0"


def _row(BM, BN, BK, WM, WN, stages, groupM):
    return "%d,%d,%d,%d,%d,%d,%d" % (BM, BN, BK, WM, WN, stages, groupM)


# The rows that the sweeps rank first somewhere, by the kind of shape they win.
SQUARE64 = [_row(64, 64, 64, 32, 32, 4, 8), _row(64, 64, 32, 32, 32, 4, 8), _row(128, 64, 64, 64, 32, 3, 8)]
MIDDLE = [_row(128, 128, 64, 64, 64, 4, 8), _row(128, 128, 64, 64, 64, 2, 8), _row(128, 128, 32, 64, 64, 4, 8),
          _row(128, 64, 128, 64, 32, 3, 8), _row(256, 128, 64, 64, 64, 3, 8)]
LARGE = [_row(256, 256, 32, 128, 64, 3, 4), _row(256, 256, 32, 128, 64, 4, 4), _row(256, 256, 32, 128, 64, 4, 8),
         _row(256, 256, 32, 64, 128, 4, 4)]
SMALL_K = [_row(256, 128, 32, 64, 64, 6, 4), _row(128, 128, 64, 64, 64, 4, 8)]
TALL = [_row(64, 128, 128, 32, 64, 3, 8), _row(128, 64, 128, 64, 32, 3, 8), _row(128, 64, 64, 64, 32, 6, 8)]

# A pass multiplies at most this much (6144 x 3072 x 6144), and a fill writes at
# most this many elements (8192 x 8192).
MOST_MNK = 6144 * 3072 * 6144
MOST_FILL = 8192 * 8192
LEAST_SPLIT_K = 1024


def _gemm(name, call, M, N, K, row, tail=""):
    return {"name": name, "kind": "gemm", "call": call, "M": M, "N": N, "K": K, "row": row, "tail": tail}


def _fill(name, fill, n):
    return {"name": name, "kind": "fill", "fill": fill, "n": n}


def listed():
    return [
        # The smallest calls: gemm(A, B, row) on a correctness-check shape, C
        # allocated by the call. Launch and host latency.
        _gemm("gemm_256x512x128", "gemm", 256, 512, 128, SQUARE64[0]),
        # The benchmark's small square: one 64 x 64 tile per CU, 16 K tiles deep.
        _gemm("launch_1024cube", "bound", 1024, 1024, 1024, SQUARE64[0]),
        # Ragged: 273 tiles of 64 x 64 (no larger tile divides it), 29 K tiles.
        _gemm("launch_1344x832x1856", "launch", 1344, 832, 1856, SQUARE64[0]),
        # The largest correctness-check shape: one 128 x 128 tile per CU.
        _gemm("launch_2048cube", "bound", 2048, 2048, 2048, MIDDLE[0]),
        # The headline benchmark: one 256 x 256 tile per CU, 128 K tiles.
        _gemm("launch_4096cube", "bound", 4096, 4096, 4096, LARGE[0]),
        # A large grid at moderate depth, of the registered sweep: four tiles per
        # CU, 32 K tiles each.
        _gemm("launch_8192x8192x1024", "bound", 8192, 8192, 1024, LARGE[0]),
        # A grid just over whole rounds of the chip (529 tiles on 256 CUs), of a
        # held-out sweep.
        _gemm("launch_5888x5888x1664", "bound", 5888, 5888, 1664, LARGE[0]),
        # The benchmark's small-K shape: writing C is the cost.
        _gemm("launch_8192x8192x128", "bound", 8192, 8192, 128, SMALL_K[0]),
        # The benchmark's tall-skinny shape: reading A is the cost.
        _gemm("launch_16384x128x8192", "bound", 16384, 128, 8192, TALL[0]),
        # The row split of the benchmark: whole rounds of 256 x 256 tiles, then
        # the other rows of C with a smaller tile.
        _gemm("split_6144x3072x6144", "split", 6144, 3072, 6144, LARGE[0], MIDDLE[0]),
        # The inputs every benchmark and sweep makes first, and those of the
        # correctness check.
        _fill("fill_uniform_8192x8192", "uniform", 8192 * 8192),
        _fill("fill_lcg_2048x2048", "lcg", 2048 * 2048),
    ]


def _log_int(rng, lo, hi):
    """An integer in [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _fields(row):
    return tuple(int(x) for x in row.split(","))


def _sized(rng, row, m, n, k):
    """M, N, K of the row's tiles within the given (low, high) ranges."""
    BM, BN, BK = _fields(row)[:3]
    return tuple(b * _log_int(rng, max(1, -(-lo // b)), max(1, hi // b)) for b, (lo, hi) in ((BM, m), (BN, n), (BK, k)))


def draw(rng):
    kind = rng.choice(["small", "small", "middle", "middle", "large", "large", "large", "small_k", "tall", "split",
                       "fill"])
    if kind == "fill":
        return {"kind": "fill", "fill": rng.choice(["uniform", "lcg"]), "n": _log_int(rng, 1 << 17, MOST_FILL)}
    rows, m, n, k = {
        "small": (SQUARE64, (64, 1536), (64, 1536), (64, 4096)),
        "middle": (MIDDLE, (256, 3072), (256, 4096), (128, 4096)),
        "large": (LARGE, (1024, 10240), (1024, 10240), (128, 8192)),
        "small_k": (SMALL_K, (1024, 16384), (1024, 8192), (64, 256)),
        "tall": (TALL, (2048, 16384), (128, 256), (1024, 8192)),
        "split": (LARGE[:3], (1024, 8192), (1024, 8192), (LEAST_SPLIT_K, 6144)),
    }[kind]
    while True:
        row = rng.choice(rows)
        M, N, K = _sized(rng, row, m, n, k)
        case = {"kind": "gemm", "call": "bound", "M": M, "N": N, "K": K, "row": row, "tail": ""}
        if kind == "split":
            # Between one and two rounds of 256 x 256 tiles on 256 CUs.
            if not 256 < (M // 256) * (N // 256) < 448:
                continue
            K = -(-K // 64) * 64
            case.update(call="split", K=K, tail=MIDDLE[0])
        elif kind == "small":
            case["call"] = rng.choice(["gemm", "launch", "bound"])
        if M * N * K <= MOST_MNK and M * N <= 8192 * 8192:
            return case


def _index(row):
    i = G.find_variant(*_fields(row))
    if i < 0:
        raise ValueError("no such row: %s" % row)
    return i


def _operands(case, seed):
    M, N, K = case["M"], case["N"], case["K"]
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    A = torch.rand((M, K), generator=g, device=DEVICE).mul_(2).sub_(1).half()
    B = torch.rand((K, N), generator=g, device=DEVICE).mul_(2).sub_(1).half()
    return A, B


def prepare(case, seed):
    if case["kind"] == "fill":
        t = torch.empty(case["n"], dtype=torch.float16, device=DEVICE)
        fill = {"uniform": G.fill_uniform, "lcg": G.fill_lcg}[case["fill"]]
        return lambda: fill(t, seed)
    M, N, K, i = case["M"], case["N"], case["K"], _index(case["row"])
    A, B = _operands(case, seed)
    if case["call"] == "gemm":
        return lambda: G.gemm(A, B, i)
    C = torch.empty((M, N), dtype=torch.float16, device=DEVICE)
    if case["call"] == "launch":
        def call():
            rc = G.launch(i, A, B, C, M, N, K)
            if rc != G.HIP_SUCCESS:
                raise RuntimeError("launch returned %d" % rc)
    elif case["call"] == "bound":
        call = G.bound_launch(i, A, B, C, M, N, K)
    else:
        call = G.bound_launch_split(i, _index(case["tail"]), G.split_rows(i, M, N, K), A, B, C, M, N, K)

    def launched():
        call()
        return C
    return launched


def run(state):
    return state()


def work(case):
    if case["kind"] == "fill":
        return {"bytes": 2 * case["n"], "flops": 0}
    M, N, K = case["M"], case["N"], case["K"]
    return {"bytes": 2 * (M * K + K * N + M * N), "flops": 2 * M * N * K}


def tolerance(case):
    """A fill is a pure function of the seed and the index. A GEMM rounds an FP32
    sum to FP16 once: against the 64-bit product it measures 2.1e-4 (2-norm) and,
    for one element, half an FP16 unit, 4.9e-4 of its value; about four times
    both."""
    return "exact" if case["kind"] == "fill" else {"rel": 8e-4, "max": 2e-3}


def _uniform_values(n, seed):
    """Element i: the top 24 bits of output i of the splitmix64 stream of `seed`,
    as a multiple of 2^-23, less 1."""
    z = np.arange(1, n + 1, dtype=np.uint64)
    z *= np.uint64(0x9e3779b97f4a7c15)
    z += np.uint64(seed)
    z ^= z >> np.uint64(30)
    z *= np.uint64(0xbf58476d1ce4e5b9)
    z ^= z >> np.uint64(27)
    z *= np.uint64(0x94d049bb133111eb)
    z ^= z >> np.uint64(31)
    return (z >> np.uint64(40)).astype(np.float64) * 2.0 ** -23 - 1.0


def _lcg_values(n, seed):
    """Element i from the state after i + 1 steps of s -> 1664525 s + 1013904223
    mod 2^32: bits 16 .. 30 over 32767, less 0.5. States are made by doubling:
    the second half of 2k states is the k-step map of the first half."""
    mul, add = 1664525, 1013904223
    s = np.array([(mul * seed + add) & 0xffffffff], dtype=np.uint32)
    while s.size < n:
        s = np.concatenate([s, s * np.uint32(mul) + np.uint32(add)])
        mul, add = (mul * mul) & 0xffffffff, (mul * add + add) & 0xffffffff
    return ((s[:n] >> np.uint32(16)) & np.uint32(0x7fff)).astype(np.float64) / 32767.0 - 0.5


def exact(case, seed):
    if case["kind"] == "fill":
        values = {"uniform": _uniform_values, "lcg": _lcg_values}[case["fill"]](case["n"], seed)
        return torch.from_numpy(values)
    A, B = _operands(case, seed)
    return A.double() @ B.double()

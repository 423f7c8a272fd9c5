"""Performance cases of the MI355X backend: what a program does with it.

Every case compiles a tforge program once (`prepare`) and launches it on device
tensors (`run`), as bench.py and the serving examples do.  Three kinds of
option strings are in use and all are here:

  * none, or plain block / thread tiles: what `--tforge-gpu-pipeline` gives
    without tile-k.  The result is one fused multiply-add chain per output in
    sequential k (the E1 numerics rows and the naive rungs run it);
  * the autotuned strings of tuned_configs.json, mask-edges for ragged shapes;
  * element-op programs (no matmul), default and row-shaped block tiles.

Inputs are uniform in [-1, 1] (the residual block: the scaled normals of
tforge_cpu.make_inputs), drawn on the GPU from the seed.
"""

import math

import torch

from tensorforge_amd import _lib
from tensorforge_amd import tforge_cpu as tc

STAGED = "block-tile={} thread-tile={} tile-k={} promote=1 vectorize=1"
SMALL_TILES = STAGED.format("32,32", "2,2", 32)       # tuned pick at 256^3 and 512^3
MID_TILES = STAGED.format("64,64", "4,4", 16)         # tuned pick at 1024^3 and the ragged shapes
WIDE_TILES = STAGED.format("128,64", "8,4", 16)       # tuned pick at 3000x2000x1000
LARGE_TILES = STAGED.format("128,128", "8,8", 16)     # tuned pick from 2048^3 up
SHORT_K_TILES = STAGED.format("128,128", "4,8", 8)    # tuned pick at 4096x4096x256
WAVE_TILES = STAGED.format("32,32", "1,1", 32) + " wave-split-k=1"   # tuned pick at 64x4096x4096
SPLIT_TILES = STAGED.format("64,64", "4,4", 16) + " split-k=4"       # the cost model's pick there
ROW_TILES = "block-tile=4,256 thread-tile=1,4"        # element ops: one 128-bit vector per thread
MASK = " mask-edges=1"

GEMM = ("matmul", "mbr", "resmlp")


def _case(workload, m, n, k, options, name=None):
    case = {"workload": workload, "m": m, "n": n, "k": k, "options": options}
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # The smallest program in the repository (examples/mbr.mlir's shape) as it compiles with no options:
        # latency of one launch and of a 128-long chain.
        _case("mbr", 256, 256, 128, "", "example_default"),
        # A small tuned layer: launch path and first loads.
        _case("mbr", 512, 512, 512, SMALL_TILES, "layer_512"),
        # An odd-sized layer with no options: the default path has no padding and no tile rules.
        _case("mbr", 777, 1111, 333, "", "ragged_default"),
        # A square matmul with register tiles but no K staging (thread-tile only, the reference's tiled naive form).
        _case("matmul", 1000, 1000, 1000, "block-tile=64,64 thread-tile=4,4", "matmul_1000_direct"),
        # The same odd-sized layer as a tuned program, edges masked in the kernel.
        _case("mbr", 777, 1111, 333, MID_TILES + MASK, "ragged_masked"),
        # A large layer one off the tile grid in every dimension.
        _case("mbr", 4095, 4097, 1023, MID_TILES + MASK, "ragged_large"),
        # The headline fused layer.
        _case("mbr", 2048, 2048, 2048, LARGE_TILES, "layer_2048"),
        # A layer on 64 rows (small-batch serving): few output tiles, long K.
        _case("mbr", 64, 4096, 4096, WAVE_TILES, "skinny_64"),
        # A short-K layer: dominated by writing C.
        _case("mbr", 4096, 4096, 256, SHORT_K_TILES, "short_k"),
        # The two-layer residual MLP block, the largest program: two fused launches, one intermediate.
        _case("resmlp", 4096, 2048, 8192, LARGE_TILES, "residual_block"),
        # A stand-alone activation chain relu(x + bias) + r on odd rows with no options.
        _case("chain", 2047, 4093, 0, "", "activation_default"),
        # A stand-alone residual add over 256 MiB tensors, row-shaped tiles: pure HBM stream.
        _case("add", 8192, 8192, 0, ROW_TILES, "add_rows_8192"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _up(x, t):
    return -(-x // t) * t


def draw(rng):
    kind = rng.choice(["direct", "direct", "tuned", "masked", "skinny", "short_k", "block", "elements", "elements"])
    if kind == "direct":
        tm, tn = rng.choice([(1, 1), (1, 1), (2, 2), (4, 4), (8, 4)])
        opts = "" if (tm, tn) == (1, 1) else f"block-tile={16 * tm},{16 * tn} thread-tile={tm},{tn}"
        m, n, k = (_log(rng, 100, 1500) for _ in range(3))
        return _case(rng.choice(["mbr", "matmul"]), m, n, k, opts)
    if kind == "tuned":
        opts, t, lo, hi = rng.choice([(SMALL_TILES, 32, 64, 700), (MID_TILES, 64, 512, 1600),
                                      (LARGE_TILES, 128, 1500, 4096)])
        m, n, k = (_up(_log(rng, lo, hi), t) for _ in range(3))
        return _case(rng.choice(["mbr", "matmul"]), m, n, k, opts)
    if kind == "masked":
        opts = rng.choice([SMALL_TILES, MID_TILES, MID_TILES, WIDE_TILES])
        lo, hi = (48, 700) if opts == SMALL_TILES else (500, 4000)
        m, n, k = _log(rng, lo, hi), _log(rng, lo, hi), _log(rng, 100, 1500)
        return _case(rng.choice(["mbr", "matmul"]), m, n, k, opts + MASK)
    if kind == "skinny":
        opts, t = rng.choice([(WAVE_TILES, 32), (WAVE_TILES, 32), (SPLIT_TILES, 64)])
        return _case("mbr", rng.choice([t, 64, 128]), _up(_log(rng, 1024, 8192), 64), _up(_log(rng, 1024, 8192), 64),
                     opts)
    if kind == "short_k":
        return _case("mbr", _up(_log(rng, 1024, 6144), 128), _up(_log(rng, 1024, 6144), 128),
                     _up(_log(rng, 64, 384), 16), SHORT_K_TILES)
    if kind == "block":
        # The residual block with no options on odd sizes, or tuned on tile multiples.
        if rng.random() < 0.5:
            return _case("resmlp", _log(rng, 64, 700), _log(rng, 64, 700), _log(rng, 100, 1500), "")
        return _case("resmlp", _up(_log(rng, 128, 2048), 128), _up(_log(rng, 256, 2048), 128),
                     _up(_log(rng, 512, 4096), 128), LARGE_TILES)
    rows, cols = _log(rng, 500, 8192), _log(rng, 500, 8192)
    return _case(rng.choice(["relu", "bias_add", "add", "chain"]), rows, cols, 0, rng.choice(["", "", ROW_TILES]))


def _program(case):
    w, m, n, k = case["workload"], case["m"], case["n"], case["k"]
    if w != "chain":
        return tc.gen_mlir(w, m, n, k if w in GEMM else None)
    t, v = f"tensor<{m}x{n}xf32>", f"tensor<{n}xf32>"
    return (f"func.func @entry(%x: {t}, %bias: {v}, %r: {t}) -> {t} {{\n"
            f"  %0 = tforge.bias_add %x, %bias : {t}, {v} -> {t}\n"
            f"  %1 = tforge.relu %0 : {t} -> {t}\n"
            f"  %2 = tforge.add %1, %r : {t}, {t} -> {t}\n"
            f"  return %2 : {t}\n}}\n")


def _inputs(case, seed):
    w, m, n, k = case["workload"], case["m"], case["n"], case["k"]
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def u(*shape):
        return torch.rand(shape, generator=gen, device="cuda", dtype=torch.float32) * 2 - 1

    def g(sigma, *shape):
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * sigma

    if w == "matmul":
        return [u(m, k), u(k, n)]
    if w == "mbr":
        return [u(m, k), u(k, n), u(n)]
    if w == "resmlp":
        return [g(1.0, m, n), g(n ** -0.5, n, k), g(0.02, k), g(k ** -0.5, k, n), g(0.02, n)]
    if w == "relu":
        return [u(m, n)]
    if w == "bias_add":
        return [u(m, n), u(n)]
    if w == "add":
        return [u(m, n), u(m, n)]
    return [u(m, n), u(n), u(m, n)]


def prepare(case, seed):
    kern = _lib.Kernel(_program(case), case["options"], "case.mlir")
    ins = _inputs(case, seed)
    out = torch.empty((case["m"], case["n"]), device="cuda", dtype=torch.float32)
    return {"kern": kern, "ins": ins, "out": out}


def run(state):
    out = state["out"]
    state["kern"].launch([t.data_ptr() for t in state["ins"]] + [out.data_ptr()],
                         torch.cuda.current_stream().cuda_stream)
    return out


def work(case):
    w, m, n, k = case["workload"], case["m"], case["n"], case["k"]
    if w == "resmlp":
        return {"bytes": 4 * (2 * m * n + 2 * n * k + n + k), "flops": 4 * m * n * k}
    if w in GEMM:
        return {"bytes": 4 * (m * k + k * n + m * n + (n if w == "mbr" else 0)), "flops": 2 * m * n * k}
    tensors, ops, vec = {"relu": (2, 1, 0), "bias_add": (2, 1, 1), "add": (3, 1, 0), "chain": (3, 3, 1)}[w]
    return {"bytes": 4 * (tensors * m * n + vec * n), "flops": ops * m * n}


def tolerance(case):
    w = case["workload"]
    if w not in GEMM:
        return "exact"  # one IEEE operation per element and op
    # Rounding of a K-long float32 sum of products of either sign grows with sqrt(K); any order of the sum.
    k = max(case["n"], case["k"]) if w == "resmlp" else case["k"]
    rel = 1e-7 * math.sqrt(max(k, 16))
    return {"rel": rel, "max": 10 * rel}


def exact(case, seed):
    w = case["workload"]
    x = [t.double() for t in _inputs(case, seed)]
    if w == "matmul":
        return x[0] @ x[1]
    if w == "mbr":
        return torch.clamp_min(x[0] @ x[1] + x[2], 0)
    if w == "resmlp":
        h = torch.clamp_min(x[0] @ x[1] + x[2], 0)
        return torch.clamp_min(h @ x[3] + x[4], 0) + x[0]
    if w == "relu":
        return torch.clamp_min(x[0], 0)
    if w == "chain":
        return torch.clamp_min(x[0] + x[1], 0) + x[2]
    return x[0] + x[1]

"""The direct kernel's chains on the matrix cores (sequential k, chosen by size
on 16-byte aligned buffers) against the one-thread-per-output kernel that runs on
unaligned buffers, and against the oracle's sequential FMA.  All three are the
same bits: one fused multiply-add per k in order from +0.0."""

import numpy as np
import pytest

from oracle import oracle as o
from tensorforge_amd import _lib
from tensorforge_amd import tforge_cpu as tc

pytestmark = pytest.mark.gpu

# relu(A @ B + bias) + R, then doubled: every epilogue op, in one chain.
CHAIN = """func.func @entry(%a: {a}, %b: {b}, %bias: {v}, %r: {c}) -> {c} {{
  %0 = tforge.matmul %a, %b : {a}, {b} -> {c}
  %1 = tforge.bias_add %0, %bias : {c}, {v} -> {c}
  %2 = tforge.relu %1 : {c} -> {c}
  %3 = tforge.add %2, %r : {c}, {c} -> {c}
  %4 = tforge.add %3, %3 : {c}, {c} -> {c}
  return %4 : {c}
}}
"""


def _program(workload, m, n, k):
    if workload != "chain":
        return tc.gen_mlir(workload, m, n, k)
    t = lambda *d: "tensor<" + "x".join(map(str, d)) + "xf32>"
    return CHAIN.format(a=t(m, k), b=t(k, n), v=t(n), c=t(m, n))


def _inputs(workload, m, n, k, scale=1.0):
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    u = lambda *s: (rng.uniform(-1, 1, s) * scale).astype(np.float32)
    ins = [u(m, k), u(k, n)]
    if workload != "matmul":
        ins.append(u(n))
    if workload == "chain":
        ins.append(u(m, n))
    return ins


def _launch(kern, ins, m, n, offset):
    """Output of kern with every buffer `offset` floats past a 256-byte boundary."""
    import torch
    dev, bufs = torch.device("cuda:0"), []
    for v in ins + [np.full((m, n), np.nan, np.float32)]:
        base = torch.zeros(v.size + offset, device=dev)
        base[offset:] = torch.from_numpy(v.ravel()).to(dev)
        bufs.append(base[offset:])
    assert all(b.data_ptr() % 16 == 4 * offset for b in bufs)
    kern.launch([b.data_ptr() for b in bufs], torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return bufs[-1].cpu().numpy().reshape(m, n)


# Tile multiples and ragged sizes of each tile (seq_entry's rule): 32x32 with
# tile-k 32 and 64, 64x64, 128x128; one row, one column, fewer columns than a
# vector, one below / above a tile, K of one, below a slab, and one past it.
SHAPES = [(1, 1, 1), (1, 500, 64), (33, 1, 17), (5, 3, 40), (32, 32, 32), (31, 33, 31), (65, 63, 97),
          (256, 256, 128), (64, 96, 2048), (65, 70, 2049), (1024, 1024, 128), (1021, 1023, 131),
          (1025, 1022, 129), (4096, 4096, 256), (4095, 4093, 270)]


@pytest.mark.parametrize("workload", ["matmul", "mbr", "chain"])
@pytest.mark.parametrize("shape", SHAPES)
def test_matrix_core_chain_is_bitwise_the_direct_kernel(workload, shape):
    m, n, k = shape
    ins = _inputs(workload, m, n, k)
    kern = _lib.Kernel(_program(workload, m, n, k), "", "t.mlir")
    got = _launch(kern, ins, m, n, 0)
    assert o.bitwise_diff(got, _launch(kern, ins, m, n, 1)) == 0
    if m * n * k <= 1 << 24:
        want = o.matmul_fma(ins[0], ins[1])
        if workload != "matmul":
            want = o.epilogue(want, ins[2], relu=True)
        if workload == "chain":
            want = o.add(want, ins[3])
            want = o.add(want, want)
        assert o.bitwise_diff(got, want) == 0


@pytest.mark.parametrize("shape", [(5, 7, 33), (32, 32, 32), (65, 130, 41), (1021, 1023, 131)])
@pytest.mark.parametrize("scale", [1e-20, 1e-23, 1e18])
def test_matrix_core_chain_denormals_signed_zeros_and_overflow(shape, scale):
    """Products around 1e-40 (denormal sums), 1e-46 (each rounds to +0.0 or -0.0, so
    the K tail's padding must leave a -0.0 accumulator alone) and 1e36."""
    m, n, k = shape
    a, b = _inputs("matmul", m, n, k, scale)
    a[0] = np.abs(a[0])
    b[:, 0] = -np.abs(b[:, 0])  # out[0, 0]: every product negative
    kern = _lib.Kernel(_program("matmul", m, n, k), "", "t.mlir")
    got = _launch(kern, [a, b], m, n, 0)
    assert o.bitwise_diff(got, _launch(kern, [a, b], m, n, 1)) == 0
    assert np.signbit(got[0, 0])
    if m * n * k <= 1 << 24:
        assert o.bitwise_diff(got, o.matmul_fma(a, b)) == 0


@pytest.mark.parametrize("shape", [(40, 36, 64), (39, 35, 61)])
def test_residual_block_without_options_is_bitwise_the_oracle(shape):
    m, n, k = shape
    ins = tc.make_inputs("resmlp", m, n, k)
    x, w1, b1, w2, b2 = (np.ascontiguousarray(v) for v in ins.values())
    kern = _lib.Kernel(tc.gen_mlir("resmlp", m, n, k), "", "t.mlir")
    h = o.epilogue(o.matmul_fma(x, w1), b1, relu=True)
    want = o.add(o.epilogue(o.matmul_fma(h, w2), b2, relu=True), x)
    assert o.bitwise_diff(_launch(kern, [x, w1, b1, w2, b2], m, n, 0), want) == 0

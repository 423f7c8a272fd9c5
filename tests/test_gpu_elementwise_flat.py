"""Element-op programs on aligned buffers run as one stream of 128-bit vectors
whatever the shape: bit-exact against the oracle where rows, vectors, segments and
the whole stream do not line up."""

import numpy as np
import pytest

from oracle import oracle as o
from tensorforge_amd import _lib
from tensorforge_amd import tforge_cpu as tc

pytestmark = pytest.mark.gpu

CHAIN = """func.func @entry(%x: {t}, %bias: {v}, %r: {t}) -> {t} {{
  %0 = tforge.bias_add %x, %bias : {t}, {v} -> {t}
  %1 = tforge.relu %0 : {t} -> {t}
  %2 = tforge.add %1, %r : {t}, {t} -> {t}
  %3 = tforge.add %2, %2 : {t}, {t} -> {t}
  return %3 : {t}
}}
"""


def _launch(program, ins, m, n, bias_offset=0):
    import torch
    dev, bufs = torch.device("cuda:0"), []
    for v in ins + [np.full((m, n), np.nan, np.float32)]:
        off = bias_offset if v.ndim == 1 else 0
        base = torch.zeros(v.size + off, device=dev)
        base[off:] = torch.from_numpy(v.ravel()).to(dev)
        bufs.append(base[off:])
    kern = _lib.Kernel(program, "", "t.mlir")
    kern.launch([b.data_ptr() for b in bufs], torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return bufs[-1].cpu().numpy().reshape(m, n)


# Less than a vector, vectors over several rows, a stream of whole vectors on odd
# rows, one wave piece (256 elements) and one more, a segment (8192), a workgroup
# span (65536) and around it, several spans.
@pytest.mark.parametrize("shape", [(1, 1), (3, 1), (1, 3), (5, 1), (7, 2), (9, 3), (4, 5), (1, 256), (1, 257), (64, 129),
                                   (8, 1024), (8, 1025), (256, 256), (255, 257), (257, 255), (1000, 333), (301, 2049)])
@pytest.mark.parametrize("bias_offset", [0, 1])
def test_chain_bit_exact(shape, bias_offset):
    m, n = shape
    rng = np.random.default_rng(m * 1009 + n)
    x, r = (rng.uniform(-1, 1, (m, n)).astype(np.float32) for _ in range(2))
    bias = rng.uniform(-1, 1, n).astype(np.float32)
    t = f"tensor<{m}x{n}xf32>"
    got = _launch(CHAIN.format(t=t, v=f"tensor<{n}xf32>"), [x, bias, r], m, n, bias_offset)
    y = o.add(o.relu(o.bias_add(x, bias)), r)
    assert o.bitwise_diff(got, o.add(y, y)) == 0


# Two biases (0, 1) or two add operands (2, 3) in a chain: read from the epilogue's own
# table instead of the preloaded arguments.
@pytest.mark.parametrize("shape", [(1, 1), (5, 1), (7, 2), (9, 3), (4, 5), (1, 257), (64, 129), (257, 255), (301, 2049)])
@pytest.mark.parametrize("ops", [(0, 1, 2, 3), (0, 1), (2, 3), (0, 2, 3), (3, 1, 0), (2, "relu", 3, 1), ("self", 0, 1)])
def test_several_biases_and_adds_bit_exact(shape, ops):
    m, n = shape
    rng = np.random.default_rng(m * 1009 + n)
    x, r1, r2 = (rng.uniform(-1, 1, (m, n)).astype(np.float32) for _ in range(3))
    b1, b2 = (rng.uniform(-1, 1, n).astype(np.float32) for _ in range(2))
    t, v = f"tensor<{m}x{n}xf32>", f"tensor<{n}xf32>"
    lines, want, cur = [], x, "%x"
    for i, op in enumerate(ops):
        if op == "relu":
            lines.append(f"  %{i} = tforge.relu {cur} : {t} -> {t}")
            want = o.relu(want)
        elif op == "self":
            lines.append(f"  %{i} = tforge.add {cur}, {cur} : {t}, {t} -> {t}")
            want = o.add(want, want)
        elif op < 2:
            lines.append(f"  %{i} = tforge.bias_add {cur}, %b{op + 1} : {t}, {v} -> {t}")
            want = o.bias_add(want, (b1, b2)[op])
        else:
            lines.append(f"  %{i} = tforge.add {cur}, %r{op - 1} : {t}, {t} -> {t}")
            want = o.add(want, (r1, r2)[op - 2])
        cur = f"%{i}"
    program = (f"func.func @entry(%x: {t}, %b1: {v}, %b2: {v}, %r1: {t}, %r2: {t}) -> {t} {{\n" + "\n".join(lines) +
               f"\n  return {cur} : {t}\n}}\n")
    kern = _lib.Kernel(program, "", "t.mlir")
    (launch,) = kern.launches()
    assert launch["run"]["kernel"] == "tf_elementwise_flat_uint32_t_false_w8s32"
    assert o.bitwise_diff(_launch(program, [x, b1, b2, r1, r2], m, n), want) == 0


@pytest.mark.parametrize("m,n,kernel", [(11585, 11587, "uint32_t_true_w4s4"), (32771, 131057, "uint32_t_true_w4s4"),
                                        (11583, 11587, "uint32_t_true_w8s32")])
def test_bias_add_of_huge_streams(m, n, kernel):
    """About 2^27 elements, on both sides of the line between the two segment sizes, and
    just below 2^32 (the 32-bit column arithmetic's largest quotients), on odd rows."""
    import torch
    assert m * n < 1 << 32
    x = torch.empty(m, n, device="cuda").uniform_(-1, 1)
    bias = torch.empty(n, device="cuda").uniform_(-1, 1)
    out = torch.full((m, n), float("nan"), device="cuda")
    kern = _lib.Kernel(tc.gen_mlir("bias_add", m, n), "", "t.mlir")
    assert kern.launches()[0]["run"]["kernel"].endswith(kernel)
    kern.launch([x.data_ptr(), bias.data_ptr(), out.data_ptr()], torch.cuda.current_stream().cuda_stream)
    for r0 in range(0, m, 1 << 13):
        rows = slice(r0, min(m, r0 + (1 << 13)))
        assert torch.equal(out[rows], x[rows] + bias)


def test_bias_add_past_32_bit_elements():
    """4.3e9 elements (17 GiB) on odd rows: 64-bit column arithmetic, and more
    pieces than the grid has workgroups."""
    import torch
    m, n = (1 << 20) + 3, 4099
    dev = torch.device("cuda:0")
    x = torch.empty(m, n, device=dev).uniform_(-1, 1)
    bias = torch.empty(n, device=dev).uniform_(-1, 1)
    out = torch.full((m, n), float("nan"), device=dev)
    kern = _lib.Kernel(tc.gen_mlir("bias_add", m, n), "", "t.mlir")
    kern.launch([x.data_ptr(), bias.data_ptr(), out.data_ptr()], torch.cuda.current_stream().cuda_stream)
    for r0 in range(0, m, 1 << 17):
        rows = slice(r0, min(m, r0 + (1 << 17)))
        assert torch.equal(out[rows], x[rows] + bias)

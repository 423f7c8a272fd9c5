"""The spread staged kernels' bounded loads: every slab of A and B comes through
buffer resources that end with the matrices.  K of less than a slab to several
slabs with every remainder, tiles at and one past the edges, NaN just past each
matrix's end and in the next row of A's K tail, and B walked in several windows
of 31-bit offsets."""

import numpy as np
import pytest

from oracle import oracle as o
from tensorforge_amd import _lib
from tensorforge_amd import tforge_cpu as tc

pytestmark = pytest.mark.gpu

STAGED = "block-tile={},{} thread-tile={},{} tile-k={} promote=1 vectorize=1 mask-edges=1"
TILES = [(32, 32, 2, 2, 32), (64, 64, 4, 4, 16), (128, 64, 8, 4, 16), (128, 128, 8, 8, 16), (128, 128, 4, 8, 8)]


def _launch(kern, ins, m, n):
    """Output of kern on buffers that each have 64 NaN right behind them."""
    import torch
    dev, bufs = torch.device("cuda:0"), []
    for v in ins + [np.full((m, n), np.nan, np.float32)]:
        base = torch.full((v.size + 64,), float("nan"), device=dev)
        base[:v.size] = torch.from_numpy(v.ravel()).to(dev)
        bufs.append(base)
    kern.launch([b.data_ptr() for b in bufs], torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.isnan(bufs[-1][m * n:]).all()  # nothing stored past C
    return bufs[-1][:m * n].cpu().numpy().reshape(m, n)


@pytest.mark.parametrize("cfg", TILES)
@pytest.mark.parametrize("slabs,rest", [(s, r) for s in range(6) for r in (0, 1, 3, 4, 7) if s or r])
def test_k_tails(cfg, slabs, rest):
    bm, bn, _, _, bk = cfg
    k = slabs * bk + rest
    for m, n in ((bm, bn), (bm + 1, bn + 1), (2 * bm - 1, bn - 3), (1, 3)):
        ins = o.make_inputs("mbr", m, n, k)
        kern = _lib.Kernel(tc.gen_mlir("mbr", m, n, k), STAGED.format(*cfg), "t.mlir")
        out = _launch(kern, [np.ascontiguousarray(v) for v in ins.values()], m, n)
        ref, bound = o.fp64_reference("mbr", ins)
        assert not np.isnan(out).any(), (m, n, k)
        assert o.e1_metrics(out, ref, bound)["max_err_over_bound"] <= 1.0, (m, n, k)
        assert o.mask_mismatches(out, o.preactivation64(ins), bound) == 0


@pytest.mark.parametrize("cfg", TILES)
@pytest.mark.parametrize("k", [45, 64, 67])
def test_nan_stays_in_its_row_and_column(cfg, k):
    """The slab that holds K's end reads the start of A's next row: a NaN there
    reaches only its own row, a NaN column of B only its own column."""
    m, n = 70, 66
    ins = o.make_inputs("matmul", m, n, k)
    a, b = ins["a"].copy(), ins["b"].copy()
    a[5, 0] = np.nan
    a[68, :] = np.inf
    b[0, 7] = np.nan
    kern = _lib.Kernel(tc.gen_mlir("matmul", m, n, k), STAGED.format(*cfg), "t.mlir")
    out = _launch(kern, [a, b], m, n)
    rows, cols = np.delete(np.arange(m), [5, 68]), np.delete(np.arange(n), 7)
    assert np.isnan(out[5]).all() and np.isnan(out[:, 7]).all()
    keep = np.ix_(rows, cols)
    ref, bound = o.fp64_reference("matmul", ins)
    assert not np.isnan(out[keep]).any()
    assert (np.abs(out[keep] - ref[keep]) <= bound[keep]).all()


# Unmasked kernels take bounded loads from five slabs on, masked ones always; the
# masked problem has one column more, and its other columns are the same bits.
@pytest.mark.parametrize("cfg", TILES + [(64, 64, 4, 4, 64), (32, 32, 2, 2, 64)])
@pytest.mark.parametrize("slabs,extra", [(1, ""), (2, ""), (3, ""), (4, ""), (5, ""), (6, ""), (4, " split-k=2"),
                                         (9, " split-k=2"), (10, " split-k=2")])
def test_few_slabs_unmasked_is_bitwise_masked(cfg, slabs, extra):
    bm, bn, _, _, bk = cfg
    m, n, k = 2 * bm, 3 * bn, slabs * bk
    ins = o.make_inputs("mbr", m, n + 1, k)
    a, b, bias = (np.ascontiguousarray(v) for v in ins.values())
    opts = STAGED.format(*cfg) + extra
    masked = _lib.Kernel(tc.gen_mlir("mbr", m, n + 1, k), opts, "t.mlir")
    plain = _lib.Kernel(tc.gen_mlir("mbr", m, n, k), opts.replace(" mask-edges=1", ""), "t.mlir")
    assert not plain.launches()[0]["run"]["kernel"].endswith("_masked")
    want = _launch(masked, [a, b, bias], m, n + 1)[:, :n]
    got = _launch(plain, [a, np.ascontiguousarray(b[:, :n]), np.ascontiguousarray(bias[:n])], m, n)
    assert not np.isnan(got).any() and o.bitwise_diff(got, np.ascontiguousarray(want)) == 0


# 2^29 elements of B fit one window; past that the loop rebases its resource, every two
# slabs at N = 5e6.  Entries in {-1, 0, 1}: exact in any order.
@pytest.mark.parametrize("shape,mask", [((128, 16384, 40000), 0), ((127, 16381, 40003), 1), ((64, 5000000, 208), 0),
                                        ((63, 4999999, 203), 1)])
def test_b_past_one_window(shape, mask):
    import torch
    m, n, k = shape
    assert k * n >= 1 << 29
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(5)
    a = torch.randint(-1, 2, (m, k), device=dev, generator=g, dtype=torch.int8).float()
    b = torch.randint(-1, 2, (k, n), device=dev, generator=g, dtype=torch.int8).float()
    out = torch.full((m, n), float("nan"), device=dev)
    opts = STAGED.format(64, 64, 4, 4, 16) if mask else STAGED.format(64, 64, 4, 4, 16).replace(" mask-edges=1", "")
    kern = _lib.Kernel(tc.gen_mlir("matmul", m, n, k), opts, "t.mlir")
    kern.launch([a.data_ptr(), b.data_ptr(), out.data_ptr()], torch.cuda.current_stream().cuda_stream)
    for j in range(0, n, 1 << 20):
        want = torch.mm(a, b[:, j:j + (1 << 20)].contiguous())
        assert torch.equal(out[:, j:j + (1 << 20)], want)

"""The matrix-core form of the direct kernel at the ends of K and of the matrices:
every tile it has, K of less than a slab to several with remainders, and B past
what one buffer resource or one window reaches.  Bit for bit the one-thread kernel,
which runs on the same values 4 bytes past a 16-byte boundary, NaN as NaN."""

import numpy as np
import pytest

from tensorforge_amd import _lib
from tensorforge_amd import tforge_cpu as tc

pytestmark = pytest.mark.gpu


def _launch(kern, ins, m, n, offset):
    """Output on buffers `offset` floats past an aligned start, 64 NaN right behind each."""
    import torch
    bufs = []
    for v in ins + [torch.full((m * n,), float("nan"), device="cuda")]:
        base = torch.full((offset + v.numel() + 64,), float("nan"), device="cuda")
        base[offset:offset + v.numel()] = v.reshape(-1)
        bufs.append(base)
    kern.launch([b.data_ptr() + 4 * offset for b in bufs], torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.isnan(bufs[-1][offset + m * n:]).all()  # nothing stored past C
    return bufs[-1][offset:offset + m * n].view(m, n)


def _same(got, want):
    import torch
    nan = torch.isnan(want)
    assert torch.equal(torch.isnan(got), nan)
    assert torch.equal(got.view(torch.int32)[~nan], want.view(torch.int32)[~nan])


def _tile(kern):
    return kern.launches()[0]["run"]["kernel"]


def _uniform(*shape):
    import torch
    g = torch.Generator(device="cuda").manual_seed(int(np.prod(shape)) % 1000003)
    return torch.rand(shape, generator=g, device="cuda") * 2 - 1


# (tile and tile-k, M x N that the size rule gives it, K)
ENDS = ([("b32x32_t2x2_k32", s, k) for s in ((32, 32), (33, 65), (1, 3))
         for k in (1, 3, 31, 32, 33, 36, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 161, 192)] +
        [("b32x32_t2x2_k64", s, k) for s in ((32, 32), (33, 65)) for k in (2048, 2049, 2051, 2111, 2112, 2113, 2240)] +
        [("b64x64_t4x4_k16", s, k) for s in ((4096, 4096), (4095, 4093))
         for k in (7, 15, 16, 17, 20, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 81, 96)] +
        [("b128x128_t8x8_k16", s, k) for s in ((8192, 8192), (8191, 8190)) for k in (63, 64, 65, 79, 80, 81, 99)])


@pytest.mark.parametrize("tile,shape,k", ENDS)
def test_k_ends(tile, shape, k):
    """One NaN at the start of a row of A and one in a column of B: the slab that holds
    K's end reads the start of A's next row, and neither may reach other outputs."""
    (m, n) = shape
    a, b, bias = _uniform(m, k), _uniform(k, n), _uniform(n)
    a[m // 2, 0] = float("nan")
    b[k - 1, n // 2] = float("nan")
    kern = _lib.Kernel(tc.gen_mlir("mbr", m, n, k), "", "t.mlir")
    assert tile in _tile(kern)
    got = _launch(kern, [a, b, bias], m, n, 0)
    assert int(got.isnan().sum()) == m + n - 1
    _same(got, _launch(kern, [a, b, bias], m, n, 1))


@pytest.mark.parametrize("tile,shape,k", [("b32x32_t2x2_k32", (70, 66), 67), ("b32x32_t2x2_k64", (70, 66), 2100),
                                          ("b64x64_t4x4_k16", (1021, 1023), 131), ("b64x64_t4x4_k16", (2048, 2048), 128),
                                          ("b128x128_t8x8_k16", (8191, 8190), 67), ("b128x128_t8x8_k16", (2048, 2048), 2048)])
def test_infinities_signed_zeros_and_denormals(tile, shape, k):
    import torch
    (m, n) = shape
    a, b = _uniform(m, k), _uniform(k, n)
    special = torch.tensor([float("inf"), float("-inf"), 0.0, -0.0, 1e-45, -1e-45, 1e-38, 3e38], device="cuda")
    g = torch.Generator(device="cuda").manual_seed(7)
    for t in (a, b):
        at = torch.randint(0, t.numel(), (max(8, t.numel() // (8 * k)),), generator=g, device="cuda")
        t.view(-1)[at] = special[torch.randint(0, 8, at.shape, generator=g, device="cuda")]
    kern = _lib.Kernel(tc.gen_mlir("matmul", m, n, k), "", "t.mlir")
    assert tile in _tile(kern)
    got = _launch(kern, [a, b], m, n, 0)
    assert got.isinf().any() and not got.isnan().all()
    _same(got, _launch(kern, [a, b], m, n, 1))


# Six slabs of B below 2^29 elements run the bounded loads, in windows where K * N
# passes that; from there on the flat loads run.
@pytest.mark.parametrize("m,n,k", [(31, 2500001, 301), (32, 2500000, 320), (31, 2796195, 200), (31, 2796211, 200)])
def test_wide_b(m, n, k):
    assert (6 * 32 * n + 32 < 1 << 29) == (n < 2796203)
    a, b = _uniform(m, k), _uniform(k, n)
    kern = _lib.Kernel(tc.gen_mlir("matmul", m, n, k), "", "t.mlir")
    assert "b32x32_t2x2_k32" in _tile(kern)
    _same(_launch(kern, [a, b], m, n, 0), _launch(kern, [a, b], m, n, 1))

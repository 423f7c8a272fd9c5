"""The 64x64 t4x4 k16 kernels' crowded-grid form (more than six workgroups per CU,
masked five, split-K included) gives the bits of the plain form: the same rows computed in two
launches of half the workgroups each, below the line."""

import numpy as np
import pytest

from oracle import oracle as o
from tensorforge_amd import _lib
from tensorforge_amd import tforge_cpu as tc

pytestmark = pytest.mark.gpu

OPTS = "block-tile=64,64 thread-tile=4,4 tile-k=16 promote=1 vectorize=1"


def _mbr(a, b, bias, opts):
    import torch
    (m, k), n = a.shape, b.shape[1]
    out = torch.full((m, n), float("nan"), device=a.device)
    kern = _lib.Kernel(tc.gen_mlir("mbr", m, n, k), opts, "t.mlir")
    kern.launch([t.data_ptr() for t in (a, b, bias, out)], torch.cuda.current_stream().cuda_stream)
    return out


# 1540 workgroups (one row of tiles more than the line's 1536; masked 1312, the line at
# 1280), the line itself and grids that several rounds of workgroups cover; K of one slab to several.
@pytest.mark.parametrize("m,n,extra", [(2240, 2816, ""), (2304, 2816, " split-k=1"), (2240, 2811, " mask-edges=1"),
                                       (2303, 4094, " mask-edges=1"), (1280, 2560, " split-k=2"),
                                       (1279, 2559, " mask-edges=1 split-k=2"), (2048, 3072, ""),
                                       (2047, 2623, " mask-edges=1"), (2047, 2559, " mask-edges=1")])
@pytest.mark.parametrize("k", [32, 48, 96, 208])
def test_crowded_form_is_bitwise_the_plain_form(m, n, extra, k):
    import torch
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    if "mask" in extra:
        k -= 3
    u = lambda *s: torch.rand(s, generator=g, device="cuda") * 2 - 1
    a, b, bias = u(m, k), u(k, n), u(n)
    got = _mbr(a, b, bias, OPTS + extra)
    half = m // 128 * 64
    want = torch.cat([_mbr(a[:half].contiguous(), b, bias, OPTS + extra),
                      _mbr(a[half:].contiguous(), b, bias, OPTS + extra)])
    assert not torch.isnan(got).any()
    assert o.bitwise_diff(got.cpu().numpy(), want.cpu().numpy()) == 0


def test_crowded_form_meets_the_bound():
    ins = o.make_inputs("mbr", 2303, 2817, 83)
    kern = _lib.Kernel(tc.gen_mlir("mbr", 2303, 2817, 83), OPTS + " mask-edges=1", "t.mlir")
    out = np.empty((2303, 2817), np.float32)
    kern.run([np.ascontiguousarray(v) for v in ins.values()], out)
    ref, bound = o.fp64_reference("mbr", ins)
    assert not np.isnan(out).any() and o.e1_metrics(out, ref, bound)["max_err_over_bound"] <= 1.0
    assert o.mask_mismatches(out, o.preactivation64(ins), bound) == 0

"""Buffers that are not 16-byte aligned, where the options' own kernels run: every
thread tile of the direct and element-op kernels, 4 bytes past a 16-byte boundary,
bit-exact against the oracle.  Sizes below, at and past the block tile, and ragged,
so that full and partial thread tiles both occur."""

import numpy as np
import pytest

from oracle import oracle as o
from tensorforge_amd import _lib
from tensorforge_amd import tforge_cpu as tc

pytestmark = pytest.mark.gpu

TILES = [(tm, tn) for tm in (1, 2, 4, 8) for tn in (1, 2, 4, 8)]


def _launch(program, options, ins, m, n):
    import torch
    bufs = []
    for v in ins + [np.full((m, n), np.nan, np.float32)]:
        base = torch.zeros(v.size + 1, device="cuda")
        base[1:] = torch.from_numpy(np.ascontiguousarray(v).ravel()).cuda()
        bufs.append(base[1:])
    assert all(b.data_ptr() % 16 == 4 for b in bufs)
    _lib.Kernel(program, options, "t.mlir").launch([b.data_ptr() for b in bufs], torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return bufs[-1].cpu().numpy().reshape(m, n)


@pytest.mark.parametrize("workload", ["mbr", "matmul"])
@pytest.mark.parametrize("tm,tn", TILES)
def test_direct_thread_tiles(workload, tm, tn):
    for m, n, k in ((8 * tm, 8 * tn, 16), (8 * tm + 1, 8 * tn - 1, 33), (1, 1, 1), (67, 131, 45)):
        ins = o.make_inputs(workload, m, n, k)
        want = o.matmul_fma(ins["a"], ins["b"])
        if workload == "mbr":
            want = o.epilogue(want, ins["bias"], relu=True)
        got = _launch(tc.gen_mlir(workload, m, n, k), f"block-tile={8 * tm},{8 * tn} thread-tile={tm},{tn}",
                      list(ins.values()), m, n)
        assert o.bitwise_diff(got, want) == 0, (m, n, k)


@pytest.mark.parametrize("workload", ["relu", "bias_add", "add"])
@pytest.mark.parametrize("tm,tn", TILES)
def test_element_op_thread_tiles(workload, tm, tn):
    for m, n in ((8 * tm, 8 * tn), (8 * tm + 1, 8 * tn - 1), (1, 1), (67, 131)):
        ins = o.make_inputs(workload, m, n, None)
        got = _launch(tc.gen_mlir(workload, m, n, None), f"block-tile={8 * tm},{8 * tn} thread-tile={tm},{tn}",
                      list(ins.values()), m, n)
        assert o.bitwise_diff(got, o.elementwise(workload, ins)) == 0, (m, n)

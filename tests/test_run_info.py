"""tf_kernel_run_info names the kernel that runs on 16-byte aligned buffers, beside the
options' own that tf_kernel_launch_info describes, and resources are the former's."""

import json

import pytest

from tensorforge_amd import _lib
from tensorforge_amd import tforge_cpu as tc
from tensorforge_amd import tforge_gpu as tg

STAGED = "block-tile={} thread-tile={} tile-k={} promote=1 vectorize=1"
MID = STAGED.format("64,64", "4,4", 16)
RES = json.loads((_lib.PKG / "kernel_resources.json").read_text())


# (workload, M, N, K, options, the options' kernel, the kernel that runs, its grid and block)
CASES = [
    ("mbr", 777, 1111, 333, "", "tf_direct_t1x1", "tf_seq_b64x64_t4x4_k16_masked", [18, 13, 1], [16, 16, 1]),
    ("mbr", 256, 256, 128, "block-tile=32,32 thread-tile=2,2", "tf_direct_t2x2", "tf_seq_b32x32_t2x2_k32", [8, 8, 1],
     [16, 16, 1]),
    ("matmul", 2048, 2048, 2048, "", "tf_direct_t1x1", "tf_seq_b128x128_t8x8_k16", [16, 16, 1], [16, 16, 1]),
    ("relu", 999, 1001, None, "block-tile=8,512 thread-tile=2,8", "tf_elementwise_t2x8",
     "tf_elementwise_flat_uint32_t_true_w8s32", [512, 1, 1], [512, 1, 1]),
    ("add", 16384, 16384, None, "", "tf_elementwise_t1x1", "tf_elementwise_flat_uint32_t_true_w4s4", [262144, 1, 1],
     [256, 1, 1]),
    # 1536 workgroups (masked 1280) and one row of tiles more; split-K ranges count
    ("mbr", 2048, 3072, 64, MID, "tf_staged_b64x64_t4x4_k16", "tf_staged_b64x64_t4x4_k16", [48, 32, 1], [16, 16, 1]),
    ("mbr", 2112, 3072, 64, MID, "tf_staged_b64x64_t4x4_k16", "tf_staged_b64x64_t4x4_k16_crowd", [48, 33, 1], [16, 16, 1]),
    ("mbr", 2047, 2559, 61, MID + " mask-edges=1", "tf_staged_b64x64_t4x4_k16_masked", "tf_staged_b64x64_t4x4_k16_masked",
     [40, 32, 1], [16, 16, 1]),
    ("mbr", 2049, 2559, 61, MID + " mask-edges=1", "tf_staged_b64x64_t4x4_k16_masked",
     "tf_staged_b64x64_t4x4_k16_masked_crowd", [40, 33, 1], [16, 16, 1]),
    ("mbr", 1025, 3000, 64, MID + " mask-edges=1 split-k=2", "tf_staged_b64x64_t4x4_k16_masked",
     "tf_staged_b64x64_t4x4_k16_masked_crowd", [47, 17, 2], [16, 16, 1]),
    ("mbr", 4096, 4096, 64, STAGED.format("64,64", "4,4", 32), "tf_staged_b64x64_t4x4_k32", "tf_staged_b64x64_t4x4_k32",
     [64, 64, 1], [16, 16, 1]),
]


@pytest.mark.parametrize("workload,m,n,k,options,own,run,grid,block", CASES)
def test_run_kernel(workload, m, n, k, options, own, run, grid, block):
    launch = _lib.Kernel(tc.gen_mlir(workload, m, n, k), options, "t.mlir").launches()[0]
    assert launch["kernel"] == own
    got = launch["run"]
    assert got["kernel"] == run and got["grid"] == grid and got["block"] == block
    if own == run:
        assert (got["grid"], got["block"], got["lds_bytes"]) == (launch["grid"], launch["block"], launch["lds_bytes"])
    assert got["lds_bytes"] == RES[run]["lds_bytes"]


@pytest.mark.parametrize("mask,per_cu", [("", 6), ("_masked", 5)])
def test_crowded_line_is_what_the_plain_form_runs_at_once(mask, per_cu):
    """Four waves a workgroup: waves per SIMD = workgroups per CU.  The crowded form
    takes the first grid past 256 CUs of them (the CASES above)."""
    assert RES[f"tf_staged_b64x64_t4x4_k16{mask}"]["occupancy_waves_per_simd"] == per_cu
    assert RES[f"tf_staged_b64x64_t4x4_k16{mask}_crowd"]["occupancy_waves_per_simd"] == 4
    for gy, crowd in ((per_cu * 8, False), (per_cu * 8 + 1, True)):
        opts = MID + (" mask-edges=1" if mask else "")
        m = gy * 64 - (1 if mask else 0)  # whole tiles run the unmasked kernel
        run = _lib.Kernel(tc.gen_mlir("mbr", m, 2048, 64), opts, "t.mlir").launches()[0]["run"]
        assert run["kernel"] == f"tf_staged_b64x64_t4x4_k16{mask}" + ("_crowd" if crowd else "")


def test_compiler_resources_are_the_run_kernels(tmp_path, monkeypatch):
    monkeypatch.setattr(tg, "ART", tmp_path)
    for wl, k in (("mbr", 333), ("relu", None)):
        d, launch = tg.compile_kernel(wl, 777, 1111, k, "", tag="t")
        rec = RES[launch["launches"][0]["run"]["kernel"]]
        res = tg.ptxas_resources(d)
        assert (res["regs"], res["agprs"], res["smem"]) == (rec["vgprs"], rec["agprs"], rec["lds_bytes"])


@pytest.mark.gpu
@pytest.mark.parametrize("workload,m,n,k,options,own,run,grid,block", CASES)
def test_device_resources_are_the_run_kernels(workload, m, n, k, options, own, run, grid, block):
    res = _lib.Kernel(tc.gen_mlir(workload, m, n, k), options, "t.mlir").resources(0)
    assert res["threads"] == block[0] * block[1] and res["static_smem"] == RES[run]["lds_bytes"]
    assert res["local_bytes"] == 0 and res["blocks_per_sm"] >= 1

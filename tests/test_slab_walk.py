"""The bounded-load kernels' slab walk, checked on the host: the scalar offset of
every load stays below its buffer resource's size (the range check subtracts it from
the size), and every slab is computed from its own bytes, once and in order, for K
of none to many slabs, split K ranges and windows of B.  No GPU needed."""

import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_every_slab_load_starts_inside_its_resource(tmp_path):
    if not pathlib.Path(HIPCC).exists():
        pytest.skip("needs hipcc")
    exe = tmp_path / "slab_walk"
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O1", "-I", str(ROOT / "include"),
                    "-I", str(ROOT / "tensorforge_amd" / "csrc"), str(ROOT / "tests" / "slab_walk_driver.cpp"),
                    "-o", str(exe)], check=True, capture_output=True, timeout=300)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip().endswith("walks ok"), r.stdout + r.stderr

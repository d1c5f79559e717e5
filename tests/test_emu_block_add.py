"""The device builder's block-wide append (block_add, j3d_amd/csrc/bvh_gpu.hip)
as the GPU runs it, on the CPU emulation (tests/emu/check_block_add.cpp)."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
EMU = os.path.join(HERE, "emu")
sys.path.insert(0, EMU)
import build_emu  # noqa: E402

pytestmark = pytest.mark.skipif(build_emu.compiler() is None, reason="needs clang++")


def test_ranges_of_a_block(tmp_path):
    s = open(os.path.join(ROOT, "j3d_amd", "csrc", "bvh_gpu.hip")).read()
    a = s.index("__device__ inline uint32_t block_add(")
    body = s[a:s.index("\n}\n", a) + 3]
    (tmp_path / "block_add.inc").write_text(body)
    exe = str(tmp_path / "check_block_add")
    subprocess.run([build_emu.compiler(), "-std=c++17", "-O1", "-fno-inline", "-fno-omit-frame-pointer", "-w",
                    "-I" + EMU, "-I" + str(tmp_path), "-o", exe, os.path.join(EMU, "check_block_add.cpp"),
                    os.path.join(EMU, "emu_runtime.cpp"), "-pthread"], check=True, timeout=300)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0 and "BLOCK ADD OK" in r.stdout, r.stdout[-2000:]

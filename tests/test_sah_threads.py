"""The device builder's host SAH (j3d_amd/csrc/bvh_gpu.hip) on its threads:
the same tree as on one thread, no data race, and neither a thread that cannot
be had nor memory that runs out ends the process."""
import os
import shutil
import subprocess

import pytest

from test_lbvh_cpu import HERE, ROOT, _lbvh_body

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.mark.parametrize("flags, args", [
    (["-fsanitize=thread"], ["trees"]),
    (["-fsanitize=address,undefined", "-fno-sanitize-recover=undefined"], ["trees"]),
    (["-DCHECK_THREADS"], ["threads", "0"]),
    (["-DCHECK_THREADS"], ["threads", "3"]),
    (["-DCHECK_MEMORY"], ["memory"]),
], ids=["tsan", "asan", "no_threads", "three_threads", "no_memory"])
def test_sah_on_threads(tmp_path, flags, args):
    (tmp_path / "lbvh_body.inc").write_text(_lbvh_body())
    exe = tmp_path / "check_sah"
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-ffp-contract=off", "-pthread"] + flags +
                   ["-I" + str(tmp_path), "-I" + HERE, "-I" + os.path.join(ROOT, "j3d_amd", "csrc"),
                    "-I" + os.path.join(ROOT, "include"), "-o", str(exe), os.path.join(HERE, "check_sah.cpp"), "-ldl"],
                   check=True, timeout=300)
    r = subprocess.run([str(exe)] + args, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0 and "SAH OK" in r.stdout, r.stdout[-3000:]

"""Scenes of many objects on the CPU emulation of the library (see
test_emu_batch.py): the object loop of up to 16 objects and the top-level tree
of more, in the tail modes, against the oracle (tests/emu/scenes_case.py)."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "emu")
sys.path.insert(0, EMU)
import build_emu  # noqa: E402

pytestmark = pytest.mark.skipif(build_emu.compiler() is None, reason="needs clang++")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return build_emu.build(str(tmp_path_factory.mktemp("emu_scenes")))


def _run(lib, what, **env_extra):
    r = subprocess.run([sys.executable, os.path.join(EMU, "scenes_case.py"), what],
                       env=dict(os.environ, J3DG_LIBRARY=lib, **env_extra), stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=600)
    print(r.stdout[-3000:])
    assert r.returncode == 0 and "SCENES OK" in r.stdout, r.stdout[-3000:]


def test_a_query_goes_on_to_the_next_object_within_a_trip(lib):
    """A loop trip has up to four traversal steps; a lane of a query that is
    done with an object uses those left for the next one."""
    _run(lib, "steps")

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


@pytest.mark.parametrize("tail,depth", [("4", "8"), ("3", "16"), ("2", "8"), ("1", "16"), ("0", "8")])
def test_many_objects_match_the_oracle(lib, tail, depth):
    """Frames and queries through a top-level tree, and queries over 16 objects."""
    _run(lib, "tails", EMU_TAIL=tail, EMU_STACK=depth, EMU_CUS="4")


def test_a_cut_top_level_walk_reads_nothing_out_of_bounds(tmp_path):
    """The walk's bound, meant for a malformed tree, brought down to eight nodes
    in a copy of the source: lanes end in the middle of the top level, and the
    split tail must not take their entries for an object's."""
    sources = build_emu.patched_sources

    def cut(out, variant=None):
        sources(out, variant)
        p = os.path.join(out, "traverse.h")
        s = open(p).read()
        assert s.count("kTopGuard = 1u << 22;") == 1
        open(p, "w").write(s.replace("kTopGuard = 1u << 22;", "kTopGuard = 8u;"))
        return out

    build_emu.patched_sources = cut
    try:
        lib = build_emu.build(str(tmp_path))
    finally:
        build_emu.patched_sources = sources
    _run(lib, "guard", EMU_CUS="4")

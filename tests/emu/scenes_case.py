"""Scenes of many objects through whichever build of libj3dg the J3DG_LIBRARY
environment variable names (the CPU emulation in tests/test_emu_scenes.py).

  tails   frames and ray queries of 24 overlapping objects (a top-level tree)
          and queries of 16 (the object loop) with the tail mode EMU_TAIL and
          the LDS stack depth EMU_STACK, bit for bit against the oracle
  steps   an any-hit query of one wave whose rays miss all of 16 objects: the
          loop trips it takes
  guard   a query over 60 objects with a build whose top-level walks are cut
          off after a few nodes: it has to report the overflow

Exit status 0 when everything holds, 1 otherwise (a memory fault in the
emulation exits 86)."""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
for p in (ROOT, os.path.join(ROOT, "oracle"), os.path.join(ROOT, "tests")):
    sys.path.insert(0, p)

import numpy as np  # noqa: E402

import j3d_amd as J  # noqa: E402
import oracle as O  # noqa: E402
from j3d_amd import ffi  # noqa: E402
from scenes import compare_gbuffers, compare_rgba, random_rays  # noqa: E402


def scene(r, n, side, seed, parts=None):
    rng = np.random.default_rng(seed)
    parts = parts or [J.icosphere(2, seed=3, amplitude=0.1), J.torus(24, 12, R=0.8, r=0.3, seed=4)]
    slots, meshes = [], []
    for i in range(n):
        v, t = parts[i % 2]
        cs = np.eye(4, dtype=np.float32)
        cs[3, :3] = rng.uniform(-side, side, 3)
        db = J.make_db_id(5, i)
        slots.append(r.upload_mesh(v, t, db_id=db, cs=cs.reshape(16)))
        meshes.append(O.Mesh(v, t, cs=cs.reshape(16), db_id=db))
    return slots, meshes


def queries(r, slots, meshes, rays):
    got, ref = r.trace_rays(slots, rays), O.closest_hits(meshes, rays)
    bad = sum(int((got[k].view(np.uint32) != ref[k].view(np.uint32)).sum()) for k in ("obj", "tri", "t", "u", "v"))
    n = int((ref["tri"] != 0xFFFFFFFF).sum())
    bad += int((r.any_hit(slots, rays) != O.any_hits(meshes, rays)).sum())
    print("queries over %d objects: %d rays, %d hits, %d mismatches" % (len(slots), len(rays), n, bad), flush=True)
    return bad + (n == 0)


def tails(r):
    r.set_tuning(**dict(r.get_tuning(), coop_tail=int(os.environ["EMU_TAIL"]), stack_depth=int(os.environ["EMU_STACK"])))
    mc, cav = J.make_matcap(0)
    r.set_matcap(mc, cav)
    slots, meshes = scene(r, 24, 1.2, 7)
    bad = 0
    light = np.array([0.3, 0.5, 0.81], np.float32)
    cs, ci = J.orbit_camera(4.5, 0.9, 0.5)
    for w, h, flags in ((1, 1, ffi.SHADING), (72, 56, ffi.EDGES | ffi.SHADOW | ffi.DIRECTIONAL_LIGHT),
                        (40, 24, ffi.SHADING | ffi.SHADOW)):
        fr = J.make_frame(w, h, J.camera_with_vertical_fov(50.0), cs, ci, np.zeros(3, np.float32), 3.0, slots,
                          flags=flags, light_dir=light / np.linalg.norm(light))
        tg = r.create_target(w, h)
        g, im = r.render(fr, tg)
        og, oim, _ = O.render(meshes, fr, mc, cav)
        mm, d = compare_gbuffers(g, og), compare_rgba(im, oim)[0]
        print("frame %dx%d: G-buffer mismatches %s, rgba %d" % (w, h, mm, d), flush=True)
        bad += sum(mm.values()) + (d > 1)
        r.destroy_target(tg)
    rays = random_rays(3001, 5, np.zeros(3), 2.5)
    rays[7, 3], rays[9, 0] = np.nan, np.inf
    bad += queries(r, slots, meshes, rays)
    bad += queries(r, slots[:16], meshes[:16], rays)
    bad += queries(r, slots[:3], meshes[:3], rays[:33])
    lib = ffi.load()
    import ctypes as C
    lib.emu_inactive_lane_reads.restype = C.c_ulonglong
    n = int(lib.emu_inactive_lane_reads())
    print("shuffles that read a lane outside the exec mask: %d" % n)
    return bad + n


def steps(r):
    slots, meshes = scene(r, 16, 0.5, 8)
    rays = np.zeros((64, 8), np.float32)
    rays[:, 0] = np.linspace(-1.0, 1.0, 64)
    rays[:, 2], rays[:, 5], rays[:, 7] = 50.0, 1.0, np.finfo(np.float32).max  # away from all of them
    r.set_tuning(**dict(r.get_tuning(), block_size=64))  # one wave in the launch
    r.set_counting(True)
    hit = r.any_hit(slots, rays)
    s = r.stats()
    r.set_counting(False)
    # one step per object; a trip has four, and the wave's last may not be full
    print("16 objects missed by a wave in %d trips, %d steps" % (s["wave_trips"], s["lane_steps"]), flush=True)
    return int(hit.any()) + (s["lane_steps"] != 16 * 64) + (s["wave_trips"] > 16 // 4 + 1)


def guard(r):
    # objects of few nodes and triangles: most top-level entries are no node or record of theirs
    small = J.icosphere(0, seed=3)
    bad = 0
    for mode in (4, 3, 2, 1, 0):
        r.set_tuning(**dict(r.get_tuning(), coop_tail=mode))
        slots, _ = scene(r, 60, 1.0, 9, [small, small])
        rays = random_rays(1500, 6, np.zeros(3), 2.5)
        for q in (r.trace_rays, r.any_hit):
            try:
                q(slots, rays)
                print("mode %d: the cut walk went unreported" % mode, flush=True)
                bad += 1
            except J.J3dgError as e:
                print("mode %d: %s" % (mode, e), flush=True)
                bad += "overflow" not in str(e)
        for s in slots:
            r.remove_mesh(s)
    return bad


def main():
    r = J.Renderer(0)
    bad = {"tails": tails, "steps": steps, "guard": guard}[sys.argv[1]](r)
    r.close()
    print("SCENES OK" if not bad else "SCENES MISMATCH %d" % bad, flush=True)
    sys.exit(0 if not bad else 1)


if __name__ == "__main__":
    main()

"""How a trace launch's rays are cut into bands of the work queue
(j3d_amd/csrc/traverse.h), compiled for the CPU from the source: the bands
cover the rays once and in order, and only a launch's last work item may be a
part of one -- an item cut by a band's end is one more item, which a launch of
as many items as waves cannot spare.  A query of few tiles is one band: all others
are marked as drained from the start, and no wave asks their counters."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MAIN = r"""
int main() {
  int bad = 0;
  auto check = [&](uint32_t n_rays, uint32_t items, BandCut cut) {
    const uint32_t batch = 64u * items, n_tiles = (n_rays + 63u) / 64u;
    const uint32_t unit = UNIT;
    uint64_t at = 0, n_items = 0;
    for (uint32_t b = 0; b < kBands; ++b) {
      const uint64_t lo = band_first_ray(b, n_tiles, unit), hi = band_first_ray(b + 1, n_tiles, unit);
      const uint64_t end = hi < n_rays ? hi : n_rays;
      if (lo != at && lo < n_rays) ++bad;
      const bool empty = bands_without_work(n_rays, cut) >> b & 1u;
      if (cut == kCutQuery && n_rays <= 64u * 64u && empty != (b + 1 < kBands)) ++bad;
      if (empty && end > lo) ++bad;
      if (end > lo) n_items += (end - lo + batch - 1) / batch, at = end;
    }
    if (at != n_rays || n_items != ((uint64_t)n_rays + batch - 1) / batch) {
      if (bad++ < 5) printf("n_rays %u items %u cut %d: up to %llu, %llu items\n", n_rays, items, (int)cut,
                            (unsigned long long)at, (unsigned long long)n_items);
    }
  };
  for (uint32_t items : {1u, 2u, 4u})
    for (BandCut cut : {kCutOrder, kCutItems, kCutQuery}) {
      for (uint32_t n = 1; n < 3000; ++n) check(n, items, cut);
      for (uint32_t t = 1; t < 3000; ++t) check(64 * t, items, cut);
      for (uint32_t n : {199999u, 200000u, 200003u, 1048576u, 2073600u, 20000001u, 0x7FFFFFFFu}) check(n, items, cut);
    }
  printf(bad ? "BAD %d\n" : "BANDS OK\n", bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_bands_cover_the_rays_in_whole_items(tmp_path):
    s = open(os.path.join(ROOT, "j3d_amd", "csrc", "traverse.h")).read()
    body = s[s.index("constexpr uint32_t kXcds"):s.index("// Wave-local pool of ray ids")]
    unit = "band_cut(n_rays, batch, cut)"
    src = tmp_path / "bands.cpp"
    src.write_text("#include <cstdint>\n#include <cstdio>\n#include <initializer_list>\n#define __host__\n#define __device__\n" + body
                   + MAIN.replace("UNIT", unit))
    exe = tmp_path / "bands"
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=undefined", "-o",
                    str(exe), str(src)], check=True, timeout=120)
    r = subprocess.run([str(exe)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0 and "BANDS OK" in r.stdout, r.stdout[-2000:]

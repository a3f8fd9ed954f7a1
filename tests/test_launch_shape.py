"""Launch shapes for every size, on the host: bear_amd/csrc/launch_shape.h
compiled by the host compiler."""

import os
import subprocess

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "bear_amd", "csrc")
LDS = 160 * 1024                                        # per workgroup on gfx950
TABLE = 16 * 1024                                       # the exponential table


def _run(folder, body):
    src = os.path.join(folder, "shapes.cpp")
    with open(src, "w") as f:
        f.write('#include <cstdio>\n#include "launch_shape.h"\nusing namespace bear_amd;\nint main() {\n' + body + "}\n")
    exe = os.path.join(folder, "shapes")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, "-I", os.path.join(ROOT, "include"), src, "-o", exe],
                   check=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return [tuple(int(v) for v in line.split()) for line in out.splitlines()]


@pytest.mark.parametrize("limit", [64 * 1024, LDS])
def test_single_transit_shapes(tmp_path, limit):
    """Two-value stencils never without their table, and every form within the
    workgroup's LDS, the table behind the sums of the tile that is launched."""
    rows = _run(str(tmp_path), """
  for (int L = 2; L <= 400; ++L)
    for (int slots = 1; slots <= 16; ++slots)
      for (int iso = 0; iso < 2; ++iso) {
        if (transitLds(L, 64, kTransitThreads) > %d) continue;      // refused when the model is configured
        const TransitShape s = transitShape(L, slots, iso, %d);
        std::printf("%%d %%d %%d %%d %%d %%d %%d %%zu %%d\\n", L, slots, iso, int(s.isothermal), s.threads, s.tile,
                    s.exp_offset, s.lds, chordSegments(L));
      }
""" % (limit, limit))
    assert rows
    forms = set()
    for levels, slots, iso, isothermal, threads, tile, offset, lds, segments in rows:
        sums = (segments + threads // tile) * tile * 8
        assert tile in (64, 128) and threads % tile == 0 and segments >= levels - 1
        assert lds <= limit
        if isothermal:
            assert iso and offset * 8 == sums and lds == sums + TABLE
            assert threads == (1024 if slots <= 12 else 512)
        else:
            assert threads == 512
            assert (offset * 8 == sums and lds == sums + TABLE) or (offset == 0 and lds == sums)
            if iso:                                          # given up only where no tile leaves room for the table
                wide = 1024 if slots <= 12 else 512
                assert (segments + wide // 64) * 64 * 8 + TABLE > limit
        forms.add((isothermal, tile, offset > 0))
    if limit == LDS:
        assert forms == {(1, 128, True), (1, 64, True), (0, 128, True), (0, 128, False), (0, 64, True), (0, 64, False)}


def test_launches_of_large_batches(tmp_path):
    """Every launch below 2^32 threads, at most 65,535 points per batch, and
    no more launches than that takes."""
    sizes = [1, 63, 64, 65, 2554, 16_500, 60_000, 65_600, 400_000, 1_000_003]
    rows = _run(str(tmp_path), """
  for (int n : {%s})
    for (int tile : {64, 128, 256})
      for (int threads : {64, 128, 256, 512})
        std::printf("%%d %%d %%d %%zu %%zu\\n", n, tile, threads, pointsPerLaunch((n + tile - 1) / tile, threads),
                    maxWorkgroups(threads));
""" % ", ".join(str(n) for n in sizes))
    assert len(rows) == len(sizes) * 12
    split = 0
    for n, tile, threads, points, groups in rows:
        per_point = (-(-n // tile) + 7) // 8 * 8
        assert points >= 1 and groups % 8 == 0 and groups * threads < 2 ** 32 <= (groups + 8) * threads
        assert points * per_point <= groups < (points + 1) * per_point
        for batch in (1, 8950, 10_737, 65_535):
            runs = [min(points, batch - m) for m in range(0, batch, points)]
            assert sum(runs) == batch and max(runs) * per_point * threads < 2 ** 32
            split += len(runs) > 1
    assert split > 0


def test_level_split_by_tiles(tmp_path):
    """Eight wavefronts per tile, then four, then one, and never fewer than
    eight wavefronts per CU where the split could give them."""
    cus = 256
    rows = _run(str(tmp_path), """
  for (size_t tiles = 1; tiles <= 8 * %d * 4; ++tiles) std::printf("%%zu %%d\\n", tiles, levelSplit(tiles, %d));
""" % (cus, cus))
    splits = [s for _, s in rows]
    assert set(splits) == {8, 4, 1} and splits == sorted(splits, reverse=True)
    assert all(tiles * split >= 8 * cus for tiles, split in rows if tiles >= cus)
    assert splits[8 * cus - 1] == 8 and splits[8 * cus] == 4 and splits[16 * cus - 1] == 4 and splits[16 * cus] == 1

"""Run-kernel launch planning on the host (no GPU): z chunks are capped so
that every raw buffer window stays within the 2 GiB reach of a 32-bit
buffer range, and grids whose planes cannot fit one window are rejected.

The shapes are those that a single-chunk plan would have windowed at 2-4 GiB
(4096x4096x64 and 8192x8192x16 FP32, 2048x2048x255 FP64); the reference's
32-bit PSIndex (include/physis/physis_common.h:33-55) admits all of them.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
REACH = 2 ** 31 - 1


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("planner") / "planner_check")
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-std=c++17",
                    "-O1", f"-I{ROOT}/include",
                    os.path.join(ROOT, "tests", "planner_check.cc"), "-o",
                    out], check=True, capture_output=True)
    return out


def _rows(text):
    return [tuple(int(v) for v in line.split())
            for line in text.strip().splitlines()]


def test_windows_stay_within_reach(planner):
    rows = _rows(subprocess.run([planner], check=True, capture_output=True,
                                text=True).stdout)
    assert len(rows) == 6
    for nx, ny, nz, elm, margin, tz, chunk, blocks, window in rows:
        assert window <= REACH, (nx, ny, nz, elm, window)
        assert tz * chunk >= nz and (tz - 1) * chunk < nz
        assert chunk >= 1
        # the window formula the run kernels use: chunk + margin per side
        assert window == (chunk + 2 * margin) * nx * ny * elm
    big = {(r[0], r[1], r[2], r[3], r[4]): r for r in rows}
    # these shapes need several chunks only because of the reach
    assert big[(8192, 8192, 16, 4, 2)][6] <= 4
    assert big[(4096, 4096, 64, 4, 2)][6] <= 28
    assert big[(2048, 2048, 255, 8, 2)][6] <= 60
    # ordinary shapes are planned for occupancy alone
    assert big[(512, 512, 512, 4, 2)][5] >= 1


def test_plane_beyond_reach_is_rejected(planner):
    # a 1 GiB plane with one halo plane per side needs a 3 GiB window
    r = subprocess.run([planner, "16384", "16384", "4", "4", "1", "256", "14",
                        "256"], capture_output=True, text=True)
    assert r.returncode != 0
    assert "2 GiB reach of a buffer window" in r.stderr


# Pairs over a domain, by the side measured faster (include/physis/hip/tile.h):
# the domain counts and not its grid, and rows that fill the 256-point tiles of
# a z-marching pass as much as the number of points.
@pytest.mark.parametrize("box,points,tiles", [
    ((1, 63) * 3, 64 ** 3, True), ((1, 255, 1, 59, 1, 59), 921600, True),
    ((1, 23, 1, 299, 1, 299), 2160000, True),
    ((40, 72) * 3, 512 ** 3, True), ((40, 72) * 3, 512 ** 3 + 1, False),
    ((1, 255, 1, 91, 1, 91), 2166784, False),
    ((1, 1023, 1, 45, 1, 45), 2166784, False),
    ((1, 255) * 3, 256 ** 3, False), ((1, 511) * 3, 512 ** 3, False)])
def test_tiles_for_pairs_over_a_domain(planner, box, points, tiles):
    r = subprocess.run([planner, "tiles", *map(str, box), str(points)],
                       check=True, capture_output=True, text=True)
    assert int(r.stdout) == tiles


# Passes of several sweeps reach further than single sweeps: where their
# windows do not fit, the run takes single sweeps (it must not be refused).
@pytest.mark.parametrize("grid,elm,margin,rows,fits", [
    ((512, 512, 512), 4, 3, 0, True), ((8755, 8755, 8), 4, 3, 0, True),
    ((9001, 9001, 8), 4, 3, 0, False), ((9001, 9001, 8), 4, 2, 0, True),
    ((6500, 6500, 8), 8, 3, 0, False), ((48000000, 3, 1), 4, 5, 1, True),
    ((49000000, 3, 1), 4, 5, 1, False), ((60000000, 3, 1), 4, 2, 1, True)])
def test_passes_of_several_sweeps_within_reach(planner, grid, elm, margin,
                                               rows, fits):
    r = subprocess.run([planner, "fits", *map(str, grid), str(elm),
                        str(margin), str(rows)], check=True,
                       capture_output=True, text=True)
    assert int(r.stdout) == fits


# Single sweeps over rows that are no multiples of 4, at one point per lane or
# ragged at four: the side measured faster (include/physis/hip/run.h).
@pytest.mark.parametrize("extents,periodic,colour,one", [
    ((63, 256, 200), 0, 0, True), ((127, 256, 200), 0, 0, True),
    ((191, 256, 200), 0, 0, False), ((255, 256, 200), 0, 0, False),
    ((290, 256, 200), 0, 0, True), ((385, 256, 200), 0, 0, False),
    ((63, 256, 200), 1, 0, True), ((127, 256, 200), 1, 0, False),
    ((255, 256, 200), 1, 0, False), ((222, 60, 60), 1, 0, True),
    ((150, 150, 150), 0, 1, False), ((255, 255, 255), 0, 1, True)])
def test_points_per_lane_of_ragged_rows(planner, extents, periodic, colour, one):
    r = subprocess.run([planner, "one", *map(str, extents), str(periodic),
                        str(colour)], check=True, capture_output=True,
                       text=True)
    assert int(r.stdout) == one


# Whole-grid and interior passes against single sweeps, which run in tiles of 64
# points on rows that are no multiples of 4: the side measured faster
# (include/physis/hip/tile.h); few: a kernel of few gets, which has tiles.
@pytest.mark.parametrize("extents,whole,interior,few", [
    ((41, 100, 100), True, True, 1), ((41, 300, 300), True, False, 1),
    ((41, 1000, 1000), False, False, 1), ((33, 500, 500), False, False, 1),
    ((40, 1000, 1000), True, True, 1), ((65, 500, 500), True, False, 1),
    ((97, 300, 300), True, False, 1), ((129, 400, 400), True, False, 1),
    ((161, 300, 300), True, True, 1), ((257, 200, 200), True, True, 1),
    ((321, 300, 200), True, True, 1),
    ((37, 256, 200), False, False, 0), ((191, 256, 200), False, False, 0),
    ((255, 256, 200), True, True, 0), ((256, 60, 60), True, True, 0),
    ((321, 256, 200), True, False, 0)])
def test_passes_where_they_pay(planner, extents, whole, interior, few):
    r = subprocess.run([planner, "pay", *map(str, extents), str(few)],
                       check=True, capture_output=True, text=True)
    assert [int(v) for v in r.stdout.split()][:2] == [whole, interior]


# The last of an odd number of red-black iterations as a pass and a copy, or as
# two colour sweeps: the side measured faster.
@pytest.mark.parametrize("extents,sweeps", [
    ((129, 129, 129), True), ((150, 150, 150), True), ((257, 257, 257), True),
    ((54, 200, 200), True), ((383, 200, 150), True), ((255, 255, 255), False),
    ((65, 65, 65), False), ((33, 100, 100), False), ((256, 256, 256), False)])
def test_last_red_black_iteration(planner, extents, sweeps):
    r = subprocess.run([planner, "pay", *map(str, extents), "0"], check=True,
                       capture_output=True, text=True)
    assert int(r.stdout.split()[2]) == sweeps


# Whole-grid passes at 4 or 2 points per lane, and in tiles: the side measured
# faster (include/physis/hip/run.h, tile.h).  Grids where the kinds of pass lie
# within 5 % of each other are left out of the second list: the rule's cost model
# is no finer than that.
@pytest.mark.parametrize("extents,periodic,colours,vx", [
    ((128, 100, 100), 0, 0, 2), ((128, 256, 256), 0, 0, 2),
    ((384, 60, 60), 0, 0, 4), ((368, 200, 150), 0, 0, 4),
    ((301, 256, 256), 0, 0, 2), ((384, 384, 384), 0, 0, 2),
    ((256, 256, 256), 0, 0, 4), ((128, 100, 100), 1, 0, 4),
    ((100, 128, 128), 1, 0, 2), ((321, 190, 157), 1, 0, 4),
    ((128, 164, 65), 0, 1, 4), ((100, 128, 128), 0, 1, 2),
    ((368, 200, 200), 0, 1, 4), ((301, 218, 400), 0, 1, 2),
    ((320, 300, 300), 0, 1, 2), ((384, 384, 384), 0, 1, 2)])
def test_points_per_lane_of_passes(planner, extents, periodic, colours, vx):
    r = subprocess.run([planner, "vx", *map(str, extents), str(periodic),
                        str(colours)], check=True, capture_output=True,
                       text=True)
    assert int(r.stdout.split()[0]) == vx


@pytest.mark.parametrize("extents,periodic,colours,tiles", [
    ((112, 112, 112), 0, 0, True), ((100, 68, 124), 0, 0, True),
    ((112, 56, 154), 0, 0, True), ((96, 24, 367), 0, 0, True),
    ((128, 128, 128), 0, 0, False), ((150, 150, 150), 0, 0, False),
    ((60, 254, 265), 1, 0, True), ((120, 36, 236), 1, 0, True),
    ((148, 124, 87), 1, 0, True), ((148, 124, 87), 0, 1, False),
    ((140, 140, 80), 1, 0, True), ((140, 140, 80), 0, 1, False),
    ((180, 110, 96), 0, 0, False), ((80, 138, 181), 0, 1, True),
    ((256, 88, 43), 0, 1, False),
    ((256, 80, 80), 0, 0, False),
    ((32, 300, 300), 0, 0, True), ((256, 256, 256), 0, 0, False)])
def test_tiles_for_whole_grids(planner, extents, periodic, colours, tiles):
    r = subprocess.run([planner, "vx", *map(str, extents), str(periodic),
                        str(colours)], check=True, capture_output=True,
                       text=True)
    assert int(r.stdout.split()[1]) == tiles


# Whole-grid red-black maps on rows that end just past a tile of the pass: colour
# sweeps or passes, as measured.
@pytest.mark.parametrize("extents,passes", [
    ((129, 422, 422), False), ((129, 622, 623), False),
    ((131, 617, 618), False), ((257, 299, 299), False),
    ((257, 441, 441), False), ((129, 152, 152), True),
    ((131, 247, 247), True), ((141, 403, 404), True),
    ((128, 422, 422), True), ((193, 508, 509), True),
    ((257, 200, 200), True), ((258, 440, 440), True),
    ((260, 441, 441), True), ((385, 360, 360), True),
    ((513, 312, 312), True)])
def test_red_black_passes_just_past_a_tile(planner, extents, passes):
    r = subprocess.run([planner, "vx", *map(str, extents), "0", "1"], check=True,
                       capture_output=True, text=True)
    assert int(r.stdout.split()[2]) == passes

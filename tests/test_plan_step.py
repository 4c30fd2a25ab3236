"""Launch plans of a whole step (strips of 56 columns) and of the first-order
schemes with two columns per lane (strips of 124, the first one starting at the
ghost column beside the domain), on the host through fvmi_substep_plan: the
segments cover every row of every strip once, at the edges of strips and row
groups and on several CU counts."""

import ctypes

import numpy as np
import pytest

from finitevolumegpu_amd import _lib

STEP, LXF2, HLL2, FORCE2 = 16, 12, 13, 14


def plan(scheme, nx, ny, tile_rows=0, waves_per_block=4, xcd_remap=True, cu_count=256, sub=(0, 0, 0, 0)):
    lib = _lib.lib()
    launch = _lib.LaunchConfig(tile_rows, waves_per_block, _lib.FVMI_MATH_FAST, 1 if xcd_remap else 2)
    n = ctypes.c_int()
    rc = lib.fvmi_substep_plan(scheme, nx, ny, *sub, ctypes.byref(launch), cu_count, None, 0, ctypes.byref(n))
    if n.value <= 0:
        return rc
    segs = np.zeros((n.value, 3), dtype=np.int32)
    rc = lib.fvmi_substep_plan(scheme, nx, ny, *sub, ctypes.byref(launch), cu_count,
                               segs.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), n.value, ctypes.byref(n))
    assert rc == 0, lib.fvmi_last_error().decode()
    return segs


@pytest.mark.parametrize("scheme", [STEP, LXF2, HLL2, FORCE2])
@pytest.mark.parametrize("nx,ny,tile_rows,waves,remap,cus", [
    (8, 8, 0, 4, True, 256), (55, 9, 0, 4, True, 256), (56, 40, 0, 4, True, 256), (57, 41, 0, 4, True, 256),
    (123, 300, 0, 4, True, 256), (124, 300, 0, 4, True, 256), (125, 1100, 1, 4, True, 256),
    (128, 128, 0, 4, True, 256), (2047, 2047, 0, 4, True, 256), (4096, 4096, 0, 4, True, 256),
    (4096, 4096, 70, 3, False, 256), (6000, 777, 0, 2, True, 256), (3000, 2500, 0, 4, True, 80),
])
def test_segments_cover_the_domain_once(scheme, nx, ny, tile_rows, waves, remap, cus):
    width, strip = (nx, 56) if scheme == STEP else (nx + 1, 124)
    strips = -(-width // strip)
    cover = np.zeros((strips, ny), dtype=np.int32)
    for s, r, c in plan(scheme, nx, ny, tile_rows, waves, remap, cus):
        if s < 0:
            assert r == 0 and c == 0
            continue
        assert 0 <= s < strips and c >= 1 and 0 <= r and r + c <= ny
        cover[s, r:r + c] += 1
    assert (cover == 1).all()


def test_second_segment_of_a_whole_step_starts_past_the_mirrored_rows():
    """A segment's march mirrors ghost rows 0 and 1 from rows 2 and 3 of the
    first segment only: every other segment starts at row 2 or later."""
    for nx, ny in ((8, 8), (64, 64), (300, 100), (2047, 2047), (4096, 4096)):
        rows = plan(STEP, nx, ny)
        starts = rows[rows[:, 0] >= 0, 1]
        assert not ((starts > 0) & (starts < 2)).any()


def test_wide_strips_of_a_workgroup_are_adjacent():
    segs = plan(LXF2, 3000, 3000)
    for b in range(0, len(segs), 4):
        live = segs[b:b + 4][segs[b:b + 4, 0] >= 0]
        if len(live) > 1:
            assert (live[:, 1:] == live[0, 1:]).all() and (np.diff(live[:, 0]) == 1).all()


@pytest.mark.parametrize("scheme", [STEP, LXF2])
def test_sub_areas_are_rejected(scheme):
    assert plan(scheme, 64, 64, sub=(1, 0, 64, 64)) < 0


@pytest.mark.parametrize("scheme,math,strip,extra", [(STEP, "fast", 56, 0), (0, "exact", 60, 0), (2, "exact", 60, 0),
                                                     (5, "fast", 62, 0), (7, "fast", 60, 0), (HLL2, "fast", 124, 1)])
@pytest.mark.parametrize("nx,ny,cus", [(8, 8, 256), (64, 3000, 256), (256, 256, 256), (1000, 1000, 256),
                                       (1500, 1500, 256), (2048, 1500, 256), (4000, 100, 256), (1500, 1500, 80),
                                       (300000, 60, 256)])
def test_equal_segments_fill_whole_waves_per_simd(scheme, math, strip, extra, nx, ny, cus):
    """Equal segments put no more than four waves on a SIMD (one workgroup of
    four beside each other on a CU), and never just a few more than a whole
    number of them: a shorter segment would not have fitted into as many."""
    lib = _lib.lib()
    launch = _lib.LaunchConfig(0, 4, _lib.FVMI_MATH_EXACT if math == "exact" else _lib.FVMI_MATH_FAST, 1)
    n = ctypes.c_int()
    lib.fvmi_substep_plan(scheme, nx, ny, 0, 0, 0, 0, ctypes.byref(launch), cus, None, 0, ctypes.byref(n))
    segs = np.zeros((n.value, 3), dtype=np.int32)
    assert lib.fvmi_substep_plan(scheme, nx, ny, 0, 0, 0, 0, ctypes.byref(launch), cus,
                                 segs.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), n.value, ctypes.byref(n)) == 0
    live = segs[segs[:, 0] >= 0]
    strips, rows = -(-(nx + extra) // strip), int(live[:, 2].max())
    band = -(-strips // 4) * 4 if scheme == HLL2 else strips
    simds = 4 * cus
    least = 4 if scheme == STEP else 2
    if len(np.unique(live[live[:, 1] + live[:, 2] < ny, 2])) > 1:
        return  # the round-weighted split
    if band > 4 * simds:
        assert rows == ny
        return
    waves = -(-band * -(-ny // rows) // simds)  # per SIMD
    assert waves <= 4 and rows >= min(least, ny)
    shorter = -(-band * -(-ny // max(rows - 1, 1)) // simds)
    assert shorter > waves or rows <= least or -(-ny // (rows - 1)) == -(-ny // rows)


@pytest.mark.parametrize("nx,ny,rounds", [(4096, 4096, True), (5500, 5500, True), (8192, 8192, False),
                                          (9500, 7000, False)])
def test_rounds_only_where_the_strips_fill_the_device(nx, ny, rounds):
    """The round-weighted split (parts in the ratio 14 : 6) where its row groups
    put at least 93 % of the equal segments' waves to work."""
    segs = plan(STEP, nx, ny)
    counts = segs[(segs[:, 0] >= 0) & (segs[:, 1] + segs[:, 2] < ny), 2]
    assert (counts.max() > 2 * counts.min()) == rounds
    if not rounds:
        assert len(np.unique(counts)) == 1
        assert (segs[:, 0] >= 0).sum() > 0.95 * 4 * 1024

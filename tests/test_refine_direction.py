"""The refinement's direction prune of (source lane, target chunk) pairs.

k_refine skips a chunk for a lane when the chunk's box and the box of the
lane's edge vertices are apart on an axis by more than 2^-8 of the reach q
and no segment of the chunk has the direction class of one of the lane's edges
(dir_bit, farm_amd/csrc/hip/device_layout.h; a segment holds the classes
within 2^-9 of its pseudo-angle).  That is only allowed if the reference
predicate (segment_intersect, src/include/geometry_computation.h:215-221) is
false for every edge of the lane and segment of the chunk: apart boxes leave
only crossings that binary32 rounding makes up, and those need an edge and a
segment whose lines meet at less than 2^-11.  These tests restate the masks in
f32 numpy and check that against the oracle's segment_intersect.
"""
import numpy as np
import pytest

import oracle
from tests.test_refine_prune import chunk_box, polyline

f32 = np.float32
BINS = 64
TOL = f32(2.0 ** -9)
ALL = (1 << BINS) - 1


def angle(u) -> tuple[np.float32, bool]:
    with np.errstate(all="ignore"):
        ux, uy = f32(u[0]), f32(u[1])
        n = f32(abs(ux) + abs(uy))
        s = f32(f32(1) - f32((-ux if uy < 0 else ux) * f32(f32(1) / n)))
    return s, bool(n >= f32(2.0 ** -60)) and bool(n < f32(2.0 ** 60))


def bit(s) -> int:
    return 1 << (int(np.floor(f32(s) * f32(BINS / 2))) & (BINS - 1))


def chunk_mask(chunk, tol=TOL) -> int:
    m = 0
    for k in range(len(chunk) - 1):
        s, ok = angle(chunk[k + 1] - chunk[k])
        m |= bit(f32(s - tol)) | bit(f32(s + tol)) if ok else ALL
    return m


def lane_mask(lane) -> int:
    m = 0
    for k in range(len(lane) - 1):
        s, ok = angle(lane[k + 1] - lane[k])
        m |= bit(s) if ok else ALL
    return m


def far(lane, box) -> bool:
    cx, cy, hx, hy = box
    with np.errstate(all="ignore"):
        ex0, ex1 = f32(cx - lane[:, 0].min()), f32(cx - lane[:, 0].max())
        ey0, ey1 = f32(cy - lane[:, 1].min()), f32(cy - lane[:, 1].max())
        q = f32(f32(f32(max(abs(ex0), abs(ex1)) + max(abs(ey0), abs(ey1))) + f32(hx + hy)) * f32(1.000001))
        hx1, hy1 = f32(hx * f32(1.000001)), f32(hy * f32(1.000001))
        sep = max(f32(max(ex1, -ex0) - hx1), f32(max(ey1, -ey0) - hy1))
        return bool(sep > f32(q * f32(2.0 ** -8))) and bool(q < f32(2.0 ** 60))


def skipped(lane, chunk, tol=TOL) -> bool:
    return far(lane, chunk_box(chunk[:, 0], chunk[:, 1])) and not (lane_mask(lane) & chunk_mask(chunk, tol))


def crossings(lane, chunk) -> int:
    return sum(oracle.segment_intersect(lane[i], lane[i + 1], chunk[k], chunk[k + 1])
               for i in range(len(lane) - 1) for k in range(len(chunk) - 1))


@pytest.mark.parametrize("edges", [1, 8])
def test_random_lanes_and_chunks(edges):
    rng = np.random.default_rng(41 + edges)
    fired = 0
    for _ in range(2000):
        chunk = polyline(rng, 17, rng.uniform(0, 40, 2), 0.02)
        lane = polyline(rng, edges + 1, chunk[rng.integers(17)] + rng.normal(0, 0.3, 2), 0.002)
        if skipped(lane, chunk):
            fired += 1
            assert not crossings(lane, chunk)
    assert fired > (300 if edges == 1 else 5)


def test_rounding_crossings_along_a_line_share_a_direction():
    # one source edge and one target segment on a common line (or an ulp off
    # it, or at a slight angle), apart along it: the regime in which the
    # reference's signs are noise and it does report crossings
    rng = np.random.default_rng(43)
    ref_true = apart = 0
    for _ in range(60000):
        scale = 2.0 ** rng.integers(-20, 21)
        o = rng.uniform(-1, 1, 2)
        th = rng.uniform(0, np.pi) if rng.random() < 0.7 else rng.choice([0, 0.25, 0.5, 0.75]) * np.pi
        u = np.array([np.cos(th), np.sin(th)])
        turn = th + rng.choice([0.0, 1.0]) * 10 ** rng.uniform(-9, -6)
        w = np.array([np.cos(turn), np.sin(turn)])
        la, lc = rng.uniform(0.1, 1, 2)
        a = o.astype(f32)
        b = (o + la * u).astype(f32)
        ab = b.astype(np.float64) - a
        nrm = np.array([-ab[1], ab[0]]) / np.linalg.norm(ab)
        c = a + (1.0 + 10 ** rng.uniform(-1.5, 0.5)) * ab + rng.uniform(-1, 1) * 1e-7 * nrm
        pts = (np.array([a, b, c, c + lc * w]) * scale).astype(f32)
        lane, chunk = pts[:2], pts[2:]
        if (chunk[0] == chunk[1]).all() or not oracle.segment_intersect(lane[0], lane[1], chunk[0], chunk[1]):
            continue
        ref_true += 1
        apart += far(lane, chunk_box(chunk[:, 0], chunk[:, 1]))
        assert not skipped(lane, chunk), (lane, chunk)
    assert ref_true > 200 and apart > 50  # the construction reaches the rounding regime


def test_the_tolerance_is_needed():
    # nearly parallel lines on both sides of a class's edge: the masks share a
    # bit with the kernel's tolerance, and some do not without it
    rng = np.random.default_rng(44)
    dropped = 0
    for _ in range(20000):
        s = rng.integers(0, BINS) / (BINS / 2) + rng.uniform(-1, 1) * 2.0 ** -12
        t = s + rng.uniform(-1, 1) * 2.0 ** -12

        def unit(v):  # a direction of pseudo-angle v
            c = 1.0 - v
            return np.array([c, 1.0 - abs(c)]) if 0 <= v <= 2 else np.array([c + (2 if v > 2 else -2), 1e-9])

        lane = np.array([[0, 0], unit(s)]).astype(f32)
        chunk = np.array([[5, 0], 5 * np.array([1, 0]) + unit(t)]).astype(f32)
        assert lane_mask(lane) & chunk_mask(chunk)
        dropped += not (lane_mask(lane) & chunk_mask(chunk, f32(0)))
    assert dropped > 0


def test_short_and_non_finite_edges_match_every_direction():
    for u in ((0.0, 0.0), (np.nan, 1.0), (np.inf, 1.0), (2.0 ** -70, 0.0), (2.0 ** 70, 1.0)):
        assert not angle(np.array(u, f32))[1]
    chunk = np.array([[0, 0], [1, np.nan], [2, 0]], f32)
    assert not far(np.array([[50, 0], [51, 0]], f32), chunk_box(chunk[:, 0], chunk[:, 1]))


def test_zero_length_segments_only_answer_with_box_overlap():
    # a repeated vertex c == d: the reference answers with the overlap of the
    # edge's box and c alone, so a chunk is kept for it only where the lane's
    # box and the chunk's are not apart (k_refine's rule for marked chunks)
    rng = np.random.default_rng(45)
    true = 0
    for _ in range(20000):
        c = rng.uniform(-1, 1, 2).astype(f32)
        lane = polyline(rng, 2, c + rng.normal(0, 0.1, 2), 0.1)
        lo, hi = lane[:2].min(0), lane[:2].max(0)
        hit = oracle.segment_intersect(lane[0], lane[1], c, c)
        assert hit == bool((lo <= c).all() and (c <= hi).all())
        true += hit
    assert true > 500

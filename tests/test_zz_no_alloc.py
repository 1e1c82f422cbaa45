"""farm_intersect_noalloc (no device allocation, the library's fixed per-GPU
scratch) against farm_intersect_dev on the same windows: two calls in a row,
the second on a smaller window, each bit-exact, with the same counters of
the filter and the same count of intersecting pairs."""
import numpy as np
import pytest

from farm_amd import capi, datagen
from tests.helpers import rings_from_list

pytestmark = pytest.mark.gpu


def _workload():
    (sa, sxy), (ta, txy) = datagen.star_pair_set(21, 600, 600, 0.0, 45.0)
    A, B = capi.HostSet.from_rings(sa, sxy), capi.HostSet.from_rings(ta, txy)
    pa, pb = capi.candidates(A, B)
    both = capi.HostSet.concat(A, B)
    both.rasterize(10)
    return both, len(A), pa, pb


def test_noalloc_matches_intersect_dev():
    from farm_amd.hipmem import DeviceBuffer

    both, na, pa, pb = _workload()
    n = len(pa)
    dev = capi.Device(0)
    ref = DeviceBuffer(n)
    got = DeviceBuffer(n)
    try:
        dev.upload_polygons(both)
        dev.upload_pairs(pa, pb + na)
        for (b, e), mode, tile in (((0, n), capi.MODE_EXACT_BATCHED, 8),
                                   ((n // 3, n // 3 + n // 4), capi.MODE_EXACT_BATCHED, 4),
                                   ((5, n // 2), capi.MODE_APPROX_HEURISTIC, 0),
                                   ((7, 200), capi.MODE_EXACT_PLAIN, 0)):
            print(f"window [{b},{e}) mode {mode} tile {tile}", flush=True)
            s_ref = dev.intersect_dev(ref.ptr, b, e, mode=mode, tile_a=tile)
            s_got = dev.intersect_noalloc(got.ptr, b, e, mode=mode, tile_a=tile)
            want = ref.to_host(np.uint8, e - b)
            have = got.to_host(np.uint8, e - b)
            diff = np.nonzero(want != have)[0]
            assert diff.size == 0, f"[{b},{e}) mode {mode}: {diff.size} pairs differ, first {diff[:10]}"
            # counters that do not depend on which wave finds a crossing first
            # (the executed segment tests of intersecting pairs do)
            for k in ("found", "in_hits", "bb_pixel_pairs", "filter_bytes"):
                assert s_ref[k] == s_got[k], (k, s_ref[k], s_got[k])
            assert 0 < s_got["found"] < e - b
        # beyond the scratch's pair capacity: a clear error, nothing launched
        with pytest.raises(capi.FarmError) as exc:
            dev.intersect_noalloc(None, 0, (1 << 18) + 1) if n > (1 << 18) else dev.intersect_noalloc(
                None, 0, n, mode=capi.MODE_APPROX_LEARNED)
        assert exc.value.code in (capi.FARM_ECAPACITY, capi.FARM_EINVAL)
    finally:
        ref.free()
        got.free()
        dev.close()


def _band(n, dx, seed):
    # a thin jagged band along a diagonal: BORDER pixels only, some with
    # hundreds of edges at 30 vertices per pixel
    rng = np.random.default_rng(seed)
    t = np.linspace(0, 1, n // 2)
    w = 0.004 * rng.uniform(-1, 1, n // 2)
    return np.concatenate([np.stack([t + dx + 1, t + 1 + w], 1),
                           np.stack([t + dx + 1.0005, t + 1 - 0.012 + w], 1)[::-1]])


def test_noalloc_default_tile_fits_what_four_edges_per_lane_fit():
    # mostly small polygons (the default is 1 edge per lane), but pairs of two
    # long ones, whose tiles fit the fixed scratch at 4 edges per lane and not
    # at 1 or 2: a call that names no tile takes 4
    from farm_amd.hipmem import DeviceBuffer

    rng = np.random.default_rng(3)
    ang = np.linspace(0, 2 * np.pi, 10, endpoint=False)
    polys = [_band(600, 0.0, 1), _band(600, 0.02, 2)]
    polys += [c + 0.05 * np.stack([np.cos(ang), np.sin(ang)], 1) for c in rng.uniform(5, 60, (2000, 2))]
    off, xy = rings_from_list(polys)
    H = capi.HostSet.from_rings(off, xy)
    H.rasterize(30)
    dev = capi.Device(0)
    try:
        dev.upload_polygons(H)
        assert dev.tuning()["tile_a"] == 1
        dev.upload_pairs(np.zeros(1, np.uint32), np.ones(1, np.uint32))
        per = dev.intersect(tile_a=4).stats["bb_pixel_pairs"]
        assert per > 8
        n = int(0.9 * (1 << 20)) // per
        a, b = np.zeros(n, np.uint32), np.ones(n, np.uint32)
        b[::2], a[::2] = 0, 1
        dev.upload_pairs(a, b)
        want = dev.intersect().bits
        out = DeviceBuffer(n)
        for tile in (1, 2):
            with pytest.raises(capi.FarmError) as exc:
                dev.intersect_noalloc(out.ptr, 0, n, tile_a=tile)
            assert exc.value.code == capi.FARM_ECAPACITY
        for tile in (4, 0):
            print(f"tile {tile}", flush=True)
            dev.intersect_noalloc(out.ptr, 0, n, tile_a=tile)
            assert np.array_equal(out.to_host(np.uint8, n), want)
        # a tile that the caller chose is kept
        dev.set_tuning(1, 16)
        with pytest.raises(capi.FarmError) as exc:
            dev.intersect_noalloc(out.ptr, 0, n)
        assert exc.value.code == capi.FARM_ECAPACITY
        out.free()
    finally:
        dev.close()

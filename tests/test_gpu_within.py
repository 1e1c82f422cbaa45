"""GPU parity: within-distance decision (hierarchical box-distance descent and
truncated segment distances) through the C ABI, bit-exact in decisions,
running minimum distances and work counters against the oracle."""
import numpy as np
import pytest

import oracle
from farm_amd import capi, datagen
from tests.helpers import rings_from_list

pytestmark = pytest.mark.gpu


def _run(dev, ro, xy, d_km=10.0, vpr=10, nlow=1, pairs=None, window=None):
    O = oracle.OracleSet(ro, xy)
    O.rasterize(vpr, hierarchy=True, nlow=nlow)
    H = capi.HostSet.from_rings(ro, xy)
    H.rasterize_h(vpr, nlow)
    if pairs is None:
        pa, pb = capi.candidates(H, H, expand_km=d_km, skip_self=True)
    else:
        pa, pb = (np.asarray(p, np.uint32) for p in pairs)
    print(f"  within d={d_km} vpr={vpr} nlow={nlow} polygons={len(O)} pairs={len(pa)}", flush=True)
    want, wmd, wst = oracle.within(O, O, pa, pb, d_km)
    dev.upload_polygons(H)
    dev.upload_pairs(pa, pb)
    lo, hi = (0, len(pa)) if window is None else window
    bits, md, st = dev.within(d_km, lo, hi)
    want, wmd = want[lo:hi], wmd[lo:hi]
    diff = np.nonzero(bits != want)[0]
    assert diff.size == 0, f"{diff.size} decisions differ, first {diff[:10]}: gpu {bits[diff[:10]]} cpu {want[diff[:10]]}"
    mdiff = np.nonzero(md.view(np.uint64) != wmd.view(np.uint64))[0]
    assert mdiff.size == 0, f"{mdiff.size} min distances differ, first {mdiff[:5]}: {md[mdiff[:5]]} vs {wmd[mdiff[:5]]}"
    assert st["found"] == int((want == 1).sum())
    if window is None:
        assert st["bb_pixel_pairs"] == wst["candidate_pixel_pairs"]
        assert st["segment_tests"] == wst["distance_evals"]
    return want, md, st


def test_lakes_10km(device):
    ro, xy = datagen.lake_set(41, 1500, hi=1.4)
    want, md, st = _run(device, ro, xy)
    assert (want == 1).sum() > 1000 and (want == 0).sum() > 1000
    assert (md != 100000.0).sum() > 1000  # the refinement path is exercised


def test_records_follow_the_polygons():
    # the pixels' and chunks' records are kept over pair lists and chunk sizes
    # and made anew for another set, larger or smaller, on the same handle
    dev = capi.Device(0)
    try:
        for n, chunk in ((300, 16), (500, 32), (200, 32), (200, 16), (400, 8)):
            dev.set_tuning(4, chunk)
            ro, xy = datagen.lake_set(60 + n + chunk, n, hi=0.7)
            _run(dev, ro, xy)
            H = capi.HostSet.from_rings(ro, xy)
            pa, pb = capi.candidates(H, H, expand_km=10.0, skip_self=True)
            want, wmd, _ = oracle.within(*[_oracle_set(ro, xy)] * 2, pa, pb, 10.0)
            for part in (slice(1, None, 3), slice(2, None, 5)):
                dev.upload_pairs(pa[part], pb[part])
                bits, md, _ = dev.within(10.0)
                assert np.array_equal(bits, want[part]) and np.array_equal(md.view(np.uint64), wmd[part].view(np.uint64))
                dev.set_tuning(4, 8)  # (other chunks, the same records)
    finally:
        dev.close()


def _oracle_set(ro, xy):
    O = oracle.OracleSet(ro, xy)
    O.rasterize(10, hierarchy=True, nlow=1)
    return O


@pytest.mark.parametrize("d_km", [0.0, 2.0, 25.0])
def test_lakes_other_distances(device, d_km):
    ro, xy = datagen.lake_set(5, 500, hi=0.8)
    _run(device, ro, xy, d_km=d_km)


def test_fine_rasters_take_the_global_path(device):
    # vpr 1: finest layers beyond 1024 pixels, so these pairs run with
    # global-memory pixel lists
    ro, xy = datagen.lake_set(9, 250, hi=0.6)
    _run(device, ro, xy, vpr=1)
    _run(device, ro, xy, vpr=3, nlow=20)


def test_mixed_sizes_and_pair_window(device):
    cro, cxy = datagen.complex_set(5, 6, hi=0.8, nv_cap=4000)
    lro, lxy = datagen.lake_set(6, 300, hi=0.8)
    ro = np.concatenate([cro, lro[1:] + cro[-1]])
    xy = np.concatenate([cxy, lxy])
    _run(device, ro, xy)
    _run(device, ro, xy, window=(100, 900))


def _square(x0, y0, s, per_edge=8):
    t = np.arange(per_edge, dtype=np.float64) / per_edge
    pts = []
    for (ax, ay), (bx, by) in [((x0, y0), (x0 + s, y0)), ((x0 + s, y0), (x0 + s, y0 + s)),
                               ((x0 + s, y0 + s), (x0, y0 + s)), ((x0, y0 + s), (x0, y0))]:
        pts.append(np.stack([ax + (bx - ax) * t, ay + (by - ay) * t], 1))
    return np.vstack(pts).astype(np.float32)


def test_hand_built_cases(device):
    # gaps around 10 km, a contained square, grid-aligned edges, identical
    # polygons and a triangle with too few vertices for a second layer
    polys = [
        _square(0.3, 0.5, 0.02, 16),
        _square(0.3 + 0.02 + 0.0898, 0.5, 0.02, 16),   # ~10.0 km east
        _square(0.3 + 0.02 + 0.0944, 0.52, 0.02, 16),  # ~10.5 km
        _square(0.013, 0.017, 1.0, 40),
        _square(0.49, 0.49, 0.04),
        _square(0.063, 0.49, 0.04),
        _square(0.0, 0.0, 1.0, 40),
        _square(0.05, 0.48, 0.04),
        np.array([[0.7, 0.7], [0.71, 0.7], [0.705, 0.71]], np.float32),
        _square(0.3, 0.5, 0.02, 16),
    ]
    ro, xy = rings_from_list(polys)
    n = len(polys)
    pa, pb = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    _run(device, ro, xy, pairs=(pa.ravel(), pb.ravel()))


def test_rejected_polygons_answer_2(device):
    # a one-pixel raster 500 degrees wide: no universal grid step is that
    # large, so MyRaster::grid_align's assertion fires in the reference; every
    # pair with that polygon answers 2
    big = np.array([[0, 0], [500, 0], [500, 50], [0, 50]], np.float32)
    ro, xy = datagen.lake_set(12, 40, hi=0.3)
    rings = [big] + [xy[int(ro[i]):int(ro[i + 1])] for i in range(len(ro) - 1)]
    n = len(rings)
    pa, pb = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    want, _, _ = _run(device, *rings_from_list(rings), pairs=(pa.ravel(), pb.ravel()))
    assert (want == 2).sum() == 2 * n - 1


def test_empty_window(device):
    ro, xy = datagen.lake_set(41, 50, hi=0.3)
    H = capi.HostSet.from_rings(ro, xy)
    H.rasterize_h(10, 1)
    device.upload_polygons(H)
    device.upload_pairs(np.zeros(1, np.uint32), np.ones(1, np.uint32))
    bits, md, st = device.within(10.0, 0, 0)
    assert len(bits) == 0 and st["found"] == 0


@pytest.mark.parametrize("chunk", [16, 32])
@pytest.mark.parametrize("vpr", [10, 150])
def test_candidates_and_rows_out_of_reach(vpr, chunk):
    # large lakes near small and large ones: hundreds of candidates a pair, most
    # of them passed over by their pixels' boxes or row by row; at vpr 150
    # sequences of many chunks (and of more than the box of a row looks at);
    # with 32-segment refinement chunks the boxes are a set of their own
    rng = np.random.default_rng(61)
    nv = np.concatenate([rng.integers(300, 1500, 30), rng.integers(20, 200, 60)])
    ro, xy = datagen.star_polygons(rng, 90, 0.0, 1.5, nv, np.log(0.12), 0.9)
    dev = capi.Device(0)
    try:
        dev.set_tuning(4, chunk, 8)
        for d_km in (4.0, 15.0):
            want, md, st = _run(dev, ro, xy, d_km=d_km, vpr=vpr)
            assert (want == 0).sum() > 50 and (want == 1).sum() > 50
        assert st["bb_pixel_pairs"] > 64 * 10
    finally:
        dev.close()

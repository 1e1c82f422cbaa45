"""GPU parity: exact intersect (plain and batched kernels, all tile widths)
and the reference -a heuristic, bit-exact against the oracle."""
import numpy as np
import pytest

import oracle
from farm_amd import capi
from tests.helpers import Workload, rings_from_list, star_pairs

pytestmark = pytest.mark.gpu

MODES = [
    (capi.MODE_EXACT_PLAIN, 0),
    (capi.MODE_EXACT_BATCHED, 1),
    (capi.MODE_EXACT_BATCHED, 2),
    (capi.MODE_EXACT_BATCHED, 4),
    (capi.MODE_EXACT_BATCHED, 8),
]


def _check(dev, w: Workload, modes=MODES, allow_ref_failures=False):
    want, st = w.oracle(0)
    # polygons on which the reference raster builder aborts or never ends:
    # the product must flag exactly the same ones (and answer false on them)
    ok = w.both.raster_ok()
    ref_failed = np.concatenate([w.OA.failed(), w.OB.failed()])
    assert np.array_equal(~ok, ref_failed)
    if not allow_ref_failures:
        assert not (want == 2).any(), "reference would abort on this input"
    done = want != 2
    w.upload(dev)
    for mode, tile in modes:
        print(f"  mode={mode} tile={tile} pairs={len(w.pa)}", flush=True)
        r = dev.intersect(mode=mode, tile_a=tile)
        diff = np.nonzero((r.bits != want) & done)[0]
        assert diff.size == 0, f"mode {mode} tile {tile}: {diff.size} pairs differ, first {diff[:10]}"
        assert not r.bits[~done].any()
        assert r.stats["found"] == int((want == 1).sum())
    return want, st


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_star_pairs_2k_full(device, seed):
    print(f"star pairs 2000 x 2000 seed={seed}", flush=True)
    w = star_pairs(seed)
    want, _ = _check(device, w)
    assert 0 < want.sum() < len(want)


def test_star_pairs_many_seeds(device):
    # 20 smaller seeded instances, every kernel variant
    for seed in range(100, 120):
        print(f"star pairs 400 x 400 seed={seed}", flush=True)
        _check(device, star_pairs(seed, n=400))


def test_heuristic_mode_matches_oracle(device):
    w = star_pairs(5)
    want, _ = w.oracle(1)
    w.upload(device)
    r = device.intersect(mode=capi.MODE_APPROX_HEURISTIC)
    assert np.array_equal(r.bits, want)


def test_autotuned_tile_is_exact(device, tmp_path):
    w = star_pairs(8, n=800)
    want, _ = w.oracle(0)
    w.upload(device)
    cache = str(tmp_path / "tune.txt")
    t = device.autotune(cache=cache)
    assert t["tile_a"] in (1, 2, 4, 8) and t["chunk"] in (8, 16, 32)
    again = device.autotune(cache=cache)  # served from the cache
    assert [again[k] for k in ("tile_a", "chunk", "blocks_per_cu", "shape_bucket")] == \
        [t[k] for k in ("tile_a", "chunk", "blocks_per_cu", "shape_bucket")]
    r = device.intersect()  # tile_a = tile_b = 0: the tuned configuration
    assert np.array_equal(r.bits, want)


@pytest.mark.parametrize("chunk", [8, 32])
def test_chunk_sizes(device, chunk):
    # the refinement with 8- and 32-step target chunks (16 is the default of
    # the tests above) on 10 small seeded instances, every tile width
    for seed in range(130, 140):
        print(f"star pairs 400 x 400 seed={seed} chunk={chunk}", flush=True)
        w = star_pairs(seed, n=400)
        want, _ = w.oracle(0)
        w.upload(device)
        for tile in (1, 2, 4, 8):
            r = device.intersect(mode=capi.MODE_EXACT_BATCHED, tile_a=tile, chunk=chunk)
            diff = np.nonzero(r.bits != want)[0]
            assert diff.size == 0, f"tile {tile} chunk {chunk}: {diff.size} pairs differ, first {diff[:10]}"


@pytest.mark.parametrize("vpr", [40, 300])
@pytest.mark.parametrize("chunk", [8, 16, 32])
def test_groups_of_chunks(device, chunk, vpr):
    # pixels of a few to hundreds of chunks, which begin and end anywhere in an
    # aligned group of them: the answers, and on pairs that all answer false
    # (so that nothing ends early) every test accounted for as run or pruned
    from farm_amd import datagen

    a, b = datagen.complex_set(41, 12, lo=0.0, hi=3.0), datagen.lake_set(42, 150, lo=0.0, hi=3.0)
    w = Workload(a, b, vpr=vpr)
    want, _ = w.oracle(0)
    w.upload(device)
    for tile in (1, 4, 8):
        r = device.intersect(mode=capi.MODE_EXACT_BATCHED, tile_a=tile, chunk=chunk)
        assert np.array_equal(r.bits, (want == 1).astype(np.uint8)), tile
    apart = want == 0
    device.upload_pairs(w.pa[apart], w.pb[apart] + len(w.A))
    full = device.intersect(mode=capi.MODE_EXACT_BATCHED, tile_a=1, chunk=chunk, flags=capi.FLAG_NO_PRUNE).stats
    assert full["pruned_tests"] == 0 and full["segment_tests"] > 0
    for tile in (1, 4, 8):
        st = device.intersect(mode=capi.MODE_EXACT_BATCHED, tile_a=tile, chunk=chunk).stats
        print(f"  -v {vpr} tile={tile} chunk={chunk}: {st['segment_tests']} run", flush=True)
        assert st["segment_tests"] + st["pruned_tests"] == full["segment_tests"]


def _collinear_slivers(seed, n):
    # pairs of thin triangles one behind the other along a line, their long
    # sides on it to within an ulp and parallel to within 1e-6: apart, so that
    # only the rounding of the f32 cross products can make them cross
    rng = np.random.default_rng(seed)
    scale = 2.0 ** rng.integers(-6, 6, n)[:, None, None]
    th = np.where(rng.random(n) < 0.7, rng.uniform(0, np.pi, n), rng.choice([0, 0.25, 0.5, 0.75], n) * np.pi)
    turn = th + rng.choice([0.0, 1.0], n) * 10 ** rng.uniform(-9, -6, n)
    o, u, w = rng.uniform(-1, 1, (n, 2)), np.stack([np.cos(th), np.sin(th)], 1), np.stack([np.cos(turn), np.sin(turn)], 1)
    a = o.astype(np.float32)
    b = (o + rng.uniform(0.1, 1, n)[:, None] * u).astype(np.float32)
    ab = b.astype(np.float64) - a
    nrm = np.stack([-ab[:, 1], ab[:, 0]], 1) / np.linalg.norm(ab, axis=1)[:, None]
    c = a + (1 + 10 ** rng.uniform(-1.5, 0.5, n))[:, None] * ab + rng.uniform(-1, 1, n)[:, None] * 1e-7 * nrm
    d = c + rng.uniform(0.1, 1, n)[:, None] * w
    A = np.stack([a, b, a + 1e-3 * nrm], 1) * scale
    B = np.stack([c, d, d - 1e-3 * nrm], 1) * scale
    return A.astype(np.float32), B.astype(np.float32)


def test_crossings_that_rounding_makes_up(device):
    # the direction prune may not drop them (its rule for k_refine, and the
    # intersection's collection, which has it too); one pixel a triangle, so
    # every pair of sides is looked at
    A, B = _collinear_slivers(47, 20000)
    k = np.arange(len(A))
    w = Workload(rings_from_list(list(A)), rings_from_list(list(B)), vpr=64, pairs=(k, k))
    want, _ = w.oracle(0)
    gap = np.maximum(B.min(1) - A.max(1), A.min(1) - B.max(1)).max(1)
    reach = (np.maximum(A.max(1), B.max(1)) - np.minimum(A.min(1), B.min(1))).sum(1)
    made_up = (want == 1) & (gap > reach * 2.0 ** -7)
    assert made_up.sum() > 300, made_up.sum()
    w.upload(device)
    for tile in (1, 2, 4, 8):
        for flags in (0, capi.FLAG_NO_PRUNE):
            r = device.intersect(mode=capi.MODE_EXACT_BATCHED, tile_a=tile, chunk=16, flags=flags)
            diff = np.nonzero(r.bits != (want == 1))[0]
            assert diff.size == 0, f"tile {tile} flags {flags}: {diff.size} pairs differ, first {diff[:10]}"
    counts, _, _ = device.intersection_area()
    assert np.array_equal(counts, oracle.intersection(w.OA, w.OB, w.pa, w.pb)[0])


@pytest.mark.parametrize("shape,vpr,tile", [("star", 10, 1), ("star", 48, 2), ("lakes", 10, 2), ("lakes", 32, 4),
                                            ("star", 300, 4)])
def test_default_tile_by_shape(shape, vpr, tile):
    # nothing tuned or set: few edges and chunks a pixel 1, up to 128 edges and
    # 24 chunks 2, beyond either 4; a chosen width stays for later sets
    from farm_amd import datagen

    if shape == "star":
        w = Workload(*datagen.star_pair_set(31, 300, 300, 0.0, 39.0), vpr=vpr)
    else:
        w = Workload(datagen.complex_set(41, 12, lo=0.0, hi=3.0), datagen.lake_set(42, 600, lo=0.0, hi=3.0), vpr=vpr)
    want, _ = w.oracle(0)
    dev = capi.Device(0)
    try:
        w.upload(dev)
        assert dev.tuning()["tile_a"] == tile
        assert np.array_equal(dev.intersect(mode=capi.MODE_EXACT_BATCHED).bits, (want == 1).astype(np.uint8))
        dev.set_tuning(8, 16)
        w.upload(dev)
        assert dev.tuning()["tile_a"] == 8
    finally:
        dev.close()


@pytest.mark.parametrize("chunk", [8, 16, 32])
def test_without_the_prune(device, chunk):
    # another kernel of its own: every chunk for every lane with an edge, in
    # rounds of 64 items and a part of one, at every tile width; on pairs that
    # all answer false, the same tests at each
    from farm_amd import datagen

    a, b = datagen.complex_set(41, 12, lo=0.0, hi=3.0), datagen.lake_set(42, 150, lo=0.0, hi=3.0)
    w = Workload(a, b, vpr=40)
    want, _ = w.oracle(0)
    w.upload(device)
    for tile in (1, 2, 4, 8):
        r = device.intersect(mode=capi.MODE_EXACT_BATCHED, tile_a=tile, chunk=chunk, flags=capi.FLAG_NO_PRUNE)
        assert np.array_equal(r.bits, (want == 1).astype(np.uint8)), tile
    apart = want == 0
    device.upload_pairs(w.pa[apart], w.pb[apart] + len(w.A))
    run = [device.intersect(mode=capi.MODE_EXACT_BATCHED, tile_a=t, chunk=chunk, flags=capi.FLAG_NO_PRUNE).stats
           for t in (1, 2, 4, 8)]
    assert run[0]["segment_tests"] > 0
    assert all(s["pruned_tests"] == 0 and s["segment_tests"] == run[0]["segment_tests"] for s in run)


def test_wide_tile_limit_holds_for_the_chunks_of_the_call(device):
    # a polygon beyond the limit in chunks of 8 segments and below it in chunks
    # of 32: which widths run is decided by the chunks that the call runs with,
    # whatever they were before it (the limit itself, 2^26 chunks, takes a ring
    # of 5e8 vertices)
    from farm_amd import datagen

    a, b = datagen.complex_set(41, 12, lo=0.0, hi=3.0), datagen.lake_set(42, 150, lo=0.0, hi=3.0)
    w = Workload(a, b, vpr=300)
    want, _ = w.oracle(0)
    w.upload(device)
    apart = want == 0
    device.upload_pairs(w.pa[apart], w.pb[apart] + len(w.A))
    nv = max(np.diff(np.asarray(r[0]).astype(np.int64)).max() for r in (a, b))

    def tiles(tile, chunk):
        r = device.intersect(mode=capi.MODE_EXACT_BATCHED, tile_a=tile, chunk=chunk)
        assert not r.bits.any()
        return r.stats["refine_items"]  # every tile runs: no pair answers true

    full = {t: tiles(t, 16) for t in (2, 4, 8)}
    assert full[2] > full[4] > full[8]
    try:
        device.set_wide_tile_limit(int(nv) // 16)
        for chunk, wide in ((32, True), (8, False), (32, True), (8, False)):
            for t in (8, 4, 2):
                got = tiles(t, chunk)
                print(f"  chunks of {chunk}, tile {t}: {got} tiles", flush=True)
                assert got == full[t if wide else 2]
    finally:
        device.set_wide_tile_limit(0)
    assert tiles(8, 8) == full[8]
    device.intersect(mode=capi.MODE_EXACT_BATCHED, chunk=16)


def test_tuning_rejects_bad_values(device):
    w = star_pairs(8, n=200)
    w.upload(device)
    with pytest.raises(capi.FarmError):
        device.set_tuning(3, 16, 8)
    with pytest.raises(capi.FarmError):
        device.set_tuning(8, 12, 8)
    with pytest.raises(capi.FarmError):
        device.intersect(mode=capi.MODE_EXACT_BATCHED, tile_a=8, chunk=24)


def test_batch_windows_concatenate(device):
    w = star_pairs(9, n=600)
    want, _ = w.oracle(0)
    w.upload(device)
    n = len(w.pa)
    cuts = [0, 1, 7, n // 3, n // 2 + 5, n]
    got = np.concatenate([device.intersect(b, e).bits for b, e in zip(cuts[:-1], cuts[1:])])
    assert np.array_equal(got, want)
    empty = device.intersect(3, 3)
    assert empty.bits.size == 0 and empty.stats["found"] == 0


def _square(x0, y0, x1, y1):
    return np.array([[x0, y0], [x1, y0], [x1, y1], [x0, y1]], dtype=np.float32)


def test_degenerate_shapes(device):
    # shared edges, touching corners, collinear overlaps, containment,
    # identical polygons, grid-aligned coordinates and one-pixel rasters
    a = [
        _square(10, 10, 20, 20),
        _square(30, 30, 31, 31),
        np.array([[50, 50], [60, 50], [55, 58]], np.float32),
        _square(70, 70, 90, 90),
        _square(1, 1, 1.5, 1.5),
        np.array([[5, 5], [6, 5], [6, 6], [5.5, 5.5], [5, 6]], np.float32),
    ]
    b = [
        _square(20, 12, 25, 18),       # shares the edge x = 20
        _square(31, 31, 32, 32),       # touches at one corner
        np.array([[55, 58], [65, 58], [60, 66]], np.float32),  # touches a vertex
        _square(75, 75, 80, 80),       # strictly inside a[3]
        _square(1, 1, 1.5, 1.5),       # identical
        _square(5.25, 5.25, 5.75, 5.75),
        _square(12, 21, 18, 22),       # near miss
        _square(20.0000001, 10, 21, 20),
    ]
    for vpr in (1, 2, 10):
        print(f"degenerate vpr={vpr}", flush=True)
        w = Workload(rings_from_list(a), rings_from_list(b), vpr=vpr)
        want, _ = _check(device, w, allow_ref_failures=True)
        assert (want != 2).sum() >= 5


def test_zero_length_target_segments(device):
    # Target rings strictly on one side of the line of a source edge, inside
    # that edge's box, each with a segment of length 0: a repeated vertex, or
    # (one-pixel raster) the reference's extra edge onto the repeated closing
    # vertex.  For c == d the reference's segment_intersect takes its
    # collinear branch and answers with the box overlap alone, so both pairs
    # are true; a prune that skipped the chunk by the line side would miss
    # them.
    a = [np.array([[0, 0], [1, 0], [1, 1]], np.float32)]
    b = [np.array([[0.45, 0.5], [0.45, 0.5], [0.40, 0.55], [0.35, 0.50]], np.float32),
         np.array([[0.45, 0.5], [0.40, 0.55], [0.35, 0.50]], np.float32)]
    w = Workload(rings_from_list(a), rings_from_list(b), pairs=([0, 0], [0, 1]))
    want, _ = _check(device, w)
    assert list(want) == [1, 1]


@pytest.mark.parametrize("bits", [3, 8])
def test_category_bits(device, bits):
    # -w b: fill classes at 2^b categories.  Exact bits do not change; the
    # reference -a decodes the finer classes (oracle mode 1 at 2^b)
    w = star_pairs(6, n=600)
    want, _ = w.oracle(0)
    import oracle

    heur, _ = oracle.intersect(w.OA, w.OB, w.pa, w.pb, 1, category_bits=bits)
    heur16, _ = oracle.intersect(w.OA, w.OB, w.pa, w.pb, 1)
    w.both.set_categories(bits)
    try:
        w.upload(device)
        assert np.array_equal(device.intersect(mode=capi.MODE_EXACT_BATCHED).bits, want)
        got = device.intersect(mode=capi.MODE_APPROX_HEURISTIC).bits
        assert np.array_equal(got, heur), int((got != heur).sum())
        assert not np.array_equal(heur, heur16) or bits == 4  # the category count matters to -a
    finally:
        w.both.set_categories(4)


def _comb(n, up, shift, tip=None):
    """A comb of n long teeth (from below, or from above), 1,200 high; tooth
    n / 2 reaches to y = tip."""
    pts = [(0.0, -60.0 if up else 1260.0), (4.0 * n, -60.0 if up else 1260.0)]
    y0, y1 = (0.0, 1080.0) if up else (1200.0, 120.0)
    for i in range(n - 1, -1, -1):
        x = 4.0 * i + shift
        yt = tip if (tip is not None and i == n // 2) else y1
        pts += [(x + 1.0, y0), (x + 0.8, yt), (x + 0.2, yt), (x, y0)]
    return np.array(pts if up else pts[1::-1] + pts[:1:-1])


@pytest.mark.parametrize("npairs", [1, 7, 64, 65, 1000])
@pytest.mark.parametrize("tile", [1, 8])
def test_window_sizes(device, npairs, tile):
    # from fewer tiles than cursors to several tiles per wave, and pixels of
    # more than 64 edge sequences of one edge (their chunks screened across
    # sequences): interlocked combs, apart or with one tooth through a spine
    combs = Workload(rings_from_list([_comb(300, True, 0.0)]),
                     rings_from_list([_comb(300, False, 2.0), _comb(300, False, 2.0, -80.0)]), vpr=48)
    assert max(np.diff(combs.both.layout()["pixoff"].astype(np.int64))) > 64
    assert combs.oracle(0)[0].tolist() == [0, 1]
    for w in (star_pairs(31, n=600), combs):
        want, _ = w.oracle(0)
        w.upload(device)
        n = len(w.pa)
        for b in range(0, n, max(npairs, n // 3)):
            e = min(b + npairs, n)
            print(f"  window {b}..{e} of {n} tile={tile}", flush=True)
            got = device.intersect(b, e, mode=capi.MODE_EXACT_BATCHED, tile_a=tile)
            assert np.array_equal(got.bits, (want[b:e] == 1).astype(np.uint8))

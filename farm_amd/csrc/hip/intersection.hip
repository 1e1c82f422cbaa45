// Intersection query on gfx950: boundary crossing points, classified
// boundary pieces and the area of A n B.
//
// Follows Ideal::intersection (src/geometry/Ideal.cpp:1440-1683) up to the
// piece statuses, where the reference returns: the crossing points of edges
// in BORDER x BORDER pixel pairs (segment_intersect_batch,
// src/include/geometry_computation.h:239-267), sorted and de-duplicated by
// point, the boundary of each polygon split at them, and every piece
// classified by Ideal::segment_contain (Ideal.cpp:1233-1327).  On top of
// those pieces the area is integrated with Green's theorem:
//   area = |sA * sum(A pieces IN B) + sB * sum(B pieces IN A)| / 2
// (cross-product sums of the piece paths relative to the low corner of the
// two MBBs' overlap; sX the orientation of ring X; a piece is IN when the
// midpoint of its longest sub-segment is).  Without two distinct crossing
// points the pair is contained (first vertex IN the other) or disjoint.
//
// One wavefront per pair, or the four of a workgroup for a pair with much work
// (k_ix_heavy) and for calls of few pairs:
//  1. the source raster's window over the target MBB; all OUT / all IN
//     windows end the pair (the reference's early return)
//  2. every edge pair of every BORDER x BORDER pixel pair: screens over the
//     pixels' 16-segment chunks (boxes and directions, then the sides of a
//     box and of each vertex against the source edge's line, with margins
//     above the f32 rounding) drop edge pairs that cannot cross; the rest
//     take the reference's exact f32 / f64 test a wave at a time; hits are
//     appended to a per-wave record slab in global memory
//  3. bitonic sorts of the slab (by point; by source edge and parameter;
//     by target edge and parameter), de-duplication, pieces, their statuses
//     (point-in-polygon tests, all of a wave's points together) and the
//     wave-cooperative path sums of the IN pieces
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cstring>
#include <vector>

#include "handle.h"
#include "wave.h"

namespace farm {

namespace {

struct Rec {
    float px, py;
    int32_t ei, ej;
    double t, u;
};

constexpr int kWaves = 4;
constexpr uint32_t kRecCap = 2048;     // records per wave slab (power of two)
constexpr uint32_t kRecCapBig = 65536;  // second pass for pairs beyond kRecCap (a third sizes to the largest)

// Point::operator== (Point.h:32)
__device__ __forceinline__ bool pt_eq(float ax, float ay, float bx, float by) {
    return fabsf(ax - bx) < 1e-9 && fabsf(ay - by) < 1e-9;
}

// key orders: 0 by point (then ei, ej, t, u); 1 by source edge and t (then
// ej, u); 2 by target edge and u (then ei, t)
template <int K>
__device__ __forceinline__ bool rec_less(const Rec &a, const Rec &b) {
    if constexpr (K == 0) {
        if (a.px != b.px) return a.px < b.px;
        if (a.py != b.py) return a.py < b.py;
        if (a.ei != b.ei) return a.ei < b.ei;
        if (a.ej != b.ej) return a.ej < b.ej;
        if (a.t != b.t) return a.t < b.t;
        return a.u < b.u;
    } else if constexpr (K == 1) {
        if (a.ei != b.ei) return a.ei < b.ei;
        if (a.t != b.t) return a.t < b.t;
        if (a.ej != b.ej) return a.ej < b.ej;
        return a.u < b.u;
    } else {
        if (a.ej != b.ej) return a.ej < b.ej;
        if (a.u != b.u) return a.u < b.u;
        if (a.ei != b.ei) return a.ei < b.ei;
        return a.t < b.t;
    }
}

__device__ __forceinline__ Rec pad_rec() {
    Rec r;
    r.px = INFINITY;
    r.py = INFINITY;
    r.ei = INT_MAX;
    r.ej = INT_MAX;
    r.t = INFINITY;
    r.u = INFINITY;
    return r;
}

// The lanes that share one pair: one wave (NW = 1), or the NW waves of a
// workgroup.
template <int NW>
struct Team {
    int lane, wv;
    __device__ __forceinline__ uint32_t tid() const { return (uint32_t)(NW == 1 ? lane : wv * 64 + lane); }
    __device__ __forceinline__ bool first() const { return NW == 1 || wv == 0; }
    __device__ __forceinline__ void sync() const {
        if constexpr (NW == 1) wave_sync();
        else __syncthreads();
    }
};

// Bitonic sort of R[0, n) in place; R has room for next_pow2(n) records.
template <int K, int NW>
__device__ void bitonic(Rec *R, uint32_t n, const Team<NW> &tm) {
    uint32_t m = 1;
    while (m < n) m <<= 1;
    for (uint32_t i = n + tm.tid(); i < m; i += 64 * NW) R[i] = pad_rec();
    tm.sync();
    for (uint32_t k = 2; k <= m; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            // pair p of this stage: i has bit j clear, l = i | j
            for (uint32_t p = tm.tid(); p < m / 2; p += 64 * NW) {
                const uint32_t i = 2 * p - (p & (j - 1)), l = i | j;
                const Rec a = R[i], b = R[l];
                const bool up = (i & k) == 0;
                if (rec_less<K>(b, a) == up) {
                    R[i] = b;
                    R[l] = a;
                }
            }
            tm.sync();
        }
    }
}

// The reference's crossing test of source edge ea and target edge eb
// (segment_intersect_batch, geometry_computation.h:239-267: f32 edge vectors
// and crosses, f64 parameters, f32 point), behind a screen that drops pairs
// whose parameters c2/dn, c1/dn lie clearly outside [-1e-6, 1 + 1e-6]
// (the f32 products in the screen are off by far less than the margins).
// Hits are appended to R through the wave's LDS counter.
__device__ __forceinline__ void edge_test(float ax, float ay, float d1x, float d1y, float bx, float by, float d2x,
                                          float d2y, uint32_t ea, uint32_t eb, Rec *R, uint32_t cap, uint32_t *cnt) {
    const float rx = bx - ax, ry = by - ay;
    const float dn = d1x * d2y - d1y * d2x;
    const float c2 = rx * d2y - ry * d2x;
    const float c1 = rx * d1y - ry * d1x;
    const float adn = fabsf(dn);
    const float s2 = dn < 0.f ? -c2 : c2, s1 = dn < 0.f ? -c1 : c1;
    const float lo = -1e-6f * adn, hi = 1.000001f * adn;
    if (!(s2 >= lo && s2 <= hi && s1 >= lo && s1 <= hi && (double)adn >= 1e-12)) return;
    const double denom = dn;
    const double t = c2 / denom;
    const double u = c1 / denom;
    if (t >= -1e-9 && t <= 1 + 1e-9 && u >= -1e-9 && u <= 1 + 1e-9) {
        const float tf = (float)t;
        Rec rec;
        rec.px = ax + tf * d1x;
        rec.py = ay + tf * d1y;
        rec.ei = (int32_t)ea;
        rec.ej = (int32_t)eb;
        rec.t = t;
        rec.u = u;
        const uint32_t pos = atomicAdd(cnt, 1u);
        if (pos < cap) R[pos] = rec;
    }
}

// ------------------------------------------------------------------------
// Collection: the edge pairs of one BORDER x BORDER pixel pair that may cross,
// narrowed down over the pixels' kIxChunk-segment chunks (a pixel's chunks are
// one consecutive range, whatever sequences they belong to) through three
// queues in LDS, each worked off 64 items or more at a time:
//   1. every (source chunk, target chunk) pair, one per lane: kept unless
//      their boxes are apart and their direction masks have no common bit;
//   2. every (edge of the source chunk, target chunk), 16 lanes to a pair:
//      kept unless the target box lies on one side of the edge's line;
//   3. every segment of the target chunk against the edge, one (edge, chunk)
//      per lane: kept unless both its ends lie on one side of the line;
//   4. the exact test (edge_test).
// On complex x lakes 1 keeps a fifth of the chunk pairs, 2 a tenth of their
// edges.  Walking the sequence pairs one by one, a wave of source edges against
// each target chunk, took 58 % of the kernel there (259 ms for 618,000 pairs,
// 138 with this), and more on jagged rings (pixels of 8 sequences of 3 edges).
//
// 1 is the refinement's direction prune.  A record needs t, u within 1e-9 of
// [0, 1]; the f32 crosses err by less than 2^-22 times the L1 lengths of their
// operands, so u puts a point of the target segment within (2^-22 3 q + 1e-9
// 2 q) sqrt 2 < 2^-20 q of the source line and t one of the source edge that
// near the target line (q the L1 reach).  With the boxes apart by g >= 2^-8 q
// the two lines then meet at less than 2 2^-20 q / g = 2^-11, and chunks that
// hold such segments share a direction bit (kDirTol = 2^-9).  Segments of
// length 0 give no record (dn = 0).
//
// 2 and 3: for the source edge a + s*d1, o(q) = (q - a) x d1 is the side of
// target vertex q.  edge_test accepts edge j only if u = o_j / dn lies in
// [-1e-9, 1 + 1e-9]; in exact arithmetic o_{j+1} = o_j - dn, and the rounding
// of o_j, o_{j+1} and dn (each product and difference rounded once, f32) moves
// o_{j+1} - (o_j - dn) by at most 2^-21 |d1|max (R_j + R_{j+1}), R = |q - a|_1,
// while 1e-9 |dn| stays below 2^-29 of the same scale.  So an accepted edge has
// min(o_j, o_{j+1}) <= M and max(o_j, o_{j+1}) >= -M for M = 2^-18 |d1|_1 Rmax,
// Rmax the reach of the chunk's box (four times the bound, which absorbs the
// rounding of M and of the fused o of the screen).  Every vertex q of a chunk
// lies in its box, so o(q) is within S = |d1y| hx + |d1x| hy of o at the centre
// c; the f32 o errs by at most M / 16 and a relative ulp.  When the f32 |o(c)|
// exceeds T = S (1 + 2^-20) + 2 M + 2^-100, every vertex lies beyond M on the
// side of o(c).  An infinite box (a non-finite vertex) makes T infinite or NaN
// and is never dropped.
// ------------------------------------------------------------------------
constexpr uint32_t kQueue = 128;  // flushed once 64 are queued, so one push always fits
struct PairQueue {
    uint32_t a[kQueue];
    uint32_t b[kQueue];
};
struct alignas(16) Queues {
    PairQueue chunks;  // source chunk, target chunk
    PairQueue lines;   // source edge's first vertex, target chunk
    PairQueue edges;   // first vertices of the source and target edge
};

// Wave-uniform state of one pair's collection.
struct Collect {
    const float4 *box;  // DevSet::ixbox / ixseg
    const uint4 *seg;
    const float *AX, *AY, *BX, *BY;
    Queues *q;
    uint32_t nc, nl, ne;  // queued items
    Rec *R;
    uint32_t cap;
    uint32_t *cnt;
    int lane;
};

__device__ __forceinline__ void push_pair(PairQueue &q, uint32_t &n, bool keep, uint32_t a, uint32_t b, int lane) {
    const uint64_t m = __ballot(keep);
    if (keep) {
        const uint32_t pos = n + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        q.a[pos] = a;
        q.b[pos] = b;
    }
    n = uni(n + (uint32_t)__popcll(m));
}

// 4: the exact test of every queued edge pair, one per lane.
__device__ __forceinline__ void flush_edges(Collect &C) {
    wave_sync();
    for (uint32_t k = C.lane; k < C.ne; k += 64) {
        const uint32_t ea = C.q->edges.a[k], eb = C.q->edges.b[k];
        const float ax = C.AX[ea], ay = C.AY[ea], bx = C.BX[eb], by = C.BY[eb];
        edge_test(ax, ay, C.AX[ea + 1] - ax, C.AY[ea + 1] - ay, bx, by, C.BX[eb + 1] - bx, C.BY[eb + 1] - by, ea, eb,
                  C.R, C.cap, C.cnt);
    }
    C.ne = 0;
    wave_sync();
}

// the margin M of edge a + s * d1 against a chunk's box
__device__ __forceinline__ float line_margin(float ax, float ay, float d1x, float d1y, float4 bb) {
    const float r = ((fabsf(bb.x - ax) + bb.z) + (fabsf(bb.y - ay) + bb.w)) * 1.000001f;
    return 0x1p-18f * (fabsf(d1x) + fabsf(d1y)) * r;
}

// 3: the first n <= 64 queued (edge, chunk) items, one per lane.
__device__ __forceinline__ void flush_lines(Collect &C, uint32_t n) {
    wave_sync();
    const bool on = (uint32_t)C.lane < n;
    const uint32_t k = on ? (uint32_t)C.lane : 0u;
    const uint32_t ea = C.q->lines.a[k], cb = C.q->lines.b[k];
    const uint4 sg = C.seg[cb];
    const float4 bb = C.box[cb];
    const uint32_t v0 = sg.x, ns = on ? sg.y & (kChunkPoint - 1u) : 0u;
    const float ax = C.AX[ea], ay = C.AY[ea];
    const float d1x = C.AX[ea + 1] - ax, d1y = C.AY[ea + 1] - ay;
    const float M = line_margin(ax, ay, d1x, d1y, bb);
    // the items behind the first 64 move up (read before they are overwritten)
    const bool more = (uint32_t)C.lane + n < C.nl;
    const uint32_t ma = more ? C.q->lines.a[C.lane + n] : 0u, mb = more ? C.q->lines.b[C.lane + n] : 0u;
    wave_sync();
    if (more) {
        C.q->lines.a[C.lane] = ma;
        C.q->lines.b[C.lane] = mb;
    }
    C.nl -= n;
    auto side = [&](uint32_t v) { return fmaf(C.BX[v] - ax, d1y, -((C.BY[v] - ay) * d1x)); };
    float o = side(v0);
    for (uint32_t m = 0; __ballot(m < ns); m++) {
        const uint32_t v = v0 + min(m + 1, ns);
        const float p = side(v);
        const bool keep = m < ns && !((o > M && p > M) || (o < -M && p < -M));
        if (__ballot(keep)) {
            push_pair(C.q->edges, C.ne, keep, ea, v0 + m, C.lane);
            if (C.ne >= 64) flush_edges(C);
        }
        o = p;
    }
}

// 2: every queued (source chunk, target chunk) pair, 4 per round: lane 16 i + e
// takes edge e of pair i.
__device__ __forceinline__ void flush_chunks(Collect &C) {
    wave_sync();
    const uint32_t e = (uint32_t)C.lane & 15u, sub = (uint32_t)C.lane >> 4;
    for (uint32_t k0 = 0; k0 < C.nc; k0 += 4) {
        const uint32_t k = k0 + sub;
        bool keep = false;
        uint32_t ea = 0, cb = 0;
        if (k < C.nc) {
            const uint4 sg = C.seg[C.q->chunks.a[k]];
            cb = C.q->chunks.b[k];
            if (e < (sg.y & (kChunkPoint - 1u))) {
                const float4 bb = C.box[cb];
                ea = sg.x + e;
                const float ax = C.AX[ea], ay = C.AY[ea];
                const float d1x = C.AX[ea + 1] - ax, d1y = C.AY[ea + 1] - ay;
                const float M = line_margin(ax, ay, d1x, d1y, bb);
                const float oc = fmaf(bb.x - ax, d1y, -((bb.y - ay) * d1x));
                const float T = fmaf(fmaf(fabsf(d1y), bb.z, fabsf(d1x) * bb.w), 1.000001f, fmaf(M, 2.f, 0x1p-100f));
                keep = !(fabsf(oc) > T);
            }
        }
        push_pair(C.q->lines, C.nl, keep, ea, cb, C.lane);
        if (C.nl >= 64) flush_lines(C, 64);
    }
    C.nc = 0;
    wave_sync();
}

// 1: the chunk pairs of source chunks [a0, a1) and target chunks [b0, b1), 64
// at a time: rounds start, start + NW, ..
template <int NW>
__device__ __forceinline__ void collect_chunks(Collect &C, uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1,
                                               uint32_t start) {
    const uint32_t na = a1 - a0, nb = b1 - b0;
    if (na == 0 || nb == 0) return;
    const uint32_t f = 64u * start + (uint32_t)C.lane;
    uint32_t i = f / nb, j = f - i * nb;
    const uint32_t qi = 64u * NW / nb, rj = 64u * NW - qi * nb;
    while (__ballot(i < na)) {
        bool keep = false;
        if (i < na) {
            const float4 A = C.box[a0 + i], B = C.box[b0 + j];
            const uint4 sa = C.seg[a0 + i], sb = C.seg[b0 + j];
            const float sx = fabsf(A.x - B.x), sy = fabsf(A.y - B.y), hx = A.z + B.z, hy = A.w + B.w;
            const float q = ((sx + hx) + (sy + hy)) * 1.000001f;
            const float gap = fmaxf(sx - hx * 1.000001f, sy - hy * 1.000001f);
            const bool far = gap > q * 0x1p-8f && q < 0x1p60f;
            keep = !far || ((sa.z & sb.z) | (sa.w & sb.w)) != 0u;
        }
        push_pair(C.q->chunks, C.nc, keep, a0 + i, b0 + j, C.lane);
        if (C.nc >= 64) flush_chunks(C);
        i += qi;
        j += rj;
        if (j >= nb) {
            j -= nb;
            i++;
        }
    }
}

// Ideal::segment_contain with count_intersection_nodes (Ideal.cpp:988-1006) for
// one point per lane (active lanes): 0 OUT, 1 BORDER (on the boundary), 2 IN.
// The serial form returns 1 at the first edge that puts the point on the
// boundary, else the parity of the crossings to the right within the pixel and
// of the sorted grid-line nodes below the point; neither depends on the order
// the edges are visited in.  So all points share the wave: (point, chunk of its
// pixel) items, one per lane, drop the chunks that cannot matter (entirely
// above, below or to the left of the point: no vertex of such a chunk is the
// point, no edge of it straddles the point's y or crosses to its right); the
// rest are queued and their edges tested, 16 lanes to a chunk, the answers
// gathered per point in LDS.  (One point after the other, the wave over its
// pixel's edges, each took a chain of six dependent loads: two thirds of the
// kernel on complex x lakes.)
__device__ __forceinline__ int contain_points(const DevSet &S, const farm_raster_hdr &h, float px, float py, bool active, int lane,
                              Queues &Q) {
    uint32_t *flag = Q.edges.a, *gx = Q.edges.a + 64;     // 1: odd crossings, 2: on the boundary; the pixel's x
    uint32_t *pre = Q.edges.b, *ch0 = Q.edges.b + 64;     // first item and first chunk of each point
    float *fx = (float *)Q.lines.a, *fy = (float *)Q.lines.b;
    int res = 0, x = 0;
    uint32_t c0 = 0, nch = 0;
    if (active) {
        x = off_axis((double)px, h.mbr[0], h.step[0], h.dimx);
        const int y = off_axis((double)py, h.mbr[1], h.step[1], h.dimy);
        const uint32_t id = (uint32_t)(y * h.dimx + x);
        const uint8_t st = S.status[h.pix_start + id];
        if (st == kCC - 1) res = 2;
        else if (st != 0) {
            const uint32_t s0 = S.pixoff[h.pixoff_start + id], s1 = S.pixoff[h.pixoff_start + id + 1];
            c0 = S.ixoff[h.seq_start + s0];
            nch = S.ixoff[h.seq_start + s1] - c0;
            res = -1;
        }
    }
    const bool todo = res < 0;
    if (!__ballot(todo)) return res;
    uint32_t total;
    const uint32_t first = wave_excl_scan(nch, lane, &total);
    flag[lane] = 0u;
    gx[lane] = (uint32_t)x;
    pre[lane] = first;
    ch0[lane] = c0;
    fx[lane] = px;
    fy[lane] = py;
    wave_sync();
    const float *X = S.x + h.vert_start, *Y = S.y + h.vert_start;
    uint32_t nq = 0;
    auto flush = [&]() {
        wave_sync();
        const uint32_t e = (uint32_t)lane & 15u, sub = (uint32_t)lane >> 4;
#pragma unroll 2
        for (uint32_t k0 = 0; k0 < nq; k0 += 4) {
            const uint32_t k = k0 + sub;
            if (k >= nq) continue;
            const uint32_t p = Q.chunks.a[k];
            const uint4 sg = S.ixseg[Q.chunks.b[k]];
            if (e >= (sg.y & (kChunkPoint - 1u))) continue;
            const uint32_t v = sg.x + e;
            const float v1x = X[v], v1y = Y[v], v2x = X[v + 1], v2y = Y[v + 1];
            const float qx = fx[p], qy = fy[p];
            bool on = pt_eq(qx, qy, v1x, v1y) || pt_eq(qx, qy, v2x, v2y), cross = false;
            if ((v1y >= qy) != (v2y >= qy)) {
                const double dx = (double)(v2x - v1x);
                const double dy = (double)(v2y - v1y);
                const double pyd = (double)(qy - v1y);
                if (fabs(dy) > 1e-9) {
                    const double ix = dx * pyd / dy + (double)v1x;
                    const double bx_high = h.mbr[0] + ((int)gx[p] + 1) * h.step[0];
                    if (fabs((double)qx - ix) < 1e-9) on = true;
                    cross = (double)qx < ix && ix <= bx_high;
                }
            } else if (v1y == qy && v2y == qy && ((v1x >= qx) != (v2x >= qx))) {
                on = true;
            }
            if (on) atomicOr(&flag[p], 2u);
            if (cross) atomicXor(&flag[p], 1u);
        }
        nq = 0;
        wave_sync();
    };
    for (uint32_t u0 = 0; u0 < total; u0 += 64) {
        const uint32_t u = u0 + (uint32_t)lane;
        bool keep = false;
        uint32_t p = 0, ch = 0;
        if (u < total) {
            // the last point whose first item is at or before u
#pragma unroll
            for (uint32_t step = 32; step > 0; step >>= 1)
                if (pre[p + step] <= u) p += step;
            ch = ch0[p] + (u - pre[p]);
            const float4 bb = S.ixbox[ch];
            const double qx = (double)fx[p], qy = (double)fy[p];
            const double ylo = (double)bb.y - (double)bb.w, yhi = (double)bb.y + (double)bb.w;
            const double xhi = (double)bb.x + (double)bb.z * 1.00001;  // (and a crossing's rounding beyond it)
            keep = !(qy > yhi + 1e-8 || qy < ylo - 1e-8 || qx > xhi + 1e-8);
        }
        push_pair(Q.chunks, nq, keep, p, ch, lane);
        if (nq >= 64) flush();
    }
    if (nq) flush();
    if (todo) {
        const uint32_t f = flag[lane];
        if (f & 2u) {
            res = 1;
        } else {
            // grid-line nodes below the point (sorted: a binary search)
            const uint32_t *vo = S.voff + h.vline_start;
            uint32_t lo = vo[x + 1], hi = vo[x + 2];
            const uint32_t i = lo;
            while (lo < hi) {
                const uint32_t mid = lo + (hi - lo) / 2;
                if (S.vnodes[h.vnode_start + mid] < (double)py) lo = mid + 1;
                else hi = mid;
            }
            res = ((f ^ (lo - i)) & 1u) ? 2 : 0;
        }
    }
    wave_sync();
    return res;
}

// The IN pieces of a pair go to buf (when requested), one atomic per wave
// and chunk; beyond cap they are only counted.
struct PieceOut {
    farm_piece *buf;
    uint32_t *cnt;
    uint32_t cap;
    uint32_t pair;
};

__device__ __forceinline__ void put_pieces(const PieceOut &po, bool mine, const farm_piece &p, int lane) {
    const uint64_t m = __ballot(mine);
    if (!po.buf || !m) return;
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(po.cnt, (uint32_t)__popcll(m));
    base = uni(__shfl(base, 0, 64));
    if (mine) {
        const uint32_t k = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        if (k < po.cap) po.buf[k] = p;
    }
}

struct PairRes {
    int32_t c[5];  // [crossing points, pieces, IN, OUT, BORDER]
    double area;
    uint64_t bb, tests, raw;
    bool over;
};

// Path point k of an area piece: 0 = a, 1..nvert = ring vertices from
// `first` (cyclic over m), nvert + 1 = b.
__device__ __forceinline__ void path_pt(const float *X, const float *Y, int m, int first, int nvert, float ax,
                                        float ay, float bx, float by, int k, float &x, float &y) {
    if (k == 0) {
        x = ax;
        y = ay;
    } else if (k == nvert + 1) {
        x = bx;
        y = by;
    } else {
        int v = first + k - 1;
        if (v >= m) v -= m;
        x = X[v];
        y = Y[v];
    }
}

constexpr int kLanePath = 16;  // area-piece paths of at most this many segments are searched by one lane

// A ring of m distinct vertices; cross products are taken relative to (ox, oy).
struct Ring {
    const float *X, *Y;
    int m;
    double ox, oy;
    // segment k of the path from a through nv vertices to b
    __device__ __forceinline__ double term(int f, int nv, float ax, float ay, float bx, float by, int k) const {
        float x0, y0, x1, y1;
        path_pt(X, Y, m, f, nv, ax, ay, bx, by, k, x0, y0);
        path_pt(X, Y, m, f, nv, ax, ay, bx, by, k + 1, x1, y1);
        return ((double)x0 - ox) * ((double)y1 - oy) - ((double)x1 - ox) * ((double)y0 - oy);
    }
};

// A path sum has one order, whatever the team: lane k adds segments k, k + 64,
// .. of one IN piece after the other.  (Its last bits are part of the area, and
// which pairs go to a team depends on the call's size.)  A team's lanes work
// out the segments of a piece each, up to `width` of them, into a row of memory
// (0 past the piece's last and for other pieces, which adds nothing; a longer
// piece's row has its vertices and ends), and one wave adds up the rows.
constexpr int kRow = 8;
constexpr int kRowLong = 0x7ff8b17e;  // high word of a longer piece's row: a NaN no arithmetic makes

// This lane's part of a ring's path sum, from the n rows.  (A call of its own:
// inlined it spills the kernel's registers.  Both rings' sums by two waves, after
// their pieces: 4,000 pairs of jagged rings, some hundred pieces each, 2.66 ms a
// call; one after the other 2.84; every wave its own pieces, in no one order, 2.74.)
__device__ __noinline__ double sum_rows(const Ring ring, const double *rows, uint32_t n, int width, int lane, Queues &Q) {
    static_assert(sizeof(Queues) >= 32 * kRow * sizeof(double), "32 rows in a wave's queues");
    double *lds = reinterpret_cast<double *>(&Q);
    double acc = 0.0;
    uint4 next[2];  // the next 32 rows, on their way
    const uint64_t nval = (uint64_t)width * n;
    const uint4 *rows4 = reinterpret_cast<const uint4 *>(rows);
    uint4 *lds4 = reinterpret_cast<uint4 *>(lds);
    auto load = [&](uint32_t p0) {
#pragma unroll
        for (uint32_t k = 0; k < 2; k++) {
            const uint64_t o = (uint64_t)width / 2 * p0 + 64 * k + lane;
            next[k] = rows4[o < nval / 2 ? o : 0];
        }
    };
    load(0);
    for (uint32_t p0 = 0; p0 < n; p0 += 32) {
        const uint32_t np = min(n - p0, 32u);
        wave_sync();
#pragma unroll
        for (uint32_t k = 0; k < 2; k++)
            if ((int)(64 * k) < 16 * width) lds4[64 * k + lane] = next[k];
        load(p0 + 32);
        wave_sync();
        uint32_t wm = (uint32_t)__ballot((uint32_t)lane < np && reinterpret_cast<const int *>(lds)[2 * width * (lane & 31) + 1] == kRowLong);
        for (uint32_t p = 0; p < np; p++) {
            // the rows up to the next longer piece
            const uint32_t end = wm ? (uint32_t)__ffs((int)wm) - 1u : np;
            if (lane < width) {
#pragma unroll 8
                for (; p < end; p++) acc += lds[width * p + lane];
            }
            p = end;
            if (!wm) break;
            wm &= wm - 1;
            const int *w = reinterpret_cast<const int *>(lds + width * p);
            const int f = uni(w[2]), nv = uni(w[3]);
            const float ax = __int_as_float(w[4]), ay = __int_as_float(w[5]);
            const float bx = __int_as_float(w[6]), by = __int_as_float(w[7]);
            for (int k = lane; k <= nv; k += 64) acc += ring.term(f, nv, ax, ay, bx, by, k);
        }
    }
    return acc;
}

// One ring's pieces: D[0, n) sorted by this ring's (edge, parameter).
// Counts the reference pieces by status into r (this wave's, of a team whose
// waves take 64 pieces each in turn) and returns this lane's part of the
// cross-product sum of the area pieces IN the other polygon, or leaves it to
// sum_rows (a team's).
template <bool SRC, int NW>
__device__ double ring_pieces(const DevSet &S, const farm_raster_hdr &hp, const farm_raster_hdr &hq, const Rec *D,
                              uint32_t n, double *rows, int width, double ox, double oy, const Team<NW> &tm, PairRes &r,
                              const PieceOut &po, Queues &Q) {
    const int lane = tm.lane;
    const float *X = S.x + hp.vert_start, *Y = S.y + hp.vert_start;
    const int m = (int)hp.nverts - 1;
    const double eps = (double)1e-6f;  // util.h:44
    double acc = 0.0;
    const Ring ring{X, Y, m, ox, oy};
    // ring vertices on the way from record i (a) to the next (b)
    auto path_len = [&](uint32_t i, const Rec &a, const Rec &b) {
        const int e0 = SRC ? a.ei : a.ej, e1 = SRC ? b.ei : b.ej;
        const double t0 = SRC ? a.t : a.u, t1 = SRC ? b.t : b.u;
        return i + 1 < n ? max(e1 - e0, 0) : (e1 - e0 + m) % m + ((e1 == e0 && t1 <= t0) ? m : 0);
    };
    for (uint32_t c0 = NW == 1 ? 0u : 64u * tm.wv; c0 < n; c0 += 64 * NW) {
        const uint32_t i = c0 + lane;
        bool piece = false, in_area = false, long_path = false;
        int st = 0, first = 0, nvert = 0;
        float ax = 0, ay = 0, bx = 0, by = 0;
        float rx = 0, ry = 0, mx = 0, my = 0;  // the two points tested against the other polygon
        if (i < n) {
            const Rec a = D[i], b = D[(i + 1) % n];
            ax = a.px;
            ay = a.py;
            bx = b.px;
            by = b.py;
            if (!pt_eq(a.px, a.py, b.px, b.py)) {
                piece = true;
                // the reference's segment (Ideal.cpp:1559-1581, 1592-1614)
                const int ea0 = SRC ? a.ei : a.ej, eb0 = SRC ? b.ei : b.ej;
                const double ta0 = SRC ? a.t : a.u, tb0 = SRC ? b.t : b.u;
                int ae = ea0, be = eb0;
                double ap = ta0, bp = tb0;
                if (fabs(ap - 1.0) < eps) {
                    ae = (ae + 1) % m;
                    ap = 0.0;
                }
                if (fabs(bp) < eps) {
                    be--;
                    bp = 1.0;
                }
                if (ae == be && ap < bp) {
                    rx = (a.px + b.px) * 0.5f;
                    ry = (a.py + b.py) * 0.5f;
                } else {
                    rx = X[ae + 1];
                    ry = Y[ae + 1];
                }
                // the area piece: a -> ring vertices ea0 + 1 .. eb0 -> b
                nvert = path_len(i, a, b);
                first = ea0 + 1;
                // the area's test point: the midpoint of the path's longest
                // sub-segment (the first on ties), well inside the piece; a
                // path of more than kLanePath segments is searched by the
                // whole wave below
                if (nvert + 1 <= kLanePath) {
                    float ux = ax, uy = ay, vx = ax, vy = ay, px = ax, py = ay;
                    double best = -1.0;
                    for (int k = 1; k <= nvert + 1; k++) {
                        float qx, qy;
                        path_pt(X, Y, m, first, nvert, ax, ay, bx, by, k, qx, qy);
                        const double dx = (double)qx - px, dy = (double)qy - py;
                        const double l = dx * dx + dy * dy;
                        if (l > best) {
                            best = l;
                            ux = px;
                            uy = py;
                            vx = qx;
                            vy = qy;
                        }
                        px = qx;
                        py = qy;
                    }
                    mx = (ux + vx) * 0.5f;
                    my = (uy + vy) * 0.5f;
                } else {
                    long_path = true;
                }
            }
        }
        // long paths, one at a time: segment k (points k - 1 -> k) on lane
        // (k - 1) % 64; each lane keeps its first longest, then the wave takes
        // the longest with the smallest k
        uint64_t lp = __ballot(long_path);
        while (lp) {
            const int src = __ffsll((unsigned long long)lp) - 1;
            lp &= lp - 1;
            const int f = uni(__shfl(first, src, 64)), nv = uni(__shfl(nvert, src, 64));
            const float pax = uni(__shfl(ax, src, 64)), pay = uni(__shfl(ay, src, 64));
            const float pbx = uni(__shfl(bx, src, 64)), pby = uni(__shfl(by, src, 64));
            double best = -1.0;
            int bk = INT_MAX;
            float ux = 0.f, uy = 0.f, vx = 0.f, vy = 0.f;
            for (int k = 1 + lane; k <= nv + 1; k += 64) {
                float x0, y0, x1, y1;
                path_pt(X, Y, m, f, nv, pax, pay, pbx, pby, k - 1, x0, y0);
                path_pt(X, Y, m, f, nv, pax, pay, pbx, pby, k, x1, y1);
                const double dx = (double)x1 - x0, dy = (double)y1 - y0;
                const double l = dx * dx + dy * dy;
                if (l > best) {
                    best = l;
                    bk = k;
                    ux = x0;
                    uy = y0;
                    vx = x1;
                    vy = y1;
                }
            }
            const double top = -wave_min(-best);
            int kk = best == top ? bk : INT_MAX;
            for (int o = 32; o > 0; o >>= 1) kk = min(kk, __shfl_xor(kk, o, 64));
            const int wl = __ffsll((unsigned long long)__ballot(best == top && bk == kk)) - 1;
            const float wmx = (__shfl(ux, wl, 64) + __shfl(vx, wl, 64)) * 0.5f;
            const float wmy = (__shfl(uy, wl, 64) + __shfl(vy, wl, 64)) * 0.5f;
            if (lane == src) {
                mx = wmx;
                my = wmy;
            }
        }
        const uint64_t pm = __ballot(piece);
        if (min(n - c0, 64u) <= 32) {
            // both points of every piece at once: lane 32 + k takes piece k's second
            const float qx = __shfl(mx, lane & 31, 64), qy = __shfl(my, lane & 31, 64);
            const bool up = lane >= 32, act = (pm >> (lane & 31)) & 1u;
            const int s = contain_points(S, hq, up ? qx : rx, up ? qy : ry, act, lane, Q);
            const int s2 = __shfl(s, (lane + 32) & 63, 64);
            if (piece) {
                st = s;
                in_area = s2 == 2;
            }
        } else {
            st = contain_points(S, hq, rx, ry, piece, lane, Q);
            in_area = contain_points(S, hq, mx, my, piece, lane, Q) == 2 && piece;
        }
        r.c[1] += __popcll(pm);
        r.c[2] += __popcll(__ballot(piece && st == 2));
        r.c[3] += __popcll(__ballot(piece && st == 0));
        r.c[4] += __popcll(__ballot(piece && st == 1));
        put_pieces(po, in_area, farm_piece{po.pair, SRC ? 0 : 1, first, nvert, ax, ay, bx, by}, lane);
        if constexpr (NW > 1) {
            if (i < n) {
                double t[kRow] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
                if (in_area && nvert < width) {
#pragma unroll
                    for (int k = 0; k < kRow; k++)
                        if (k <= nvert) t[k] = ring.term(first, nvert, ax, ay, bx, by, k);
                    // a NaN vertex keeps its low bits through the arithmetic
                    // and could read as a longer piece's row
                    if (!(t[0] == t[0])) t[0] = NAN;
                } else if (in_area) {
                    t[0] = __hiloint2double(kRowLong, 0);
                    t[1] = __hiloint2double(nvert, first);
                    t[2] = __hiloint2double(__float_as_int(ay), __float_as_int(ax));
                    t[3] = __hiloint2double(__float_as_int(by), __float_as_int(bx));
                }
#pragma unroll
                for (int k = 0; k < kRow; k++)
                    if (k < width) rows[(uint64_t)width * i + k] = t[k];
            }
        } else {
            // the wave over one IN piece after the other
            uint64_t inm = __ballot(in_area);
            while (inm) {
                const int src = __ffsll((unsigned long long)inm) - 1;
                inm &= inm - 1;
                const int f = __shfl(first, src, 64), nv = __shfl(nvert, src, 64);
                const float pax = __shfl(ax, src, 64), pay = __shfl(ay, src, 64);
                const float pbx = __shfl(bx, src, 64), pby = __shfl(by, src, 64);
                for (int k = lane; k <= nv; k += 64) acc += ring.term(f, nv, pax, pay, pbx, pby, k);
            }
        }
    }
    return acc;
}

// What the waves of a team add up over a pair, in LDS.
struct TeamSum {
    uint32_t cnt, nk;
    int32_t c[5];
    double side[2][kWaves];
};

// Ideal::intersection for one pair plus the area; R / D: the team's two record
// slabs of cap records each (cap a power of two).  Every wave of the team
// returns the same result.
template <int NW>
__device__ __forceinline__ PairRes intersection_pair(const DevSet &S, const double *ring2a, uint32_t ia, uint32_t ib,
                                                     Rec *R, Rec *D, uint32_t cap, TeamSum &T, Queues &Q,
                                                     const Team<NW> &tm, const PieceOut &po) {
    const int lane = tm.lane;
    PairRes r;
    for (int k = 0; k < 5; k++) r.c[k] = 0;
    r.area = 0.0;
    r.bb = r.tests = r.raw = 0;
    r.over = false;
    const farm_raster_hdr &hA = S.hdr[ia];
    const farm_raster_hdr &hB = S.hdr[ib];
    // 1. source pixels over the target MBB (retrieve_pixels, +-1e-6)
    const Window w = window_of(hA, hB.mbr[0], hB.mbr[1], hB.mbr[2], hB.mbr[3]);
    const int wx = w.x1 - w.x0 + 1, wy = w.y1 - w.y0 + 1;
    const uint32_t npx = (wx > 0 && wy > 0) ? (uint32_t)(wx * wy) : 0u;
    uint32_t etn = 0, itn = 0;
    for (uint32_t c0 = 0; c0 < npx; c0 += 64) {
        const uint32_t k = c0 + lane;
        uint8_t st = 1;
        if (k < npx) {
            const int x = w.x0 + (int)(k / wy), y = w.y0 + (int)(k % wy);
            st = S.status[hA.pix_start + y * hA.dimx + x];
        }
        etn += __popcll(__ballot(k < npx && st == 0));
        itn += __popcll(__ballot(k < npx && st == kCC - 1));
    }
    if (etn == npx) {
        r.c[0] = -1;
        return r;
    }
    if (itn == npx) {
        r.c[0] = -2;
        r.area = fabs(ring2a[ib]) / 2.0;
        put_pieces(po, tm.tid() == 0, farm_piece{po.pair, 1, 0, -1, 0.f, 0.f, 0.f, 0.f}, lane);  // all of B
        return r;
    }
    // 2. crossing points of the edges of BORDER x BORDER pixel pairs.  Lanes
    // take 64 source pixels, then the window of one of them, so that a pixel
    // pair needs no loads of its own before its chunks.
    const float *AX = S.x + hA.vert_start, *AY = S.y + hA.vert_start;
    const float *BX = S.x + hB.vert_start, *BY = S.y + hB.vert_start;
    if (tm.tid() == 0) {
        T.cnt = 0u;
        T.nk = 0u;
        for (int k = 0; k < 5; k++) T.c[k] = 0;
    }
    tm.sync();
    Collect C{S.ixbox, S.ixseg, AX, AY, BX, BY, &Q, 0u, 0u, 0u, R, cap, &T.cnt, lane};
    uint32_t turn = NW == 1 ? 0u : (uint32_t)tm.wv;  // the team's waves start at different rounds
    for (uint32_t k0 = 0; k0 < npx; k0 += 64) {
        const uint32_t k = k0 + lane;
        bool live = false;
        uint32_t ca0 = 0, ca1 = 0, na = 0;
        Window v{0, -1, 0, -1};
        if (k < npx) {
            const int x = w.x0 + (int)(k / wy), y = w.y0 + (int)(k % wy);
            const uint32_t pa = (uint32_t)(y * hA.dimx + x);
            live = show(S.status[hA.pix_start + pa]) == 1;
            if (live) {
                double lx, ly, hx, hy;
                pixel_box(hA, x, y, lx, ly, hx, hy);
                v = window_of(hB, lx, ly, hx, hy);
                const uint32_t s0 = S.pixoff[hA.pixoff_start + pa], s1 = S.pixoff[hA.pixoff_start + pa + 1];
                ca0 = S.ixoff[hA.seq_start + s0];
                ca1 = S.ixoff[hA.seq_start + s1];
                na = S.pixedges[hA.pix_start + pa];
            }
        }
        uint64_t lm = __ballot(live);
        while (lm) {
            const int src = __ffsll((unsigned long long)lm) - 1;
            lm &= lm - 1;
            const int vx0 = __builtin_amdgcn_readlane(v.x0, src), vx1 = __builtin_amdgcn_readlane(v.x1, src);
            const int vy0 = __builtin_amdgcn_readlane(v.y0, src), vy1 = __builtin_amdgcn_readlane(v.y1, src);
            const uint32_t a0 = __builtin_amdgcn_readlane(ca0, src), a1 = __builtin_amdgcn_readlane(ca1, src);
            const uint64_t ea = (uint32_t)__builtin_amdgcn_readlane(na, src);
            const uint32_t hgt = (uint32_t)(vy1 - vy0 + 1);
            const uint32_t nt = vx1 >= vx0 && vy1 >= vy0 ? (uint32_t)(vx1 - vx0 + 1) * hgt : 0u;
            for (uint32_t t0 = 0; t0 < nt; t0 += 64) {
                const uint32_t t = t0 + lane;
                bool tl = false;
                uint32_t cb0 = 0, cb1 = 0, nb = 0;
                if (t < nt) {
                    const uint32_t pb = (uint32_t)((vy0 + (int)(t % hgt)) * hB.dimx + vx0 + (int)(t / hgt));
                    tl = show(S.status[hB.pix_start + pb]) == 1;
                    if (tl) {
                        const uint32_t s0 = S.pixoff[hB.pixoff_start + pb], s1 = S.pixoff[hB.pixoff_start + pb + 1];
                        cb0 = S.ixoff[hB.seq_start + s0];
                        cb1 = S.ixoff[hB.seq_start + s1];
                        nb = S.pixedges[hB.pix_start + pb];
                    }
                }
                uint64_t bm = __ballot(tl);
                while (bm) {
                    const int s2 = __ffsll((unsigned long long)bm) - 1;
                    bm &= bm - 1;
                    r.bb++;
                    r.tests += ea * (uint32_t)__builtin_amdgcn_readlane(nb, s2);
                    collect_chunks<NW>(C, a0, a1, (uint32_t)__builtin_amdgcn_readlane(cb0, s2),
                                       (uint32_t)__builtin_amdgcn_readlane(cb1, s2), turn);
                    if (NW > 1) turn = turn + 1 == NW ? 0 : turn + 1;
                }
            }
        }
    }
    if (C.nc) flush_chunks(C);
    while (C.nl) flush_lines(C, min(C.nl, 64u));
    if (C.ne) flush_edges(C);
    tm.sync();
    const uint32_t nrec = uni(T.cnt);
    r.raw = nrec;
    if (nrec > cap) {
        r.over = true;
        return r;
    }
    const double ox = fmax(hA.mbr[0], hB.mbr[0]), oy = fmax(hA.mbr[1], hB.mbr[1]);
    uint32_t nk = 0;
    if (nrec > 0) {
        // 3. sort by point, keep the first of each run of equal points
        bitonic<0>(R, nrec, tm);
        bool small = false;
        if (tm.first()) {
            for (uint32_t k = lane; k < nrec; k += 64) {
                const Rec e = R[k];
                small |= fabsf(e.px) < 0.015625f || fabsf(e.py) < 0.015625f;
            }
            if (!wave_any(small)) {
                // above 2^-6 the 1e-9 tolerance is float equality: a record is
                // kept when it differs from its predecessor
                for (uint32_t c0 = 0; c0 < nrec; c0 += 64) {
                    const uint32_t k = c0 + lane;
                    bool keep = false;
                    Rec e;
                    if (k < nrec) {
                        e = R[k];
                        keep = k == 0 || !pt_eq(R[k - 1].px, R[k - 1].py, e.px, e.py);
                    }
                    const uint64_t km = __ballot(keep);
                    if (keep) D[nk + (uint32_t)__popcll(km & ((1ull << lane) - 1ull))] = e;
                    nk += (uint32_t)__popcll(km);
                }
            } else if (lane == 0) {
                // std::unique: compare with the last kept record
                for (uint32_t k = 0; k < nrec; k++) {
                    const Rec e = R[k];
                    if (nk == 0 || !pt_eq(D[nk - 1].px, D[nk - 1].py, e.px, e.py)) D[nk++] = e;
                }
            }
            if (lane == 0) T.nk = nk;
        }
        tm.sync();
        nk = uni(T.nk);
    }
    r.c[0] = (int32_t)nk;
    double acc_a = 0.0, acc_b = 0.0;
    if (nk > 0) {
        // a team's rows take the place of the raw records, which are done with:
        // both rings', and one wave adds up either; or one ring's at a time
        static_assert(kRow * sizeof(double) == 2 * sizeof(Rec), "two records to a row");
        double *rows = reinterpret_cast<double *>(R);
        const int width = 4 * (uint64_t)nk <= cap ? kRow : kRow / 2;
        const bool both = 2 * (uint64_t)nk <= cap;
        const Ring ra{AX, AY, (int)hA.nverts - 1, ox, oy}, rb{BX, BY, (int)hB.nverts - 1, ox, oy};
        bitonic<1>(D, nk, tm);
        acc_a = ring_pieces<true>(S, hA, hB, D, nk, rows, width, ox, oy, tm, r, po, Q);
        tm.sync();
        if (NW > 1 && !both) {
            if (tm.wv == 0) acc_a = sum_rows(ra, rows, nk, width, lane, Q);
            tm.sync();
        }
        bitonic<2>(D, nk, tm);
        double *rows_b = both ? rows + (uint64_t)width * nk : rows;
        acc_b = ring_pieces<false>(S, hB, hA, D, nk, rows_b, width, ox, oy, tm, r, po, Q);
        if constexpr (NW > 1) {
            tm.sync();
            if (both && tm.wv == 0) acc_a = sum_rows(ra, rows, nk, width, lane, Q);
            if (tm.wv == 1) acc_b = sum_rows(rb, rows_b, nk, width, lane, Q);
        }
    }
    double side_a = wave_sum(acc_a), side_b = wave_sum(acc_b);
    if constexpr (NW > 1) {
        if (lane == 0) {
            for (int k = 1; k < 5; k++)
                if (r.c[k]) atomicAdd(&T.c[k], r.c[k]);
            T.side[0][tm.wv] = side_a;
            T.side[1][tm.wv] = side_b;
        }
        tm.sync();
        for (int k = 1; k < 5; k++) r.c[k] = T.c[k];
        side_a = side_b = 0.0;
        for (int k = 0; k < NW; k++) {
            side_a += T.side[0][k];
            side_b += T.side[1][k];
        }
    }
    if (r.c[1] == 0) {
        // containment or disjoint: the first vertex of A in B, of B in A
        const int in_b = uni(__shfl(contain_points(S, hB, AX[0], AY[0], lane == 0, lane, Q), 0, 64));
        const int in_a = in_b == 2 ? 0 : uni(__shfl(contain_points(S, hA, BX[0], BY[0], lane == 0, lane, Q), 0, 64));
        const bool mine = tm.tid() == 0;
        if (in_b == 2) {
            r.area = fabs(ring2a[ia]) / 2.0;
            put_pieces(po, mine, farm_piece{po.pair, 0, 0, -1, 0.f, 0.f, 0.f, 0.f}, lane);  // all of A
        } else if (in_a == 2) {
            r.area = fabs(ring2a[ib]) / 2.0;
            put_pieces(po, mine, farm_piece{po.pair, 1, 0, -1, 0.f, 0.f, 0.f, 0.f}, lane);  // all of B
        }
        return r;
    }
    const double sa = ring2a[ia] < 0 ? -1.0 : 1.0, sb = ring2a[ib] < 0 ? -1.0 : 1.0;
    r.area = fabs(sa * side_a + sb * side_b) / 2.0;
    return r;
}

}  // namespace

// Twice the signed area of every ring, relative to its MBB's low corner
// (one wave per polygon).
__global__ __launch_bounds__(256) void k_ring_area(DevSet S, int64_t npolys, double *__restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int64_t p = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (p >= npolys) return;
    const farm_raster_hdr &h = S.hdr[p];
    const float *X = S.x + h.vert_start, *Y = S.y + h.vert_start;
    const double ox = h.mbr[0], oy = h.mbr[1];
    double acc = 0.0;
    for (uint32_t k = lane; k + 1 < h.nverts; k += 64)
        acc += ((double)X[k] - ox) * ((double)Y[k + 1] - oy) - ((double)X[k + 1] - ox) * ((double)Y[k] - oy);
    acc = wave_sum(acc);
    if (lane == 0) out[p] = acc;
}

// Pairs for a whole workgroup: their indices to list (count at ctr[kIxHeavy]),
// and flags[k] = 1.  A pair's collection runs over up to (chunks of A in the
// overlap of the boxes) x (chunks of B in it) chunk pairs, estimated from the
// overlap's share of each box.  Beyond kHeavyChunks one wave is at it too long,
// or its crossing records outgrow the wave's slab and the pair is done again.
// Measured, ms at 256 / 1,024 / 4,096 / 16,384 chunk pairs: complex x lakes
// (479,000 pairs) -v 256 47.1 45.3 47.3 48.1, -v 64 51.2 47.1 45.4 45.7; jagged
// rings -v 10 (237,000 pairs) 70.0 67.6 67.3 174; -v 33 (63,000) 14.0 14.5 18.3
// 18.2.  (Chunks as they are: a jagged ring at 10 vertices per pixel has a third
// of its vertices, not a sixteenth.)
// all: every pair, in a call of fewer than kTeamPairs pairs to a workgroup, which
// would not fill the chip evenly with one wave per pair.  Measured, ms with all
// by workgroups and without, 1,024 workgroups: jagged rings -v 100 8,000 pairs
// 2.93 / 5.02, 16,000 4.95 / 7.45, 32,000 9.09 / 9.22, 48,000 13.2 / 12.3;
// complex x lakes -v 256 2,000 pairs 1.76 / 4.22, 8,000 6.58 / 6.39, 16,000 7.09 /
// 6.58, 32,000 18.5 / 17.6.
enum : int { kIxHead = 0, kIxOver = 1, kIxPieces = 2, kIxHeavy = 3, kIxHeavyHead = 4 };
constexpr float kHeavyChunks = 1024.f;
constexpr uint32_t kTeamPairs = 16;

__global__ __launch_bounds__(256) void k_ix_heavy(DevSet S, const uint32_t *__restrict__ pa,
                                                  const uint32_t *__restrict__ pb, uint32_t n, int all,
                                                  uint8_t *__restrict__ flags, uint32_t *__restrict__ list,
                                                  uint32_t *__restrict__ ctr) {
    const int lane = threadIdx.x & 63;
    for (uint64_t k0 = (uint64_t)blockIdx.x * blockDim.x; k0 < n; k0 += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t k = k0 + threadIdx.x;
        bool heavy = false;
        if (k < n) {
            const farm_raster_hdr &A = S.hdr[pa[k]], &B = S.hdr[pb[k]];
            auto part = [&](int lo, int hi, float &fa, float &fb) {
                const float w = (float)(fmin(A.mbr[hi], B.mbr[hi]) - fmax(A.mbr[lo], B.mbr[lo]));
                fa *= fminf(fmaxf(w, 0.f) / fmaxf((float)(A.mbr[hi] - A.mbr[lo]), 1e-30f), 1.f);
                fb *= fminf(fmaxf(w, 0.f) / fmaxf((float)(B.mbr[hi] - B.mbr[lo]), 1e-30f), 1.f);
            };
            float fa = 1.f, fb = 1.f;
            part(0, 2, fa, fb);
            part(1, 3, fa, fb);
            const float ca = (float)(S.ixoff[A.seq_start + A.nseqs] - S.ixoff[A.seq_start]);
            const float cb = (float)(S.ixoff[B.seq_start + B.nseqs] - S.ixoff[B.seq_start]);
            heavy = all || (ca * fa) * (cb * fb) > kHeavyChunks;
            flags[k] = heavy ? 1 : 0;
        }
        const uint64_t m = __ballot(heavy);
        uint32_t base = 0;
        if (lane == 0 && m) base = atomicAdd(&ctr[kIxHeavy], (uint32_t)__popcll(m));
        base = uni(__shfl(base, 0, 64));
        if (heavy) list[base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint32_t)k;
    }
}

// Persistent workgroups: first the pairs of list[0 .. *nlist), all four waves
// on one pair (records in slabs of kWaves * cap), then, wave by wave, the other
// pairs of the window (flags; slabs of cap).  BIG: pairs that overflowed the
// first launch's slabs, all on the list (n = 0).
// Four waves per SIMD (128 registers, 20 of them spilled): 56.0 ms for 618,000
// complex x lakes pairs against 63.6 ms at three, 4,000 jagged pairs 2.55 and 2.67.
template <bool BIG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_intersection(DevSet S, const double *__restrict__ ring2a,
                                                      const uint32_t *__restrict__ pa, const uint32_t *__restrict__ pb,
                                                      uint32_t n, const uint8_t *__restrict__ flags,
                                                      const uint32_t *__restrict__ list,
                                                      const uint32_t *__restrict__ nlist,
                                                      int32_t *__restrict__ counts, double *__restrict__ area,
                                                      Rec *__restrict__ slab, uint32_t cap,
                                                      uint32_t *__restrict__ ctr, uint32_t *__restrict__ ovf,
                                                      unsigned long long *__restrict__ stats,
                                                      farm_piece *__restrict__ pcs, uint32_t pcap) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    Rec *block_slab = slab + (uint64_t)blockIdx.x * kWaves * 2ull * cap;
    __shared__ TeamSum sums[kWaves];
    __shared__ Queues queues[kWaves];
    __shared__ uint32_t s_next;
    unsigned long long bb = 0, tests = 0, raw = 0, found = 0;
    // one pair by a team; `writer` stores its results
    auto run = [&](auto tm, uint32_t idx, Rec *R, Rec *D, uint32_t rcap, TeamSum &T, bool writer) {
        const uint32_t ia = pa[idx], ib = pb[idx];
        if ((S.hdr[ia].flags | S.hdr[ib].flags) & FARM_HDR_REJECTED) {
            if (writer && lane < 5) counts[5ull * idx + lane] = lane == 0 ? -3 : 0;
            if (writer && lane == 0) area[idx] = 0.0;
            return;
        }
        const PieceOut po{pcs, ctr + kIxPieces, pcap, idx};
        const PairRes r = intersection_pair(S, ring2a, ia, ib, R, D, rcap, T, queues[wv], tm, po);
        if (!writer) return;
        if (r.over) {
            if (lane == 0) {
                if (BIG) {  // still too many: the host reruns it with larger slabs
                    counts[5ull * idx] = -4;
                    counts[5ull * idx + 1] = (int32_t)min(r.raw, (uint64_t)INT_MAX);
                } else {
                    ovf[atomicAdd(&ctr[kIxOver], 1u)] = idx;
                }
            }
            return;
        }
        bb += r.bb;
        tests += r.tests;
        raw += r.raw;
        found += r.area > 0.0;
        if (lane < 5) counts[5ull * idx + lane] = r.c[lane];
        if (lane == 0) area[idx] = r.area;
    };
    const uint32_t nl = *nlist;
    for (;;) {
        __syncthreads();  // the team's last pair is done with the shared state
        if (threadIdx.x == 0) s_next = atomicAdd(&ctr[kIxHeavyHead], 1u);
        __syncthreads();
        const uint32_t k = uni(s_next);
        if (k >= nl) break;
        run(Team<kWaves>{lane, wv}, list[k], block_slab, block_slab + (uint64_t)kWaves * cap, kWaves * cap, sums[0],
            wv == 0);
    }
    if constexpr (!BIG) {
        Rec *R = block_slab + wv * 2ull * cap;
        const uint32_t grab = min(max(n / (gridDim.x * kWaves * 16u), 1u), 8u);
        for (;;) {
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(&ctr[kIxHead], grab);
            base = uni(__shfl(base, 0, 64));
            if (base >= n) break;
            const uint32_t end = min(base + grab, n);
            for (uint32_t k = base; k < end; k++)
                if (!flags[k]) run(Team<1>{lane, wv}, k, R, R + cap, cap, sums[wv], true);
        }
    }
    if (lane == 0 && (bb || tests || raw || found)) {
        atomicAdd(&stats[0], bb);
        atomicAdd(&stats[1], tests);
        atomicAdd(&stats[2], raw);
        atomicAdd(&stats[3], found);
    }
}

template __global__ void k_intersection<false>(DevSet, const double *, const uint32_t *, const uint32_t *, uint32_t,
                                               const uint8_t *, const uint32_t *, const uint32_t *, int32_t *,
                                               double *, Rec *, uint32_t, uint32_t *, uint32_t *,
                                               unsigned long long *, farm_piece *, uint32_t);
template __global__ void k_intersection<true>(DevSet, const double *, const uint32_t *, const uint32_t *, uint32_t,
                                              const uint8_t *, const uint32_t *, const uint32_t *, int32_t *,
                                              double *, Rec *, uint32_t, uint32_t *, uint32_t *,
                                              unsigned long long *, farm_piece *, uint32_t);

}  // namespace farm

using namespace farm;

namespace farm {
int build_ix_boxes(farm_handle h);
}  // namespace farm

namespace {

int run_intersection(farm_handle h, uint64_t begin, uint64_t end, int32_t *counts_dev, double *area_dev,
                     farm_stats *st, farm_piece *pcs_dev = nullptr, uint32_t pcap = 0, uint64_t *npcs = nullptr) {
    if (!h) return FARM_EINVAL;
    if (h->npolys <= 0) return fail(h, FARM_ESTATE, "no polygons uploaded");
    if (h->has_layers) return fail(h, FARM_ESTATE, "intersection needs a set rasterized without -h");
    if (begin > end || end > h->npairs)
        return fail(h, FARM_EINVAL, "pair window [%llu,%llu) outside [0,%llu)", (unsigned long long)begin,
                    (unsigned long long)end, (unsigned long long)h->npairs);
    const uint64_t n64 = end - begin;
    if (n64 > 0xffffffffull) return fail(h, FARM_ECAPACITY, "batch larger than 2^32 pairs");
    const uint32_t n = (uint32_t)n64;
    HIPCHK(h, hipSetDevice(h->device));
    if (st) memset(st, 0, sizeof *st);
    if (st) st->pairs = n;
    if (n == 0) return FARM_OK;
    int rc;
    if ((rc = build_ix_boxes(h))) return rc;
    DevSet S = devset(h);
    if (!h->ring_area_ready) {
        if ((rc = ensure(h, h->ring2a, 8ull * h->npolys))) return rc;
        hipLaunchKernelGGL(k_ring_area, dim3((unsigned)((h->npolys + 3) / 4)), dim3(256), 0, h->stream, S, h->npolys,
                           P<double>(h->ring2a));
        HIPCHK(h, hipGetLastError());
        h->ring_area_ready = true;
    }
    const uint32_t *pa = P<uint32_t>(h->pa) + begin;
    const uint32_t *pb = P<uint32_t>(h->pb) + begin;
    if ((rc = ensure(h, h->wctr, 64))) return rc;
    if ((rc = ensure(h, h->wovf, 4ull * n))) return rc;
    if ((rc = ensure(h, h->ixlist, 4ull * n))) return rc;
    if ((rc = ensure(h, h->ixflag, n))) return rc;
    uint32_t *ctr = P<uint32_t>(h->wctr);
    unsigned long long *ist = reinterpret_cast<unsigned long long *>(ctr + 8);
    if ((rc = fill_u32(h, ctr, 16, 0))) return rc;
    const unsigned nblocks = (unsigned)h->num_cus * 4;
    const uint64_t nwaves = (uint64_t)nblocks * kWaves;
    if ((rc = ensure(h, h->wslab, nwaves * 2ull * kRecCap * sizeof(Rec)))) return rc;
    HIPCHK(h, hipEventRecord(h->ev[0], h->stream));
    hipLaunchKernelGGL(k_ix_heavy, dim3((unsigned)std::min<uint64_t>(blocks_for(n), kMaxLaunchGroups)), dim3(256), 0, h->stream, S, pa, pb, n,
                       n < kTeamPairs * nblocks ? 1 : 0,
                       P<uint8_t>(h->ixflag), P<uint32_t>(h->ixlist), ctr);
    HIPCHK(h, hipGetLastError());
    hipLaunchKernelGGL(k_intersection<false>, dim3(nblocks), dim3(64 * kWaves), 0, h->stream, S,
                       (const double *)P<double>(h->ring2a), pa, pb, n, (const uint8_t *)P<uint8_t>(h->ixflag),
                       (const uint32_t *)P<uint32_t>(h->ixlist), (const uint32_t *)(ctr + kIxHeavy), counts_dev,
                       area_dev, P<Rec>(h->wslab), kRecCap, ctr, P<uint32_t>(h->wovf), ist, pcs_dev, pcap);
    HIPCHK(h, hipGetLastError());
    uint32_t novf = 0;
    HIPCHK(h, hipMemcpyAsync(&novf, ctr + kIxOver, 4, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));
    if (novf) {
        // pairs with more raw crossing records than the first slabs hold
        const unsigned bblocks = 16;
        if ((rc = ensure(h, h->wslab_big, (uint64_t)bblocks * kWaves * 2ull * kRecCapBig * sizeof(Rec)))) return rc;
        if ((rc = fill_u32(h, ctr + kIxHeavyHead, 1, 0))) return rc;
        hipLaunchKernelGGL(k_intersection<true>, dim3(bblocks), dim3(64 * kWaves), 0, h->stream, S,
                           (const double *)P<double>(h->ring2a), pa, pb, 0u, (const uint8_t *)nullptr,
                           (const uint32_t *)P<uint32_t>(h->wovf), (const uint32_t *)(ctr + kIxOver), counts_dev,
                           area_dev, P<Rec>(h->wslab_big), kRecCapBig, ctr, P<uint32_t>(h->wovf), ist, pcs_dev, pcap);
        HIPCHK(h, hipGetLastError());
    }
    HIPCHK(h, hipEventRecord(h->ev[1], h->stream));
    unsigned long long hst[4] = {0, 0, 0, 0};
    HIPCHK(h, hipMemcpyAsync(hst, ist, sizeof hst, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));
    if (novf) {
        // pairs beyond the second slabs: once more, with slabs sized to the
        // largest of them (fewer waves, at most 8 GiB of slabs)
        std::vector<uint32_t> list(novf), big;
        HIPCHK(h, hipMemcpy(list.data(), P<uint32_t>(h->wovf), 4ull * novf, hipMemcpyDeviceToHost));
        uint32_t most = 0;
        for (uint32_t idx : list) {
            int32_t c[2];
            HIPCHK(h, hipMemcpy(c, counts_dev + 5ull * idx, 8, hipMemcpyDeviceToHost));
            if (c[0] == -4) {
                big.push_back(idx);
                most = std::max(most, (uint32_t)c[1]);
            }
        }
        if (!big.empty()) {
            if (most > (1u << 26))
                return fail(h, FARM_ECAPACITY, "a pair has %u crossing records (limit 2^26)", most);
            uint64_t cap = 2ull * kRecCapBig;  // a workgroup's slabs hold kWaves * cap records each
            while (kWaves * cap < most) cap <<= 1;
            const uint64_t per_wave = 2ull * cap * sizeof(Rec);
            const uint64_t waves = std::max<uint64_t>(kWaves, std::min<uint64_t>(64, (8ull << 30) / per_wave));
            const unsigned blocks = (unsigned)(waves / kWaves);
            if ((rc = ensure(h, h->wslab_big, (uint64_t)blocks * kWaves * per_wave))) return rc;
            HIPCHK(h, hipMemcpyAsync(P<uint32_t>(h->wovf), big.data(), 4ull * big.size(), hipMemcpyHostToDevice,
                                     h->stream));
            const uint32_t nbig = (uint32_t)big.size();
            HIPCHK(h, hipMemcpyAsync(ctr + kIxOver, &nbig, 4, hipMemcpyHostToDevice, h->stream));
            if ((rc = fill_u32(h, ctr + kIxHeavyHead, 1, 0))) return rc;
            hipLaunchKernelGGL(k_intersection<true>, dim3(blocks), dim3(64 * kWaves), 0, h->stream, S,
                               (const double *)P<double>(h->ring2a), pa, pb, 0u, (const uint8_t *)nullptr,
                               (const uint32_t *)P<uint32_t>(h->wovf), (const uint32_t *)(ctr + kIxOver), counts_dev,
                               area_dev, P<Rec>(h->wslab_big), (uint32_t)cap, ctr, P<uint32_t>(h->wovf), ist, pcs_dev, pcap);
            HIPCHK(h, hipGetLastError());
            HIPCHK(h, hipEventRecord(h->ev[1], h->stream));
            HIPCHK(h, hipMemcpyAsync(hst, ist, sizeof hst, hipMemcpyDeviceToHost, h->stream));
            HIPCHK(h, hipStreamSynchronize(h->stream));
            for (uint32_t idx : big) {
                int32_t c0 = 0;
                HIPCHK(h, hipMemcpy(&c0, counts_dev + 5ull * idx, 4, hipMemcpyDeviceToHost));
                if (c0 == -4)
                    return fail(h, FARM_ECAPACITY, "pair %llu: more than %llu crossing records",
                                (unsigned long long)(begin + idx), (unsigned long long)(kWaves * cap));
            }
        }
    }
    if (npcs) {
        uint32_t np = 0;
        HIPCHK(h, hipMemcpy(&np, ctr + kIxPieces, 4, hipMemcpyDeviceToHost));
        *npcs = np;
    }
    if (st) {
        float ms = 0;
        HIPCHK(h, hipEventElapsedTime(&ms, h->ev[0], h->ev[1]));
        st->bb_pixel_pairs = hst[0];
        st->segment_tests = hst[1];
        st->refine_items = hst[2];
        st->found = hst[3];
        st->refine_ms = ms;
        st->total_ms = ms;
    }
    return FARM_OK;
}

}  // namespace

extern "C" {

int farm_intersection_area_dev(farm_handle h, uint64_t begin, uint64_t end, int32_t *counts_dev, double *area_dev,
                               farm_stats *st) {
    if (!counts_dev || !area_dev) return fail(h, FARM_EINVAL, "null output buffer");
    return run_intersection(h, begin, end, counts_dev, area_dev, st);
}

int farm_intersection_pieces(farm_handle h, uint64_t begin, uint64_t end, int32_t *counts, double *area,
                             farm_piece *pieces, uint64_t cap, uint64_t *npieces, farm_stats *st) {
    if (!h) return FARM_EINVAL;
    if (begin > end || !npieces || (cap && !pieces)) return fail(h, FARM_EINVAL, "bad arguments");
    if (cap > 0xffffffffull) cap = 0xffffffffull;
    const uint64_t n = end - begin;
    int rc;
    if ((rc = ensure(h, h->icounts, 20 * n + 16))) return rc;
    if ((rc = ensure(h, h->iarea, 8 * n + 16))) return rc;
    if ((rc = ensure(h, h->ipieces, sizeof(farm_piece) * (cap ? cap : 1)))) return rc;
    if ((rc = run_intersection(h, begin, end, P<int32_t>(h->icounts), P<double>(h->iarea), st,
                               P<farm_piece>(h->ipieces), (uint32_t)cap, npieces)))
        return rc;
    if (n && counts) HIPCHK(h, hipMemcpy(counts, h->icounts.p, 20 * n, hipMemcpyDeviceToHost));
    if (n && area) HIPCHK(h, hipMemcpy(area, h->iarea.p, 8 * n, hipMemcpyDeviceToHost));
    if (*npieces > cap)
        return fail(h, FARM_ECAPACITY, "%llu pieces, room for %llu", (unsigned long long)*npieces,
                    (unsigned long long)cap);
    if (*npieces) HIPCHK(h, hipMemcpy(pieces, h->ipieces.p, sizeof(farm_piece) * *npieces, hipMemcpyDeviceToHost));
    return FARM_OK;
}

int farm_intersection_area(farm_handle h, uint64_t begin, uint64_t end, int32_t *counts, double *area,
                           farm_stats *st) {
    if (!h) return FARM_EINVAL;
    if (begin > end) return fail(h, FARM_EINVAL, "bad pair window");
    const uint64_t n = end - begin;
    int rc;
    if ((rc = ensure(h, h->icounts, 20 * n + 16))) return rc;
    if ((rc = ensure(h, h->iarea, 8 * n + 16))) return rc;
    if ((rc = run_intersection(h, begin, end, P<int32_t>(h->icounts), P<double>(h->iarea), st))) return rc;
    if (n && counts) HIPCHK(h, hipMemcpy(counts, h->icounts.p, 20 * n, hipMemcpyDeviceToHost));
    if (n && area) HIPCHK(h, hipMemcpy(area, h->iarea.p, 8 * n, hipMemcpyDeviceToHost));
    return FARM_OK;
}

}  // extern "C"

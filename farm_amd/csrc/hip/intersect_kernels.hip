// Exact and approximate intersect kernels for gfx950 (wave64).
//
// Semantics: Ideal::intersect of the reference CPU path (Ideal.cpp:1329-1422):
//   TRUE iff some non-OUT source pixel pa in the source window of the target
//   MBB and some non-OUT target pixel pb in the target window of pa's box have
//   an IN pixel on either side, or some BORDER x BORDER pair (pa, pb) has an
//   edge of one of pa's edge sequences crossing an edge of one of pb's
//   (segment_intersect, geometry_computation.h:215-237, binary32).
// The answer is an OR, so any evaluation order (and any early exit) returns
// the reference's bit.
#include <type_traits>

#include "device_layout.h"
#include "isect_work.h"
#include "wave.h"

namespace farm {

// ------------------------------------------------------------------------
// Raster filter: one lane per candidate pair (grid-stride over the window).
// pass 0: count BORDER x BORDER pixel pairs, decide IN hits (and the
//         reference -a heuristic when approx != 0); the 64-bit total of the
//         pixel pairs goes to the shards of kCtrPixPairs (the scan's second
//         kernel folds them into ctr)
// pass 1: emit the pixel pairs at the offsets of an exclusive scan; it does
//         nothing when that total exceeds cap_pp (the buffer's capacity: the
//         host grows it or fails the call, and no offset has wrapped).
// A lane stops walking its pair's windows at the first IN overlap (or, in
// approximate mode, the first decisive BORDER pair): the pair is decided and
// its count is not used.  An undecided pair's windows are walked in full.
// skip (optional): pairs already decided by the caller (their result is left
// untouched and they emit no pixel pairs).
// ------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_filter(DevSet S, const uint32_t *__restrict__ pa_all,
                                                 const uint32_t *__restrict__ pb_all,
                                                 const IsxDesc *__restrict__ desc, int pass, int approx,
                                                 const uint8_t *__restrict__ skip, uint32_t *__restrict__ npp,
                                                 const uint32_t *__restrict__ pp_off, PixPair *__restrict__ pps,
                                                 uint64_t cap_pp, uint32_t *__restrict__ result,
                                                 const unsigned long long *__restrict__ ctr,
                                                 unsigned long long *__restrict__ shards) {
    if (pass == 1 && ctr[kCtrPixPairs] > cap_pp) return;
    const uint64_t n = desc->n;
    const uint32_t *pa_ids = pa_all + desc->begin;
    const uint32_t *pb_ids = pb_all + desc->begin;
    uint32_t *tests = desc->pair_tests;
    unsigned long long bytes = 0, inhit = 0, bb = 0;
    for (uint64_t kk = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; kk < n;
         kk += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t k = (uint32_t)kk;
        if (pass == 0 && tests) tests[k] = 0;
        if (skip && skip[k]) {
            if (pass == 0) npp[k] = 0;
            continue;
        }
        if (pass == 1 && npp[k] == 0) continue;  // decided by the count pass or no BORDER pair
        const uint32_t ia = pa_ids[k], ib = pb_ids[k];
        const farm_raster_hdr A = S.hdr[ia];
        const farm_raster_hdr B = S.hdr[ib];
        const uint8_t *sa = S.status + A.pix_start;
        const uint8_t *sb = S.status + B.pix_start;
        const uint32_t *ea = S.pixedges + A.pix_start;
        const uint32_t *pofa = S.pixoff + A.pixoff_start;
        // the reference's -a (its GPU filter) takes the source window over
        // the target MBB without the 1e-6 shrink (query_intersect.cu:51-54);
        // Ideal::intersect shrinks it (MyRaster.cpp:332-337)
        const Window wa = approx ? window_of(A, B.mbr[0], B.mbr[1], B.mbr[2], B.mbr[3], 0.0)
                                 : window_of(A, B.mbr[0], B.mbr[1], B.mbr[2], B.mbr[3]);
        const double area_a = A.step[0] * A.step[1], area_b = B.step[0] * B.step[1];
        const double amax = fmax(area_a, area_b);
        bool in_hit = false, heur = false;
        uint32_t cnt = 0;
        const uint32_t base = pass == 1 ? pp_off[k] : 0u;
        bytes += 8 + 2 * 56;
        for (int x = wa.x0; x <= wa.x1 && !(in_hit || heur); x++) {
            for (int y = wa.y0; y <= wa.y1 && !(in_hit || heur); y++) {
                const int pa = y * A.dimx + x;
                const uint8_t fa = sa[pa];
                bytes += 1;
                const int st_a = show(fa);
                if (st_a == 0) continue;
                double lx, ly, hx, hy;
                pixel_box(A, x, y, lx, ly, hx, hy);
                const Window wb = window_of(B, lx, ly, hx, hy);
                for (int u = wb.x0; u <= wb.x1 && !(in_hit || heur); u++) {
                    for (int v = wb.y0; v <= wb.y1 && !(in_hit || heur); v++) {
                        const int pb = v * B.dimx + u;
                        const uint8_t fb = sb[pb];
                        bytes += 1;
                        const int st_b = show(fb);
                        if (st_b == 0) continue;
                        if (st_a == 2 || st_b == 2) {
                            in_hit = true;
                            continue;
                        }
                        if (approx) {
                            // fill classes at the set's category count (-w)
                            const double prob = (apx_area_cc(S.fill[A.pix_start + pa], area_a, S.cc) +
                                                 apx_area_cc(S.fill[B.pix_start + pb], area_b, S.cc)) /
                                                amax;
                            if (prob > 1.0) heur = true;
                            continue;
                        }
                        if (pass == 1) {
                            // edge slots of pa: sum of (len + 1) over its sequences
                            const uint32_t nseq = pofa[pa + 1] - pofa[pa];
                            pps[base + cnt] = PixPair{k, (uint32_t)pa, (uint32_t)pb, ea[pa] + nseq};
                        }
                        cnt++;
                    }
                }
            }
        }
        if (pass == 0) {
            const bool decided = in_hit || heur;
            npp[k] = decided ? 0u : cnt;
            result[k] = decided ? 1u : 0u;
            inhit += in_hit ? 1 : 0;
            bb += decided ? 0u : cnt;
        }
    }
    if (pass == 0) {
        // wave-level reduction of the counters, one atomic per wave
        for (int o = 32; o > 0; o >>= 1) {
            bytes += __shfl_xor(bytes, o);
            inhit += __shfl_xor(inhit, o);
            bb += __shfl_xor(bb, o);
        }
        if ((threadIdx.x & 63) == 0) {
            unsigned long long *sh = ctr_shard(shards, blockIdx.x * 4u + (threadIdx.x >> 6));
            if (bytes) atomicAdd(&sh[kCtrFilterBytes], bytes);
            if (inhit) atomicAdd(&sh[kCtrInHits], inhit);
            if (bb) atomicAdd(&sh[kCtrPixPairs], bb);
        }
    }
}

// ------------------------------------------------------------------------
// Exclusive scan of n u32 values, n = bounded_count(nsrc, cap): out[0..n)
// gets the prefix sums and out[n] the (32-bit) total.  Three kernels:
// kScanParts blocks sum one contiguous segment each, one block scans the
// segment sums, and every block rescans its segment from its offset.
// ------------------------------------------------------------------------
__device__ __forceinline__ void scan_segment(uint64_t n, uint32_t b, uint64_t &s0, uint64_t &s1) {
    const uint64_t seg = (n + kScanParts - 1) / kScanParts;
    s0 = min(n, (uint64_t)b * seg);
    s1 = min(n, s0 + seg);
}

// block-wide sum (256 lanes) delivered to every lane
__device__ __forceinline__ uint32_t block_sum256(uint32_t v, uint32_t *lds4) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) lds4[threadIdx.x >> 6] = v;
    __syncthreads();
    return lds4[0] + lds4[1] + lds4[2] + lds4[3];
}

__global__ __launch_bounds__(256) void k_scan_sums(const uint32_t *__restrict__ in,
                                                    const unsigned long long *__restrict__ nsrc, uint64_t cap,
                                                    uint32_t *__restrict__ part) {
    __shared__ uint32_t lds[4];
    uint64_t s0, s1;
    scan_segment(bounded_count(nsrc, cap), blockIdx.x, s0, s1);
    uint32_t s = 0;
    for (uint64_t i = s0 + threadIdx.x; i < s1; i += 256) s += in[i];
    s = block_sum256(s, lds);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// one block of kScanParts lanes; it also folds the shards of counter `slot`,
// whose total the kernels after the scan read
__global__ __launch_bounds__(kScanParts) void k_scan_parts(uint32_t *__restrict__ part,
                                                            const unsigned long long *__restrict__ nsrc,
                                                            uint64_t cap, uint32_t *__restrict__ out,
                                                            unsigned long long *__restrict__ ctr,
                                                            unsigned long long *__restrict__ shards, int slot) {
    if (threadIdx.x < 64) {
        const unsigned long long v = fold_shards(shards, slot, threadIdx.x, true);
        if (threadIdx.x == 0) ctr[slot] = v;
    }
    __shared__ uint32_t wsum[kScanParts / 64];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const uint32_t v = part[t];
    uint32_t tot;
    const uint32_t ex = wave_excl_scan(v, lane, &tot);
    if (lane == 0) wsum[w] = tot;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int i = 0; i < kScanParts / 64; i++) {
        before += i < w ? wsum[i] : 0u;
        all += wsum[i];
    }
    part[t] = before + ex;
    if (t == 0) {
        part[kScanParts] = all;
        out[bounded_count(nsrc, cap)] = all;
    }
}

__global__ __launch_bounds__(256) void k_scan_apply(const uint32_t *__restrict__ in,
                                                     const unsigned long long *__restrict__ nsrc, uint64_t cap,
                                                     const uint32_t *__restrict__ part, uint32_t *__restrict__ out) {
    __shared__ uint32_t wsum[4];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    uint64_t s0, s1;
    scan_segment(bounded_count(nsrc, cap), blockIdx.x, s0, s1);
    uint32_t carry = part[blockIdx.x];
    for (uint64_t base = s0; base < s1; base += 1024) {
        // four consecutive values per lane
        uint32_t v[4], sum = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint64_t i = base + 4 * (uint64_t)t + j;
            v[j] = i < s1 ? in[i] : 0u;
            sum += v[j];
        }
        uint32_t wtot;
        const uint32_t ex = wave_excl_scan(sum, lane, &wtot);
        __syncthreads();
        if (lane == 0) wsum[w] = wtot;
        __syncthreads();
        uint32_t before = 0;
        for (int i = 0; i < w; i++) before += wsum[i];
        uint32_t run = carry + before + ex;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint64_t i = base + 4 * (uint64_t)t + j;
            if (i < s1) out[i] = run;
            run += v[j];
        }
        carry += wsum[0] + wsum[1] + wsum[2] + wsum[3];
    }
}

// the call's window, and its counters cleared
__global__ __launch_bounds__(256) void k_set_desc(IsxDesc *d, unsigned long long begin, unsigned long long n,
                                                  uint8_t *out, uint32_t *pair_tests, uint32_t *__restrict__ clear) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kIsxClear) clear[i] = 0;
    if (i == 0) {
        d->begin = begin;
        d->n = n;
        d->out = out;
        d->pair_tests = pair_tests;
    }
}

// ------------------------------------------------------------------------
// Cost order: counting sort of the pixel pairs by floor(log2(cost)),
// heaviest bucket first.  cost = edge slots of pa x edges of pb.
// ------------------------------------------------------------------------
constexpr int kBuckets = 40;

__device__ __forceinline__ int cost_bucket(uint64_t cost) {
    int b = cost ? 63 - __builtin_clzll(cost) : 0;
    return min(b, kBuckets - 1);
}

__global__ __launch_bounds__(256) void k_bucket_hist(DevSet S, const uint32_t *__restrict__ pb_all,
                                                      const IsxDesc *__restrict__ desc,
                                                      const PixPair *__restrict__ pps,
                                                      const unsigned long long *__restrict__ ctr, uint64_t cap_pp,
                                                      const float *__restrict__ pred_cost,
                                                      uint8_t *__restrict__ bucket, uint32_t *__restrict__ hist) {
    __shared__ uint32_t h[kBuckets];
    for (int i = threadIdx.x; i < kBuckets; i += blockDim.x) h[i] = 0;
    __syncthreads();
    const uint64_t n = bounded_count(&ctr[kCtrPixPairs], cap_pp);
    const uint32_t *pb_ids = pb_all + desc->begin;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const PixPair p = pps[i];
        int b;
        if (pred_cost) {
            // learned order: the MLP cost head predicts log2(1 + tests) of
            // the pair; predictions are (logit, cost) pairs, hence stride 2
            const float c = fmaxf(pred_cost[2 * (size_t)p.pair], 0.f);
            b = min((int)c, kBuckets - 1);
        } else {
            const farm_raster_hdr B = S.hdr[pb_ids[p.pair]];
            const uint64_t eb = S.pixedges[B.pix_start + p.pb];
            b = cost_bucket((uint64_t)p.slots * eb);
        }
        bucket[i] = (uint8_t)b;
        atomicAdd(&h[b], 1u);
    }
    __syncthreads();
    for (int j = threadIdx.x; j < kBuckets; j += blockDim.x)
        if (h[j]) atomicAdd(&hist[j], h[j]);
}

// one block: descending-bucket exclusive scan of the histogram
__global__ void k_bucket_scan(uint32_t *__restrict__ hist, uint32_t *__restrict__ cursor) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        uint32_t acc = 0;
        for (int b = kBuckets - 1; b >= 0; b--) {
            cursor[b] = acc;
            acc += hist[b];
        }
    }
}

// positions are reserved per block round and bucket (one global atomic per
// non-empty bucket per round), then handed out from LDS
__global__ __launch_bounds__(256) void k_bucket_scatter(const uint8_t *__restrict__ bucket,
                                                         const unsigned long long *__restrict__ ctr, uint64_t cap_pp,
                                                         uint32_t *__restrict__ cursor, uint32_t *__restrict__ order) {
    constexpr int kPer = 8;  // items per lane and round: a global atomic per bucket serves 2,048 items
    __shared__ uint32_t cnt[kBuckets], base[kBuckets];
    const uint64_t n = bounded_count(&ctr[kCtrPixPairs], cap_pp);
    for (uint64_t b0 = (uint64_t)blockIdx.x * 256 * kPer; b0 < n; b0 += (uint64_t)gridDim.x * 256 * kPer) {
        for (int j = threadIdx.x; j < kBuckets; j += blockDim.x) cnt[j] = 0;
        __syncthreads();
        int b[kPer];
        uint32_t local[kPer];
#pragma unroll
        for (int q = 0; q < kPer; q++) {
            const uint64_t i = b0 + (uint64_t)q * 256 + threadIdx.x;
            b[q] = i < n ? bucket[i] : 0;
        }
#pragma unroll
        for (int q = 0; q < kPer; q++)
            if (b0 + (uint64_t)q * 256 + threadIdx.x < n) local[q] = atomicAdd(&cnt[b[q]], 1u);
        __syncthreads();
        for (int j = threadIdx.x; j < kBuckets; j += blockDim.x)
            if (cnt[j]) base[j] = atomicAdd(&cursor[j], cnt[j]);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kPer; q++) {
            const uint64_t i = b0 + (uint64_t)q * 256 + threadIdx.x;
            if (i < n) order[base[b[q]] + local[q]] = (uint32_t)i;
        }
        __syncthreads();
    }
}

// tiles per ordered pixel pair (written at position i, scanned afterwards);
// the 64-bit total goes to the shards of kCtrTiles
template <int E>
__global__ __launch_bounds__(256) void k_tiles(const PixPair *__restrict__ pps, const uint32_t *__restrict__ order,
                                                const unsigned long long *__restrict__ ctr,
                                                unsigned long long *__restrict__ shards, uint64_t cap_pp,
                                                uint32_t *__restrict__ tiles) {
    const uint64_t n = bounded_count(&ctr[kCtrPixPairs], cap_pp);
    unsigned long long t = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t slots = pps[order[i]].slots;
        const uint32_t per = 64u * E;
        const uint32_t ti = slots > 1 ? (slots - 1 + per - 1) / per : 0u;
        tiles[i] = ti;
        t += ti;
    }
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o);
    if ((threadIdx.x & 63) == 0 && t)
        atomicAdd(&ctr_shard(shards, blockIdx.x * 4u + (threadIdx.x >> 6))[kCtrTiles], t);
}

// The descriptor of every tile (its ordered pixel pair, the tile within it,
// the two pixels' sequence ranges and polygons), from the scanned counts;
// nothing is written when the tiles exceed the map's capacity
__global__ __launch_bounds__(256) void k_tile_map(DevSet S, const uint32_t *__restrict__ pa_all,
                                                  const uint32_t *__restrict__ pb_all,
                                                  const IsxDesc *__restrict__ desc, const PixPair *__restrict__ pps,
                                                  const uint32_t *__restrict__ order,
                                                  const uint32_t *__restrict__ tile_off,
                                                  const unsigned long long *__restrict__ ctr, uint64_t cap_pp,
                                                  uint64_t cap_tiles, TileDesc *__restrict__ map) {
    const uint64_t npp = bounded_count(&ctr[kCtrPixPairs], cap_pp);
    if (ctr[kCtrTiles] > cap_tiles) return;
    const uint32_t *pa_ids = pa_all + desc->begin;
    const uint32_t *pb_ids = pb_all + desc->begin;
    for (uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; q < npp; q += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t t0 = tile_off[q], t1 = tile_off[q + 1];
        if (t0 == t1) continue;
        const PixPair P = pps[order[q]];
        const farm_raster_hdr &A = S.hdr[pa_ids[P.pair]];
        const farm_raster_hdr &B = S.hdr[pb_ids[P.pair]];
        TileDesc d;
        d.pair = P.pair;
        d.a_s0 = A.seq_start + S.pixoff[A.pixoff_start + P.pa];
        d.a_s1 = A.seq_start + S.pixoff[A.pixoff_start + P.pa + 1];
        const uint32_t b_s0 = B.seq_start + S.pixoff[B.pixoff_start + P.pb];
        const uint32_t b_s1 = B.seq_start + S.pixoff[B.pixoff_start + P.pb + 1];
        d.b_c0 = S.choff[b_s0];
        d.b_c1 = S.choff[b_s1];
        d.a_vert = A.vert_start;
        d.b_vert = B.vert_start;
        // the target pixel's sequences once: offsets, sequence entries, vertices
        const uint32_t nb = b_s1 - b_s0;
        d.rbytes = 16 + 8u * nb + 8u * (S.pixedges[B.pix_start + P.pb] + nb);
        d.pad[0] = d.pad[1] = d.pad[2] = 0;
        for (uint32_t t = t0; t < t1; t++) {
            d.tile = t - t0;
            map[t] = d;
        }
    }
}

// ------------------------------------------------------------------------
// Persistent refinement over the tiles of the window.  A tile is 64 lanes x W consecutive edge slots of one source
// pixel's sequences (consecutive lanes share one vertex), refined against
// the edge sequences of one target pixel, walked in chunks of C segments
// (C = 8, 16 or 32, chosen per call; the autotuner picks it).  The chunks of
// all the pixel's sequences are one consecutive range of the box and chunk
// arrays, so kRefScreen of them are screened per round whatever sequences
// they belong to: at 10 vertices per pixel a pixel of a jagged ring holds 8
// sequences of 3 edges, and walking them one by one (a dependent chain of
// sequence, chunk offset and box loads each) took most of the kernel.
// Per chunk every lane first tests its W edges against the chunk's box (an
// exact prune: no edge whose line keeps the whole box at a safe distance can
// meet a segment of the chunk under the reference predicate); the (lane,
// chunk) pairs that survive are queued in LDS and evaluated kDrain at a time:
// the lane's edges (read from LDS) against the chunk's segments (loads of the
// evaluating lane), with the screen below and, for the rare candidates, the
// exact reference predicate.
//
// The line test alone keeps 6 % of the (lane, chunk) pairs on complex x lakes.
// A second exact test drops four fifths of those: boxes apart on an axis leave
// only crossings that rounding makes up, and those need lines that are nearly
// parallel.  Let the lane's vertex box and the chunk's be apart by g >= 2^-8 q
// on an axis (q the L1 reach).  The collinear branch needs box overlap, so a
// true answer needs the computed signs of c, d against line ab and of a, b
// against line cd to differ.  The f32 cross products err by less than 2^-22
// times the L1 lengths of their two differences, i.e. by a distance below
// delta = 2^-21.4 q to the line, so some point X of cd lies within delta of
// line ab and some point Y of ab within delta of line cd.  X and Y are at
// least g apart, so both lines make an angle below delta / g = 2^-13.4 with
// XY, and less than 2^-12.4 with each other.  A chunk's direction mask holds
// the classes within kDirTol = 2^-9 (>= 2^-10 in angle) of each of its
// segments, so masks without a common bit rule the crossing out.
// ------------------------------------------------------------------------

// Boxes of the refinement's target chunks.  A sequence (first, len) is walked
// in chunks c = 0, 1, ..: steps base = 1 + C c .. min(len, base + C - 1), whose
// segments span vertices first + base - 1 .. first + base + n - 1.  The box is
// stored as a centre and half extents rounded up, so [c - h, c + h] holds
// every vertex of the chunk in exact arithmetic.  Infinite extents (the prune
// never applies) go to a box that reaches past 2^40 or holds a non-finite
// vertex.  A chunk that holds a segment of length 0 is marked (kChunkPoint):
// for c == d the reference's c.cross(a, d) is 0 for every a, so
// segment_intersect takes its collinear branch and answers with the
// bounding-box overlap alone, on either side of line ab.  Such a segment is
// in play only for a lane whose box is not apart from the chunk's.  (Every
// closed ring has one, its repeated first vertex; as a box that is never
// pruned it put its chunk against all 512 edges of every tile, all of them
// through the exact replay: half of the kernel's time.)
__global__ __launch_bounds__(256) void k_chunk_count(DevSet S, int64_t npolys, uint32_t C,
                                                     uint32_t *__restrict__ cnt) {
    const int64_t p = blockIdx.x;
    if (p >= npolys) return;
    const farm_raster_hdr H = S.hdr[p];
    for (uint32_t s = threadIdx.x; s < H.nseqs; s += blockDim.x)
        cnt[H.seq_start + s] = (S.seqs[H.seq_start + s].y + C - 1) / C;
}

__global__ __launch_bounds__(256) void k_chunk_box(DevSet S, int64_t npolys, uint32_t C,
                                                   const uint32_t *__restrict__ choff, float4 *__restrict__ box,
                                                   uint4 *__restrict__ seg) {
    const int64_t p = blockIdx.x;
    if (p >= npolys) return;
    const farm_raster_hdr H = S.hdr[p];
    const float *x = S.x + H.vert_start, *y = S.y + H.vert_start;
    // chunk o of sequence sq, whose segments start at step base
    auto put = [&](uint2 sq, uint32_t base, uint32_t o) {
        const uint32_t n = min(C, sq.y - base + 1);
        float x0 = x[sq.x + base - 1], x1 = x0, y0 = y[sq.x + base - 1], y1 = y0;
        bool open = isfinite(x0) && isfinite(y0);  // false: never prune this chunk
        float lx = x0, ly = y0;
        uint64_t dirs = 0;
        uint32_t mark = 0;
        for (uint32_t m = 0; m < n; m++) {
            const float vx = x[sq.x + base + m], vy = y[sq.x + base + m];
            open = open && isfinite(vx) && isfinite(vy);
            float s;
            if (vx == lx && vy == ly) mark = kChunkPoint;
            else dirs |= dir_angle(vx - lx, vy - ly, s) ? dir_bit(s - kDirTol) | dir_bit(s + kDirTol) : ~0ull;
            lx = vx;
            ly = vy;
            x0 = fminf(x0, vx);
            x1 = fmaxf(x1, vx);
            y0 = fminf(y0, vy);
            y1 = fmaxf(y1, vy);
        }
        const float cx = 0.5f * x0 + 0.5f * x1, cy = 0.5f * y0 + 0.5f * y1;
        // a rounded difference is within 2^-24 of the exact one; the
        // factor and the smallest normal cover it and the product's rounding
        float hx = fmaxf(x1 - cx, cx - x0) * 1.0000003f + 1.1754944e-38f;
        float hy = fmaxf(y1 - cy, cy - y0) * 1.0000003f + 1.1754944e-38f;
        const float big = 0x1p40f;
        if (!(open && fabsf(cx) + hx < big && fabsf(cy) + hy < big)) hx = hy = INFINITY;
        box[o] = make_float4(cx, cy, hx, hy);
        seg[o] = make_uint4(sq.x + base - 1, n | mark, (uint32_t)dirs, (uint32_t)(dirs >> 32));
    };
    // a lane takes a short sequence whole; the chunks of a longer one are
    // shared by the wave (1.18 -> 0.58 ms for 400 rings of 1.6 M vertices in
    // all and 10,000 lakes, where one lane had sequences of 10,000 segments)
    const int lane = threadIdx.x & 63;
    for (uint32_t s0 = threadIdx.x & ~63u; s0 < H.nseqs; s0 += blockDim.x) {
        const uint32_t s = s0 + lane;
        const uint2 sq = s < H.nseqs ? S.seqs[H.seq_start + s] : make_uint2(0u, 0u);
        const uint32_t o = s < H.nseqs ? choff[H.seq_start + s] : 0u;
        const bool wide = sq.y > 4 * C;
        if (!wide)
            for (uint32_t k = 0; k * C < sq.y; k++) put(sq, 1 + k * C, o + k);
        for (uint64_t m = __ballot(wide); m; m &= m - 1) {
            const int src = __ffsll((unsigned long long)m) - 1;
            const uint2 w = make_uint2((uint32_t)__builtin_amdgcn_readlane((int)sq.x, src),
                                       (uint32_t)__builtin_amdgcn_readlane((int)sq.y, src));
            const uint32_t wo = (uint32_t)__builtin_amdgcn_readlane((int)o, src);
            for (uint32_t k = lane; k * C < w.y; k += 64) put(w, 1 + k * C, wo + k);
        }
    }
}

// Most chunks of one polygon.
__global__ __launch_bounds__(256) void k_most_chunks(DevSet S, int64_t npolys, const uint32_t *__restrict__ choff,
                                                     uint32_t *__restrict__ most) {
    uint32_t n = 0;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < npolys;
         p += (int64_t)gridDim.x * blockDim.x) {
        const farm_raster_hdr H = S.hdr[p];
        n = max(n, choff[H.seq_start + H.nseqs] - choff[H.seq_start]);
    }
    for (int o = 32; o > 0; o >>= 1) n = max(n, __shfl_xor(n, o));
    if ((threadIdx.x & 63) == 0 && n) atomicMax(most, n);
}

// Groups of kGroup consecutive chunks: the box that holds theirs, their
// steps, directions and mark.
__global__ __launch_bounds__(256) void k_chunk_group(const float4 *__restrict__ box, const uint4 *__restrict__ seg,
                                                     uint32_t nchunks, float4 *__restrict__ gbox,
                                                     uint4 *__restrict__ gseg) {
    const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t c0 = g * kGroup;
    if (g >= (nchunks + kGroup - 1) / kGroup) return;
    float x0 = INFINITY, x1 = -INFINITY, y0 = INFINITY, y1 = -INFINITY;
    bool open = true;
    uint4 s = make_uint4(0u, 0u, 0u, 0u);
    for (uint32_t c = c0; c < min(c0 + kGroup, nchunks); c++) {
        const float4 b = box[c];
        const uint4 q = seg[c];
        open = open && b.z < INFINITY && b.w < INFINITY;
        x0 = fminf(x0, b.x - b.z);
        x1 = fmaxf(x1, b.x + b.z);
        y0 = fminf(y0, b.y - b.w);
        y1 = fmaxf(y1, b.y + b.w);
        s.x += q.y & ~kChunkPoint;
        s.y |= q.y & kChunkPoint;
        s.z |= q.z;
        s.w |= q.w;
    }
    // the chunk's ends are off by a rounding each of c - h and c + h (2^-24 of
    // the larger of the two: at most 2^-24 (|x0| + |x1|) a side), the new
    // centre and extent by a few more of the same
    const float cx = 0.5f * x0 + 0.5f * x1, cy = 0.5f * y0 + 0.5f * y1;
    const float ex = (fabsf(x0) + fabsf(x1)) * 0x1p-22f, ey = (fabsf(y0) + fabsf(y1)) * 0x1p-22f;
    float hx = fmaxf(x1 - cx, cx - x0) + ex + 1.1754944e-38f, hy = fmaxf(y1 - cy, cy - y0) + ey + 1.1754944e-38f;
    if (!(open && hx < 0x1p42f && hy < 0x1p42f)) hx = hy = INFINITY;
    gbox[g] = make_float4(open ? cx : 0.f, open ? cy : 0.f, hx, hy);
    gseg[g] = s;
}

// Chunk boxes read through the constant address space: they do not change
// during a launch, and uniform addresses then become scalar loads.
typedef __attribute__((address_space(4))) const float cfloat;
typedef __attribute__((address_space(4))) const uint32_t cuint;

// Queued items are evaluated kDrain at a time, 2^kSplit lanes or more to an
// item: measured on complex x lakes (496,000 pairs, 8 edges per lane, 16
// segments per chunk) 9.87, 9.22 and 9.5 ms with 1, 2 and 4 lanes, as a wave
// usually holds a few dozen items and fewer steps follow each other.
constexpr uint32_t kSplit = 1, kDrain = 64u >> kSplit;
constexpr uint32_t kRefQueue = 512;  // queued items per wave: a power of 2 above 63 + 64 kRefScreen (or kGroup)

template <int W, int C, bool PRUNE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_refine(DevSet S, const uint32_t *__restrict__ pa_all,
                                                 const uint32_t *__restrict__ pb_all,
                                                 const IsxDesc *__restrict__ desc,
                                                 const TileDesc *__restrict__ tile_map, uint64_t cap_pp,
                                                 uint64_t cap_tiles, uint32_t *__restrict__ cursor,
                                                 uint32_t *__restrict__ result,
                                                 const unsigned long long *__restrict__ ctr,
                                                 unsigned long long *__restrict__ shards) {
    // the tile total, unless a buffer of an earlier phase overflowed (the
    // host then grows the workspace and repeats the call, or fails it)
    if (ctr[kCtrPixPairs] > cap_pp || ctr[kCtrTiles] > cap_tiles) return;
    const uint32_t total = (uint32_t)ctr[kCtrTiles];
    uint32_t *pair_tests = desc->pair_tests;
    // per wave: the tile's source slots (x then y, W + 1 each) and edge bits
    // of every lane, and the ring of queued items (first vertex of the target
    // chunk, source lane | steps << 8)
    __shared__ float s_src[4][64][2 * (W + 1)];
    __shared__ uint32_t s_ev[4][64];
    // (with groups: chunk of the pixel and source lane in one word each, and
    // in the other half a ring of groups and source lanes; sets with a
    // polygon of 2^26 chunks or more run at 2 edges per lane)
    constexpr bool groups = PRUNE && W >= 4;
    __shared__ uint2 s_ring[4][kRefQueue];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    float(*src)[2 * (W + 1)] = s_src[wv];
    uint32_t *sev = s_ev[wv];
    uint2 *ring = s_ring[wv];
    uint32_t *ring4 = (uint32_t *)s_ring[wv], *ringg = ring4 + kRefQueue;
    // and the directions of every lane's edges (dir_bit)
    __shared__ uint2 s_dir[4][64];
    uint2 *sdir = s_dir[wv];
    // work counters: per tile in 32-bit lane registers, summed at its end
    // into wave-uniform totals (64-bit lane totals push the kernel past its
    // register budget)
    unsigned long long items = 0, rbytes = 0, tests_w = 0, pruned_w = 0;
    // A wave takes `grab` consecutive tiles at a time, whose pairs' flags are
    // looked up together, one per lane (on jagged small polygons 70 % of the
    // tiles belong to pairs already decided; a descriptor and a flag load for
    // each, one tile after the other, was most of their time).  Grab k of
    // cursor c covers tiles (k * kCtrShards + c) * grab onwards, so every
    // cursor runs through the cost order.  A wave stays with its own cursor
    // until that has run out, then looks at all of them (one load) and moves
    // on to the next that has not.  One cursor for all waves took 0.6 ms to
    // hand out the 26,000 tiles of a 4,000-pair call; handing tiles out by
    // position alone left waves idle (a call of 1.3e6 tiles of uneven cost
    // took 17.5 ms instead of 13.9).
    const uint32_t nwaves = gridDim.x * 4u, wid = blockIdx.x * 4u + (uint32_t)wv;
    const uint32_t grab = min(max(total / (nwaves * 16u), 1u), 16u);
    uint32_t home = wid & (kCtrShards - 1);
    uint32_t tbase = 0;
    unsigned long long live = 0;  // the batch's tiles still to run
    for (;;) {
        if (!live) {
            // (an opaque copy of the lane: the addresses below are computed
            // here, not kept in registers across the tiles)
            uint32_t ln = (uint32_t)lane;
            asm volatile("" : "+v"(ln));
            uint32_t c = 0;
            if (ln == 0) c = atomicAdd(&cursor[home * kCursorStride], 1u);
            c = __builtin_amdgcn_readfirstlane(c);
            const uint64_t b = ((uint64_t)c * kCtrShards + home) * grab;
            if (b >= total) {
                const uint32_t at = __hip_atomic_load(&cursor[ln * kCursorStride], __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT);
                const unsigned long long left =
                    __ballot(((uint64_t)at * kCtrShards + ln) * grab < total);
                if (!left) break;  // every cursor has run out
                // the first cursor after home with tiles left
                const unsigned long long after = home < 63u ? left >> (home + 1u) << (home + 1u) : 0ull;
                home = (uint32_t)__ffsll(after ? after : left) - 1u;
                continue;
            }
            tbase = (uint32_t)b;
            bool open = false;
            if (ln < grab && tbase + (uint64_t)ln < total)
                open = !__hip_atomic_load(&result[tile_map[tbase + ln].pair], __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
            live = __ballot(open);
            continue;
        }
        const uint32_t t = tbase + (uint32_t)__ffsll(live) - 1u;
        live &= live - 1;
        uint32_t tests = 0, queued = 0, dropped = 0;
        // the tile's descriptor (one uniform load), then its pair's flag
        // again (an earlier tile of the grab may have decided it)
        const TileDesc td = tile_map[t];
        const uint32_t pair = uni(td.pair), tile = uni(td.tile);
        if (__hip_atomic_load(&result[pair], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) continue;
        items++;
        const uint2 *sqa = S.seqs;  // absolute sequence indices
        const uint32_t a_s0 = uni(td.a_s0), a_s1 = uni(td.a_s1);
        const uint32_t b_c0 = uni(td.b_c0), b_c1 = uni(td.b_c1);
        const float *ax_ = S.x + uni(td.a_vert);
        const float *ay_ = S.y + uni(td.a_vert);
        const float4 *bq_ = S.xyd + uni(td.b_vert);
        const uint32_t td_rbytes = uni(td.rbytes);
        // the tile's body, invoked once below (as a lambda it is allocated
        // to fewer registers than as a plain block: 128 against 155 VGPRs at
        // W = 8, four waves per SIMD instead of three)
        auto run = [&](auto width_tag) {
            constexpr int E = decltype(width_tag)::value;
            // source vertices of this lane: slots first .. first + E
            const uint32_t first = tile * 64u * W + (uint32_t)lane * E;
            float px[E + 1], py[E + 1];
            bool ev[E];
            const uint32_t nsq = a_s1 - a_s0;
            if (nsq <= 64) {
                // every lane loads one of the pixel's sequences and its first
                // slot (a wave prefix sum of len + 1) into the wave's LDS slot
                // array (free until this tile's slots are published); a slot's
                // sequence is then found by a binary search there and the
                // lane's later slots by stepping on (LDS reads only, so lanes
                // may diverge)
                const uint2 mine = (uint32_t)lane < nsq ? sqa[a_s0 + lane] : make_uint2(0u, 0u);
                uint32_t nslots;
                const uint32_t sstart = wave_excl_scan((uint32_t)lane < nsq ? mine.y + 1 : 0u, lane, &nslots);
                src[lane][0] = __uint_as_float(mine.x);  // (bit copies: the array holds floats)
                src[lane][1] = __uint_as_float(mine.y);
                src[lane][2] = __uint_as_float(sstart);
                wave_sync();
                auto ent = [&](int j, int f) { return __float_as_uint(src[j][f]); };
                int k = 0;
#pragma unroll
                for (int step = 32; step > 0; step >>= 1) {
                    const int c = k + step;
                    if (c < (int)nsq && ent(c, 2) <= first) k = c;
                }
                uint32_t sbase = ent(k, 2);
                uint2 sq = make_uint2(ent(k, 0), ent(k, 1));
                for (int m = 0; m <= E; m++) {
                    const uint32_t s = first + m;
                    while (k + 1 < (int)nsq && s >= sbase + sq.y + 1) {
                        sbase += sq.y + 1;
                        k++;
                        sq = make_uint2(ent(k, 0), ent(k, 1));
                    }
                    uint32_t o = s - sbase;
                    const bool inside = s < sbase + sq.y + 1;
                    if (!inside) o = sq.y;  // past the last slot: clamp (no edge)
                    const uint32_t v = sq.x + o;
                    px[m] = ax_[v];
                    py[m] = ay_[v];
                    if (m < E) ev[m] = inside && o < sq.y;
                }
                wave_sync();  // every lane's reads done before the slots overwrite the array
            } else {
                uint32_t k = a_s0, sbase = 0;
                uint2 sq = sqa[k];
                for (int m = 0; m <= E; m++) {
                    const uint32_t s = first + m;
                    while (k + 1 < a_s1 && s >= sbase + sq.y + 1) {
                        sbase += sq.y + 1;
                        k++;
                        sq = sqa[k];
                    }
                    uint32_t o = s - sbase;
                    const bool inside = s < sbase + sq.y + 1;
                    if (!inside) o = sq.y;  // past the last slot: clamp (no edge)
                    const uint32_t v = sq.x + o;
                    px[m] = ax_[v];
                    py[m] = ay_[v];
                    if (m < E) ev[m] = inside && o < sq.y;
                }
            }
            int nvalid = 0;
            uint32_t evb = 0;
#pragma unroll
            for (int e = 0; e < E; e++) {
                nvalid += ev[e] ? 1 : 0;
                evb |= (ev[e] ? 1u : 0u) << e;
            }
            // publish this lane's slots for the lanes that evaluate its items
#pragma unroll
            for (int v = 0; v <= E; v++) {
                src[lane][v] = px[v];
                src[lane][E + 1 + v] = py[v];
            }
            sev[lane] = evb;
            {
                uint64_t dirs = 0;
#pragma unroll
                for (int e = 0; e < E; e++) {
                    float s;
                    const uint64_t b = dir_angle(px[e + 1] - px[e], py[e + 1] - py[e], s) ? dir_bit(s) : ~0ull;
                    dirs |= ev[e] ? b : 0ull;
                }
                sdir[lane] = make_uint2((uint32_t)dirs, (uint32_t)(dirs >> 32));
            }
            __builtin_amdgcn_wave_barrier();
            bool hit = false;
            bool stop = false;
            uint32_t qhead = 0, qn = 0, screened = 0;  // wave-uniform
            uint32_t ghead = 0, gn = 0;
            const uint32_t g0 = groups ? b_c0 & ~(kGroup - 1) : b_c0, lo = b_c0 - g0, nch = b_c1 - g0;
            const float4 *vbox = S.chbox + g0;
            const uint4 *vseg = S.chseg + g0;
            uint32_t scr_steps = 0, queued_steps = 0;  // target steps screened (uniform) / queued by this lane

            // Evaluate source lane sl's E edges against the ns <= C segments from
            // target vertex vs on.  Per target vertex q and source edge (a, b):
            //   O(q) = a.cross(b, q)   -- o1/o2 of consecutive steps
            //   o(p) = c.cross(p, d)   -- per source vertex p, for the segment (c, d)
            // carried from step to step: tx/ty = p - c serves O(c) and, by the
            // antisymmetry of rounded subtraction, o(p) of the next step.  A
            // superset filter (o1*o2 <= 0 or o3 == 0, and o3*o4 <= 0) sends
            // the rare candidates to the exact reference predicate.
            auto eval = [&](uint32_t sl, uint32_t vs, uint32_t ns) {
                float qpx[E + 1], qpy[E + 1];
#pragma unroll
                for (int v = 0; v <= E; v++) {
                    qpx[v] = src[sl][v];
                    qpy[v] = src[sl][E + 1 + v];
                }
                const uint32_t eb = sev[sl];
                float qbax[E], qbay[E], qinv[E];
                int qnv = 0;
#pragma unroll
                for (int e = 0; e < E; e++) {
                    qbax[e] = qpx[e + 1] - qpx[e];
                    qbay[e] = qpy[e + 1] - qpy[e];
                    const bool ve = (eb >> e) & 1u;
                    qinv[e] = ve ? -INFINITY : INFINITY;  // lifts a slot without an edge out of the screen
                    qnv += ve ? 1 : 0;
                }
                const float4 c04 = bq_[vs];
                const float c0x = c04.x, c0y = c04.y;
                float tx[E + 1], ty[E + 1], Op[E];
#pragma unroll
                for (int v = 0; v <= E; v++) {
                    tx[v] = qpx[v] - c0x;
                    ty[v] = qpy[v] - c0y;
                }
#pragma unroll
                for (int e = 0; e < E; e++) {
                    float l = qbay[e] * tx[e];
                    float r = qbax[e] * ty[e];
                    Op[e] = l - r;  // a.cross(b, c), bit-identical to the reference form
                }
                // running minimum of the screen, even and odd edges apart
                float gmin[2] = {INFINITY, INFINITY};
#pragma unroll 4
                for (int m = 0; m < C; m++) {
                    if ((uint32_t)m < ns) {
                        // the step's end q and direction (q - c), precomputed with
                        // the same rounding, in one load
                        const float4 q4 = bq_[vs + 1 + m];
                        const float qx = q4.x, qy = q4.y, ddx = q4.z, ddy = q4.w;
                        float o[E + 1];
#pragma unroll
                        for (int v = 0; v <= E; v++) {
                            float l = tx[v] * ddy;
                            float r = ty[v] * ddx;
                            o[v] = l - r;  // c.cross(p_v, d)
                            tx[v] = qpx[v] - qx;
                            ty[v] = qpy[v] - qy;
                        }
#pragma unroll
                        for (int e = 0; e < E; e++) {
                            float l = qbay[e] * tx[e];
                            float r = qbax[e] * ty[e];
                            const float On = l - r;  // a.cross(b, d)
                            // superset of segment_intersect: both pairs of
                            // orientations have opposite (or zero) signs, or the
                            // collinear branch may apply (o3 == 0).  A slot
                            // without an edge enters only through o3 == 0, a
                            // false candidate the exact replay discards.
                            const float h = fmaxf(fmaxf(o[e] * o[e + 1], Op[e] * On), qinv[e]);
                            gmin[e & 1] = fminf(fminf(gmin[e & 1], h), fabsf(o[e]));
                            Op[e] = On;
                        }
                    }
                }
                const bool maybe = fminf(gmin[0], gmin[1]) <= 0.f;
                if (__any(maybe)) {
                    // rare: re-evaluate the item with the reference predicate
                    if (maybe) {
                        float ccx = c0x, ccy = c0y;
                        for (uint32_t m = 0; m < ns; m++) {
                            const float4 d4 = bq_[vs + 1 + m];
                            const float dx = d4.x, dy = d4.y;
#pragma unroll
                            for (int e = 0; e < E; e++)
                                if (((eb >> e) & 1u) &&
                                    seg_intersect(qpx[e], qpy[e], qpx[e + 1], qpy[e + 1], ccx, ccy, dx, dy))
                                    hit = true;
                            ccx = dx;
                            ccy = dy;
                        }
                    }
                }
                tests += (uint32_t)qnv * ns;
            };

            // Evaluate the n <= kDrain (without the prune 64) oldest queued items: the source
            // lane's E edges against the chunk's nstep target segments.
            //
            // An item is split over k = 64 / n lanes, rounded down to a power
            // of two (at most C), part j taking its steps j C / k .. (j + 1) C
            // / k - 1.  A part is the item's segments from its own first vertex
            // on, so the split evaluates the same tests in C / k steps instead
            // of C.
            auto drain = [&](uint32_t n) {
                uint32_t lk = PRUNE ? kSplit : 0u;  // log2 k (uniform)
                while ((1u << lk) < (uint32_t)C && (n << (lk + 1)) <= 64u) lk++;
                const uint32_t seg = (uint32_t)C >> lk;
                const uint32_t item = (uint32_t)lane >> lk, m0 = ((uint32_t)lane & ((1u << lk) - 1u)) * seg;
                uint2 it;
                if constexpr (groups) {
                    const uint32_t w = ring4[(qhead + min(item, n - 1)) & (kRefQueue - 1)];
                    const uint4 sg = vseg[w >> 6];
                    it = make_uint2(sg.x, (w & 63u) | ((sg.y & ~kChunkPoint) << 8));
                } else {
                    it = ring[(qhead + item) & (kRefQueue - 1)];
                }
                const uint32_t nsf = item < n ? (it.y >> 8) : 0u;
                const uint32_t ns = nsf > m0 ? min(seg, nsf - m0) : 0u;
                const bool has = ns > 0u;
                const uint32_t sl = has ? (it.y & 63u) : (uint32_t)lane;
                const uint32_t vs = has ? it.x + m0 : 0u;  // the part's first vertex c
                eval(sl, vs, ns);
                qhead = (qhead + n) & (kRefQueue - 1);
                qn -= n;
                if (__any(hit)) stop = true;
            };

            // Exact prune of a lane's edges against a chunk (or a group of
            // them, by the box that holds theirs).  q >= Q, the L1 reach from any vertex of the lane's
            // edges to the chunk box, is taken from the box of those
            // vertices.  If every box point p has
            // |a.cross(b, p)| > M_lin = 2^-18 q |b - a|_1 in exact
            // arithmetic, the reference's f32 a.cross(b, p) has one
            // nonzero sign on the whole chunk (rounding <= 3 2^-24 Q
            // |b - a|_1), so its sign test is false for every segment of
            // the chunk.  Its collinear branch (c.cross(a, d) ==
            // c.cross(b, d) == 0) answers with inter1's exact bounding-box
            // overlap, impossible when the chunk box and the box of the
            // lane's vertices are apart on an axis; otherwise it needs a
            // and b within rounding of line cd, which puts c within
            // 2^-20.7 Q (|b - a|_1 + 2Q) of line ab, and the margin is
            // M = 2^-18 q (|b - a|_1 + 2q).  Both margins get 2^-80 added.
            // The cross product at the box centre is evaluated relative
            // to the lane's first vertex o: C = s.cross(a - o) per edge
            // (s = b - a), then s.cross(c - o) - C in two fmas; with the
            // spread over the box and M in two more fmas the f32
            // evaluation errs by at most about 13 2^-24 q |b - a|_1
            // (every operand is within 2q of o), which M covers twice
            // over.  (A segment of length 0 only answers with box
            // overlap: its chunk is kept for the lanes not apart.)
            struct Lines {
                float sbx[E], sby[E], scc[E];
                float ox, oy, lxl, lxh, lyl, lyh;  // first vertex, box of the slot vertices
                uint2 dir;
            };
            auto lines = [&](uint32_t sl, uint32_t eb) {
                Lines L;
                L.ox = src[sl][0];
                L.oy = src[sl][E + 1];
                float nx = L.ox, ny = L.oy;
                L.lxl = L.lxh = nx;
                L.lyl = L.lyh = ny;
#pragma unroll
                for (int e = 0; e < E; e++) {
                    const float ax = nx, ay = ny;
                    nx = src[sl][e + 1];
                    ny = src[sl][E + 2 + e];
                    L.lxl = fminf(L.lxl, nx);
                    L.lxh = fmaxf(L.lxh, nx);
                    L.lyl = fminf(L.lyl, ny);
                    L.lyh = fmaxf(L.lyh, ny);
                    const bool ve = (eb >> e) & 1u;
                    // a slot without an edge gets s = 0 and C = +inf: its
                    // centre cross is -inf and the box is "pruned" for it
                    // (an infinite box makes the threshold NaN instead,
                    // which queues the item; the evaluation skips the slot)
                    L.sbx[e] = ve ? nx - ax : 0.f;
                    L.sby[e] = ve ? ny - ay : 0.f;
                    const float axo = ax - L.ox, ayo = ay - L.oy;
                    L.scc[e] = ve ? fmaf(L.sbx[e], ayo, -(L.sby[e] * axo)) : INFINITY;
                }
                L.dir = sdir[sl];
                return L;
            };
            auto needs = [&](const Lines &L, float4 bb, uint32_t mark, uint32_t cdl, uint32_t cdh) -> bool {
                // the reach q (rounded up), and whether the boxes are apart
                // on an axis (by more than the f32 rounding of the tests)
                const float ex0 = bb.x - L.lxl, ex1 = bb.x - L.lxh;
                const float ey0 = bb.y - L.lyl, ey1 = bb.y - L.lyh;
                const float q = ((fmaxf(fabsf(ex0), fabsf(ex1)) + fmaxf(fabsf(ey0), fabsf(ey1))) + (bb.z + bb.w)) *
                                1.000001f;
                const float hx1 = bb.z * 1.000001f, hy1 = bb.w * 1.000001f;
                // (ex1 > hx1 or -ex0 > hx1 or ey1 > hy1 or -ey0 > hy1, as two
                // maxima and two compares)
                const float sepx = fmaxf(ex1, -ex0), sepy = fmaxf(ey1, -ey0);
                const bool apart = (sepx > hx1) | (sepy > hy1);
                // Direction prune: apart by more than 2^-8 q on an axis
                // and no segment of the chunk within kDirTol of the
                // direction of any of the lane's edges.
                const bool far = fmaxf(sepx - hx1, sepy - hy1) > q * 0x1p-8f && q < 0x1p60f;
                const bool cand = !far || ((L.dir.x & cdl) | (L.dir.y & cdh)) != 0u;
                if (!__ballot(cand)) return false;  // no lane's lines need a look
                const float k1 = q * 0x1p-18f;
                const float k2 = apart ? 0x1p-80f : fmaf(q, q * 0x1p-17f, 0x1p-80f);
                // |s_y| hx + |s_x| hy + (|s_x| + |s_y|) k1 + k2 as
                // |s_y| (hx + k1) + |s_x| (hy + k1) + k2
                const float hxk = bb.z + k1, hyk = bb.w + k1;
                const float cxo = bb.x - L.ox, cyo = bb.y - L.oy;
                bool line = false;
#pragma unroll
                for (int e = 0; e < E; e++) {
                    const float oc = fmaf(L.sbx[e], cyo, -fmaf(L.sby[e], cxo, L.scc[e]));  // at the box centre
                    const float thr = fmaf(fabsf(L.sby[e]), hxk, fmaf(fabsf(L.sbx[e]), hyk, k2));
                    line = line | !(fabsf(oc) > thr);  // bitwise: no branch per edge
                }
                return (line & cand) | (!apart && (mark & kChunkPoint));
            };
            // bits of the lanes below this one in m
            auto below = [](unsigned long long m) {
                return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            };
            // The chunks of the n <= 64 oldest queued groups, each for the
            // source lane that queued it; 64 / n lanes (a power of 2, at most
            // kGroup) share a group's chunks.
            auto look = [&](uint32_t n) {
                uint32_t lk = 0;
                while ((1u << lk) < kGroup && (n << (lk + 1)) <= 64u) lk++;
                const uint32_t item = (uint32_t)lane >> lk, part = kGroup >> lk;
                const bool has = item < n;
                const uint32_t w = ringg[(ghead + min(item, n - 1)) & (kRefQueue - 1)];
                const uint32_t sl = w & 63u, eb = sev[sl];
                const uint32_t c0 = (w >> 6) * kGroup + ((uint32_t)lane & ((1u << lk) - 1u)) * part;
                const Lines L = lines(sl, eb);
                for (uint32_t i = 0; i < part; i++) {
                    const uint32_t c = c0 + i;
                    const float4 bb = vbox[c];
                    const uint4 sg = vseg[c];
                    const bool mine = has && c >= lo && c < nch;
                    const bool need = needs(L, bb, sg.y, sg.z, sg.w) && mine;
                    const unsigned long long bm = __ballot(need);
                    if (need) ring4[(qhead + qn + below(bm)) & (kRefQueue - 1)] = c << 6 | sl;
                    else if (mine) dropped += (uint32_t)__popc(eb) * (sg.y & ~kChunkPoint);
                    qn += (uint32_t)__popcll(bm);
                }
                ghead = (ghead + n) & (kRefQueue - 1);
                gn -= n;
            };

            if constexpr (!PRUNE) {
                // every chunk for every lane that has an edge, 64 items at a
                // time (straight from the chunks, each lane its own edges, a
                // tile's empty lanes idle: 91 ms instead of 75 at 8 edges per
                // lane on complex x lakes)
                const cuint *cseg = (const cuint *)S.chseg;
                const unsigned long long bm = __ballot(evb != 0);
                for (uint32_t c = b_c0; c < b_c1 && !stop; c++) {
                    const uint32_t v0 = cseg[4 * c], nstep = cseg[4 * c + 1] & ~kChunkPoint;
                    scr_steps += nstep;
                    if (evb) {
                        ring[(qhead + qn + below(bm)) & (kRefQueue - 1)] = make_uint2(v0, (uint32_t)lane | (nstep << 8));
                        queued_steps += nstep;
                    }
                    qn += (uint32_t)__popcll(bm);
                    while (!stop && (qn >= 64 || (c + 1 == b_c1 && qn))) {
                        __builtin_amdgcn_wave_barrier();
                        drain(min(qn, 64u));
                    }
                    if ((++screened & 31u) == 0 &&
                        __hip_atomic_load(&result[pair], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                        break;
                }
            } else {
                // kRefScreen boxes at a time against every lane's edges (scalar
                // loads; entries past the pixel's last are read, the arrays keep
                // spare ones, but not used): of chunks at narrow tiles, whose
                // pixels hold few of them; at 4 edges per lane and more of
                // aligned groups of kGroup chunks (the first and last may hold
                // chunks of other pixels, which are not used).  Nearly every
                // group is needed by one of the 64 lanes or another, but by few
                // of them, so the (lane, group) items are queued and their chunks
                // looked at with every lane at work (skipping the groups that no
                // lane needs gave 7 % only).  Measured, k_refine at 8 edges per
                // lane on 400 complex rings x 9,973 lakes (-v 256): 9.2 ms
                // without groups, 6.4 with groups of 4, 6.1 of 8; with chunks of
                // 32 segments 7.45, 6.7 and 6.9.  For 4,000 x 100,000 of
                // them, 16 segments: 110.5, 76.9, 74.5 ms.  (All with the prune
                // still a switch in the kernel; without it 6.03 and 72.7 with
                // groups of 4.)
                const cfloat *cbox = (const cfloat *)(groups ? S.cgbox + g0 / kGroup : vbox);
                const cuint *cseg = (const cuint *)(groups ? S.cgseg + g0 / kGroup : vseg);
                const uint32_t nbox = groups ? (nch + kGroup - 1) / kGroup : nch;
                for (uint32_t g = 0;;) {
                    if (g < nbox) {
                        // this lane's slots again, from LDS (not kept in registers
                        // across the evaluation of queued items: the lane's index
                        // is made opaque, or the loads would move out of the loop)
                        uint32_t sln = (uint32_t)lane;
                        asm volatile("" : "+v"(sln));
                        const Lines L = lines(sln, evb);
                        bool need[kRefScreen];
#pragma unroll
                        for (int i = 0; i < (int)kRefScreen; i++) {
                            const uint32_t c = 4 * (g + i);
                            need[i] = needs(L, make_float4(cbox[c], cbox[c + 1], cbox[c + 2], cbox[c + 3]), cseg[c + 1],
                                            cseg[c + 2], cseg[c + 3]);
                        }
#pragma unroll
                        for (int i = 0; i < (int)kRefScreen; i++) {
                            const uint32_t c = g + i;
                            if (c >= nbox) break;
                            const uint32_t v0 = cseg[4 * c], nstep = cseg[4 * c + 1] & ~kChunkPoint;
                            const unsigned long long bm = __ballot(need[i]);
                            if constexpr (groups) {
                                uint32_t steps = v0;  // the group's
                                if (c * kGroup < lo || (c + 1) * kGroup > nch) {
                                    steps = 0;
                                    for (uint32_t k = max(c * kGroup, lo); k < min((c + 1) * kGroup, nch); k++)
                                        steps += ((const cuint *)vseg)[4 * k + 1] & ~kChunkPoint;
                                }
                                scr_steps += steps;
                                queued_steps += need[i] ? steps : 0u;
                                if (need[i]) ringg[(ghead + gn + below(bm)) & (kRefQueue - 1)] = c << 6 | (uint32_t)lane;
                                gn += (uint32_t)__popcll(bm);
                            } else {
                                scr_steps += nstep;
                                if (bm) {
                                    // append this chunk for every lane that needs it
                                    if (need[i]) {
                                        ring[(qhead + qn + below(bm)) & (kRefQueue - 1)] =
                                            make_uint2(v0, (uint32_t)lane | (nstep << 8));
                                        queued_steps += nstep;
                                    }
                                    qn += (uint32_t)__popcll(bm);
                                }
                            }
                        }
                        g += kRefScreen;
                    }
                    const bool last = g >= nbox;
                    do {
                        if constexpr (groups) {
                            if (gn >= 64 || (last && gn)) {
                                __builtin_amdgcn_wave_barrier();
                                look(min(gn, 64u));
                            }
                        }
                        while (!stop && (qn >= kDrain || (last && !gn && qn))) {
                            __builtin_amdgcn_wave_barrier();
                            drain(min(qn, kDrain));
                        }
                    } while (!stop && (gn >= 64 || (last && gn)));
                    if (last || stop) break;
                    if ((++screened & (groups ? 1u : 7u)) == 0 &&
                        __hip_atomic_load(&result[pair], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                        break;
                }
            }
            if (__any(hit)) {
                if (lane == 0) __hip_atomic_fetch_or(&result[pair], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }

            // algorithmic refine bytes of this tile: its source vertices plus
            // the target pixel's sequences once
            uint32_t edges = 0;
#pragma unroll
            for (int e = 0; e < E; e++) edges += (uint32_t)__popcll(__ballot((evb >> e) & 1u));
            rbytes += td_rbytes + edges * 8u;
            // tests the prune skipped: every edge's every screened step that was
            // not queued
            queued += (uint32_t)nvalid * queued_steps;
            pruned_w += (unsigned long long)edges * scr_steps;
        };
        run(std::integral_constant<int, W>());
        const unsigned long long t64 = wave_sum_u64(tests);
        tests_w += t64;
        pruned_w -= wave_sum_u64(queued);
        if constexpr (groups) pruned_w += wave_sum_u64(dropped);
        // executed tests of this tile, for the cost labels
        if (pair_tests && lane == 0) atomicAdd(&pair_tests[pair], (uint32_t)min(t64, 0xffffffffull));
    }
    if (lane == 0 && items) {
        unsigned long long *sh = ctr_shard(shards, wid);
        atomicAdd(&sh[kCtrTests], tests_w);
        atomicAdd(&sh[kCtrItems], items);
        atomicAdd(&sh[kCtrRefineBytes], rbytes);
        atomicAdd(&sh[kCtrPruned], pruned_w);
    }
}

// ------------------------------------------------------------------------
// Plain kernel: one workgroup (256 lanes) per candidate pair, the direct
// formulation with no pruning and no queue.  The window is scanned for IN
// overlaps by all lanes; then each BORDER x BORDER pixel pair is refined in
// full: both pixels' edges are flattened into LDS (a block scan over the
// sequence lengths, then every lane fills edges, finding its sequence by a
// binary search over the scanned starts), as coordinates, up to kPlainCap
// edges per side at a time, and the lanes sweep the source x target edge
// grid in 16 x 16 blocks (lane t tests source edge t / 16 and target edge
// t % 16 of each block), with a block-wide early exit every 8 blocks.
// ------------------------------------------------------------------------
constexpr int kPlainCap = 1024;   // edges per side held in LDS per chunk
constexpr int kPlainSeqs = 256;   // sequences per pixel scanned per pass

// Fills dst[0 .. len) with the coordinates (a.x, a.y, b.x, b.y) of edges
// first .. first + len of the concatenation of a pixel's sequences
// sq[0 .. nseq), seq_off[k] the scanned start of sequence k.
__device__ void plain_fill(const uint2 *__restrict__ sq, const uint32_t *seq_off, uint32_t nseq, uint32_t first,
                           uint32_t len, const float *__restrict__ X, const float *__restrict__ Y, float4 *dst) {
    for (uint32_t i = threadIdx.x; i < len; i += blockDim.x) {
        const uint32_t g = first + i;
        uint32_t lo = 0, hi = nseq;  // last k with seq_off[k] <= g
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (seq_off[mid] <= g) lo = mid;
            else hi = mid;
        }
        const uint32_t v = sq[lo].x + (g - seq_off[lo]);
        dst[i] = make_float4(X[v], Y[v], X[v + 1], Y[v + 1]);
    }
}

// Exclusive block scan of the lengths of sequences sq[0 .. n) (n <=
// kPlainSeqs): seq_off[k] for k < n, returns the total.
__device__ uint32_t plain_scan(const uint2 *__restrict__ sq, uint32_t n, uint32_t *seq_off, uint32_t *wsum) {
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const uint32_t v = (uint32_t)t < n ? sq[t].y : 0u;
    uint32_t tot;
    const uint32_t ex = wave_excl_scan(v, lane, &tot);
    if (lane == 0) wsum[w] = tot;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int i = 0; i < 4; i++) {
        before += i < w ? wsum[i] : 0u;
        all += wsum[i];
    }
    if ((uint32_t)t < n) seq_off[t] = before + ex;
    __syncthreads();
    return all;
}

__global__ __launch_bounds__(256) void k_plain(DevSet S, const uint32_t *__restrict__ pa_ids,
                                                const uint32_t *__restrict__ pb_ids, uint32_t npairs,
                                                uint32_t *__restrict__ result, unsigned long long *__restrict__ ctr) {
    __shared__ float4 ea[kPlainCap];
    __shared__ float4 eb[kPlainCap];
    __shared__ uint32_t offa[kPlainSeqs], offb[kPlainSeqs], wsum[4];
    __shared__ int s_flag;
    const uint32_t k = blockIdx.x;
    if (k >= npairs) return;
    const int tid = threadIdx.x;
    const farm_raster_hdr A = S.hdr[pa_ids[k]];
    const farm_raster_hdr B = S.hdr[pb_ids[k]];
    const uint8_t *sa = S.status + A.pix_start;
    const uint8_t *sb = S.status + B.pix_start;
    const uint32_t *pofa = S.pixoff + A.pixoff_start;
    const uint32_t *pofb = S.pixoff + B.pixoff_start;
    const uint2 *sqa = S.seqs + A.seq_start;
    const uint2 *sqb = S.seqs + B.seq_start;
    const float *AX = S.x + A.vert_start, *AY = S.y + A.vert_start;
    const float *BX = S.x + B.vert_start, *BY = S.y + B.vert_start;
    const Window wa = window_of(A, B.mbr[0], B.mbr[1], B.mbr[2], B.mbr[3]);
    const int nwx = wa.x1 - wa.x0 + 1, nwy = wa.y1 - wa.y0 + 1;
    const int nwa = nwx * nwy;
    if (tid == 0) s_flag = 0;
    __syncthreads();
    // IN overlap scan: lanes over source window pixels
    for (int w = tid; w < nwa; w += blockDim.x) {
        const int x = wa.x0 + w / nwy, y = wa.y0 + w % nwy;
        const int st_a = show(sa[y * A.dimx + x]);
        if (st_a == 0) continue;
        double lx, ly, hx, hy;
        pixel_box(A, x, y, lx, ly, hx, hy);
        const Window wb = window_of(B, lx, ly, hx, hy);
        for (int u = wb.x0; u <= wb.x1; u++)
            for (int v = wb.y0; v <= wb.y1; v++) {
                const int st_b = show(sb[v * B.dimx + u]);
                if (st_b != 0 && (st_a == 2 || st_b == 2)) s_flag = 1;
            }
    }
    __syncthreads();
    if (s_flag) {
        if (tid == 0) {
            result[k] = 1;
            atomicAdd(&ctr[kCtrInHits], 1ull);
        }
        return;
    }
    unsigned long long tests = 0;
    bool hit = false;
    const int ti = tid >> 4, tj = tid & 15;  // this lane's place in a 16 x 16 block
    // refinement: uniform loop over the BORDER x BORDER pixel pairs
    for (int w = 0; w < nwa && !hit; w++) {
        const int x = wa.x0 + w / nwy, y = wa.y0 + w % nwy;
        const int pa = y * A.dimx + x;
        if (show(sa[pa]) != 1) continue;
        double lx, ly, hx, hy;
        pixel_box(A, x, y, lx, ly, hx, hy);
        const Window wb = window_of(B, lx, ly, hx, hy);
        for (int u = wb.x0; u <= wb.x1 && !hit; u++)
            for (int v = wb.y0; v <= wb.y1 && !hit; v++) {
                const int pb = v * B.dimx + u;
                if (show(sb[pb]) != 1) continue;
                // the pixels' sequences, kPlainSeqs at a time on each side
                for (uint32_t s0a = pofa[pa]; s0a < pofa[pa + 1] && !hit; s0a += kPlainSeqs) {
                    const uint32_t nsa = min((uint32_t)kPlainSeqs, pofa[pa + 1] - s0a);
                    const uint32_t na = plain_scan(sqa + s0a, nsa, offa, wsum);
                    for (uint32_t s0b = pofb[pb]; s0b < pofb[pb + 1] && !hit; s0b += kPlainSeqs) {
                        const uint32_t nsb = min((uint32_t)kPlainSeqs, pofb[pb + 1] - s0b);
                        const uint32_t nb = plain_scan(sqb + s0b, nsb, offb, wsum);
                        for (uint32_t ca = 0; ca < na && !hit; ca += kPlainCap) {
                            const uint32_t la = min((uint32_t)kPlainCap, na - ca);
                            __syncthreads();
                            plain_fill(sqa + s0a, offa, nsa, ca, la, AX, AY, ea);
                            for (uint32_t cb = 0; cb < nb && !hit; cb += kPlainCap) {
                                const uint32_t lb = min((uint32_t)kPlainCap, nb - cb);
                                __syncthreads();
                                plain_fill(sqb + s0b, offb, nsb, cb, lb, BX, BY, eb);
                                __syncthreads();
                                const uint32_t bi = (la + 15) / 16, bj = (lb + 15) / 16;
                                uint32_t blk = 0;
                                bool done = false;  // block-uniform: set only from __syncthreads_or
                                for (uint32_t i0 = 0; i0 < bi && !done; i0++) {
                                    const uint32_t i = 16 * i0 + ti;
                                    const float4 a = ea[min(i, la - 1)];
                                    for (uint32_t j0 = 0; j0 < bj; j0++, blk++) {
                                        const uint32_t j = 16 * j0 + tj;
                                        if (i < la && j < lb) {
                                            const float4 b = eb[j];
                                            tests++;
                                            if (seg_intersect(a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w)) hit = true;
                                        }
                                        if ((blk & 7) == 7 && __syncthreads_or(hit)) {
                                            done = true;
                                            break;
                                        }
                                    }
                                }
                                hit = __syncthreads_or(hit);
                            }
                        }
                    }
                }
            }
    }
    for (int o = 32; o > 0; o >>= 1) tests += __shfl_xor(tests, o);
    if ((tid & 63) == 0) atomicAdd(&ctr[kCtrTests], tests);
    if (tid == 0 && hit) result[k] = 1;
}

// xyd[v] = (x[v], y[v], x[v] - x[v - 1], y[v] - y[v - 1]) over n padded
// vertices: the vertex and the same rounded f32 difference the refinement
// would form for the step arriving at it
__global__ __launch_bounds__(256) void k_vdiff(const float *__restrict__ x, const float *__restrict__ y, uint64_t n,
                                               float4 *__restrict__ xyd) {
    const uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    const float vx = x[v], vy = y[v];
    xyd[v] = v == 0 ? make_float4(vx, vy, 0.f, 0.f) : make_float4(vx, vy, vx - x[v - 1], vy - y[v - 1]);
}

// per-pixel edge count of every BORDER pixel (sum of its sequence lengths)
__global__ __launch_bounds__(256) void k_pixedges(DevSet S, int64_t npolys, uint32_t *__restrict__ out) {
    const int64_t p = blockIdx.x;
    if (p >= npolys) return;
    const farm_raster_hdr H = S.hdr[p];
    const int n = H.dimx * H.dimy;
    const uint32_t *pof = S.pixoff + H.pixoff_start;
    const uint2 *sq = S.seqs + H.seq_start;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        uint32_t c = 0;
        if (show(S.status[H.pix_start + i]) == 1)
            for (uint32_t s = pof[i]; s < pof[i + 1]; s++) c += sq[s].y;
        out[H.pix_start + i] = c;
    }
}

__global__ __launch_bounds__(256) void k_finalize(const uint32_t *__restrict__ result,
                                                   const IsxDesc *__restrict__ desc,
                                                   unsigned long long *__restrict__ ctr,
                                                   unsigned long long *__restrict__ shards) {
    __shared__ uint32_t lds[4];
    const uint64_t n = desc->n;
    uint8_t *out = desc->out;
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        // what the earlier kernels counted
        for (int s = 0; s < kCtrSlots; s++) {
            const unsigned long long v = fold_shards(shards, s, threadIdx.x, false);
            if (threadIdx.x == 0 && v) atomicAdd(&ctr[s], v);
        }
    }
    uint32_t f = 0;  // a block's part of at most 2^31 pairs
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t r = result[i] ? 1u : 0u;
        if (out) out[i] = (uint8_t)r;
        f += r;
    }
    f = block_sum256(f, lds);
    if (threadIdx.x == 0 && f) atomicAdd(&ctr[kCtrFound], (unsigned long long)f);
}

#define FARM_TILES_INST(EE)                                                                                    \
    template __global__ void k_tiles<EE>(const PixPair *, const uint32_t *, const unsigned long long *,          \
                                         unsigned long long *, uint64_t, uint32_t *);
#define FARM_REFINE_INST(EE, CC, PP)                                                                           \
    template __global__ void k_refine<EE, CC, PP>(DevSet, const uint32_t *, const uint32_t *, const IsxDesc *,  \
                                                  const TileDesc *, uint64_t, uint64_t, uint32_t *, uint32_t *, \
                                                  const unsigned long long *, unsigned long long *);
#define FARM_REFINE_INSTS(EE)     \
    FARM_REFINE_INST(EE, 8, true)  \
    FARM_REFINE_INST(EE, 16, true) \
    FARM_REFINE_INST(EE, 32, true) \
    FARM_REFINE_INST(EE, 8, false) \
    FARM_REFINE_INST(EE, 16, false) \
    FARM_REFINE_INST(EE, 32, false)
FARM_TILES_INST(1)
FARM_TILES_INST(2)
FARM_TILES_INST(4)
FARM_TILES_INST(8)
FARM_REFINE_INSTS(1)
FARM_REFINE_INSTS(2)
FARM_REFINE_INSTS(4)
FARM_REFINE_INSTS(8)
#undef FARM_REFINE_INSTS
#undef FARM_TILES_INST
#undef FARM_REFINE_INST

}  // namespace farm

// The learned part: pair features and an 80-128-128-2 MLP (intersect logit,
// log refinement cost) trained and evaluated on the GPU.
//
// The products run on MFMA (v_mfma_f32_16x16x16_bf16): operands are rounded
// to bf16 when staged (round to nearest even), products accumulate in fp32.
// Inference is one kernel (k_mlp_infer); a training step is three: k_mlp_rows
// (forward and backward of 32 rows at a time), k_mlp_wgrad (the sums over the
// rows: weight and bias gradients, the loss) and k_mlp_step (Adam).  The reference has no learned component; the features come from the
// same raster windows as the filter (Ideal::intersect, Ideal.cpp:1329-1357).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "handle.h"

namespace farm {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ short f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even (inputs are finite)
    return (short)(u >> 16);
}

// ------------------------------------------------------------------------
// Pair features (one lane per candidate pair).  decided: 1 = an IN pixel
// overlap (the exact answer is true), 0 = no BORDER x BORDER pixel pair and
// no IN overlap (the exact answer is false), -1 = needs refinement.
// ------------------------------------------------------------------------
__global__ __launch_bounds__(128) void k_features(DevSet S, const uint32_t *__restrict__ pa_ids,
                                                   const uint32_t *__restrict__ pb_ids, uint32_t n,
                                                   float *__restrict__ feat, int8_t *__restrict__ decided) {
    __shared__ uint32_t hist_all[128][64];  // 32 KB: per-lane 32-bit bins (no wrap on huge pairs)
    uint32_t *hist = hist_all[threadIdx.x];
    for (int i = 0; i < 64; i++) hist[i] = 0;
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const farm_raster_hdr A = S.hdr[pa_ids[k]];
    const farm_raster_hdr B = S.hdr[pb_ids[k]];
    const uint8_t *sa = S.status + A.pix_start;
    const uint8_t *sb = S.status + B.pix_start;
    const uint32_t *ea = S.pixedges + A.pix_start;
    const uint32_t *eb = S.pixedges + B.pix_start;
    const Window wa = window_of(A, B.mbr[0], B.mbr[1], B.mbr[2], B.mbr[3]);
    const double area_a = A.step[0] * A.step[1], area_b = B.step[0] * B.step[1];
    const double amax = fmax(area_a, area_b);
    uint32_t n_in = 0, n_bb = 0, wa_border = 0, wa_in = 0, wa_total = 0;
    double sum_cost = 0, sum_ea = 0, sum_eb = 0, max_prob = 0, sum_prob = 0;
    for (int x = wa.x0; x <= wa.x1; x++) {
        for (int y = wa.y0; y <= wa.y1; y++) {
            const int pa = y * A.dimx + x;
            const uint8_t fa = sa[pa];
            const int st_a = show(fa);
            wa_total++;
            if (st_a == 0) continue;
            if (st_a == 1) wa_border++;
            else wa_in++;
            double lx, ly, hx, hy;
            pixel_box(A, x, y, lx, ly, hx, hy);
            const Window wb = window_of(B, lx, ly, hx, hy);
            for (int u = wb.x0; u <= wb.x1; u++)
                for (int v = wb.y0; v <= wb.y1; v++) {
                    const int pb = v * B.dimx + u;
                    const uint8_t fb = sb[pb];
                    const int st_b = show(fb);
                    if (st_b == 0) continue;
                    if (st_a == 2 || st_b == 2) {
                        n_in++;
                        continue;
                    }
                    n_bb++;
                    const double xa = apx_area_cc(S.fill[A.pix_start + pa], area_a, S.cc);
                    const double xb = apx_area_cc(S.fill[B.pix_start + pb], area_b, S.cc);
                    const double prob = (xa + xb) / amax;
                    max_prob = fmax(max_prob, prob);
                    sum_prob += prob;
                    const double p = (xa / area_a) * (xb / area_b);
                    hist[min(63, (int)(p * 64.0))]++;
                    sum_cost += (double)ea[pa] * (double)eb[pb];
                    sum_ea += ea[pa];
                    sum_eb += eb[pb];
                }
        }
    }
    float *f = feat + (size_t)k * kNFeat;
    const float inv = n_bb ? 1.0f / n_bb : 0.f;
    for (int i = 0; i < 64; i++) f[i] = hist[i] * inv;
    const double ix = fmax(0.0, fmin(A.mbr[2], B.mbr[2]) - fmax(A.mbr[0], B.mbr[0]));
    const double iy = fmax(0.0, fmin(A.mbr[3], B.mbr[3]) - fmax(A.mbr[1], B.mbr[1]));
    const double ma = (A.mbr[2] - A.mbr[0]) * (A.mbr[3] - A.mbr[1]);
    const double mb = (B.mbr[2] - B.mbr[0]) * (B.mbr[3] - B.mbr[1]);
    f[64] = log1pf((float)n_in);
    f[65] = log1pf((float)n_bb);
    f[66] = log1pf((float)A.nverts);
    f[67] = log1pf((float)B.nverts);
    f[68] = (float)(ix * iy / fmax(fmin(ma, mb), 1e-30));
    f[69] = (float)log1p(sum_cost);
    f[70] = (float)max_prob;
    f[71] = n_bb ? (float)(sum_prob / n_bb) : 0.f;
    f[72] = (float)log1p(sum_ea);
    f[73] = (float)log1p(sum_eb);
    f[74] = (float)log(area_a / area_b);
    f[75] = wa_total ? (float)wa_border / wa_total : 0.f;
    f[76] = wa_total ? (float)wa_in / wa_total : 0.f;
    f[77] = f[78] = f[79] = 0.f;
    decided[k] = n_in ? 1 : (n_bb ? -1 : 0);
}

// ------------------------------------------------------------------------
// Inference in one pass: normalisation and the three layers of 64 pairs at a
// time, the weights staged in LDS once per workgroup, the activations never
// leaving it.  norm may be null (rows that are normalised already).  Every
// output takes one MFMA sequence over K (16 at a time, ascending).
// MFMA 16x16x16 operand layout (lane l): A row l%16, k 4*(l/16)+j;
// B col l%16, k 4*(l/16)+j; D row 4*(l/16)+j, col l%16.
// Wave w owns rows 16w .. 16w + 15 of the tile.
// ------------------------------------------------------------------------
constexpr int kInferRows = 64;

template <int K, bool RELU>
__device__ __forceinline__ void infer_layer(const short (*A)[K], const short (*B)[kHidden], const float *bias,
                                            short (*H)[kHidden], int w, int l) {
    f32x4 acc[kHidden / 16];
#pragma unroll
    for (int tt = 0; tt < kHidden / 16; tt++) acc[tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int ar = 16 * w + (l & 15), ak = 4 * (l >> 4);
#pragma unroll
    for (int k0 = 0; k0 < K; k0 += 16) {
        bf16x4 a;
#pragma unroll
        for (int j = 0; j < 4; j++) a[j] = A[ar][k0 + ak + j];
#pragma unroll
        for (int tt = 0; tt < kHidden / 16; tt++) {
            bf16x4 b;
#pragma unroll
            for (int j = 0; j < 4; j++) b[j] = B[k0 + ak + j][16 * tt + (l & 15)];
            acc[tt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[tt], 0, 0, 0);
        }
    }
#pragma unroll
    for (int tt = 0; tt < kHidden / 16; tt++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int col = 16 * tt + (l & 15);
            float v = acc[tt][j] + bias[col];
            if (RELU) v = fmaxf(v, 0.f);
            H[16 * w + 4 * (l >> 4) + j][col] = f2bf(v);
        }
}

__global__ __launch_bounds__(256) void k_mlp_infer(const float *__restrict__ feat, const float *__restrict__ norm,
                                                    const float *__restrict__ W, uint64_t n,
                                                    float *__restrict__ pred) {
    __shared__ short sW1[kNFeat][kHidden];
    __shared__ short sW2[kHidden][kHidden];
    __shared__ short sW3[kHidden][16];  // columns >= kOut are zero
    __shared__ float sb[2 * kHidden + kOut];
    __shared__ short sX[kInferRows][kNFeat];
    __shared__ short sH1[kInferRows][kHidden];
    __shared__ short sH2[kInferRows][kHidden];
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    for (int i = t; i < kNFeat * kHidden; i += 256) sW1[i / kHidden][i % kHidden] = f2bf(W[kOffW1 + i]);
    for (int i = t; i < kHidden * kHidden; i += 256) sW2[i / kHidden][i % kHidden] = f2bf(W[kOffW2 + i]);
    for (int i = t; i < kHidden * 16; i += 256) {
        const int k = i / 16, c = i % 16;
        sW3[k][c] = c < kOut ? f2bf(W[kOffW3 + k * kOut + c]) : (short)0;
    }
    for (int i = t; i < kHidden; i += 256) {
        sb[i] = W[kOffB1 + i];
        sb[kHidden + i] = W[kOffB2 + i];
    }
    if (t < kOut) sb[2 * kHidden + t] = W[kOffB3 + t];
    __syncthreads();
    for (uint64_t r0 = (uint64_t)blockIdx.x * kInferRows; r0 < n; r0 += (uint64_t)gridDim.x * kInferRows) {
        for (int i = t; i < kInferRows * kNFeat; i += 256) {
            const int r = i / kNFeat, c = i % kNFeat;
            float v = 0.f;
            if (r0 + r < n) {
                v = feat[(r0 + r) * kNFeat + c];
                if (norm) v = (v - norm[c]) * norm[kNFeat + c];
            }
            sX[r][c] = f2bf(v);
        }
        __syncthreads();
        infer_layer<kNFeat, true>(sX, sW1, sb, sH1, w, l);
        __syncthreads();
        infer_layer<kHidden, true>(sH1, sW2, sb + kHidden, sH2, w, l);
        __syncthreads();
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        const int ar = 16 * w + (l & 15), ak = 4 * (l >> 4);
#pragma unroll
        for (int k0 = 0; k0 < kHidden; k0 += 16) {
            bf16x4 a, b;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                a[j] = sH2[ar][k0 + ak + j];
                b[j] = sW3[k0 + ak + j][l & 15];
            }
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
        }
        const int col = l & 15;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint64_t row = r0 + 16 * w + 4 * (l >> 4) + j;
            if (col < kOut && row < n) pred[2 * row + col] = acc[j] + sb[2 * kHidden + col];
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------
// Training.  loss = mean(BCE-with-logits(z0, y)) + lambda * mean((z1 - c)^2).
//
// Three kernels a step.  k_mlp_rows takes 32 rows a workgroup through the
// forward pass and back: the operands of the next product row-major in LDS as
// bf16, padded so that a wave's 8-byte fragment reads fall two to a bank; the
// weights as bf16 from L2, in the layout each product reads with one 8-byte
// load per fragment (MlpPacked).  Every activation and dL/dactivation leaves
// it transposed, ready to be an operand of a weight gradient, whose inner
// dimension is the rows (MlpAct).  k_mlp_wgrad sums over the rows: a wave per
// 16 x 16 tile of a weight gradient and chunk of about 1,024 rows, one MFMA
// chain in row order; a workgroup per bias; the loss.  k_mlp_step adds the
// chunks up and applies Adam.
//
// The orders of these sums are part of the result: a last bit of dL/dh turns a
// bf16 rounding, Adam's division amplifies it, and a run's weights then differ
// by 1e-3 in norm.  So a step's sums do not depend on how its rows are spread
// over the chip: chunks of the rows as grad_chunk() cuts them, and within one
// 16 rows an MFMA in ascending order.  (Gradients kept per workgroup gave
// other weights and were no faster.)
//
// A step of 2,048 rows is bound by latency: a chain of five dependent products
// for 64 workgroups (16.3 us), then one of 64 MFMAs a wave (8.0 us; 10.2 with
// 8 blocks' loads in flight instead of 32), then Adam (5 us).  65,536 rows in
// batches of 2,048, two epochs: 2.85 ms, as with gradients per workgroup.
// ------------------------------------------------------------------------
constexpr int kGradRows = 32;
constexpr int kGradParts = 256;  // most chunks whose sums are kept apart

// What k_mlp_rows leaves for k_mlp_wgrad, M rows padded to Mp (a multiple of
// kGradRows).  xt .. dzt: bf16, in blocks of 16 rows, [block][column][row], so
// that a fragment (4 rows of a column) is one 8-byte load and a wave's 64
// fragments are 512 consecutive bytes; rows past M are 0.  f2, f1, fz:
// dL/d(layer output) before its rounding to bf16, z: the logits, [column][row].
struct MlpAct {
    short *xt, *h1t, *h2t, *d2t, *d1t, *dzt;
    float *f2, *f1, *fz, *z;
    size_t Mp;
};
constexpr uint64_t kActBytesPerRow = 2ull * (kNFeat + 4 * kHidden + kOut) + 4ull * (2 * kHidden + 2 * kOut);

// bf16 copies of the weights: W1^T, W2^T, W2, W3^T (16 rows, 2 used), W3
struct MlpPacked {
    short w1t[kHidden * kNFeat];
    short w2t[kHidden * kHidden];
    short w2[kHidden * kHidden];
    short w3t[16 * kHidden];
    short w3[kHidden * kOut];
};

// parameter i's copies
__device__ __forceinline__ void pack_param(MlpPacked *__restrict__ P, int i, float v) {
    const short b = f2bf(v);
    if (i < kOffB1) {
        P->w1t[(i % kHidden) * kNFeat + i / kHidden] = b;
    } else if (i >= kOffW2 && i < kOffB2) {
        const int k = (i - kOffW2) / kHidden, n = (i - kOffW2) % kHidden;
        P->w2t[n * kHidden + k] = b;
        P->w2[k * kHidden + n] = b;
    } else if (i >= kOffW3 && i < kOffB3) {
        const int k = (i - kOffW3) / kOut, o = (i - kOffW3) % kOut;
        P->w3t[o * kHidden + k] = b;
        P->w3[k * kOut + o] = b;
    }
}

__global__ __launch_bounds__(256) void k_mlp_pack(const float *__restrict__ W, MlpPacked *__restrict__ P) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kNParams) pack_param(P, i, W[i]);
    if (i < (16 - kOut) * kHidden) P->w3t[kOut * kHidden + i] = 0;
}

__device__ __forceinline__ bf16x4 frag(const short *p) { return *reinterpret_cast<const bf16x4 *>(p); }
__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// One layer's product for this wave: both 16-row tiles x its two 16-column
// tiles 2w, 2w + 1; A row-major in LDS (stride SA), B column-major in memory.
template <int K, int SA>
__device__ __forceinline__ void tile_product(const short *A, const short *__restrict__ B, int w, int l,
                                             f32x4 (&acc)[2][2]) {
    const int c = l & 15, q = 4 * (l >> 4);
    bf16x4 b[2][K / 16];
#pragma unroll
    for (int n = 0; n < 2; n++)
#pragma unroll
        for (int k = 0; k < K / 16; k++) b[n][k] = frag(B + (16 * (2 * w + n) + c) * K + 16 * k + q);
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int n = 0; n < 2; n++) acc[m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < K / 16; k++)
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const bf16x4 a = frag(A + (16 * m + c) * SA + 16 * k + q);
#pragma unroll
            for (int n = 0; n < 2; n++) acc[m][n] = mfma(a, b[n][k], acc[m][n]);
        }
}

// rows: the rows' indices into X, y and c (null: rows 0 .. M - 1).
__global__ __launch_bounds__(256) void k_mlp_rows(const float *__restrict__ X, const uint32_t *__restrict__ rows,
                                                   const float *__restrict__ y, const float *__restrict__ cst, int M,
                                                   float lambda, const float *__restrict__ W,
                                                   const MlpPacked *__restrict__ P, MlpAct act) {
    constexpr int SX = kNFeat + 8, SH = kHidden + 8;
    __shared__ __align__(16) short sX[kGradRows * SX], sH1[kGradRows * SH], sH2[kGradRows * SH], sD2[kGradRows * SH];
    __shared__ __align__(16) short sDz[kGradRows * 4];
    __shared__ uint32_t sRow[kGradRows];
    const int t = threadIdx.x, w = t >> 6, l = t & 63, c = l & 15, q = 4 * (l >> 4);
    const int r0 = blockIdx.x * kGradRows;
    const bf16x4 zero = {0, 0, 0, 0};
    if (t < kGradRows) sRow[t] = r0 + t < M ? (rows ? rows[r0 + t] : (uint32_t)(r0 + t)) : 0xffffffffu;
    __syncthreads();
    for (int i = t; i < kGradRows * (kNFeat / 4); i += 256) {
        const int r = i / (kNFeat / 4), k = 4 * (i % (kNFeat / 4));
        const uint32_t src = sRow[r];
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (src != 0xffffffffu) v = *reinterpret_cast<const float4 *>(X + (size_t)src * kNFeat + k);
        *reinterpret_cast<bf16x4 *>(sX + r * SX + k) = bf16x4{f2bf(v.x), f2bf(v.y), f2bf(v.z), f2bf(v.w)};
    }
    __syncthreads();
    // fragment f of ncol columns: rows 16 m + q .. + 3 of this lane's column
    auto at = [&](short *T, int ncol, int m, int col, int rq) {
        return reinterpret_cast<bf16x4 *>(T + (((size_t)2 * blockIdx.x + m) * ncol + col) * 16 + rq);
    };
    for (int i = t; i < 2 * kNFeat * 4; i += 256) {
        const int rq = 4 * (i & 3), col = (i >> 2) % kNFeat, m = (i >> 2) / kNFeat;
        bf16x4 b;
#pragma unroll
        for (int j = 0; j < 4; j++) b[j] = sX[(16 * m + rq + j) * SX + col];
        *at(act.xt, kNFeat, m, col, rq) = b;
    }
    // this wave's tile of a layer's output, staged for the next product (R) and
    // for the weight gradients (T; rows past M as 0)
    auto put = [&](const f32x4 v, int m, int n, short *R, short *T) {
        const int col = 16 * (2 * w + n) + c;
        bf16x4 b;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            b[j] = f2bf(v[j]);
            if (R) R[(16 * m + q + j) * SH + col] = b[j];
            if (r0 + 16 * m + q + j >= M) b[j] = 0;
        }
        *at(T, kHidden, m, col, q) = b;
    };
    f32x4 h1[2][2], h2[2][2], d[2][2];
    auto relu_layer = [&](f32x4(&h)[2][2], const float *bias, short *R, short *T) {
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int n = 0; n < 2; n++) {
                const float b = bias[16 * (2 * w + n) + c];
#pragma unroll
                for (int j = 0; j < 4; j++) h[m][n][j] = fmaxf(h[m][n][j] + b, 0.f);
                put(h[m][n], m, n, R, T);
            }
    };
    tile_product<kNFeat, SX>(sX, P->w1t, w, l, h1);
    relu_layer(h1, W + kOffB1, sH1, act.h1t);
    __syncthreads();
    tile_product<kHidden, SH>(sH1, P->w2t, w, l, h2);
    relu_layer(h2, W + kOffB2, sH2, act.h2t);
    __syncthreads();
    if (w < 2) {
        // logits of rows 16w ..: lane column 0 the logit, 1 the cost
        f32x4 z = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < kHidden / 16; k++)
            z = mfma(frag(sH2 + (16 * w + c) * SH + 16 * k + q), frag(P->w3t + c * kHidden + 16 * k + q), z);
        bf16x4 dz = zero;
        if (c < kOut) {
            f32x4 g = f32x4{0.f, 0.f, 0.f, 0.f};
            const float b = W[kOffB3 + c];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                z[j] += b;
                const uint32_t src = sRow[16 * w + q + j];
                if (src == 0xffffffffu) continue;
                if (c == 0) {
                    const float s = 1.f / (1.f + expf(-z[j]));
                    g[j] = (s - y[src]) / M;
                } else {
                    g[j] = 2.f * lambda * (z[j] - cst[src]) / M;
                }
                dz[j] = f2bf(g[j]);
            }
            const size_t o = (size_t)c * act.Mp + r0 + 16 * w + q;
            *reinterpret_cast<f32x4 *>(act.z + o) = z;
            *reinterpret_cast<f32x4 *>(act.fz + o) = g;
            *at(act.dzt, kOut, w, c, q) = dz;
        }
        if (c < 4)
#pragma unroll
            for (int j = 0; j < 4; j++) sDz[(16 * w + q + j) * 4 + c] = dz[j];
    }
    __syncthreads();
    // dL/dh2 = dz W3^T (two inner terms, the rest of the 16 zero), masked
#pragma unroll
    for (int n = 0; n < 2; n++) {
        const int col = 16 * (2 * w + n) + c;
        bf16x4 b = zero;
        if (q == 0) {
            const short *p = P->w3 + col * kOut;
            b[0] = p[0];
            b[1] = p[1];
        }
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const bf16x4 a = q == 0 ? frag(sDz + (16 * m + c) * 4) : zero;
            f32x4 v = mfma(a, b, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = h2[m][n][j] > 0.f ? v[j] : 0.f;
            *reinterpret_cast<f32x4 *>(act.f2 + (size_t)col * act.Mp + r0 + 16 * m + q) = v;
            put(v, m, n, sD2, act.d2t);
        }
    }
    __syncthreads();
    tile_product<kHidden, SH>(sD2, P->w2, w, l, d);
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int n = 0; n < 2; n++) {
            const int col = 16 * (2 * w + n) + c;
#pragma unroll
            for (int j = 0; j < 4; j++) d[m][n][j] = h1[m][n][j] > 0.f ? d[m][n][j] : 0.f;
            *reinterpret_cast<f32x4 *>(act.f1 + (size_t)col * act.Mp + r0 + 16 * m + q) = d[m][n];
            put(d[m][n], m, n, nullptr, act.d1t);
        }
}

// Weight gradient tiles of 16 x 16: 5 x 8 of W1, 8 x 8 of W2, 8 x 1 of W3.
constexpr int kTilesW1 = (kNFeat / 16) * (kHidden / 16), kTilesW2 = (kHidden / 16) * (kHidden / 16),
              kGradTiles = kTilesW1 + kTilesW2 + kHidden / 16;
constexpr int kBiases = 2 * kHidden + kOut;

// Workgroups [0, gw): the weight gradients, a wave per tile and part p of np,
// which takes the row chunks p, p + np, ..; [gw, gw + kBiases): a bias each;
// the rest: 256 rows' losses, one sum per wave.
__global__ __launch_bounds__(256) void k_mlp_wgrad(MlpAct act, const uint32_t *__restrict__ rows,
                                                    const float *__restrict__ y, const float *__restrict__ cst, int M,
                                                    float lambda, int chunk, int np, int gw, float *__restrict__ part,
                                                    float *__restrict__ loss_part) {
    const int t = threadIdx.x, w = t >> 6, l = t & 63, c = l & 15, q = 4 * (l >> 4);
    const int b = blockIdx.x;
    if (b < gw) {
        const int task = 4 * b + w, tile = task % kGradTiles, p = task / kGradTiles;
        if (p >= np) return;
        // operands and output of this tile
        const short *A, *B;
        int na, nb, mt, nt, off, ld;
        if (tile < kTilesW1) {
            A = act.xt, B = act.d1t, na = kNFeat, nb = kHidden, off = kOffW1, ld = kHidden;
            mt = tile / (kHidden / 16), nt = tile % (kHidden / 16);
        } else if (tile < kTilesW1 + kTilesW2) {
            A = act.h1t, B = act.d2t, na = nb = kHidden, off = kOffW2, ld = kHidden;
            mt = (tile - kTilesW1) / (kHidden / 16), nt = (tile - kTilesW1) % (kHidden / 16);
        } else {
            A = act.h2t, B = act.dzt, na = kHidden, nb = kOut, off = kOffW3, ld = kOut;
            mt = tile - kTilesW1 - kTilesW2, nt = 0;
        }
        const bool col = 16 * nt + c < nb;  // W3 has 2 of the 16 columns
        const bf16x4 zero = {0, 0, 0, 0};
        A += (size_t)(16 * mt + c) * 16 + q;
        B += col ? (size_t)(16 * nt + c) * 16 + q : 0;
        f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int k0 = p * chunk; k0 < M; k0 += np * chunk) {
            const int rb1 = (min(M, k0 + chunk) + 15) / 16;
            f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
            // (32 blocks' loads together, then their products in turn)
            for (int rb = k0 / 16; rb < rb1; rb += 32) {
                bf16x4 fa[32], fb[32];
#pragma unroll
                for (int u = 0; u < 32; u++) {
                    const size_t r = min(rb + u, rb1 - 1);
                    fa[u] = frag(A + r * na * 16);
                    fb[u] = frag(B + r * nb * 16);
                }
#pragma unroll
                for (int u = 0; u < 32; u++)
                    if (rb + u < rb1) acc = mfma(fa[u], col ? fb[u] : zero, acc);
            }
            sum += acc;
        }
        if (!col) return;
        float *G = part + (size_t)p * kNParams + off;
#pragma unroll
        for (int j = 0; j < 4; j++) G[(16 * mt + q + j) * ld + 16 * nt + c] = sum[j];
        return;
    }
    if (b < gw + kBiases) {
        // the column's sum in f32: rows t, t + 256, .. a lane
        __shared__ float sum[4];
        const int k = b - gw;
        const float *f;
        int i;
        if (k < kHidden) f = act.f1 + (size_t)k * act.Mp, i = kOffB1 + k;
        else if (k < 2 * kHidden) f = act.f2 + (size_t)(k - kHidden) * act.Mp, i = kOffB2 + k - kHidden;
        else f = act.fz + (size_t)(k - 2 * kHidden) * act.Mp, i = kOffB3 + k - 2 * kHidden;
        float s = 0.f;
#pragma unroll 8
        for (int64_t r = t; r < M; r += 256) s += f[r];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (l == 0) sum[w] = s;
        __syncthreads();
        if (t == 0) part[i] = sum[0] + sum[1] + sum[2] + sum[3];
        return;
    }
    const int g = b - gw - kBiases, r = 256 * g + t;
    float L = 0.f;
    if (r < M) {
        const uint32_t src = rows ? rows[r] : (uint32_t)r;
        const float z0 = act.z[r], e = act.z[act.Mp + r] - cst[src];
        L = (fmaxf(z0, 0.f) - z0 * y[src] + log1pf(expf(-fabsf(z0)))) / M + lambda * e * e / M;
    }
    for (int o = 32; o > 0; o >>= 1) L += __shfl_xor(L, o);
    if (l == 0) loss_part[4 * g + w] = L;
}

// The step's gradients (the chunks' parts, summed in order) into g when given,
// and Adam on w and its bf16 copies when adam != 0; the loss, the sum of nloss
// parts, to *loss.
__global__ __launch_bounds__(256) void k_mlp_step(const float *__restrict__ part, const float *__restrict__ loss_part,
                                                   int np, int nloss, float *__restrict__ g, float *__restrict__ loss,
                                                   int adam, float *__restrict__ w, MlpPacked *__restrict__ P,
                                                   float *__restrict__ m, float *__restrict__ v, float lr, float b1,
                                                   float b2, float eps, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        float L = 0.f;
        for (int k = threadIdx.x; k < nloss; k += 64) L += loss_part[k];
        for (int o = 32; o > 0; o >>= 1) L += __shfl_xor(L, o);
        if (threadIdx.x == 0) *loss = L;
    }
    if (i >= kNParams) return;
    // (a bias is one sum over all rows, in the first part)
    const bool bias = (i >= kOffB1 && i < kOffW2) || (i >= kOffB2 && i < kOffW3) || i >= kOffB3;
    float gi = 0.f;
#pragma unroll 8
    for (int k = 0; k < (bias ? 1 : np); k++) gi += part[(size_t)k * kNParams + i];
    if (g) g[i] = gi;
    if (!adam) return;
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    pack_param(P, i, wi);
}

}  // namespace farm

using namespace farm;

namespace {

// Rows of a chunk of the weight gradients: M / (M / 1024) of them, to a whole
// number of 16.
int grad_chunk(int M) {
    const int n = std::max(1, M / 1024);
    return ((M + n - 1) / n + 15) / 16 * 16;
}
int grad_parts(int M) {
    const int chunk = grad_chunk(M);
    return std::min((M + chunk - 1) / chunk, kGradParts);
}
uint64_t grad_rows(int M) { return ((uint64_t)M + kGradRows - 1) / kGradRows * kGradRows; }
int loss_blocks(int M) { return (M + 255) / 256; }

int grad_buffers(farm_handle h, int M, uint64_t losses) {
    int rc;
    if ((rc = ensure(h, h->mlp_act, kActBytesPerRow * grad_rows(M)))) return rc;
    if ((rc = ensure(h, h->mlp_part, 4ull * kNParams * grad_parts(M)))) return rc;
    if ((rc = ensure(h, h->mlp_lpart, 16ull * loss_blocks(M)))) return rc;
    return ensure(h, h->mlp_loss, 4ull * losses);
}

// the arrays of M rows in mlp_act (Mp is a multiple of 32: each is aligned to 64 bytes)
MlpAct carve_act(farm_handle h, int M) {
    MlpAct a;
    const size_t Mp = a.Mp = grad_rows(M);
    float *f = P<float>(h->mlp_act);
    auto floats = [&](int ncol) {
        float *p = f;
        f += Mp * ncol;
        return p;
    };
    a.f2 = floats(kHidden);
    a.f1 = floats(kHidden);
    a.fz = floats(kOut);
    a.z = floats(kOut);
    short *s = reinterpret_cast<short *>(f);
    auto shorts = [&](int ncol) {
        short *p = s;
        s += Mp * ncol;
        return p;
    };
    a.xt = shorts(kNFeat);
    a.h1t = shorts(kHidden);
    a.h2t = shorts(kHidden);
    a.d2t = shorts(kHidden);
    a.d1t = shorts(kHidden);
    a.dzt = shorts(kOut);
    return a;
}

// loss (to mlp_loss[slot]) and gradients of M rows of X, y, c (device; rows:
// their indices, or null), then Adam (step adam_t) or the gradients to mlp_g
int mlp_step(farm_handle h, const float *X, const uint32_t *rows, const float *y, const float *c, int M, float lambda,
             uint64_t slot, bool adam, float lr) {
    const MlpAct act = carve_act(h, M);
    const int np = grad_parts(M), gw = (np * kGradTiles + 3) / 4, gl = loss_blocks(M);
    hipLaunchKernelGGL(k_mlp_rows, dim3((unsigned)(act.Mp / kGradRows)), dim3(256), 0, h->stream, X, rows, y, c, M,
                       lambda, (const float *)P<float>(h->mlp_w), (const MlpPacked *)P<MlpPacked>(h->mlp_wb), act);
    HIPCHK(h, hipGetLastError());
    hipLaunchKernelGGL(k_mlp_wgrad, dim3(gw + kBiases + gl), dim3(256), 0, h->stream, act, rows, y, c, M, lambda,
                       grad_chunk(M), np, gw, P<float>(h->mlp_part), P<float>(h->mlp_lpart));
    HIPCHK(h, hipGetLastError());
    const float c1 = 1.f - powf(0.9f, (float)h->adam_t), c2 = 1.f - powf(0.999f, (float)h->adam_t);
    hipLaunchKernelGGL(k_mlp_step, dim3(blocks_for(kNParams)), dim3(256), 0, h->stream,
                       (const float *)P<float>(h->mlp_part), (const float *)P<float>(h->mlp_lpart), np, 4 * gl,
                       adam ? (float *)nullptr : P<float>(h->mlp_g), P<float>(h->mlp_loss) + slot, adam ? 1 : 0,
                       P<float>(h->mlp_w), P<MlpPacked>(h->mlp_wb), P<float>(h->mlp_m), P<float>(h->mlp_v), lr, 0.9f,
                       0.999f, 1e-8f, c1, c2);
    HIPCHK(h, hipGetLastError());
    return FARM_OK;
}

// the three layers of n rows of X (device, normalised unless norm is given)
int mlp_infer(farm_handle h, const float *X, const float *norm, uint64_t n, float *out) {
    const unsigned grid = (unsigned)std::min<uint64_t>((n + kInferRows - 1) / kInferRows, 2ull * h->num_cus);
    hipLaunchKernelGGL(k_mlp_infer, dim3(grid), dim3(256), 0, h->stream, X, norm, (const float *)P<float>(h->mlp_w), n,
                       out);
    HIPCHK(h, hipGetLastError());
    return FARM_OK;
}

int require_mlp(farm_handle h) {
    if (!h) return FARM_EINVAL;
    if (!h->mlp_ready) return fail(h, FARM_ESTATE, "MLP parameters not set (farm_mlp_set_params)");
    return FARM_OK;
}

}  // namespace

extern "C" {

int farm_mlp_set_params(farm_handle h, const float *params, uint64_t n, const float *norm) {
    if (!h || !params || n != (uint64_t)kNParams)
        return fail(h, FARM_EINVAL, "expected %d parameters", kNParams);
    HIPCHK(h, hipSetDevice(h->device));
    int rc;
    if ((rc = upload(h, h->mlp_w, params, 4ull * kNParams))) return rc;
    if ((rc = ensure(h, h->mlp_m, 4ull * kNParams))) return rc;
    if ((rc = ensure(h, h->mlp_v, 4ull * kNParams))) return rc;
    if ((rc = ensure(h, h->mlp_g, 4ull * kNParams))) return rc;
    if ((rc = ensure(h, h->mlp_wb, sizeof(MlpPacked)))) return rc;
    hipLaunchKernelGGL(k_mlp_pack, dim3(blocks_for(kNParams)), dim3(256), 0, h->stream,
                       (const float *)P<float>(h->mlp_w), P<MlpPacked>(h->mlp_wb));
    HIPCHK(h, hipGetLastError());
    if ((rc = fill_u32(h, h->mlp_m.p, kNParams, 0))) return rc;
    if ((rc = fill_u32(h, h->mlp_v.p, kNParams, 0))) return rc;
    std::vector<float> nm(2 * kNFeat);
    for (int i = 0; i < kNFeat; i++) {
        nm[i] = norm ? norm[i] : 0.f;
        nm[kNFeat + i] = norm ? norm[kNFeat + i] : 1.f;
    }
    if ((rc = upload(h, h->mlp_norm, nm.data(), 4ull * nm.size()))) return rc;
    HIPCHK(h, hipStreamSynchronize(h->stream));
    h->adam_t = 0;
    h->mlp_ready = true;
    return FARM_OK;
}

int farm_mlp_get_params(farm_handle h, float *params, uint64_t n) {
    int rc = require_mlp(h);
    if (rc) return rc;
    if (n != (uint64_t)kNParams) return fail(h, FARM_EINVAL, "expected %d parameters", kNParams);
    HIPCHK(h, hipMemcpy(params, h->mlp_w.p, 4ull * kNParams, hipMemcpyDeviceToHost));
    return FARM_OK;
}

int farm_mlp_forward(farm_handle h, const float *X, uint64_t n, float *out) {
    int rc = require_mlp(h);
    if (rc) return rc;
    HIPCHK(h, hipSetDevice(h->device));
    const int chunk = 1 << 16;
    for (uint64_t s = 0; s < n; s += chunk) {
        const int M = (int)std::min<uint64_t>(chunk, n - s);
        if ((rc = ensure(h, h->mlp_z3, 4ull * M * kOut))) return rc;
        if ((rc = upload(h, h->mlp_x, X + s * kNFeat, 4ull * M * kNFeat))) return rc;
        if ((rc = mlp_infer(h, P<float>(h->mlp_x), nullptr, M, P<float>(h->mlp_z3)))) return rc;
        HIPCHK(h, hipMemcpyAsync(out + s * kOut, h->mlp_z3.p, 4ull * M * kOut, hipMemcpyDeviceToHost, h->stream));
        HIPCHK(h, hipStreamSynchronize(h->stream));
    }
    return FARM_OK;
}

int farm_mlp_loss_grad(farm_handle h, const float *X, const float *y, const float *c, uint64_t n, float lambda,
                       float *loss, float *grad) {
    int rc = require_mlp(h);
    if (rc) return rc;
    if (n == 0 || n > (1u << 24)) return fail(h, FARM_EINVAL, "batch of %llu rows", (unsigned long long)n);
    HIPCHK(h, hipSetDevice(h->device));
    const int M = (int)n;
    if ((rc = grad_buffers(h, M, 1))) return rc;
    if ((rc = upload(h, h->mlp_x, X, 4ull * M * kNFeat))) return rc;
    if ((rc = upload(h, h->mlp_y, y, 4ull * M))) return rc;
    if ((rc = upload(h, h->mlp_c, c, 4ull * M))) return rc;
    if ((rc = mlp_step(h, P<float>(h->mlp_x), nullptr, P<float>(h->mlp_y), P<float>(h->mlp_c), M, lambda, 0, false,
                       0.f)))
        return rc;
    if (loss) HIPCHK(h, hipMemcpyAsync(loss, h->mlp_loss.p, 4, hipMemcpyDeviceToHost, h->stream));
    if (grad) HIPCHK(h, hipMemcpyAsync(grad, h->mlp_g.p, 4ull * kNParams, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));
    return FARM_OK;
}

int farm_mlp_train(farm_handle h, const float *X, const float *y, const float *c, uint64_t n, int epochs, int batch,
                   float lr, float lambda, uint64_t seed, float *epoch_loss) {
    int rc = require_mlp(h);
    if (rc) return rc;
    if (n == 0 || batch <= 0 || epochs <= 0) return fail(h, FARM_EINVAL, "bad training arguments");
    HIPCHK(h, hipSetDevice(h->device));
    // batches of an epoch: whole ones only (one short one when n < batch)
    const int M = (int)std::min<uint64_t>((uint64_t)batch, n);
    const uint64_t nb = n / M;
    DevBuf dX, dy, dc, dperm;
    auto cleanup = [&]() {
        (void)hipStreamSynchronize(h->stream);
        free_buf(dX);
        free_buf(dy);
        free_buf(dc);
        free_buf(dperm);
    };
    // two orders in turn: one may still be in transfer while the next is made
    std::vector<uint32_t> perms[2] = {std::vector<uint32_t>(n), std::vector<uint32_t>(n)};
    uint64_t s = seed * 6364136223846793005ull + 1442695040888963407ull;
    auto shuffle = [&](std::vector<uint32_t> &perm) {
        for (uint64_t i = 0; i < n; i++) perm[i] = (uint32_t)i;
        for (uint64_t i = n - 1; i > 0; i--) {  // Fisher-Yates, PCG-style LCG
            s = s * 6364136223846793005ull + 1442695040888963407ull;
            const uint64_t j = (s >> 33) % (i + 1);
            std::swap(perm[i], perm[j]);
        }
    };
    if ((rc = upload(h, dX, X, 4ull * n * kNFeat)) || (rc = upload(h, dy, y, 4ull * n)) ||
        (rc = upload(h, dc, c, 4ull * n)) || (rc = ensure(h, dperm, 4ull * n)) || (rc = grad_buffers(h, M, nb))) {
        cleanup();
        return rc;
    }
    shuffle(perms[0]);
    std::vector<float> losses(nb);
    for (int ep = 0; ep < epochs; ep++) {
        if ((rc = upload(h, dperm, perms[ep & 1].data(), 4ull * n))) {
            cleanup();
            return rc;
        }
        // the epoch's steps are queued without a wait; the next shuffle runs
        // on the host meanwhile
        for (uint64_t b = 0; b < nb; b++) {
            h->adam_t++;
            if ((rc = mlp_step(h, P<float>(dX), P<uint32_t>(dperm) + b * M, P<float>(dy), P<float>(dc), M, lambda, b,
                               true, lr))) {
                cleanup();
                return rc;
            }
        }
        if (ep + 1 < epochs) shuffle(perms[(ep + 1) & 1]);
        hipError_t e = hipMemcpyAsync(losses.data(), h->mlp_loss.p, 4ull * nb, hipMemcpyDeviceToHost, h->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
        if (e != hipSuccess) {
            cleanup();
            return fail(h, FARM_EDEVICE, "training step failed: %s", hipGetErrorString(e));
        }
        double ep_loss = 0;
        for (float L : losses) ep_loss += L;
        if (epoch_loss) epoch_loss[ep] = (float)(ep_loss / nb);
    }
    cleanup();
    return FARM_OK;
}

// features of pairs [begin, end) on the device (normalised copy in h->feat
// when the MLP norm is set); optional host copies of raw features / flags
int farm_pair_features(farm_handle h, uint64_t begin, uint64_t end, float *feat_out, int8_t *decided_out) {
    if (!h) return FARM_EINVAL;
    if (h->npolys <= 0) return fail(h, FARM_ESTATE, "no polygons uploaded");
    if (begin > end || end > h->npairs) return fail(h, FARM_EINVAL, "bad pair window");
    const uint64_t n = end - begin;
    HIPCHK(h, hipSetDevice(h->device));
    int rc;
    if ((rc = ensure(h, h->feat, 4ull * (n ? n : 1) * kNFeat))) return rc;
    if ((rc = ensure(h, h->decided, n ? n : 1))) return rc;
    if (n) {
        hipLaunchKernelGGL(k_features, dim3(blocks_for(n, 128)), dim3(128), 0, h->stream, devset(h),
                           (const uint32_t *)P<uint32_t>(h->pa) + begin, (const uint32_t *)P<uint32_t>(h->pb) + begin,
                           (uint32_t)n, P<float>(h->feat), P<int8_t>(h->decided));
        HIPCHK(h, hipGetLastError());
        if (feat_out)
            HIPCHK(h, hipMemcpyAsync(feat_out, h->feat.p, 4ull * n * kNFeat, hipMemcpyDeviceToHost, h->stream));
        if (decided_out) HIPCHK(h, hipMemcpyAsync(decided_out, h->decided.p, n, hipMemcpyDeviceToHost, h->stream));
    }
    HIPCHK(h, hipStreamSynchronize(h->stream));
    return FARM_OK;
}

// MLP predictions (logit, log-cost) of pairs [begin, end): features, norm,
// forward on the device; results stay in h->pred (2 floats per pair) and are
// copied to `out` when given
int farm_mlp_predict_pairs(farm_handle h, uint64_t begin, uint64_t end, float *out) {
    int rc = require_mlp(h);
    if (rc) return rc;
    if ((rc = farm_pair_features(h, begin, end, nullptr, nullptr))) return rc;
    const uint64_t n = end - begin;
    if ((rc = ensure(h, h->pred, 8ull * (n ? n : 1)))) return rc;
    if (!n) return FARM_OK;
    if ((rc = mlp_infer(h, P<float>(h->feat), P<float>(h->mlp_norm), n, P<float>(h->pred)))) return rc;
    if (out) HIPCHK(h, hipMemcpyAsync(out, h->pred.p, 8ull * n, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(h, hipStreamSynchronize(h->stream));
    return FARM_OK;
}

}  // extern "C"

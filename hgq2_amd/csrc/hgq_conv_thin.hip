// Convolutions of unit stride over few input values per pixel (kh * kw * C <= 31: an image's first layer) on
// v_mfma_f32_32x32x16_bf16 over exact bf16 parts (hgq_device.h).
//
// Such a layer reads and writes a [.., F] tensor and little else, and its contraction fits one 32-deep block.  A workgroup
// takes a band of whole rows of one image; its pixels, counted along the band, are the rows of the products:
//
//   forward    Y[m, f]  = act(sum_k X[m, k] W[k, f] + b[f])       X[m, k] gathered from the input patch in LDS
//   backward   dW[k, f] = sum_m X[m, k] dZ[m, f],  db[f] likewise with a column of ones
//              G[m, k]  = sum_f dZ[m, f] W[k, f],  dx[p, c] = sum of the G of the kh kw pixels and taps that read p
//
// The backward pass does both from one reading of dy (and of the mask): dZ of the band and of the kh - 1 rows above it sits in
// LDS as fp32 words; every wavefront contracts a share of the pixels for dW and a block of 32 pixels for G; G then takes
// dZ's place and each input value adds up its taps.  (An infinity is not the sum of its bf16 parts: a band whose dZ is not
// all finite is contracted on the fp32 instruction.)  A row of dZ is owned (for dW) by one band; the rows above it are
// contracted again for G, which costs a quarter of the matrix work and no memory traffic beyond L2.
//
// 300 x 24 x 24 x 3 onto 40 filters of 3 x 3: backward 30 us with its reduction (47 MB; gathered kernels for the two gradients
// 150 us), forward 11.6 us (implicit GEMM 26 us).  1024 x 28 x 28 x 1 onto 32, behind a pooling: backward 54 us (multiply-adds per
// pixel and filter 57 us; few filters or wide rows are theirs, see thin_bwd_shape).  Bound by vector instructions, 50 for every
// matrix instruction: staging, splitting and the nine taps.
#include "hgq_device.h"
#include "hgq_host.h"

namespace hgq {

#define TH_GS 33      // words per pixel of G
#define THIN_TAIL 24  // pixels behind the input patch that the last batch of sixteen reads: 14 + KK - 1 at most

struct ThinPlan {
    int rows;       // rows of a band: output rows (forward), input rows (backward)
    int bands;      // per image
    int patch;      // LDS words of the largest input patch (backward)
    int xw;         // pixels per patch row: OW + kw - 1
    int64_t tiles;  // B * bands
};

static bool thin_shape(const hgq_conv_geom &g, int F) {
    const int K = g.kh * g.kw * g.C;
    return ((g.kh == 3 && g.kw == 3) || (g.kh == 5 && g.kw == 5)) && K <= 31 && F >= 1 && F <= 64 && g.sy == 1 && g.sx == 1 && g.dly == 1 &&
           g.dlx == 1 && g.py < g.kh && g.px < g.kw && g.OH <= g.H + g.py && g.OW <= g.W + g.px && g.OW + g.kw - 1 >= g.W + g.px && g.OW <= 64 && g.W <= 4096 &&
           (int64_t)g.B * g.OH * g.OW * F * 4 < (1ll << 31) &&
           (int64_t)g.B * g.H * g.W * g.C * 4 < (1ll << 31);
}
// rows of a band that fit `pixels` pixels at `width` per row, evened out over the image; the whole image where it fits
static ThinPlan thin_plan(const hgq_conv_geom &g, int pixels, int width, int total, int halo, int step) {
    ThinPlan p = {};
    int most = g.OH * width <= pixels ? total : pixels / width - halo;
    if (most < total) most = most / step * step;
    if (most < 1) most = 1;
    p.bands = (total + most - 1) / most;
    p.rows = (total + p.bands - 1) / p.bands;
    if (p.bands > 1) p.rows = (p.rows + step - 1) / step * step;
    p.bands = (total + p.rows - 1) / p.rows;
    p.xw = g.OW + g.kw - 1;
    p.tiles = (int64_t)g.B * p.bands;
    return p;
}
// LDS words of the input patch of `rows` output rows
static int thin_patch(const hgq_conv_geom &g, const ThinPlan &p, int rows) { return ((rows + g.kh - 1) * p.xw * g.C + 3) & ~3; }

// ------------------------------------------------------------------------------------------ forward
// Four wavefronts, 128 pixels; a lane's pixel (A row) is the same in every tile, so its patch offsets sit in registers.
template <int KK, int C, int NB>
__global__ __launch_bounds__(256, 3) void thin_fwd_kernel(const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
                                                          float *__restrict__ y, const hgq_conv_geom g, const ThinPlan p, int F, int act) {
    constexpr int K = KK * KK * C, KS = (K + 15) / 16;
    extern __shared__ float xs[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5;
    const int xwc = p.xw * C, wc = g.W * C;
    const int m = wave * 32 + (lane & 31);
    const FastDiv by_ow((uint32_t)g.OW), by_xwc((uint32_t)xwc);
    const int my = (int)by_ow.div((uint32_t)m), base = m < p.rows * g.OW ? (my * p.xw + m - my * g.OW) * C : 0;
    float b[KS][NB][8], w0 = 0.f;  // w0: zero times every kernel entry, a NaN if one of them is not finite
    int at[KS][8];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int k = 16 * s + 2 * u + half, tap = k / C;
            at[s][u] = base + (k < K ? (tap / KK) * xwc + (tap % KK) * C + k - tap * C : 0);
#pragma unroll
            for (int n = 0; n < NB; ++n) {
                const int f = n * 32 + (lane & 31);
                b[s][n][u] = k < K && f < F ? w[k * F + f] : 0.f;
                w0 = __fmaf_rn(b[s][n][u], 0.f, w0);
            }
        }
    const bool wild_w = __any(!(w0 == 0.f));
    float bv[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) bv[n] = bias && n * 32 + (lane & 31) < F ? bias[n * 32 + (lane & 31)] : 0.f;
    const __amdgpu_buffer_rsrc_t rs_x = buf_rsrc(x, (int64_t)g.B * g.H * wc * 4);
    for (int64_t tile = blockIdx.x; tile < p.tiles; tile += gridDim.x) {
        const int img = (int)(tile / p.bands), oy0 = (int)(tile - (int64_t)img * p.bands) * p.rows;
        const int n_rows = min(p.rows, g.OH - oy0), n_px = n_rows * g.OW, n_x = (n_rows + KK - 1) * xwc;
        __syncthreads();
        for (int e0 = tid; e0 < n_x; e0 += 4 * 256) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = e0 + u * 256, r = (int)by_xwc.div((uint32_t)e), q = e - r * xwc, iy = oy0 - g.py + r, ixc = q - g.px * C;
                const bool ok = e < n_x && (unsigned)iy < (unsigned)g.H && (unsigned)ixc < (unsigned)wc;
                v[u] = buf_ld1(rs_x, ok ? (uint32_t)((img * g.H + iy) * wc + ixc) * 4u : BUF_OOB);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (e0 + u * 256 < n_x) xs[e0 + u * 256] = v[u];
        }
        __syncthreads();
        if (wave * 32 >= n_px) continue;
        floatx16 acc[NB];
        float sum0 = 0.f;  // zero times this lane's inputs
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[n] = floatx16{0};
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            float a[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const float v = m < n_px ? xs[at[s][u]] : 0.f;  // (the LDS behind a short band may hold anything)
                a[u] = 16 * s + 2 * u + 1 < K ? v : (16 * s + 2 * u + half < K ? v : 0.f);
                sum0 = __fmaf_rn(a[u], 0.f, sum0);
            }
#pragma unroll
            for (int n = 0; n < NB; ++n) acc[n] = mfma_batch_bf16<false, false>(acc[n], a, b[s][n]);
        }
        // (an infinity is not the sum of its bf16 parts)
        if (wild_w || __any(!(sum0 == 0.f))) {
#pragma unroll
            for (int n = 0; n < NB; ++n) acc[n] = floatx16{0};
#pragma unroll
            for (int s = 0; s < KS; ++s)
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const float v = m < n_px && 16 * s + 2 * u + half < K ? xs[at[s][u]] : 0.f;
#pragma unroll
                    for (int n = 0; n < NB; ++n) acc[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, b[s][n][u], acc[n], 0, 0, 0);
                }
        }
        float *out = y + ((int64_t)img * g.OH + oy0) * g.OW * F;
        const int left = n_px * F;
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            const int f = n * 32 + (lane & 31);
            const int e0 = f < F ? (wave * 32 + half * 4) * F + f : left;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int e = e0 + ((r >> 2) * 8 + (r & 3)) * F;
                float v = acc[n][r] + bv[n];
                if (act == HGQ_ACT_RELU) v = v > 0.f ? v : 0.f;
                if (e < left) out[e] = v;
            }
        }
    }
}

// ------------------------------------------------------------------------------------------ backward
// POOL 0: dy [B, OH, OW, F], masked by mask > 0 where mask is given (POOL 3: F not a multiple of four or misaligned).  The gradient behind a 2 x 2 maximum pooling of stride
// 2 otherwise (dyp, F a multiple of four, bands that start on even rows): the pixel of the window's first maximum takes it,
// named by `code` (POOL 1) or found in the forward output `mask` (POOL 2); relu: and only where that maximum is positive.
//
// The band's raster is the input patch's: KK - 1 columns of zeros behind each row of dZ.  Pixel m and tap (ky, kx) then meet
// input value m + ky * xw + kx (no index arithmetic in the contraction), and in G the columns left of a row are the zeros
// behind the one above.
struct ThinBwd {
    const float *dy, *mask, *x, *w;
    const uint8_t *code;
    float *dx, *part;
    int F, relu;
};
#define TH_NT 512  // eight wavefronts, 256 pixels
template <int KK, int C, int NB, int POOL>
__global__ __launch_bounds__(TH_NT, 4) void thin_bwd_kernel(const ThinBwd a, const hgq_conv_geom g, const ThinPlan p) {
    constexpr int FP = 32 * NB, FS = FP + 1, K = KK * KK * C, TOP = KK - 1, TAIL = THIN_TAIL;
    extern __shared__ float lds[];
    float *zs = lds, *xs = lds + 256 * FS + TOP * TH_GS;  // dZ [256][FS], later G [TOP + 256][33], at the end dW; input patch
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5;
    const int F = a.F, xw = p.xw, xwc = xw * C, wc = g.W * C, PHo = g.OH >> 1, PWo = g.OW >> 1;
    const FastDiv by_ow((uint32_t)g.OW), by_xw((uint32_t)xw), by_xwc((uint32_t)xwc), by_wc((uint32_t)wc);
    // lane = entry k of the kernel: its place in the patch; 31 stands for the bias (a column of ones)
    const int k = lane & 31, tap = k / C, koff = k < K ? (tap / KK) * xwc + (tap % KK) * C + k - tap * C : 0;
    // the kernel's transpose: in registers, or for two blocks of filters in LDS (32 registers more spill 47)
    float wt[NB == 1 ? 2 : 1][8];
    float *ws = xs + p.patch;
    if (NB == 1) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int f = 16 * s + 2 * u + half;
                wt[s][u] = k < K && f < F ? a.w[k * F + f] : 0.f;
            }
    } else {
        for (int e = tid; e < 32 * FP; e += TH_NT) {
            const int f = e % FP, kk = e / FP;
            ws[kk * FS + f] = kk < K && f < F ? a.w[kk * F + f] : 0.f;
        }
    }
    floatx16 dw[NB];
#pragma unroll
    for (int n = 0; n < NB; ++n) dw[n] = floatx16{0};
    const int64_t y_bytes = (int64_t)g.B * g.OH * g.OW * F * 4, p_bytes = (int64_t)g.B * PHo * PWo * F * 4;
    const __amdgpu_buffer_rsrc_t rs_x = buf_rsrc(a.x, (int64_t)g.B * g.H * wc * 4), rs_dy = buf_rsrc(a.dy, POOL == 1 || POOL == 2 ? p_bytes : y_bytes),
                                 rs_mask = buf_rsrc(a.mask ? a.mask : a.dy, a.mask ? y_bytes : 0),
                                 rs_code = buf_rsrc(POOL == 1 ? (const void *)a.code : (const void *)a.dy, POOL == 1 ? p_bytes / 4 : 0);
    // A band: rows [z0, z1) of dZ are read, those before own1 are owned; input rows [iy0, iy1) get their gradient.
    struct Band {
        int img, iy0, iy1, z0, z1, own1;
    };
    auto band_at = [&](int64_t tile) {
        Band t;
        t.img = (int)(tile / p.bands);
        const int band = (int)(tile - (int64_t)t.img * p.bands);
        t.iy0 = band * p.rows, t.iy1 = min(g.H, t.iy0 + p.rows);
        t.z0 = max(0, t.iy0 + g.py - (KK - 1)), t.z1 = max(t.z0, min(g.OH, t.iy1 + g.py));
        t.own1 = band + 1 == p.bands ? t.z1 : max(t.z0, min(t.z1, t.iy1 + g.py - (KK - 1)));
        return t;
    };
    // Staging of dZ in units: a window x four filters, a pixel x four filters, or a pixel x one filter.  ask(): the loads of
    // U units from e0 on; put(): their values into LDS.  (Asking for the next band's first units ahead of the contraction
    // changes nothing with one unit and spills with more: the wavefronts are bound by what they issue.)
    constexpr bool WINDOWS = POOL == 1 || POOL == 2, VEC = POOL == 0;
    constexpr int U = WINDOWS || (POOL == 3 && NB == 2) ? 1 : VEC ? 4 : 2;
    const int f4 = F >> 2, wpr = (g.OW + 1) >> 1;
    const FastDiv by_f4((uint32_t)max(f4, 1)), by_wpr((uint32_t)wpr);
    auto units = [&](const Band &t) {
        const int zr = t.z1 - t.z0;
        return WINDOWS ? ((zr + 1) >> 1) * wpr * f4 : VEC ? zr * g.OW * f4 : zr * g.OW * FP;
    };
    f32x4_t gv[U], yv[U][POOL == 2 ? 4 : 1];
    auto ask = [&](const Band &t, int e0) {
        const int n_u = units(t);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = e0 + u * TH_NT;
            if (WINDOWS) {
                const int wi = (int)by_f4.div((uint32_t)e), f0 = (e - wi * f4) * 4, wr = (int)by_wpr.div((uint32_t)wi), wx = wi - wr * wpr,
                          wy = (t.z0 >> 1) + wr;
                const bool in = e < n_u && wy < PHo && wx < PWo;
                const uint32_t off = in ? (uint32_t)(((t.img * PHo + wy) * PWo + wx) * F + f0) : BUF_OOB;
                gv[u] = buf_ld4(rs_dy, in ? off * 4u : BUF_OOB);
                if (POOL == 1) {
                    yv[u][0][0] = buf_ld1(rs_code, off);
                } else {
                    const uint32_t oy = (uint32_t)(((t.img * g.OH + 2 * wy) * g.OW + 2 * wx) * F + f0) * 4u;
#pragma unroll
                    for (int j = 0; j < (POOL == 2 ? 4 : 1); ++j)
                        yv[u][j] = buf_ld4(rs_mask, in ? oy + (uint32_t)(((j >> 1) * g.OW + (j & 1)) * F) * 4u : BUF_OOB);
                }
            } else if (VEC) {
                const uint32_t off = e < n_u ? (uint32_t)((t.img * g.OH + t.z0) * g.OW * F) * 4u + (uint32_t)e * 16u : BUF_OOB;
                gv[u] = buf_ld4(rs_dy, off);
                yv[u][0] = buf_ld4(rs_mask, off);
            } else {  // four pixels a quarter of the trip apart, lanes along the filters
                const int f = e % FP;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int px = e / FP + ((e0 - tid) / FP) * 3 + c * (U * TH_NT / FP);
                    const uint32_t off = px * FP < n_u && f < F ? (uint32_t)(((t.img * g.OH + t.z0) * g.OW + px) * F + f) * 4u : BUF_OOB;
                    gv[u][c] = buf_ld1(rs_dy, off);
                    yv[u][0][c] = buf_ld1(rs_mask, off);
                }
            }
        }
    };
    float sum0;  // zero times every value staged: a NaN if one of them is not finite
    auto put = [&](const Band &t, int e0) {
        const int n_u = units(t), zr = t.z1 - t.z0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = e0 + u * TH_NT;
            if (WINDOWS) {
                const int wi = (int)by_f4.div((uint32_t)e), f0 = (e - wi * f4) * 4, wr = (int)by_wpr.div((uint32_t)wi), wx = wi - wr * wpr;
                if (e >= n_u) continue;
                const bool right = 2 * wx + 1 < g.OW, below = 2 * wr + 1 < zr;  // the band has the window's second column / row
                float *z0 = zs + (2 * wr * xw + 2 * wx) * FS + f0;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    int first;
                    bool positive;
                    if (POOL == 1) {
                        const uint32_t cb = __float_as_uint(yv[u][0][0]) >> (8 * c);
                        first = (int)(cb & 3u), positive = (cb & 4u) != 0u;
                    } else {
                        float best = yv[u][0][c];
                        first = 0;
#pragma unroll
                        for (int j = 1; j < (POOL == 2 ? 4 : 1); ++j)
                            if (yv[u][j][c] > best) best = yv[u][j][c], first = j;
                        positive = best > 0.f;
                    }
                    const float gz = !a.relu || positive ? gv[u][c] : 0.f;
                    sum0 = __fmaf_rn(gz, 0.f, sum0);
                    float *z = z0 + c;
                    z[0] = first == 0 ? gz : 0.f;
                    if (right) z[FS] = first == 1 ? gz : 0.f;
                    if (below) z[xw * FS] = first == 2 ? gz : 0.f;
                    if (right && below) z[(xw + 1) * FS] = first == 3 ? gz : 0.f;
                }
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const float v = a.mask && !(yv[u][0][c] > 0.f) ? 0.f : gv[u][c];
                    sum0 = __fmaf_rn(v, 0.f, sum0);
                    gv[u][c] = v;
                }
                if (VEC) {
                    const int px = (int)by_f4.div((uint32_t)e), r = (int)by_ow.div((uint32_t)px);
                    float *z = zs + (px + r * TOP) * FS + (e - px * f4) * 4;
                    if (e < n_u) z[0] = gv[u][0], z[1] = gv[u][1], z[2] = gv[u][2], z[3] = gv[u][3];
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int px = e / FP + ((e0 - tid) / FP) * 3 + c * (U * TH_NT / FP), r = (int)by_ow.div((uint32_t)px);
                        if (px * FP < n_u) zs[(px + r * TOP) * FS + e % FP] = gv[u][c];
                    }
                }
            }
        }
    };
    const int trip = U * TH_NT;
    for (int64_t tile = blockIdx.x; tile < p.tiles; tile += gridDim.x) {
        const Band t = band_at(tile);
        const int img = t.img, iy0 = t.iy0, iy1 = t.iy1, z0 = t.z0, own1 = t.own1, zr = t.z1 - z0;
        const int n_z = zr * xw, n_own = (own1 - z0) * xw, n_x = own1 > z0 ? (own1 - z0 + KK - 1) * xwc : 0;
        const int n_z32 = (n_z + 31) & ~31, n_u = WINDOWS || VEC ? units(t) : (units(t) + 3) / 4;
        sum0 = 0.f;
        __syncthreads();  // the previous tile is done with the LDS
        // ---- dZ, with zeros behind the rows, the last pixel and the last filter
        for (int e = tid; e < zr * TOP * FP; e += TH_NT) {
            const int f = e % FP, c = e / FP;
            zs[((c / TOP) * xw + g.OW + c % TOP) * FS + f] = 0.f;
        }
        for (int e = tid; e < (n_z32 - n_z) * FP; e += TH_NT) zs[(n_z + e / FP) * FS + e % FP] = 0.f;
        if (WINDOWS || VEC)
            for (int f = F + (tid >> 8); f < FP; f += TH_NT / 256)
                if ((tid & 255) < n_z) zs[(tid & 255) * FS + f] = 0.f;
        for (int e0 = tid; e0 - tid < n_u; e0 += trip) {
            ask(t, e0);
            put(t, e0);
        }
        // ---- the input patch under the owned rows, and zeros for what the zero columns behind the last one meet
        for (int e = tid; e < n_x + TAIL * C; e += TH_NT) {
            const int r = (int)by_xwc.div((uint32_t)e), q = e - r * xwc, iy = z0 - g.py + r, ixc = q - g.px * C;
            const bool ok = e < n_x && (unsigned)iy < (unsigned)g.H && (unsigned)ixc < (unsigned)wc;
            const float v = buf_ld1(rs_x, ok ? (uint32_t)((img * g.H + iy) * wc + ixc) * 4u : BUF_OOB);
            sum0 = __fmaf_rn(v, 0.f, sum0);
            xs[e] = v;
        }
        const bool wild = __syncthreads_or(!(sum0 == 0.f));
        // ---- dW: sixteen owned pixels at a time, the batches dealt out over the wavefronts
        if (a.part) {
            for (int s = wave; s * 16 < n_own; s += TH_NT / 64) {
                float xv[8], zv[NB][8];
                const float *xp = xs + koff + (16 * s + half) * C, *zp = zs + (16 * s + half) * FS + k;
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    xv[u] = xp[2 * u * C];
#pragma unroll
                    for (int n = 0; n < NB; ++n) zv[n][u] = zp[2 * u * FS + n * 32];
                }
                if (16 * s + 16 > n_own) {  // (wavefront-uniform) the rest belongs to the next band, or lies behind the patch
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const bool own = 16 * s + 2 * u + half < n_own;
                        xv[u] = own ? xv[u] : 0.f;
#pragma unroll
                        for (int n = 0; n < NB; ++n) zv[n][u] = own ? zv[n][u] : 0.f;
                    }
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) xv[u] = k == 31 ? 1.f : xv[u];
#pragma unroll
                for (int n = 0; n < NB; ++n) {
                    if (wild) {
                        // (an infinite input value against a zero behind a row is not a term of the sum)
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            const uint32_t m = (uint32_t)(16 * s + 2 * u + half);
                            xv[u] = k != 31 && (int)by_xw.mod(m) >= g.OW ? 0.f : xv[u];
                        }
#pragma unroll
                        for (int u = 0; u < 8; ++u) dw[n] = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[u], zv[n][u], dw[n], 0, 0, 0);
                    } else {
                        dw[n] = mfma_batch_bf16<false, true>(dw[n], xv, zv[n], k < K);
                    }
                }
            }
        }
        if (!a.dx) continue;
        // ---- G: a block of 32 pixels per wavefront
        floatx16 gacc = {0};
        if (wave * 32 < n_z32) {
            const float *zp = zs + (wave * 32 + (lane & 31)) * FS + half;
#pragma unroll
            for (int s = 0; s < 2 * NB; ++s) {
                float zv[8], wv[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) zv[u] = zp[16 * s + 2 * u], wv[u] = NB == 1 ? wt[NB == 1 ? s : 0][u] : ws[k * FS + 16 * s + 2 * u + half];
                if (wild) {
#pragma unroll
                    for (int u = 0; u < 8; ++u) gacc = __builtin_amdgcn_mfma_f32_32x32x2f32(zv[u], wv[u], gacc, 0, 0, 0);
                } else {
                    gacc = mfma_batch_bf16<true, false>(gacc, zv, wv);
                }
            }
        }
        __syncthreads();  // everyone has read dZ
        if (tid < TOP * TH_GS) zs[tid] = 0.f;
        if (wave * 32 < n_z32) {
            float *gp = zs + (TOP + wave * 32 + half * 4) * TH_GS + k;
#pragma unroll
            for (int r = 0; r < 16; ++r) gp[((r >> 2) * 8 + (r & 3)) * TH_GS] = gacc[r];
        }
        __syncthreads();
        const int n_dx = (iy1 - iy0) * wc;
        float *dst = a.dx + ((int64_t)img * g.H + iy0) * wc;
        for (int e = tid; e < n_dx; e += TH_NT) {
            const int r = (int)by_wc.div((uint32_t)e), q = e - r * wc, ix = q / C, c = q - ix * C;
            const int ty = iy0 + r + g.py - z0;
            const float *gp = zs + (TOP + ty * xw + ix + g.px) * TH_GS + c;
            float v = 0.f;
#pragma unroll
            for (int ky = 0; ky < KK; ++ky) {
                if ((unsigned)(ty - ky) < (unsigned)zr) {
                    const float *t = gp - ky * xw * TH_GS;
                    float s[KK];
#pragma unroll
                    for (int kx = 0; kx < KK; ++kx) s[kx] = t[(ky * KK + kx) * C - kx * TH_GS];
#pragma unroll
                    for (int kx = 0; kx < KK; ++kx) v += s[kx];
                }
            }
            dst[e] = v;
        }
    }
    if (!a.part) return;
    // the wavefronts' sums in a fixed order
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) zs[((wave * NB + n) * 32 + (r >> 2) * 8 + half * 4 + (r & 3)) * 32 + (lane & 31)] = dw[n][r];
    __syncthreads();
    float *out = a.part + (int64_t)blockIdx.x * (K * F + F);
    for (int e = tid; e < 32 * FP; e += TH_NT) {
        const int row = e / FP, f = e % FP;
        float s = 0.f;
#pragma unroll
        for (int v = 0; v < TH_NT / 64; ++v) s += zs[((v * NB + f / 32) * 32 + row) * 32 + (f & 31)];
        if (f < F && (row < K || row == 31)) out[(row == 31 ? K : row) * F + f] = s;
    }
}

static ThinPlan bwd_plan(const hgq_conv_geom &g) {  // (bands of whole pooling windows, whether or not there is a pooling: same sums)
    ThinPlan p = thin_plan(g, 256, g.OW + g.kw - 1, g.H, g.kh - 1, 2);
    const int rows = p.bands == 1 ? g.OH : (p.rows + g.kh - 1 < g.OH ? p.rows + g.kh - 1 : g.OH);
    p.patch = thin_patch(g, p, rows) + THIN_TAIL * g.C;
    return p;
}
static size_t bwd_lds(int F, const ThinPlan &p) { return (size_t)((F > 32 ? (256 + 32) * 65 : 256 * 33) + 4 * TH_GS + p.patch) * sizeof(float); }

bool conv_thin_fwd_ok(const hgq_conv_geom &g, int F) {
    if (!thin_shape(g, F) || !hgq_dense_use_bf16_parts(-1)) return false;
    const ThinPlan p = thin_plan(g, 128, g.OW, g.OH, 0, 1);
    return p.rows * g.OW <= 128 && thin_patch(g, p, p.rows) * sizeof(float) <= 48 * 1024;
}
bool conv_thin_bwd_shape(const hgq_conv_geom &g, int F) {
    if (!thin_shape(g, F)) return false;
    const ThinPlan p = bwd_plan(g);
    return (p.bands == 1 ? g.OH : p.rows + g.kh - 1) * p.xw <= 256 && bwd_lds(F, p) <= 120 * 1024 && (int64_t)p.rows * g.W * g.C < (1 << 20);
}
int64_t conv_thin_bwd_tiles(const hgq_conv_geom &g) { return bwd_plan(g).tiles; }
int conv_thin_slices(const hgq_conv_geom &g) { return persistent_grid(bwd_plan(g).tiles, 2); }

int conv_thin_fwd(const float *x, const float *w, const float *bias, float *y, const hgq_conv_geom &g, int F, int act, hipStream_t s) {
    const ThinPlan p = thin_plan(g, 128, g.OW, g.OH, 0, 1);
    const size_t lds = thin_patch(g, p, p.rows) * sizeof(float);
    const dim3 grid((unsigned)persistent_grid(p.tiles, 3));
#define HGQ_THIN(KK, CC)                                                                                                              \
    do {                                                                                                                              \
        if (F <= 32) hipLaunchKernelGGL((thin_fwd_kernel<KK, CC, 1>), grid, dim3(256), lds, s, x, w, bias, y, g, p, F, act);          \
        else hipLaunchKernelGGL((thin_fwd_kernel<KK, CC, 2>), grid, dim3(256), lds, s, x, w, bias, y, g, p, F, act);                  \
    } while (0)
    if (g.kh == 5) HGQ_THIN(5, 1);
    else if (g.C == 1) HGQ_THIN(3, 1);
    else if (g.C == 2) HGQ_THIN(3, 2);
    else HGQ_THIN(3, 3);
#undef HGQ_THIN
    return check_launch("hgq_conv2d_fwd(thin)");
}

template <int KK, int C, int NB, int POOL>
static int thin_bwd_launch(const ThinBwd &a, const hgq_conv_geom &g, const ThinPlan &p, hipStream_t s) {
    const size_t lds = bwd_lds(a.F, p);
    if (lds > 60 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void *)thin_bwd_kernel<KK, C, NB, POOL>, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
        if (e != hipSuccess) return fail(HGQ_ERR_LAUNCH, "hgq_conv2d_bwd: hipFuncSetAttribute: %s", hipGetErrorString(e));
    }
    hipLaunchKernelGGL((thin_bwd_kernel<KK, C, NB, POOL>), dim3((unsigned)conv_thin_slices(g)), dim3(TH_NT), lds, s, a, g, p);
    return check_launch("hgq_conv2d_bwd(thin)");
}

// dyp: the gradient behind the 2 x 2 pooling instead of dy, with `code` or the forward output in `mask`
int conv_thin_bwd(const float *dy, const float *mask, const float *dyp, const uint8_t *code, const float *x, const float *w, float *dx,
                  float *part, const hgq_conv_geom &g, int F, int act, hipStream_t s) {
    const ThinPlan p = bwd_plan(g);
    ThinBwd a = {};
    a.dy = dyp ? dyp : dy, a.mask = mask, a.x = x, a.w = w, a.code = code, a.dx = dx, a.part = part, a.F = F, a.relu = act == HGQ_ACT_RELU;
    if (dyp && F > 32) return fail(HGQ_ERR_UNSUPPORTED, "hgq_conv2d_maxpool_bwd: more than 32 filters");
    const bool vec = F % 4 == 0 && (((uintptr_t)dy | (uintptr_t)mask) & 15u) == 0;
#define HGQ_THIN(KK, CC)                                                                                                              \
    return dyp ? (code ? thin_bwd_launch<KK, CC, 1, 1>(a, g, p, s) : thin_bwd_launch<KK, CC, 1, 2>(a, g, p, s))                       \
           : F <= 32 ? (vec ? thin_bwd_launch<KK, CC, 1, 0>(a, g, p, s) : thin_bwd_launch<KK, CC, 1, 3>(a, g, p, s))                  \
                     : (vec ? thin_bwd_launch<KK, CC, 2, 0>(a, g, p, s) : thin_bwd_launch<KK, CC, 2, 3>(a, g, p, s))
    if (g.kh == 5) HGQ_THIN(5, 1);
    if (g.C == 1) HGQ_THIN(3, 1);
    if (g.C == 2) HGQ_THIN(3, 2);
    HGQ_THIN(3, 3);
#undef HGQ_THIN
}

}  // namespace hgq

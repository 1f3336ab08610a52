// Contractions of dense layers beyond the streaming kernels' 64 x 64 (K or N > 64): forward, data gradient and weight
// gradient as tiled matrix products on v_mfma_f32_32x32x16_bf16 over exact bf16 parts (hgq_device.h).
//
//   forward        Y[m, n]  = act(sum_k X[m, k] W[k, n] + b[n])
//   data gradient  dX[m, k] = sum_n dZ[m, n] W[k, n]              dZ = dY where Y > 0 (ReLU), else dY
//   weight grad.   dW[k, n] = sum_m X[m, k] dZ[m, n],  db[n] = sum_m dZ[m, n]      (split along m, one slice per split)
//
// and, with the gathered operand read through the image's geometry (CONV), the same three products of a convolution: X[m, k] is
// the input value tap k = (ky, kx, c) of pixel m meets, the data gradient gathers dZ around an input pixel (unit stride).
// Depths of a tap are padded to a multiple of four, so a thread's four consecutive steps are one 128-bit load.
//
// An operand element is split into its parts ONCE per tile, on its way into LDS, where each part has a plane of its own with
// eight consecutive contraction steps of a row in 16 bytes: an operand of the matrix instruction is one 128-bit LDS read.
// (The implicit-GEMM kernels these replaced read their operands as single fp32 words - 32 LDS reads per instruction - and
// split them again in every wavefront that multiplied by them.)
// Planes that would be zero are neither written nor multiplied: the workgroup agrees on the number of parts of a tile step
// from the low bits of its values (quantized operands of up to 8 bits: one part each, one matrix instruction per product);
// gradients are arbitrary fp32 numbers and always take three.
//
// What bounds them: 50 000 x 256 onto 512 (153 MB, 13 GFLOP) takes 56 us, 50 000 x 512 onto 256 47 us (implicit GEMM: 167 and
// 153 us) - 3 TB/s and 240 - 280 TFLOP/s, in between the two roofs: the chain load -> agree -> stage -> multiply of a tile step,
// hidden by the second workgroup of a CU alone (matrix cores busy 8 % of the time, wavefronts waiting 47 %; 22 vector
// instructions per matrix instruction).  4096 x 256 x 512: forward 9.4, data gradient 14.5, weight gradient 20.8 us with its
// reduction (16.6, 34.3, 24.7 us).  Below some 300 rows the weight gradient is 0.7 - 1 us behind the gathered kernel it
// replaced (256 x 256 x 512 15.0 / 14.0 us); the data gradient beside it is 20 us ahead.
#include "hgq_device.h"
#include "hgq_host.h"

namespace hgq {

enum { GP_FWD = 0, GP_DGRAD = 1, GP_WGRAD = 2 };

// A load at voff + soff bytes; beyond the descriptor's range a lane gets zeros, dword by dword (soff counts towards the range).
__device__ __forceinline__ f32x4_t gp_ld4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
__device__ __forceinline__ float gp_ld1(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

struct GpArgs {
    const float *a, *b;     // operands: FWD x, w; DGRAD dy, w; WGRAD x, dy
    const float *mask;      // DGRAD / WGRAD: the forward output where the activation is a ReLU, else NULL
    const float *bias;      // FWD
    float *out;             // FWD / DGRAD [mo, no]; WGRAD slices [splits][mo * no + no]
    int64_t rows;           // samples: FWD / DGRAD output rows, WGRAD contraction length
    int64_t chunk;          // WGRAD: samples per split (a multiple of the contraction step)
    int mo, no, kc;         // WGRAD: mo x no outputs; FWD / DGRAD: no output columns, kc contraction steps
    int ntm, ntn;           // output tiles
    int total;              // workgroups with work (tiles x splits)
    int per_xcd;            // workgroups per XCD: consecutive ones (same rows, next columns) share an L2
    int act;
    hgq_stack_quant oq;     // FWD: quantizer of the output's columns (oq.i NULL: none)
    hgq_conv_geom cg;       // CONV
    int depth, dp;          // CONV, FWD / DGRAD: values of a tap (C / F), padded to a multiple of four; kc = taps * dp
    int64_t a_bytes;        // CONV: size of the gathered tensor
};

// Staging of one operand tile of S rows (output index) x BK contraction steps by 256 threads.
// KMAJOR = false: contraction steps are adjacent in memory: 128-bit loads (dword-aligned), four steps of a row each.
// KMAJOR = true: output indices are adjacent in memory: a thread takes one output index and CPT consecutive steps, dword
// loads that are whole cache lines per wavefront; it then holds what one 128-bit LDS write needs.  No alignment rule.
template <int S, int BK, bool KMAJOR, bool MASKED>
struct GpTile {
    static constexpr int N = S * BK / 256;  // values per thread
    static constexpr int LW = BK / 2 + 4;   // words per LDS row: 16-byte rows reads spread over all banks
    static constexpr int QPR = BK / 4, RPP = 256 / QPR, NP = S / RPP;
    float v[N], m[MASKED ? N : 1];

    // base: the first element of the tile (row0 / step0 already applied by the caller), range in bytes from there
    __device__ __forceinline__ void fetch(const float *base, const float *mbase, int64_t bytes, int ld, int cols_left, int step0) {
        const __amdgpu_buffer_rsrc_t r = buf_rsrc(base, bytes), rm = buf_rsrc(MASKED && mbase ? mbase : base, MASKED && mbase ? bytes : 0);
        const int tid = threadIdx.x;
        if (KMAJOR) {
            const int col = tid % S, grp = tid / S;
            const uint32_t voff = col < cols_left ? (uint32_t)(grp * N * ld + col) * 4u : 0x80000000u;
#pragma unroll
            for (int c = 0; c < N; ++c) {
                v[c] = gp_ld1(r, voff, (uint32_t)(c * ld) * 4u);
                if (MASKED) m[c] = gp_ld1(rm, voff, (uint32_t)(c * ld) * 4u);
            }
        } else {
            const int cq = tid % QPR, row = tid / QPR;
            const uint32_t voff = (uint32_t)(row * ld + 4 * cq) * 4u;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const f32x4_t t = gp_ld4(r, voff, (uint32_t)(p * RPP * ld + step0) * 4u);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[4 * p + j] = t[j];
                if (MASKED) {
                    const f32x4_t u = gp_ld4(rm, voff, (uint32_t)(p * RPP * ld + step0) * 4u);
#pragma unroll
                    for (int j = 0; j < 4; ++j) m[4 * p + j] = u[j];
                }
            }
        }
    }
    // ---- gathered operands of a convolution
    // rows of this thread (KMAJOR false): place of the window's first tap, ~0 in `px` for rows past the end
    int px[KMAJOR ? 1 : NP], yx[KMAJOR ? 1 : NP];
    template <bool TRANSPOSED>
    __device__ __forceinline__ void locate(const hgq_conv_geom &g, int64_t row0, int64_t rows) {
        const int w = TRANSPOSED ? g.W : g.OW, per = TRANSPOSED ? g.H * g.W : g.OH * g.OW;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int64_t m = row0 + (int)threadIdx.x / QPR + p * RPP;
            const int b = (int)(m / per), rem = (int)(m - (int64_t)b * per), y = rem / w, x = rem - y * w;
            px[p] = m < rows ? b * (TRANSPOSED ? g.OH * g.OW : g.H * g.W) : -1;
            const int y0 = TRANSPOSED ? y + g.py : y * g.sy - g.py, x0 = TRANSPOSED ? x + g.px : x * g.sx - g.px;
            yx[p] = (int)(((uint32_t)y0 << 16) | ((uint32_t)x0 & 0xffffu));
        }
    }
    // four consecutive steps (tap, d0 ..) of this thread's rows from the image `base`
    template <bool TRANSPOSED>
    __device__ __forceinline__ void gather(__amdgpu_buffer_rsrc_t r, __amdgpu_buffer_rsrc_t rm, const hgq_conv_geom &g, int depth, int dp,
                                           const FastDiv &by_dp, const FastDiv &by_kw, int step0, int kc) {
        const int k = step0 + 4 * ((int)threadIdx.x % QPR), tap = (int)by_dp.div((uint32_t)k), d0 = k - tap * dp;
        const int ky = (int)by_kw.div((uint32_t)tap), kx = tap - ky * g.kw;
        const int h = TRANSPOSED ? g.OH : g.H, w = TRANSPOSED ? g.OW : g.W;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int y0 = yx[p] >> 16, x0 = (int)(int16_t)(yx[p] & 0xffff);
            const int y = TRANSPOSED ? y0 - ky * g.dly : y0 + ky * g.dly, x = TRANSPOSED ? x0 - kx * g.dlx : x0 + kx * g.dlx;
            const bool ok = px[p] >= 0 && k < kc && (unsigned)y < (unsigned)h && (unsigned)x < (unsigned)w;
            const uint32_t off = ok ? (uint32_t)((px[p] + y * w + x) * depth + d0) * 4u : BUF_OOB;
            const f32x4_t t = gp_ld4(r, off, 0);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[4 * p + j] = depth == dp || d0 + j < depth ? t[j] : 0.f;
            if (MASKED) {
                const f32x4_t u = gp_ld4(rm, off, 0);
#pragma unroll
                for (int j = 0; j < 4; ++j) m[4 * p + j] = u[j];
            }
        }
    }
    // DGRAD: kernel entries w[tap][c][f], rows c of this tile from c0, four consecutive f
    __device__ __forceinline__ void kernel_rows(__amdgpu_buffer_rsrc_t r, int c0, int C, int F, int dp, const FastDiv &by_dp, int step0, int kc) {
        const int k = step0 + 4 * ((int)threadIdx.x % QPR), tap = (int)by_dp.div((uint32_t)k), f0 = k - tap * dp;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int c = c0 + (int)threadIdx.x / QPR + p * RPP;
            const f32x4_t t = gp_ld4(r, c < C && k < kc ? (uint32_t)((tap * C + c) * F + f0) * 4u : BUF_OOB, 0);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[4 * p + j] = f0 + j < F ? t[j] : 0.f;
        }
    }
    // FWD: kernel entries w[tap][c][n], column n of this tile, consecutive steps
    __device__ __forceinline__ void kernel_cols(__amdgpu_buffer_rsrc_t r, int n0, int C, int F, int dp, const FastDiv &by_dp, int step0, int kc) {
        const int n = n0 + (int)threadIdx.x % S, k0 = step0 + ((int)threadIdx.x / S) * N;
#pragma unroll
        for (int q = 0; q < N / 4; ++q) {
            const int k = k0 + 4 * q, tap = (int)by_dp.div((uint32_t)k), c0 = k - tap * dp;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[4 * q + j] = gp_ld1(r, n < F && k < kc && c0 + j < C ? (uint32_t)((tap * C + c0 + j) * F + n) * 4u : BUF_OOB, 0);
        }
    }
    // WGRAD: this thread's kernel entry (output row) against consecutive pixels from m0 on
    __device__ __forceinline__ void pixels(__amdgpu_buffer_rsrc_t r, const hgq_conv_geom &g, int k, int K, int64_t m0, int64_t m_end) {
        const int tap = k / g.C, c = k - tap * g.C, ky = tap / g.kw, kx = tap - ky * g.kw;
        const int dy = ky * g.dly - g.py, dx = kx * g.dlx - g.px;
        // the pixels are the same for a whole wavefront (S >= 64 columns)
        const int mm = (int)m0 + __builtin_amdgcn_readfirstlane((int)threadIdx.x / S) * N, per = g.OH * g.OW;
        int b = mm / per, oy = (mm - b * per) / g.OW, ox = mm - b * per - oy * g.OW;
#pragma unroll
        for (int e = 0; e < N; ++e) {
            const int y = oy * g.sy + dy, x = ox * g.sx + dx;
            const bool ok = k < K && mm + e < (int)m_end && (unsigned)y < (unsigned)g.H && (unsigned)x < (unsigned)g.W;
            v[e] = gp_ld1(r, ok ? (uint32_t)(((b * g.H + y) * g.W + x) * g.C + c) * 4u : BUF_OOB, 0);
            if (++ox == g.OW) {
                ox = 0;
                if (++oy == g.OH) oy = 0, ++b;
            }
        }
    }
    // steps past the end of the contraction read the next row: zeros instead (only the last tile step can hold any)
    __device__ __forceinline__ void clip(int steps_left) {
        if (!KMAJOR && steps_left < BK) {
            const int c0 = 4 * (threadIdx.x % QPR);
#pragma unroll
            for (int p = 0; p < NP; ++p) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (c0 + j >= steps_left) v[4 * p + j] = 0.f;
            }
        }
    }
    __device__ __forceinline__ void mask(bool on) {
        if (MASKED && on) {
#pragma unroll
            for (int e = 0; e < N; ++e) v[e] = m[e] > 0.f ? v[e] : 0.f;
        }
    }
    __device__ __forceinline__ uint32_t low_bits() const {
        uint32_t low = 0u;
#pragma unroll
        for (int e = 0; e < N; ++e) low |= __float_as_uint(v[e]);
        return low;
    }
    // word index of this thread's unit u of four steps
    __device__ __forceinline__ int at(int u) const {
        const int tid = threadIdx.x;
        if (KMAJOR) return (tid % S) * LW + (tid / S) * (N / 2) + 2 * u;
        return (tid / QPR + RPP * u) * LW + 2 * (tid % QPR);
    }
    __device__ __forceinline__ void put(uint32_t *plane, const uint32_t (&w)[N / 2]) const {
        if (KMAJOR && N % 8 == 0) {
#pragma unroll
            for (int u = 0; u < N / 8; ++u) *(u32x4_t *)(plane + at(2 * u)) = u32x4_t{w[4 * u], w[4 * u + 1], w[4 * u + 2], w[4 * u + 3]};
        } else {
#pragma unroll
            for (int u = 0; u < N / 4; ++u) *(uint2 *)(plane + at(u)) = make_uint2(w[2 * u], w[2 * u + 1]);
        }
    }
    // the first `parts` planes of the tile
    __device__ __forceinline__ void stash(uint32_t *planes, int parts) const {
        uint32_t w[N / 2];
#pragma unroll
        for (int e = 0; e < N; e += 2) w[e / 2] = bf16_pair(__float_as_uint(v[e]), __float_as_uint(v[e + 1]));
        put(planes, w);
        if (parts > 1) {
            uint32_t l[N / 2];
#pragma unroll
            for (int e = 0; e < N; e += 2) {
                uint32_t h0, m0, l0, h1, m1, l1;
                bf16_parts(v[e], h0, m0, l0), bf16_parts(v[e + 1], h1, m1, l1);
                w[e / 2] = bf16_pair(m0, m1), l[e / 2] = bf16_pair(l0, l1);
            }
            put(planes + S * LW, w);
            if (parts > 2) put(planes + 2 * S * LW, l);
        }
    }
};

template <int OP, int BM, int BN, int BK, bool CONV>
__global__ __launch_bounds__(256, 2) void gemm_parts_kernel(const GpArgs g) {
    constexpr bool A_KMAJOR = OP == GP_WGRAD, B_KMAJOR = OP != GP_DGRAD;
    constexpr int WN = BN >= 64 ? 2 : 1, WM = 4 / WN;    // wavefronts along the rows / columns of the tile
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;  // 32 x 32 blocks per wavefront
    using TA = GpTile<BM, BK, A_KMAJOR, OP == GP_DGRAD>;
    using TB = GpTile<BN, BK, B_KMAJOR, OP == GP_WGRAD>;
    constexpr int LW = TA::LW;
    __shared__ uint32_t as[3 * BM * LW], bs[3 * BN * LW], fl[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave / WN, wn = wave % WN;
    const int t = (int)(blockIdx.x % 8u) * g.per_xcd + (int)(blockIdx.x / 8u);
    if (t >= g.total || (int)(blockIdx.x / 8u) >= g.per_xcd) return;  // the whole workgroup
    const int tile = OP == GP_WGRAD ? t % (g.ntm * g.ntn) : t, split = OP == GP_WGRAD ? t / (g.ntm * g.ntn) : 0;
    const int mt = tile / g.ntn, nt = tile - mt * g.ntn;
    const int64_t r0 = (int64_t)mt * BM;  // first output row
    const int n0 = nt * BN;               // first output column
    const bool relu = g.mask != nullptr;
    // contraction range
    const int64_t c_begin = OP == GP_WGRAD ? (int64_t)split * g.chunk : 0;
    const int64_t c_end = OP == GP_WGRAD ? min(g.rows, c_begin + g.chunk) : (int64_t)g.kc;
    const int n_steps = c_end > c_begin ? (int)((c_end - c_begin + BK - 1) / BK) : 0;

    floatx16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = floatx16{0};
    TA ta;
    TB tb;
    float bsum = 0.f;
    const FastDiv by_dp((uint32_t)(CONV ? g.dp : 1)), by_kw((uint32_t)(CONV ? g.cg.kw : 1));
    const int64_t w_bytes = CONV ? (int64_t)g.cg.kh * g.cg.kw * g.cg.C * (OP == GP_DGRAD ? g.depth : g.no) * 4 : 0;
    const __amdgpu_buffer_rsrc_t rs_a = buf_rsrc(g.a, CONV ? g.a_bytes : 0), rs_w = buf_rsrc(g.b, w_bytes),
                                 rs_m = buf_rsrc(CONV && relu ? g.mask : g.a, CONV && relu ? g.a_bytes : 0);
    if (CONV && OP != GP_WGRAD) ta.template locate<OP == GP_DGRAD>(g.cg, r0, g.rows);
    auto fetch = [&](int st) {
        if (CONV && OP == GP_FWD) {
            ta.template gather<false>(rs_a, rs_m, g.cg, g.depth, g.dp, by_dp, by_kw, st * BK, g.kc);
            tb.kernel_cols(rs_w, n0, g.depth, g.no, g.dp, by_dp, st * BK, g.kc);
        } else if (CONV && OP == GP_DGRAD) {
            ta.template gather<true>(rs_a, rs_m, g.cg, g.depth, g.dp, by_dp, by_kw, st * BK, g.kc);
            tb.kernel_rows(rs_w, n0, g.no, g.depth, g.dp, by_dp, st * BK, g.kc);
        } else if (CONV) {
            const int64_t m0 = c_begin + (int64_t)st * BK, left = c_end - m0;
            ta.pixels(rs_a, g.cg, (int)r0 + tid % BM, g.mo, m0, c_end);
            tb.fetch(g.b + m0 * g.no + n0, relu ? g.mask + m0 * g.no + n0 : nullptr, (left * g.no - n0) * 4, g.no, g.no - n0, 0);
        } else if (OP == GP_WGRAD) {
            const int64_t m0 = c_begin + (int64_t)st * BK;
            const int64_t left = c_end - m0;
            ta.fetch(g.a + m0 * g.mo + r0, nullptr, (left * g.mo - r0) * 4, g.mo, g.mo - (int)r0, 0);
            tb.fetch(g.b + m0 * g.no + n0, relu ? g.mask + m0 * g.no + n0 : nullptr, (left * g.no - n0) * 4, g.no, g.no - n0, 0);
        } else {
            const int64_t left = g.rows - r0;
            ta.fetch(g.a + r0 * g.kc, relu ? g.mask + r0 * g.kc : nullptr, left * g.kc * 4, g.kc, 0, st * BK);
            if (OP == GP_FWD) {
                const int k0 = st * BK;
                tb.fetch(g.b + (int64_t)k0 * g.no + n0, nullptr, ((int64_t)(g.kc - k0) * g.no - n0) * 4, g.no, g.no - n0, 0);
            } else {
                tb.fetch(g.b + (int64_t)n0 * g.kc, nullptr, (int64_t)(g.no - n0) * g.kc * 4, g.kc, 0, st * BK);
            }
        }
    };
    if (n_steps > 0) fetch(0);
    for (int st = 0; st < n_steps; ++st) {
        const int left = (int)min((int64_t)BK, c_end - c_begin - (int64_t)st * BK);
        if (!CONV) ta.clip(left), tb.clip(left);
        ta.mask(relu), tb.mask(relu);
        if (OP == GP_WGRAD) {
            if (mt == 0) {
#pragma unroll
                for (int e = 0; e < TB::N; ++e) bsum += tb.v[e];
            }
        }
        // how many parts the operands of this step have, agreed on by the workgroup: a word whose low half is zero is its
        // own first part, one whose low byte is zero has at most two
        uint32_t low_a = OP == GP_DGRAD ? 0u : ta.low_bits(), low_b = OP == GP_WGRAD ? 0u : tb.low_bits();
        uint32_t f = 0u;
        if (OP != GP_DGRAD) f |= (__any((low_a & 0xffffu) != 0u) ? 1u : 0u) | (__any((low_a & 0xffu) != 0u) ? 2u : 0u);
        if (OP != GP_WGRAD) f |= (__any((low_b & 0xffffu) != 0u) ? 4u : 0u) | (__any((low_b & 0xffu) != 0u) ? 8u : 0u);
        if (lane == 0) fl[wave] = f;
        __syncthreads();  // the previous step's operand reads are over; the flags are there
        f = (uint32_t)__builtin_amdgcn_readfirstlane((int)(fl[0] | fl[1] | fl[2] | fl[3]));
        const int pa = OP == GP_DGRAD ? 3 : 1 + (int)(f & 1u) + (int)((f >> 1) & 1u);
        const int pb = OP == GP_WGRAD ? 3 : 1 + (int)((f >> 2) & 1u) + (int)((f >> 3) & 1u);
        ta.stash(as, pa), tb.stash(bs, pb);
        __syncthreads();
        if (st + 1 < n_steps) fetch(st + 1);
        const int arow = wm * 32 * TM + (lane & 31), brow = wn * 32 * TN + (lane & 31), half = lane >> 5;
#pragma unroll
        for (int ks = 0; ks < BK / 16; ++ks) {
            const uint32_t *ap = as + arow * LW + ks * 8 + half * 4, *bp = bs + brow * LW + ks * 8 + half * 4;
            auto products = [&](const u32x4_t (&fa)[TM], const u32x4_t (&fb)[TN]) {
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) acc[i][j] = mfma_bf16(fa[i], fb[j], acc[i][j]);
            };
            auto load_a = [&](u32x4_t (&fa)[TM], int p) {
#pragma unroll
                for (int i = 0; i < TM; ++i) fa[i] = *(const u32x4_t *)(ap + p * BM * LW + i * 32 * LW);
            };
            auto load_b = [&](u32x4_t (&fb)[TN], int p) {
#pragma unroll
                for (int j = 0; j < TN; ++j) fb[j] = *(const u32x4_t *)(bp + p * BN * LW + j * 32 * LW);
            };
            // the gradient's three parts against the parts of the quantized operand (or the parts of two quantized operands)
            if (OP == GP_WGRAD) {
                u32x4_t b0[TN], b1[TN], b2[TN];
                load_b(b0, 0), load_b(b1, 1), load_b(b2, 2);
                for (int p = 0; p < pa; ++p) {
                    u32x4_t fa[TM];
                    load_a(fa, p);
                    products(fa, b0), products(fa, b1), products(fa, b2);
                }
            } else if (OP == GP_DGRAD) {
                u32x4_t a0[TM], a1[TM], a2[TM];
                load_a(a0, 0), load_a(a1, 1), load_a(a2, 2);
                for (int p = 0; p < pb; ++p) {
                    u32x4_t fb[TN];
                    load_b(fb, p);
                    products(a0, fb), products(a1, fb), products(a2, fb);
                }
            } else {
                u32x4_t a0[TM], b0[TN];
                load_a(a0, 0), load_b(b0, 0);
                products(a0, b0);
                for (int p = 1; p < pb; ++p) {
                    u32x4_t fb[TN];
                    load_b(fb, p);
                    products(a0, fb);
                }
                for (int p = 1; p < pa; ++p) {
                    u32x4_t fa[TM];
                    load_a(fa, p);
                    products(fa, b0);
                    for (int q = 1; q < pb; ++q) {
                        u32x4_t fb[TN];
                        load_b(fb, q);
                        products(fa, fb);
                    }
                }
            }
        }
    }
    // An infinity is not the sum of its bf16 parts (Inf - Inf) and a zero part turns it into a NaN: where a result is not
    // finite the wavefront contracts its blocks again on the fp32 instruction, from memory.
    bool bad = false;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) bad |= !(fabsf(acc[i][j][r]) < INFINITY);
    if (__any(bad)) {
        // CONV: value of the gathered tensor that pixel m and depth d of tap `tap` meet
        auto tap_at = [&](int64_t m, int tap, int d) -> float {
            const hgq_conv_geom &q = g.cg;
            const int ky = tap / q.kw, kx = tap - ky * q.kw;
            const int per = OP == GP_DGRAD ? q.H * q.W : q.OH * q.OW, w = OP == GP_DGRAD ? q.W : q.OW;
            const int b = (int)(m / per), rem = (int)(m - (int64_t)b * per), y = rem / w, x = rem - y * w;
            const int sy = OP == GP_DGRAD ? y + q.py - ky * q.dly : y * q.sy - q.py + ky * q.dly;
            const int sx = OP == GP_DGRAD ? x + q.px - kx * q.dlx : x * q.sx - q.px + kx * q.dlx;
            const int sh = OP == GP_DGRAD ? q.OH : q.H, sw = OP == GP_DGRAD ? q.OW : q.W, depth = OP == GP_WGRAD ? q.C : g.depth;
            if ((unsigned)sy >= (unsigned)sh || (unsigned)sx >= (unsigned)sw) return 0.f;
            const int64_t e = (((int64_t)b * sh + sy) * sw + sx) * depth + d;
            return OP == GP_DGRAD && relu && !(g.mask[e] > 0.f) ? 0.f : g.a[e];
        };
        auto a_at = [&](int64_t i, int64_t c) -> float {  // output row i of the tile's matrix, contraction step c
            if (c >= c_end || i >= (OP == GP_WGRAD ? (int64_t)g.mo : g.rows)) return 0.f;
            if (CONV && OP == GP_WGRAD) return tap_at(c, (int)i / g.cg.C, (int)i % g.cg.C);
            if (CONV) return (int)c % g.dp < g.depth ? tap_at(i, (int)c / g.dp, (int)c % g.dp) : 0.f;
            const int64_t e = A_KMAJOR ? c * g.mo + i : i * g.kc + c;
            return OP == GP_DGRAD && relu && !(g.mask[e] > 0.f) ? 0.f : g.a[e];
        };
        auto b_at = [&](int64_t j, int64_t c) -> float {
            if (c >= c_end || j >= g.no) return 0.f;
            if (CONV && OP != GP_WGRAD) {
                const int tap = (int)c / g.dp, d = (int)c - tap * g.dp;
                if (d >= g.depth) return 0.f;
                return OP == GP_FWD ? g.b[((int64_t)tap * g.depth + d) * g.no + j] : g.b[((int64_t)tap * g.no + j) * g.depth + d];
            }
            const int64_t e = B_KMAJOR ? c * g.no + j : j * g.kc + c;
            return OP == GP_WGRAD && relu && !(g.mask[e] > 0.f) ? 0.f : g.b[e];
        };
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int64_t ai = r0 + wm * 32 * TM + i * 32 + (lane & 31), bj = n0 + wn * 32 * TN + j * 32 + (lane & 31);
                floatx16 s = {0};
                for (int64_t c = c_begin; c < c_end; c += 2)
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(a_at(ai, c + (lane >> 5)), b_at(bj, c + (lane >> 5)), s, 0, 0, 0);
                acc[i][j] = s;
            }
    }
    const int64_t out_rows = OP == GP_WGRAD ? (int64_t)g.mo : g.rows;
    float *out = g.out + (OP == GP_WGRAD ? (int64_t)split * ((int64_t)g.mo * g.no + g.no) : 0);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn * 32 * TN + j * 32 + (lane & 31);
        const float bv = (OP == GP_FWD && g.bias && n < g.no) ? g.bias[n] : 0.f;
        const bool quant = OP == GP_FWD && g.oq.i;
        const Mode qm(g.oq.mode);
        KIF qp = {0.f, 0.f, 0.f};
        if (quant && n < g.no) {
            const int e = g.oq.size == 1 ? 0 : n;
            qp = resolve_kif(load_k(g.oq.k, e, qm.k_u8), g.oq.i[e], g.oq.fb[e], qm.kbi, qm.round_params);
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t m = r0 + wm * 32 * TM + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
                float v = acc[i][j][r];
                if (OP == GP_FWD) {
                    v += bv;
                    if (g.act == HGQ_ACT_RELU) v = v > 0.f ? v : 0.f;
                    if (quant) v = quantize_dyn(v, qp, qm.round_mode, qm.overflow_mode, qm.training);
                }
                if (m < out_rows && n < g.no) out[m * g.no + n] = v;
            }
        }
    }
    if (OP == GP_WGRAD && mt == 0) {
        // bias gradient: the threads of a column add up in a fixed order
        float *red = (float *)bs;
        __syncthreads();
        red[tid] = bsum;
        __syncthreads();
        if (tid < BN && n0 + tid < g.no) {
            float s = 0.f;
#pragma unroll
            for (int u = 0; u < 256 / BN; ++u) s += red[tid + u * BN];
            out[(int64_t)g.mo * g.no + n0 + tid] = s;
        }
    }
}

template <int OP, int BM, int BN, int BK, bool CONV = false>
static void gp_launch(GpArgs g, int splits, hipStream_t s) {
    g.ntm = (int)(((OP == GP_WGRAD ? (int64_t)g.mo : g.rows) + BM - 1) / BM);
    g.ntn = (g.no + BN - 1) / BN;
    g.total = g.ntm * g.ntn * splits;
    g.per_xcd = (g.total + 7) / 8;
    hipLaunchKernelGGL((gemm_parts_kernel<OP, BM, BN, BK, CONV>), dim3((unsigned)g.per_xcd * 8u), dim3(256), 0, s, g);
}

// Tile of a product with `m` x `n` outputs.  128 x 128 tiles split and stage each operand value half as often, but a launch
// needs two of them per CU to cover the staging of one with the products of the other; fewer outputs go to 64 x 64 tiles.
// 64 x 64 against 128 x 128, forward: 4096 x 256 -> 512 (128 large tiles) 9.8 / 15.2 us, 8192 x 256 -> 512 (256) 16.7 / 16.7 us,
// 12 288 x 256 -> 512 (384) 23.0 / 18.3 us, 32 768 x 256 -> 512 (1024) 53.4 / 32.7 us; data gradients have the same line.
template <int OP>
static void gp_dispatch(const GpArgs &g, int64_t m, int64_t n, int splits, hipStream_t s) {
    const int64_t big = ((m + 127) / 128) * ((n + 127) / 128) * splits;
    if (n <= 32) gp_launch<OP, 128, 32, 32>(g, splits, s);
    else if (big >= 384) gp_launch<OP, 128, 128, 32>(g, splits, s);
    else gp_launch<OP, 64, 64, 64>(g, splits, s);
}

bool gemm_parts_shape(int64_t rows, int K, int N) {
    return K >= 8 && N >= 1 && K <= (1 << 20) && N <= (1 << 20) && ((rows + 63) / 64) * (((int64_t)(K > N ? K : N) + 31) / 32) < (1ll << 30);
}

int64_t gemm_parts_splits(int64_t rows, int K, int N) {
    const int64_t tiles = N <= 32 ? (K + 127) / 128 : (int64_t)((K + 63) / 64) * ((N + 63) / 64);
    int64_t s = (512 + tiles - 1) / tiles;
    const int64_t cap = N <= 32 ? (rows + 127) / 128 : (rows + 255) / 256;  // at least four tile steps each
    if (s > cap) s = cap;
    if (s > 512) s = 512;
    return s < 1 ? 1 : s;
}

int gemm_parts_fwd(const float *x, const float *w, const float *bias, float *y, int64_t rows, int K, int N, int act, hipStream_t s,
                   const hgq_stack_quant *oq) {
    GpArgs g = {};
    if (oq) g.oq = *oq;
    g.a = x, g.b = w, g.bias = bias, g.out = y, g.rows = rows, g.no = N, g.kc = K, g.act = act;
    gp_dispatch<GP_FWD>(g, rows, N, 1, s);
    return check_launch("gemm_parts(forward)");
}

int gemm_parts_dgrad(const float *dy, const float *mask, const float *w, float *dx, int64_t rows, int K, int N, hipStream_t s) {
    GpArgs g = {};
    g.a = dy, g.b = w, g.mask = mask, g.out = dx, g.rows = rows, g.no = K, g.kc = N;
    gp_dispatch<GP_DGRAD>(g, rows, K, 1, s);
    return check_launch("gemm_parts(data gradient)");
}

int gemm_parts_wgrad(const float *x, const float *dy, const float *mask, float *part, int64_t rows, int K, int N, int64_t splits, hipStream_t s) {
    GpArgs g = {};
    g.a = x, g.b = dy, g.mask = mask, g.out = part, g.rows = rows, g.mo = K, g.no = N;
    g.chunk = ((rows + splits - 1) / splits + 63) / 64 * 64;
    if (N <= 32) gp_launch<GP_WGRAD, 128, 32, 32>(g, (int)splits, s);
    else gp_launch<GP_WGRAD, 64, 64, 64>(g, (int)splits, s);
    return check_launch("gemm_parts(weight gradient)");
}

// ---- convolutions.  Pixel indices and places in a window are 32- and 16-bit numbers, tensors below 2 GiB.
bool conv_parts_shape(const hgq_conv_geom &g, int F) {
    const int lim = 16384;
    return g.H <= lim && g.W <= lim && g.OH <= lim && g.OW <= lim && g.py <= lim / 2 && g.px <= lim / 2 &&
           (int64_t)g.OH * g.sy <= lim && (int64_t)g.OW * g.sx <= lim && (int64_t)g.kh * g.dly <= lim && (int64_t)g.kw * g.dlx <= lim &&
           (int64_t)g.kh * g.kw * (g.C + 3) < (1 << 20) && (int64_t)g.kh * g.kw * (F + 3) < (1 << 20) && F <= (1 << 16) &&
           (int64_t)g.kh * g.kw * g.C * F * 4 < (1ll << 31) && (int64_t)g.B * g.H * g.W * g.C * 4 < (1ll << 31) &&
           (int64_t)g.B * g.OH * g.OW * F * 4 < (1ll << 31);
}

int conv_parts_fwd(const float *x, const float *w, const float *bias, float *y, const hgq_conv_geom &cg, int F, int act, hipStream_t s) {
    GpArgs g = {};
    g.a = x, g.b = w, g.bias = bias, g.out = y, g.rows = (int64_t)cg.B * cg.OH * cg.OW, g.no = F, g.act = act, g.cg = cg;
    g.depth = cg.C, g.dp = (cg.C + 3) & ~3, g.kc = cg.kh * cg.kw * g.dp, g.a_bytes = (int64_t)cg.B * cg.H * cg.W * cg.C * 4;
    if (F <= 32) gp_launch<GP_FWD, 128, 32, 32, true>(g, 1, s);
    else gp_launch<GP_FWD, 64, 64, 64, true>(g, 1, s);
    return check_launch("hgq_conv2d_fwd(parts)");
}

int conv_parts_dgrad(const float *dy, const float *mask, const float *w, float *dx, const hgq_conv_geom &cg, int F, hipStream_t s) {
    GpArgs g = {};
    g.a = dy, g.b = w, g.mask = mask, g.out = dx, g.rows = (int64_t)cg.B * cg.H * cg.W, g.no = cg.C, g.cg = cg;
    g.depth = F, g.dp = (F + 3) & ~3, g.kc = cg.kh * cg.kw * g.dp, g.a_bytes = (int64_t)cg.B * cg.OH * cg.OW * F * 4;
    if (cg.C <= 32) gp_launch<GP_DGRAD, 128, 32, 32, true>(g, 1, s);
    else gp_launch<GP_DGRAD, 64, 64, 64, true>(g, 1, s);
    return check_launch("hgq_conv2d_bwd(data, parts)");
}

int conv_parts_wgrad(const float *x, const float *dy, const float *mask, float *part, const hgq_conv_geom &cg, int F, int64_t splits, hipStream_t s) {
    GpArgs g = {};
    g.a = x, g.b = dy, g.mask = mask, g.out = part, g.rows = (int64_t)cg.B * cg.OH * cg.OW, g.mo = cg.kh * cg.kw * cg.C, g.no = F, g.cg = cg;
    g.a_bytes = (int64_t)cg.B * cg.H * cg.W * cg.C * 4;
    g.chunk = ((g.rows + splits - 1) / splits + 63) / 64 * 64;
    if (F <= 32) gp_launch<GP_WGRAD, 128, 32, 32, true>(g, (int)splits, s);
    else gp_launch<GP_WGRAD, 64, 64, 64, true>(g, (int)splits, s);
    return check_launch("hgq_conv2d_bwd(weights, parts)");
}

}  // namespace hgq

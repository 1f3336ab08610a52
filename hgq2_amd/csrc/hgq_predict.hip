// Inference of a stack of QDense layers in one call: y = L_n(... L_1(x)), L(x) = act(q_in(x) q_w(W) + q_b(b)).
//
// Two forms.
//
// * Every width up to 64 (`stack_chain_kernel`): ONE launch.  A workgroup quantizes all kernels and biases into LDS, then
//   takes tiles of 64 samples through every layer; between layers a tile stays in LDS and the next layer's input quantizer
//   runs on the accumulator registers.  One event through 16-64-32-32-5 is bound by latency: four loads and one rounding
//   per kernel entry, then a short matrix-instruction chain per layer (19 us); the call takes 75 us, most of it the host's (a
//   launch per quantizer and contraction, sixteen in all: 512 us).
// * Wider layers, or many rows: one launch quantizes all kernels and biases into the workspace, one the input; then per layer
//   a tiled product whose epilogue applies the next layer's input quantizer (a pass over [rows, N] each way less), the
//   streaming kernel of up to 64 x 64, or what hgq_conv2d_fwd has for a product of few tiles.  50 000 rows through
//   256-512-256-128-10: 195 us (a launch per quantizer and contraction: 484 us).
//
// Arithmetic per value is that of hgq_quantize_fwd and of the layer's own contraction; the variables are quantized again on
// every call (they may have been written in between).
#include "hgq_device.h"
#include "hgq_host.h"

namespace hgq {

#define CHAIN_BM 64
#define CHAIN_LD 65   // odd row stride: the 32 rows of an operand read fall into different banks
#define CHAIN_LDS (160 * 1024)  // of a CU; seven layers of 64 x 64 fit
// Eight wavefronts stage, quantize and store; four of them contract, row half x column half of a tile.  Quantizing the kernels is
// what a call of few samples waits for, two wavefronts per SIMD issue it nearly twice as fast as one: 64 x 64 on one sample
// 14.9 -> 10.4 us, seven such layers 67.3 -> 44.6 us, 16-64-32-32-5 22.0 -> 19.3 us.  (Sixteen wavefronts: 8.9, 35.7, 19.2 us, and
// one workgroup per CU instead of two: 39 against 23 us for the last on 32 768 samples.)
#define CHAIN_NT 512

struct ChainDev {
    hgq_stack_layer l[HGQ_STACK_MAX_LAYERS];
    int off_w[HGQ_STACK_MAX_LAYERS];  // kernel [Kp][Np], zero padded (Kp: multiple of 16, Np: of 32), then the bias [Np]
    int n_layers, off_q, off_a;       // off_q: (k, i, f) of the input quantizers, [n_layers][3][64]; off_a: two tiles
    uint32_t how;                     // two bits per layer, CHAIN_*
};
// How a layer multiplies.  An infinity is not the sum of its bf16 parts (times a part that is zero it is a NaN): where an operand
// may hold one a tile whose sums are not all finite is contracted again on the fp32 instruction.  A quantizer outside training
// leaves none: it saturates them or wraps them to NaNs.
enum { CHAIN_BF16 = 0, CHAIN_CHECKED = 1, CHAIN_FP32 = 2 };

__device__ __forceinline__ KIF stack_entry(const hgq_stack_quant &q, int e) {
    const Mode m(q.mode);
    return resolve_kif(load_k(q.k, e, m.k_u8), q.i[e], q.fb[e], m.kbi, m.round_params);
}
// bit-width entry of element e of a tensor with n elements
__device__ __forceinline__ int stack_index(const hgq_stack_quant &q, int e, int n) {
    return q.size == n ? e : (e / q.inner) % q.size;
}
__device__ __forceinline__ float stack_quantize(float v, const KIF &p, int mode) {
    const Mode m(mode);
    return quantize_dyn(v, p, m.round_mode, m.overflow_mode, m.training);
}

__global__ __launch_bounds__(CHAIN_NT) void stack_chain_kernel(const ChainDev d, const float *__restrict__ x, float *__restrict__ y,
                                                               int64_t rows) {
    extern __shared__ float lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int L = d.n_layers;
    float *qt = lds + d.off_q, *tiles = lds + d.off_a;
    for (int e = tid; e < d.off_a; e += CHAIN_NT) lds[e] = 0.f;
    for (int e = tid; e < 2 * CHAIN_BM * CHAIN_LD; e += CHAIN_NT) tiles[e] = 0.f;
    __syncthreads();
    for (int l = 0; l < L; ++l) {
        const hgq_stack_layer &h = d.l[l];
        const int n = h.K * h.N, Np = (h.N + 31) & ~31, Kp = (h.K + 15) & ~15;
        const FastDiv by_n((uint32_t)h.N);
        float *w = lds + d.off_w[l];
        for (int e0 = tid; e0 < n; e0 += 4 * CHAIN_NT) {
            float v[4];
            KIF p[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {  // (four entries in flight; the last trip repeats its own entry)
                const int e = e0 + u * CHAIN_NT < n ? e0 + u * CHAIN_NT : e0;
                v[u] = h.w[e];
                p[u] = stack_entry(h.kq, stack_index(h.kq, e, n));
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = e0 + u * CHAIN_NT < n ? e0 + u * CHAIN_NT : e0;
                const int k = (int)by_n.div((uint32_t)e);
                w[k * Np + (e - k * h.N)] = stack_quantize(v[u], p[u], h.kq.mode);
            }
        }
        if (h.bias && tid < h.N) w[Kp * Np + tid] = stack_quantize(h.bias[tid], stack_entry(h.bq, stack_index(h.bq, tid, h.N)), h.bq.mode);
        if (h.iq.i && h.iq.size <= h.K && tid >= 64 && tid < 64 + h.K) {
            const int c = tid - 64;
            const KIF p = stack_entry(h.iq, h.iq.size == 1 ? 0 : c);
            qt[l * 192 + c] = p.k, qt[l * 192 + 64 + c] = p.i, qt[l * 192 + 128 + c] = p.f;
        }
    }
    __syncthreads();
    const int64_t n_tiles = (rows + CHAIN_BM - 1) / CHAIN_BM;
    const int K0 = d.l[0].K, NL = d.l[L - 1].N;
    const FastDiv by_k0((uint32_t)K0), by_nl((uint32_t)NL);
    const int rh = wave & 1, cb = wave >> 1, half = lane >> 5;
    for (int64_t tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int64_t r0 = tile * CHAIN_BM;
        const int live = (int)(rows - r0 < CHAIN_BM ? rows - r0 : CHAIN_BM);
        {
            // the input tile: rows are contiguous; zeros past the last one (their results are not stored)
            const __amdgpu_buffer_rsrc_t rs = buf_rsrc(x + r0 * K0, (int64_t)live * K0 * 4);
            const hgq_stack_quant &iq = d.l[0].iq;
            const bool quant = iq.i != nullptr, table = quant && iq.size > K0;  // (a table of several rows is read per element)
            const int t0 = table ? (int)(r0 * K0 % iq.size) : 0;
            for (int e0 = tid; e0 < CHAIN_BM * K0; e0 += 4 * CHAIN_NT) {
                float v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = buf_ld1(rs, e0 + u * CHAIN_NT < CHAIN_BM * K0 ? (uint32_t)(e0 + u * CHAIN_NT) * 4u : BUF_OOB);
                KIF p[4];
                if (table) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) p[u] = stack_entry(iq, (t0 + e0 + u * CHAIN_NT) % iq.size);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int e = e0 + u * CHAIN_NT;
                    if (e < CHAIN_BM * K0) {
                        const int row = (int)by_k0.div((uint32_t)e), c = e - row * K0;
                        if (!table) p[u] = KIF{qt[c], qt[64 + c], qt[128 + c]};
                        tiles[row * CHAIN_LD + c] = quant ? stack_quantize(v[u], p[u], iq.mode) : v[u];
                    }
                }
            }
            // columns that pad the contraction to sixteen steps: a deeper layer of the previous tile has been here
            const int pad = ((K0 + 15) & ~15) - K0;
            for (int e = tid; e < CHAIN_BM * pad; e += CHAIN_NT) tiles[(e & (CHAIN_BM - 1)) * CHAIN_LD + K0 + e / CHAIN_BM] = 0.f;
        }
        for (int l = 0; l < L; ++l) {
            const hgq_stack_layer &h = d.l[l];
            const int Np = (h.N + 31) & ~31, batches = (h.K + 15) >> 4;
            const float *src = tiles + (l & 1) * CHAIN_BM * CHAIN_LD;
            float *dst = tiles + ((l + 1) & 1) * CHAIN_BM * CHAIN_LD;
            const bool last = l + 1 == L;
            __syncthreads();  // the source tile is complete
            if (wave < 4 && cb * 32 < Np) {
                const float *w = lds + d.off_w[l];
                const floatx16 zero = {0};
                const float *ap = src + (rh * 32 + (lane & 31)) * CHAIN_LD + half, *bp = w + half * Np + cb * 32 + (lane & 31);
                const uint32_t how = (d.how >> (2 * l)) & 3u;
                floatx16 acc = zero;
                if (how != CHAIN_FP32) acc = mfma_chain_bf16<false, false>(zero, ap, 1, bp, Np, batches);
                if (how != CHAIN_BF16) {
                    bool bad = how == CHAIN_FP32;
#pragma unroll
                    for (int r = 0; r < 16; ++r) bad |= !(fabsf(acc[r]) < INFINITY);
                    if (__any(bad)) acc = mfma_chain(zero, ap, 1, bp, Np, batches);
                }
                const int c = cb * 32 + (lane & 31);
                const float b = w[batches * 16 * Np + c];
                // the next layer's input quantizer, column c (nothing is read past its table: c < N = next K)
                const bool quant = !last && d.l[last ? l : l + 1].iq.i != nullptr;
                const int nm = d.l[last ? l : l + 1].iq.mode;
                const float *qn = qt + (last ? 0 : l + 1) * 192;
                const KIF p = {qn[c], qn[64 + c], qn[128 + c]};
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    float v = acc[r] + b;
                    if (h.act == HGQ_ACT_RELU) v = v > 0.f ? v : 0.f;
                    if (quant) v = stack_quantize(v, p, nm);
                    dst[(rh * 32 + (r >> 2) * 8 + half * 4 + (r & 3)) * CHAIN_LD + c] = c < h.N ? v : 0.f;
                }
            }
        }
        __syncthreads();
        const float *out = tiles + (L & 1) * CHAIN_BM * CHAIN_LD;
        const hgq_stack_quant &oq = d.l[L - 1].oq;
        const int t0 = oq.i ? (int)(r0 * NL % oq.size) : 0;
        for (int e0 = tid; e0 < live * NL; e0 += 4 * CHAIN_NT) {
            float v[4];
            KIF p[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = e0 + u * CHAIN_NT < live * NL ? e0 + u * CHAIN_NT : e0, row = (int)by_nl.div((uint32_t)e);
                v[u] = out[row * CHAIN_LD + (e - row * NL)];
                if (oq.i) p[u] = stack_entry(oq, oq.size == 1 ? 0 : (t0 + e) % oq.size);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (e0 + u * CHAIN_NT < live * NL) y[r0 * NL + e0 + u * CHAIN_NT] = oq.i ? stack_quantize(v[u], p[u], oq.mode) : v[u];
        }
        __syncthreads();  // the next input tile goes into the first buffer
    }
}

// All kernels and biases of a stack, quantized into the workspace.
struct StackPrep {
    hgq_stack_quant q[2 * HGQ_STACK_MAX_LAYERS];
    const float *src[2 * HGQ_STACK_MAX_LAYERS];
    float *dst[2 * HGQ_STACK_MAX_LAYERS];
    int n[2 * HGQ_STACK_MAX_LAYERS];
};
__global__ __launch_bounds__(256) void stack_prep_kernel(const StackPrep p) {
    const int it = blockIdx.y, n = p.n[it];
    const hgq_stack_quant q = p.q[it];
    for (int e = blockIdx.x * 256 + threadIdx.x; e < n; e += gridDim.x * 256)
        p.dst[it][e] = stack_quantize(p.src[it][e], stack_entry(q, stack_index(q, e, n)), q.mode);
}

static bool quant_ok(const hgq_stack_quant &q, int64_t n) {
    const Mode m(q.mode);
    return q.k && q.i && q.fb && q.size >= 1 && q.inner >= 1 && n % ((int64_t)q.size * q.inner) == 0 && m.round_mode <= HGQ_RND_CONV &&
           m.overflow_mode <= HGQ_SAT_SYM;
}

static int chain_layout(const hgq_stack_layer *layers, int n, ChainDev &d) {
    int at = 0;
    for (int l = 0; l < n; ++l) {
        d.l[l] = layers[l];
        d.off_w[l] = at;
        at += (((layers[l].K + 15) & ~15) + 1) * ((layers[l].N + 31) & ~31);
    }
    d.n_layers = n;
    d.off_q = at;
    d.off_a = at + n * 192;
    return (d.off_a + 2 * CHAIN_BM * CHAIN_LD) * (int)sizeof(float);
}

// 0: refused, 1: one launch, 2: a launch per layer (a function of the arguments alone: what hgq_dense_stack_workspace answered
// holds for the launch, also where another thread has changed the matrix instruction in between)
static int stack_form(const hgq_stack_layer *layers, int n, int64_t rows) {
    if (!layers || n < 1 || n > HGQ_STACK_MAX_LAYERS || rows < 1) return 0;
    bool chain = true, wide = true, tables = false;
    for (int l = 0; l < n; ++l) {
        const hgq_stack_layer &h = layers[l];
        if (h.K < 1 || h.N < 1 || (int64_t)h.K * h.N > (1 << 26) || (l && h.K != layers[l - 1].N)) return 0;
        if (!h.w || !quant_ok(h.kq, (int64_t)h.K * h.N) || (h.bias && !quant_ok(h.bq, h.N))) return 0;
        if (h.iq.i && (!quant_ok(h.iq, l ? h.K : rows * h.K) || h.iq.inner != 1 || (h.iq.size != 1 && (l ? h.iq.size != h.K : h.iq.size % h.K)))) return 0;
        if (h.oq.i && (l + 1 < n || !quant_ok(h.oq, rows * h.N) || h.oq.inner != 1 || (h.oq.size != 1 && h.oq.size % h.N))) return 0;
        chain = chain && h.K <= 64 && h.N <= 64;
        wide = wide && gemm_parts_shape(rows, h.K < 8 ? 8 : h.K, h.N);
        tables = tables || (h.iq.i && h.iq.size > h.K) || (h.oq.i && h.oq.size > h.N);
    }
    ChainDev d;
    chain = chain && chain_layout(layers, n, d) <= CHAIN_LDS;
    // One launch where the host and the launches are what a call costs, and as long as it is not the slower one on the device
    // either.  Device time of recorded calls, one launch against a launch per layer: 16-64-32-32-5 on 65 536 rows 32 / 54 us,
    // seven layers of 64 units 118 / 117 us; 64 onto 64 with tables for input and output on 32 768 rows 21.8 / 25.4 us, on
    // 65 536 36.3 / 30.9 us.  (On a few rows 64 onto 64 alone is 10.4 / 8.5 us, with both tables 16.7 / 11.3 us, and an eager call
    // of two or three launches more takes the host 7 us longer.)
    if (chain && (!wide || rows <= (tables ? 32768 : 65536))) return 1;
    return wide ? 2 : 0;
}

static int64_t image_floats(const hgq_stack_layer *layers, int n) {
    int64_t at = 0;
    for (int l = 0; l < n; ++l) at += ((int64_t)layers[l].K * layers[l].N + 3) / 4 * 4 + (layers[l].N + 3) / 4 * 4;
    return at;
}
// A product of few output tiles behind a long contraction, which one workgroup per tile would leave to a handful of CUs and a
// chain of tile steps (32 contraction steps each up to 32 columns, 64 beyond): the forms of hgq_conv2d_fwd that spread it along
// k, from sixteen tile steps on, with the quantizer behind it as a launch of its own.  Tiled product against those, whole
// calls: 1024 rows of 3872 -> 10 126 / 28 us, 300 of 2048 -> 512 50 / 34 us, 1024 of 520 -> 3 25.0 / 20.4 us; below the line 1024
// of 512 -> 512 19.4 / 27.1 us, 64 of 600 -> 64 -> 5 23.9 / 26.7 us, 64 of 784 -> 128 -> 10 28.8 / 28.5 us.
static bool few_tiles(const hgq_stack_layer &h, int64_t rows) {
    return (h.K > 64 || h.N > 64) && h.K >= (h.N <= 32 ? 512 : 1024) && dense_split_k(rows, h.K, h.N);
}
static hgq_conv_geom dense_geom(const hgq_stack_layer &h, int64_t rows) { return {(int)rows, 1, 1, h.K, 1, 1, 1, 1, 0, 0, 1, 1, 1, 1}; }
// scratch of such products: the partial sums along k and the result that a quantizer reads
static int64_t few_floats(const hgq_stack_layer *layers, int n, int64_t rows) {
    int64_t most = 0;
    for (int l = 0; l < n; ++l) {
        if (!few_tiles(layers[l], rows)) continue;
        const hgq_conv_geom g = dense_geom(layers[l], rows);
        const int64_t w = (rows * layers[l].N + 3) / 4 * 4 + hgq_conv2d_fwd_workspace(&g, layers[l].N);
        if (w > most) most = w;
    }
    return most;
}
// an output quantizer the last product's epilogue does not apply (it takes one entry or one per column)
static bool table_out(const hgq_stack_layer &h) { return h.oq.i && h.oq.size > h.N; }
// widest tensor that goes into buffer `which` (0: inputs of even layers, 1: of odd layers, and a last output to be quantized)
static int64_t buffer_floats(const hgq_stack_layer *layers, int n, int64_t rows, int which) {
    int64_t w = table_out(layers[n - 1]) && (n & 1) == which ? layers[n - 1].N : 0;
    for (int l = which; l < n; l += 2)
        if ((l || layers[0].iq.i) && layers[l].K > w) w = layers[l].K;
    return (w * rows + 3) / 4 * 4;
}

}  // namespace hgq

using namespace hgq;

extern "C" int64_t hgq_dense_stack_workspace(const hgq_stack_layer *layers, int n_layers, int64_t rows) {
    const int form = stack_form(layers, n_layers, rows);
    if (form != 2) return form == 1 ? 0 : -1;
    if (!hgq_dense_use_bf16_parts(-1)) return -1;  // the tiled products know one instruction: layer by layer on the other
    return image_floats(layers, n_layers) + buffer_floats(layers, n_layers, rows, 0) + buffer_floats(layers, n_layers, rows, 1) +
           few_floats(layers, n_layers, rows);
}

extern "C" int hgq_dense_stack_predict(const hgq_stack_layer *layers, int n_layers, const float *x, float *y, int64_t rows,
                                       float *workspace, void *stream) {
    const int form = stack_form(layers, n_layers, rows);
    if (!form) return fail(HGQ_ERR_UNSUPPORTED, "hgq_dense_stack_predict: these layers are not covered (ask hgq_dense_stack_workspace)");
    if (!x || !y || (form == 2 && !workspace)) return fail(HGQ_ERR_ARG, "hgq_dense_stack_predict: null argument");
    hipStream_t s = (hipStream_t)stream;
    if (form == 1) {
        ChainDev d = {};
        const int bytes = chain_layout(layers, n_layers, d);
        for (int l = 0; l < n_layers; ++l) {
            const Mode mi(layers[l].iq.mode), mk(layers[l].kq.mode);
            const bool open = !layers[l].iq.i || (mi.overflow_mode == HGQ_WRAP && mi.training) || (mk.overflow_mode == HGQ_WRAP && mk.training);
            d.how |= (uint32_t)(!hgq_dense_use_bf16_parts(-1) ? CHAIN_FP32 : open ? CHAIN_CHECKED : CHAIN_BF16) << (2 * l);
        }
        if (bytes > 64 * 1024) {
            hipError_t e = hipFuncSetAttribute((const void *)stack_chain_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, CHAIN_LDS);
            if (e != hipSuccess) return fail(HGQ_ERR_LAUNCH, "hgq_dense_stack_predict: hipFuncSetAttribute: %s", hipGetErrorString(e));
        }
        const int per_cu = CHAIN_LDS / bytes;  // each workgroup quantizes the kernels once: no more of them than fit at a time
        const int grid = persistent_grid((rows + CHAIN_BM - 1) / CHAIN_BM, per_cu > 2 ? 2 : per_cu);
        hipLaunchKernelGGL(stack_chain_kernel, dim3((unsigned)grid), dim3(CHAIN_NT), bytes, s, d, x, y, rows);
        return check_launch("hgq_dense_stack_predict(chain)");
    }
    StackPrep p = {};
    float *at = workspace, *qw[HGQ_STACK_MAX_LAYERS], *qb[HGQ_STACK_MAX_LAYERS];
    int items = 0, most = 0;
    for (int l = 0; l < n_layers; ++l) {
        const hgq_stack_layer &h = layers[l];
        const int n = h.K * h.N;
        p.q[items] = h.kq, p.src[items] = h.w, p.dst[items] = qw[l] = at, p.n[items++] = n;
        at += ((int64_t)n + 3) / 4 * 4;
        if (n > most) most = n;
        qb[l] = h.bias ? at : nullptr;
        if (h.bias) p.q[items] = h.bq, p.src[items] = h.bias, p.dst[items] = at, p.n[items++] = h.N;
        at += (h.N + 3) / 4 * 4;
    }
    const int gx = (most + 255) / 256 < 512 ? (most + 255) / 256 : 512;
    hipLaunchKernelGGL(stack_prep_kernel, dim3((unsigned)gx, (unsigned)items), dim3(256), 0, s, p);
    int rc = check_launch("hgq_dense_stack_predict(kernels)");
    if (rc) return rc;
    float *buf[2] = {at, at + buffer_floats(layers, n_layers, rows, 0)}, *few = buf[1] + buffer_floats(layers, n_layers, rows, 1);
    const float *cur = x;
    if (const hgq_stack_quant &q = layers[0].iq; q.i) {
        if ((rc = hgq_quantize_fwd(x, q.k, q.i, q.fb, buf[0], nullptr, nullptr, rows * layers[0].K, q.size, 1, q.mode, stream))) return rc;
        cur = buf[0];
    }
    for (int l = 0; l < n_layers; ++l) {
        const hgq_stack_layer &h = layers[l];
        const bool last = l + 1 == n_layers, later = last && table_out(h);
        float *out = last && !later ? y : buf[(l + 1) & 1];
        const hgq_stack_quant *oq = last ? (h.oq.i && !later ? &h.oq : nullptr) : layers[l + 1].iq.i ? &layers[l + 1].iq : nullptr;
        if (few_tiles(h, rows)) {
            const hgq_conv_geom g = dense_geom(h, rows);
            float *z = oq ? few : out, *ws = few + (rows * h.N + 3) / 4 * 4;
            rc = hgq_conv2d_fwd(cur, qw[l], qb[l], z, ws, &g, h.N, h.act, stream);
            if (!rc && oq) rc = hgq_quantize_fwd(z, oq->k, oq->i, oq->fb, out, nullptr, nullptr, rows * h.N, oq->size, 1, oq->mode, stream);
        } else if (!oq && h.K <= 64 && h.N <= 64) {
            rc = hgq_qdense_fwd(cur, nullptr, nullptr, nullptr, 0, qw[l], qb[l], out, nullptr, rows, h.K, h.N, h.act, 0, stream);
        } else {
            rc = gemm_parts_fwd(cur, qw[l], qb[l], out, rows, h.K, h.N, h.act, s, oq);
        }
        if (rc) return rc;
        if (later) return hgq_quantize_fwd(out, h.oq.k, h.oq.i, h.oq.fb, y, nullptr, nullptr, rows * h.N, h.oq.size, 1, h.oq.mode, stream);
        cur = out;
    }
    return HGQ_OK;
}

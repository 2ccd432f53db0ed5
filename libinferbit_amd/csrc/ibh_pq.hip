// ibh_pq.hip -- product-quantised (PQ) LUT matvec, ib_pq_matmul_fp32
// (src/pq_decode.c:1504-1686) on gfx950.
//
// Tensor layout is the reference's (src/pq_decode.h:39-87), uploaded as is:
// fp16 codebooks [K][G/2] per side (one L and one R codebook shared by all
// chunks, plus the level-2 pair), uint8 indices [M][C] per side (level-2:
// uint8, uint16 or 4-bit packed), fp16 row scales, outlier sidecar.
//
// out[r] = row_scale[r] * sum_c (T_L[c][iL[r,c]] + T_R[c][iR[r,c]] (+ L2))
//          + outlier terms,
// T_side[c][k] = codebook_side[k] . x[inner columns of chunk c, that side].
//
// Kernel 1 (tables): block per chunk: its tables (K entries x 2 sides, in the
// reference's operation order) and its max|x|, written once to a workspace.
// Kernel 2 (gather): block (row tile, slab of CS chunks): the global max|x|
// over the inner columns from the chunk maxima (chunk-skipping rule of
// pq_decode.c:1569-1616: chunks whose max|x| is below 1% of it are left
// out), the slab's tables into LDS, then each thread walks its rows: CS index
// bytes per side from one 16-byte load, 2*CS LDS gathers.  The per-slab
// partial sums go to the workspace.
// Kernel 3 (reduce): sums the slabs in order, applies the row scale and the
// outlier sidecar (the x86 rules of pq_decode.c:1233-1421: int8-quantised
// dot for >= 32 outliers, fp32 otherwise).
// The chunk sum is associated slab by slab instead of strictly serially, so
// results differ from the CPU by fp32 rounding only.
#include "ibh_common.h"

using namespace ibh;

namespace {

constexpr int kRowsPerBlock = 512;    // rows of one slab block (2 per thread)
constexpr int kThreads = 256;

struct PqDev {
    int M, N, G, K, K2, n_levels, n_outlier, C, l2_idx_bytes;
    // chunk selection: 0 every chunk; 1 kept iff max|x_c| >= skip_val * max|x|
    // (matmul_impl); 2 kept iff max|x_c| > skip_val when skip_val > 0
    // (streaming_sparse)
    int skip_mode;
    float skip_val;
    int q8;                  // int8 codebooks and chunk activations (streaming_int8_cached)
    int l2skip;              // per-(row, chunk) level-2 skip (l2skip_cached) with threshold l2_thr
    float l2_thr;
    int pyramid;             // per-cluster level-2 norm bound (format 4)
    const float* cnorm;      // [C][2] |x_L|, |x_R| per chunk (l2skip)
    const float* c2max;      // [2][n_outer] max level-2 codeword norm per cluster (l2skip)
    const uint16_t *cb1l, *cb1r, *cb2l, *cb2r;
    const uint8_t *i1l, *i1r, *i2l, *i2r;
    const uint16_t* row_scale;
    const int32_t* ocols;
    const int8_t* oside;
    const uint16_t* oscale;
    const int32_t* inner;    // inner (non-outlier) columns, null when n_outlier == 0
    int slab_sh;             // log2 of the three-kernel path's chunks per slab (two levels: 8 or 16)
};

__device__ __forceinline__ int inner_col(const PqDev& t, int j) { return t.inner ? t.inner[j] : j; }

__device__ __forceinline__ int l2_at(const PqDev& t, const uint8_t* row, int c) {
    if (t.K2 == 16) { const uint8_t b = row[c >> 1]; return (c & 1) ? (b >> 4) : (b & 0xf); }
    if (t.l2_idx_bytes == 2) return ((const uint16_t*)row)[c];
    return row[c];
}

__device__ __forceinline__ size_t l2_stride(const PqDev& t) {
    if (t.K2 == 16) return (size_t)(t.C + 1) / 2;
    return (size_t)t.C * (t.l2_idx_bytes == 2 ? 2 : 1);
}

// sum_i cb[i] * x[i]: products of the first hf&~3 terms rounded then added
// in order, remaining terms fused (the x86 build's evaluation of
// pq_decode.c:1621-1659).
__device__ __forceinline__ float table_entry(const uint16_t* cb, const float* xv, int hf) {
    float s = 0.f;
    const int v = hf & ~3;
    int i = 0;
    for (; i < v; i++) s = s + f16_to_f32(cb[i]) * xv[i];
    for (; i < hf; i++) s = fmaf(f16_to_f32(cb[i]), xv[i], s);
    return s;
}

// Tables of one chunk, built once: T1[c][side][k] (and T2) written to global
// memory with the chunk's max|x| (the skipping rule is applied by the
// gather, which has every chunk's max).
// Round-half-away int8 code of v * inv, clamped to +-127
// (pq_quantize_codebook_int8 / pq_quantize_chunk_int8, pq_decode.c:2766-2856).
__device__ __forceinline__ int q8_code(float v, float inv) {
    const float u = v * inv;
    const int q = (int)(u >= 0.0f ? u + 0.5f : u - 0.5f);
    return q > 127 ? 127 : (q < -127 ? -127 : q);
}

// int8 table entry (pq_chunk_dot_table_int8, pq_decode.c:2817-2836): the
// codeword quantised with its own scale, exact int32 dot with the chunk's
// codes, then (float)dot * cb_scale * x_scale.
__device__ __forceinline__ float table_entry_q8(const uint16_t* cb, const int8_t* xq, float xsc, int hf) {
    float m = 0.f;
    for (int i = 0; i < hf; i++) m = fmaxf(m, fabsf(f16_to_f32(cb[i])));
    const float cs = m > 0.f ? m / 127.0f : 1.0f;
    const float inv = 1.0f / cs;
    int sum = 0;
    for (int i = 0; i < hf; i++) sum += q8_code(f16_to_f32(cb[i]), inv) * (int)xq[i];
    return (float)sum * cs * xsc;
}

template <bool TWO>
__global__ __launch_bounds__(kThreads) void pq_tables(PqDev t, const float* __restrict__ x, float* __restrict__ tab1,
                                                      float* __restrict__ tab2, float* __restrict__ cmax,
                                                      float* __restrict__ cnorm) {
    __shared__ float xs[64];
    __shared__ int8_t xq[2][32];
    __shared__ float xsc[2];
    const int K = t.K, K2 = t.K2, G = t.G, hf = G / 2;
    const int c = blockIdx.x;
    if (threadIdx.x < G) xs[threadIdx.x] = x[inner_col(t, c * G + threadIdx.x)];
    __syncthreads();
    if (threadIdx.x == 0) {
        float cm = 0.f;
        for (int i = 0; i < G; i++) cm = fmaxf(cm, fabsf(xs[i]));
        cmax[c] = cm;
    }
    if (threadIdx.x < 2 && (t.l2skip || t.q8)) {
        // this side's |x| (l2skip) and int8 codes (q8)
        const float* v = xs + threadIdx.x * hf;
        float n2 = 0.f, m = 0.f;
        for (int i = 0; i < hf; i++) {
            n2 = fmaf(v[i], v[i], n2);
            m = fmaxf(m, fabsf(v[i]));
        }
        if (t.l2skip) cnorm[2 * c + threadIdx.x] = sqrtf(n2);
        const float sc = m > 0.f ? m / 127.0f : 1.0f;
        const float inv = 1.0f / sc;
        for (int i = 0; i < hf; i++) xq[threadIdx.x][i] = (int8_t)q8_code(v[i], inv);
        xsc[threadIdx.x] = sc;
    }
    if (t.q8) __syncthreads();
    for (int e = threadIdx.x; e < 2 * K; e += kThreads) {
        const int side = e / K, k = e % K;
        const uint16_t* cb = (side ? t.cb1r : t.cb1l) + (size_t)k * hf;
        tab1[(size_t)c * 2 * K + e] = t.q8 ? table_entry_q8(cb, xq[side], xsc[side], hf) : table_entry(cb, xs + side * hf, hf);
    }
    if (TWO) {
        for (int e = threadIdx.x; e < 2 * K2; e += kThreads) {
            const int side = e / K2, k = e % K2;
            const uint16_t* cb = (side ? t.cb2r : t.cb2l) + (size_t)k * hf;
            tab2[(size_t)c * 2 * K2 + e] =
                t.q8 ? table_entry_q8(cb, xq[side], xsc[side], hf) : table_entry(cb, xs + side * hf, hf);
        }
    }
}

// Max level-2 codeword norm per cluster (ib_pq_lut_cache_create,
// pq_decode.c:2655-2675): block per cluster; c2max[0][k1] (L), [1][k1] (R).
__global__ __launch_bounds__(kThreads) void pq_c2max(PqDev t, float* __restrict__ c2max, int n_outer, int k_inner) {
    __shared__ float red[2][kThreads / 64];
    const int k1 = blockIdx.x, hf = t.G / 2, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float ml = 0.f, mr = 0.f;
    for (int k = k1 * k_inner + (int)threadIdx.x; k < (k1 + 1) * k_inner; k += kThreads) {
        float nl = 0.f, nr = 0.f;
        for (int j = 0; j < hf; j++) {
            const float a = f16_to_f32(t.cb2l[(size_t)k * hf + j]), b = f16_to_f32(t.cb2r[(size_t)k * hf + j]);
            nl = fmaf(a, a, nl);
            nr = fmaf(b, b, nr);
        }
        ml = fmaxf(ml, sqrtf(nl));
        mr = fmaxf(mr, sqrtf(nr));
    }
    ml = wave_max(ml);
    mr = wave_max(mr);
    if (lane == 0) { red[0][wave] = ml; red[1][wave] = mr; }
    __syncthreads();
    if (threadIdx.x < 2) {
        float m = 0.f;
        for (int w = 0; w < kThreads / 64; w++) m = fmaxf(m, red[threadIdx.x][w]);
        c2max[threadIdx.x * n_outer + k1] = m;
    }
}

// Rows [r0, r1): the slab partials summed in slab order, the row scale, and
// the outlier sidecar (the x86 rules of pq_decode.c:1233-1421: int8-quantised
// dot for >= 32 outliers, fp32 otherwise).  Whole block.
__device__ void finish_rows(const PqDev& t, const float* __restrict__ x, const float* __restrict__ part, int nslabs,
                            float* __restrict__ out, int r0, int r1, int8_t* qq_s, float* meta_s) {
    const int no = t.n_outlier;
    const bool quant = no >= 32;
    if (quant) {
        // x * col_scale quantised with one meta scale (pq_decode.c:274-301)
        if (threadIdx.x == 0) {
            float mx = 0.f;
            for (int j = 0; j < no; j++) {
                const float v = x[t.ocols[j]] * f16_to_f32(t.oscale[j]);
                const float a = v < 0 ? -v : v;
                if (a > mx) mx = a;
            }
            *meta_s = mx > 0.f ? mx / 127.0f : 1.0f;
        }
        __syncthreads();
        const float inv = 1.0f / *meta_s;
        for (int j = threadIdx.x; j < no; j += kThreads) {
            const float sv = (x[t.ocols[j]] * f16_to_f32(t.oscale[j])) * inv;
            const int v = (int)(sv >= 0 ? sv + 0.5f : sv - 0.5f);
            qq_s[j] = (int8_t)(v > 127 ? 127 : (v < -128 ? -128 : v));
        }
        __syncthreads();
    }
    for (int r = r0 + (int)threadIdx.x; r < r1; r += kThreads) {
        float acc = 0.f;
        int s = 0;
        for (; s + 16 <= nslabs; s += 16) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) v[u] = part[(size_t)(s + u) * t.M + r];
#pragma unroll
            for (int u = 0; u < 16; u++) acc += v[u];
        }
        for (; s < nslabs; s++) acc += part[(size_t)s * t.M + r];
        float y = acc * f16_to_f32(t.row_scale[r]);
        if (no > 0) {
            const int8_t* side = t.oside + (size_t)r * no;
            if (quant) {
                int32_t sum = 0;
                for (int j = 0; j < no; j++) sum += (int32_t)side[j] * (int32_t)qq_s[j];
                y = fmaf((float)sum, *meta_s, y);
            } else {
                for (int j = 0; j < no; j++)
                    y = fmaf((float)side[j] * f16_to_f32(t.oscale[j]), x[t.ocols[j]], y);
            }
        }
        out[r] = y;
    }
}

// Level-2 skip of one (row, chunk) (l2skip_cached, pq_decode.c:3203-3214):
// |l1| > thr * (c2L * |x_L| + c2R * |x_R|), with per-cluster bounds for a
// pyramid tensor (cluster = the row's level-1 code of that side).
__device__ __forceinline__ bool l2_skipped(const PqDev& t, float l1, const float (*c2)[256], const float* nrm, int a,
                                           int b) {
    const float bound = t.l2_thr * fmaf(c2[0][t.pyramid ? a : 0], nrm[0], c2[1][t.pyramid ? b : 0] * nrm[1]);
    return fabsf(l1) > bound;
}

// Block (row tile, slab): the slab's tables into LDS, then each thread walks
// its rows (CS index bytes per side from one 16-byte load, 2 CS gathers).
template <bool TWO>
__global__ __launch_bounds__(kThreads) void pq_gather(PqDev t, const float* __restrict__ tab1,
                                                      const float* __restrict__ tab2, const float* __restrict__ cmax,
                                                      float* __restrict__ part, int CS) {
    extern __shared__ __align__(16) float sm[];
    __shared__ float red[kThreads / 64];
    __shared__ int act_s[64];
    __shared__ float nrm_s[64][2];            // l2skip: |x_L|, |x_R| of the slab's chunks
    __shared__ float c2_s[2][256];            // l2skip: cluster bounds (pyramid: per level-1 code)
    const int K = t.K, K2 = t.K2, C = t.C;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float* T1 = sm;                                   // [CS][2][K]
    float* T2 = T1 + (size_t)CS * 2 * K;              // [CS][2][K2]  (TWO)
    const int c0 = blockIdx.y * CS;
    const int cn = min(CS, C - c0);
    {
        const int n1 = cn * 2 * K, n2 = TWO ? cn * 2 * K2 : 0;
        const float* g1 = tab1 + (size_t)c0 * 2 * K;
        const float* g2 = TWO ? tab2 + (size_t)c0 * 2 * K2 : nullptr;
        if ((n1 & 3) == 0 && (n2 & 3) == 0 && (((uintptr_t)g1 | (uintptr_t)g2) & 15) == 0) {
            for (int i = threadIdx.x; i < n1 / 4; i += kThreads) ((float4*)T1)[i] = ((const float4*)g1)[i];
            for (int i = threadIdx.x; i < n2 / 4; i += kThreads) ((float4*)T2)[i] = ((const float4*)g2)[i];
        } else {
            for (int i = threadIdx.x; i < n1; i += kThreads) T1[i] = g1[i];
            for (int i = threadIdx.x; i < n2; i += kThreads) T2[i] = g2[i];
        }
    }
    // chunk-skipping rule (pq_decode.c:1569-1616): the global max|x| over the
    // inner columns is the max of the chunk maxima
    float mx = 0.f;
    for (int c0_ = 0; c0_ < C; c0_ += 4 * kThreads) {
        float v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = cmax[min(c0_ + u * kThreads + (int)threadIdx.x, C - 1)];
#pragma unroll
        for (int u = 0; u < 4; u++) mx = fmaxf(mx, v[u]);
    }
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    float gmax = 0.f;
    for (int w = 0; w < kThreads / 64; w++) gmax = fmaxf(gmax, red[w]);
    if (threadIdx.x < cn) {
        const float cm = cmax[c0 + threadIdx.x];
        act_s[threadIdx.x] = t.skip_mode == 1 ? (gmax > 0.f ? cm >= gmax * t.skip_val : 1)
                           : t.skip_mode == 2 ? (t.skip_val > 0.f ? cm > t.skip_val : 1) : 1;
    }
    const bool l2skip = TWO && t.l2skip && t.l2_thr > 0.f;
    if (l2skip) {
        const int no = t.pyramid ? K : 1;
        for (int i = threadIdx.x; i < 2 * no; i += kThreads) c2_s[i / no][i % no] = t.c2max[i];
        if (threadIdx.x < 2 * cn) nrm_s[threadIdx.x >> 1][threadIdx.x & 1] = t.cnorm[2 * c0 + threadIdx.x];
    }
    __syncthreads();

    const size_t l2s = TWO ? l2_stride(t) : 0;
    for (int rr = threadIdx.x; rr < kRowsPerBlock; rr += kThreads) {
        const int r = blockIdx.x * kRowsPerBlock + rr;
        if (r >= t.M) break;
        const uint8_t* il = t.i1l + (size_t)r * C + c0;
        const uint8_t* ir = t.i1r + (size_t)r * C + c0;
        const uint8_t* i2l = TWO ? t.i2l + (size_t)r * l2s : nullptr;
        const uint8_t* i2r = TWO ? t.i2r + (size_t)r * l2s : nullptr;
        float acc = 0.f;
        if (cn == 16 && (((uintptr_t)il | (uintptr_t)ir) & 15) == 0) {
            // a full slab: both index rows in one 16-byte load each
            const uint4 a4 = *(const uint4*)il, b4 = *(const uint4*)ir;
            const uint32_t aw[4] = {a4.x, a4.y, a4.z, a4.w}, bw[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
            for (int c = 0; c < 16; c++) {
                if (!act_s[c]) continue;
                const float* tc = T1 + (size_t)c * 2 * K;
                const int a = (aw[c >> 2] >> (8 * (c & 3))) & 0xff, b = (bw[c >> 2] >> (8 * (c & 3))) & 0xff;
                const float l1 = tc[a] + tc[K + b];
                acc = acc + l1;
                if (TWO && !(l2skip && l2_skipped(t, l1, c2_s, nrm_s[c], a, b))) {
                    const float* t2 = T2 + (size_t)c * 2 * K2;
                    acc = acc + (t2[l2_at(t, i2l, c0 + c)] + t2[K2 + l2_at(t, i2r, c0 + c)]);
                }
            }
        } else {
            for (int c = 0; c < cn; c++) {
                if (!act_s[c]) continue;
                const float* tc = T1 + (size_t)c * 2 * K;
                const int a = il[c], b = ir[c];
                const float l1 = tc[a] + tc[K + b];
                acc = acc + l1;
                if (TWO && !(l2skip && l2_skipped(t, l1, c2_s, nrm_s[c], a, b))) {
                    const float* t2 = T2 + (size_t)c * 2 * K2;
                    acc = acc + (t2[l2_at(t, i2l, c0 + c)] + t2[K2 + l2_at(t, i2r, c0 + c)]);
                }
            }
        }
        part[(size_t)blockIdx.y * t.M + r] = acc;
    }
}

// Kernel 3: block per 256 rows.
__global__ __launch_bounds__(kThreads) void pq_reduce(PqDev t, const float* __restrict__ x,
                                                      const float* __restrict__ part, int nslabs,
                                                      float* __restrict__ out) {
    __shared__ int8_t qq_s[1024];
    __shared__ float meta_s;
    finish_rows(t, x, part, nslabs, out, blockIdx.x * kThreads, min(t.M, (int)(blockIdx.x + 1) * kThreads), qq_s,
                &meta_s);
}


// ── one-launch PQ matvec (G <= 16, up to 256 codes a level) ────────────────
// Block = (tile of 512 rows, slab of 32 chunks), 1024 threads: two per row,
// thread q of a row owns chunks 16q..16q+15 of the slab on both sides.  The
// two slabs that share the 64-byte index segments of a row run on one XCD,
// back to back (its L2 serves the second).
//  1. Global loads first: the slab's x, the codebooks, x for the max|x|
//     scan, and last the row's index bytes (one 16-byte load per side), so
//     the table phase does not wait for those HBM reads.
//  2. The slab's tables T[c][side][k] = cb_side[k] . x[chunk c, side] on the
//     matrix cores: per side, a 32-code x 32-chunk tile is one
//     v_mfma_f32_32x32x16_f16 with A = [cb | cb] (the fp16 codewords, exact)
//     and B = [x_hi ; x_lo], x scaled per (chunk, side) by a power of two
//     (exact) and split into two fp16 parts; products are exact and sums
//     fp32.  The power of two takes the 8 elements' max|x| to the top of fp16:
//     an element's two parts then keep 2^-23 of the element itself down to
//     2^-17 of that max.  (Scaled to 1 instead, small elements lost their low
//     parts: error against 64 bits 3.0e-7 -> 1.5e-7, 3489 rows of 201 chunks.
//     With one power of two a slab, one large channel took bits from every
//     other chunk of it: 520 x 1536, rows whose codewords are 0 on a channel
//     2^20 / 2^26 / 2^32 times the others, error 6e-7 / 4e-5 / 3e-3 -> 1.1e-7 /
//     1.1e-7 / 6e-7, the three kernels 1.1e-7.)
//  3. Max|x| over the inner columns (the skipping rule of
//     pq_decode.c:1569-1616) and sum|x|, the slab's chunk maxima.
//  4. Gather: 32 LDS lookups per thread, the row's two partials summed.
//  5. Slabs meet per row in one 64-bit word: each slab adds
//     2^58 + round(partial * 2^q) + 2^50 (an agent-scope atomic with return,
//     performed where every XCD sees it).  2^q maps the largest sum the
//     inputs allow (max|cb| * sum|x|, doubled; with N * max|x| in place of
//     the sum one large channel cost the other rows bits) to 2^50, so every
//     term is an exact integer below 2^51 and the sum of at most 63 slabs stays
//     below 2^58; the count sits above.  The slab whose add completes the
//     count has the whole row in the returned value: it applies the row scale
//     and the outliers, writes y and clears the word for the next call.
//     Integer addition is associative: y does not depend on arrival order.
//     The words belong to the caller's workspace (its first 1 MB + 256 B),
//     zeroed once by ibh_pq_workspace_init, which also writes a stamp the
//     kernel checks: a workspace without it gives NaN rows and raises
//     IBH_DEVERR_PQ_WS instead of adding into unknown words.  Calls on the
//     library workspace (ws == NULL) use a library array of words.
//     A non-finite x (or a bound that overflows) would make the fixed-point
//     terms meaningless: every slab then writes NaN to its rows (the CPU
//     gives +-Inf or NaN there); two-level calls, which had the three-kernel
//     path's fp32 sums there, take them from direct_rows.
//  Two levels double the tables, the lookups and the index bytes and keep the
//  rest: 4096 x 14336, 256 + 256 codes, streaming: 75.3 us in three launches
//  (68 of them the gather, 16 chunks' tables re-read by every block of 512
//  rows and two byte loads per lookup) -> 12.4 us, error 2.1e-7 -> 1.2e-7.
constexpr int kFThreads = 1024;
constexpr int kFRows = 512;
constexpr int kFCS = 32;
constexpr int kFMaxS = 63;
constexpr int kFMaxRows = 131072;
constexpr int kMinExp = -100;   // exponents of x below it share its scale
constexpr int kXS = 20;   // LDS floats per slab chunk: 8 per side (zero padded) + 4 (bank spread)
__device__ unsigned long long pq_row_acc[kFMaxRows];   // ws == NULL calls: zero at load, each row's last slab clears it
__device__ unsigned int ibh_pq_err;                    // IBH_DEVERR_* bits of this file's kernels
__device__ uint4 pq_spare;                             // what a block without 16-byte index rows loads in their place
constexpr unsigned long long kPqStamp = 0x49424850515753ull;   // "IBHPQWS"
constexpr size_t kPqFront = 256 + (size_t)kFMaxRows * 8;       // stamp + row words at the front of a caller workspace

// Phase probes, compiled only with -DIBH_PQ_TRACE (a development build
// outside the library): s_memrealtime of thread 0 of each block.
#ifdef IBH_PQ_TRACE
__device__ unsigned long long ibh_pq_tt[4096][8];
#define PQ_TT(i) do { if (tid == 0 && blockIdx.x < 4096) ibh_pq_tt[blockIdx.x][i] = __builtin_amdgcn_s_memrealtime(); } while (0)
#else
#define PQ_TT(i) ((void)0)
#endif

// 16 (8) bytes from any address in one load: indices lie where a file put
// them, codebooks and x on multiples of their element
typedef uint32_t u4a_t __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u2a_t __attribute__((ext_vector_type(2), aligned(1)));
typedef float f4a_t __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ uint4 ld16(const void* p) {
    const u4a_t v = *(const u4a_t*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float4 ld4f(const float* p) {
    const f4a_t v = *(const f4a_t*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f16x_t __attribute__((ext_vector_type(16)));

// The slab's tables from the block's LDS copies of the codebooks (fp16, rows
// padded to 8) and of the slab's x.  A wavefront has one side: it scales and
// splits that side's x once (a lane has a chunk's whole) and takes every eighth
// 32-code tile of both levels.  (Split again for each tile, 4096 x 14336 at 256
// + 256 codes: 13.3 us; 12.4 so.)  Scales are a power of two of each (chunk,
// side); the entries leave as T * 2^-ex, so that the row sums are rescaled once.
// Records each (chunk, side)'s max|x|.
template <bool KA, bool TWO>
__device__ __forceinline__ void slab_tables(int K, int K2, const h8_t* cbs, const float* xsl, int cn, int wave, int lane,
                                            int ex, float* T1, float* T2, float (*cmax_s)[kFCS]) {
    static_assert(kFCS == 32);
    const int sd = wave & 1, cc = lane & 31;
    const float4* xp = (const float4*)(xsl + min(cc, cn - 1) * kXS + sd * 8);
    const float4 x0 = xp[0], x1 = xp[1];
    const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) m = fmaxf(m, fabsf(xv[i]));
    if (wave < 2 && lane < cn) cmax_s[sd][lane] = m;
    const int ec = m > 0.f ? max(__builtin_amdgcn_frexp_expf(m), kMinExp) - 15 : ex;   // m < 2^(ec + 15)
    const float xscale = ldexpf(1.0f, -ec), es = ldexpf(1.0f, ec - ex);
    const bool lo = lane >= 32;
    h8_t b;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float v = xv[i] * xscale;                       // exact: a power of two
        const _Float16 h = (_Float16)v;
        b[i] = lo ? (_Float16)(v - (float)h) : h;
    }
    const int KT1 = (K + 31) / 32, KT = KT1 + (TWO ? (K2 + 31) / 32 : 0);
    for (int j = wave >> 1; j < KT; j += kFThreads / 128) {
        const bool second = TWO && j >= KT1;
        const int k0 = 32 * (second ? j - KT1 : j), Kj = second ? K2 : K;
        const h8_t a = cbs[(second ? 2 * K : 0) + sd * Kj + min(k0 + (lane & 31), Kj - 1)];
        const f16x_t d = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, f16x_t{}, 0, 0, 0) * es;
        // D[k][n]: lane (n = lane & 31), register r: row 8*(r>>2) + 4*(lane>>5) + (r&3)
        if (cc < cn) {
            float* dst = (second ? T2 : T1) + (size_t)cc * (2 * Kj + 4) + sd * Kj + k0 + 4 * (lane >> 5);
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int kk = k0 + 8 * g + 4 * (lane >> 5);
                const float4 v = make_float4(d[4 * g], d[4 * g + 1], d[4 * g + 2], d[4 * g + 3]);
                if (KA || kk + 3 < Kj) *(float4*)(dst + 8 * g) = v;
                else {
                    const float vv[4] = {v.x, v.y, v.z, v.w};
                    for (int u = 0; u < 4; u++)
                        if (kk + u < Kj) dst[8 * g + u] = vv[u];
                }
            }
        }
    }
}

// Rows' sums from the codebooks and x directly, no tables and no row words:
// two-level calls with a non-finite or tiny x or a non-finite codeword, sums
// past the fixed-point range, or a workspace without the stamp, all of which the three-kernel path
// served.  The sums are that path's bit for bit: a lane sums the entries of
// one of its slabs of 8 or 16 chunks, the slabs are added in order.  Rows
// [lo, hi) of the block's tiles, two per group of lanes, into sums[row - tile
// start].  Bound by the LDS reads of codewords at random (four of 16 bytes per
// row and chunk) and of x, staged once with the slabs 4 floats apart so that
// the lanes' reads spread over the banks.  A workspace without the stamp, 4096
// x 14336, 256 + 256 codes: 53 us; 1024 x 3216 with 16 outliers, 256 + 64
// codes: 42 us (the three kernels 79 and 45, a thread per row 10072 and 2299).
constexpr int kDPad = 4;

template <bool P4>
__device__ __forceinline__ void direct_rows(const PqDev& t, const float* __restrict__ x, const h8_t* cbs, float* xd,
                                            float* sums, int base, int lo, int hi, float gmax, int tid) {
    const int hf = t.G / 2, C = t.C, K = t.K, K2 = t.K2, lane = tid & 63, wave = tid >> 6;
    const int CS = 1 << t.slab_sh, dxs = 16 * CS + kDPad;
    const size_t l2s = l2_stride(t);
    for (int i = tid; i < C * 16; i += kFThreads) {
        const int c = i >> 4, sd = (i >> 3) & 1, e = i & 7;
        xd[(c >> t.slab_sh) * dxs + (i & (16 * CS - 1))] = e < hf ? x[inner_col(t, c * t.G + sd * hf + e)] : 0.f;
    }
    __syncthreads();
    // sum_i cb[i] * x[i] in table_entry's order, over the hf values that exist
    auto entry = [&](const h8_t cb, const float* xv) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if (i >= hf) break;
            const float c = (float)cb[i];
            s = i < (hf & ~3) ? s + c * xv[i] : fmaf(c, xv[i], s);
        }
        return s;
    };
    const int ns = (C + CS - 1) >> t.slab_sh;
    // lanes per row: the power of two that holds the slabs, up to 64
    int lsh = 0;
    while (lsh < 6 && (1 << lsh) < ns) lsh++;
    const int sub = lane & ((1 << lsh) - 1), first = lane - sub, nrow = 2 << (6 - lsh);
    for (int r0 = lo + nrow * wave; r0 < hi; r0 += nrow * (kFThreads / 64)) {
        const int r = r0 + 2 * (lane >> lsh);
        const uint8_t* ip[2][4];
        float tot[2] = {0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const size_t rr = (size_t)min(base + min(r + u, hi - 1), t.M - 1);
            ip[u][0] = t.i1l + rr * C;
            ip[u][1] = t.i1r + rr * C;
            ip[u][2] = t.i2l + rr * l2s;
            ip[u][3] = t.i2r + rr * l2s;
        }
        for (int s0 = 0; s0 < ns; s0 += 64) {
            const int sl = min(s0 + sub, ns - 1);             // lanes past the last slab are not added
            float acc[2] = {0.f, 0.f};
            int k[2][4];
            auto load = [&](int j) {                          // the chunk's codes
                const int c = min(CS * sl + j, C - 1);
#pragma unroll
                for (int u = 0; u < 2; u++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        k[u][i] = P4 && i > 1 ? (ip[u][i][c >> 1] >> (4 * (c & 1))) & 15 : ip[u][i][c];
            };
            load(0);
            for (int j = 0; j < CS; j++) {
                h8_t cw[2][4];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    cw[u][0] = cbs[k[u][0]];
                    cw[u][1] = cbs[K + k[u][1]];
                    cw[u][2] = cbs[2 * K + k[u][2]];
                    cw[u][3] = cbs[2 * K + K2 + k[u][3]];
                }
                load(min(j + 1, CS - 1));                     // in flight during the sums
                float xv[16], cm = 0.f;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float4 f = *(const float4*)(xd + sl * dxs + 16 * j + 4 * v);
                    xv[4 * v] = f.x; xv[4 * v + 1] = f.y; xv[4 * v + 2] = f.z; xv[4 * v + 3] = f.w;
                }
#pragma unroll
                for (int v = 0; v < 16; v++) cm = fmaxf(cm, fabsf(xv[v]));
                const bool keep = t.skip_mode == 1 ? (gmax > 0.f ? cm >= gmax * t.skip_val : true)
                                : t.skip_mode == 2 ? (t.skip_val > 0.f ? cm > t.skip_val : true) : true;
                if (!keep || CS * sl + j >= C) continue;
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    acc[u] = acc[u] + (entry(cw[u][0], xv) + entry(cw[u][1], xv + 8));
                    acc[u] = acc[u] + (entry(cw[u][2], xv) + entry(cw[u][3], xv + 8));
                }
            }
            const int n = min(64, ns - s0);
#pragma unroll
            for (int u = 0; u < 2; u++)
                for (int l = 0; l < n; l++) tot[u] = tot[u] + __shfl(acc[u], first + l, 64);
        }
#pragma unroll
        for (int u = 0; u < 2; u++)
            if (sub == 0 && r + u < hi) sums[r + u] = tot[u];
    }
    __syncthreads();
}

// KA: every codebook a multiple of 32 codes (every table row of a tile is
// stored).  LV: 1 one level; 2 both, the second's tables beside the first's in
// LDS (132 KB at 256 codes each) and its index bytes behind the first's; 3 the
// second's indices packed 4-bit (16 codes).  NR: row
// tiles per block, the tables shared by both (used where one tile each would
// need a second round of blocks: 32000 x 4096, level 1, 504 blocks of one 17.7
// us, 256 of two 13.5 us).
template <bool KA, int LV, int NR>
__global__ __launch_bounds__(kFThreads) void pq_fused(PqDev t, const float* __restrict__ x, float* __restrict__ out,
                                                      int S, unsigned long long* __restrict__ racc,
                                                      const unsigned long long* __restrict__ hdr) {
    constexpr int CS = kFCS;
    constexpr bool TWO = LV > 1, P4 = LV == 3;
    extern __shared__ __align__(16) float T[];            // [CS][TS]
    __shared__ float red[kFThreads / 64], redc[kFThreads / 64], redc2[TWO ? kFThreads / 64 : 1];
    __shared__ float cmax_s[2][CS];
    __shared__ int8_t qq_s[1024];
    __shared__ float ox_s[32], os_s[32];                   // fewer than 32 outliers: their x and scales
    __shared__ h8_t cbs[(TWO ? 4 : 2) * 256];              // the codebooks, fp16 rows padded to 8
    __shared__ __align__(16) float xsl[CS * kXS];          // the slab's x: [chunk][side][8], zero padded
    const int K = t.K, C = t.C, G = t.G, M = t.M, hf = G / 2;
    const int TS = 2 * K + 4;                              // padded chunk stride (bank spread)
    const int K2 = TWO ? t.K2 : 0, TS2 = 2 * K2 + 4;
    float* T2 = T + (size_t)CS * TS;                       // TWO: [CS][TS2]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // XCD-aware order: dispatch puts block b on XCD b % 8, so logical block
    // (b % 8) * (nb / 8) + b / 8 keeps consecutive slabs of a tile on one XCD
    const int nb = gridDim.x, bx = blockIdx.x;
    const int lb = (nb & 7) ? bx : (bx & 7) * (nb >> 3) + (bx >> 3);
    const int rt = lb / S, sl = lb - rt * S;
    const int c0 = sl * CS, cn = min(CS, C - c0);
    const int q = tid & 1;
    const int r0 = rt * (kFRows * NR) + (tid >> 1);        // row of tile h: r0 + h * kFRows
    // the workspace stamp (caller workspaces): its address, and the magic
    const bool wsok = !hdr || (hdr[0] == kPqStamp && hdr[1] == (unsigned long long)(uintptr_t)hdr);
    if (!TWO && S > 1 && !wsok) {
#pragma unroll
        for (int h = 0; h < NR; h++)
            if (q == 0 && r0 + h * kFRows < M) out[r0 + h * kFRows] = __builtin_nanf("");
        if (tid == 0) __hip_atomic_fetch_or(&ibh_pq_err, (unsigned)IBH_DEVERR_PQ_WS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    unsigned long long* const words = racc ? racc : pq_row_acc;

    // 1. loads: the slab's x, the codebooks, x for the max|x| scan, the index
    // bytes (in the order they are needed; loads complete in issue order)
    const int ninner = C * G;
    const bool x4ok = !t.inner && (ninner & 3) == 0 && ninner <= 16 * kFThreads;
    const bool slab4 = x4ok && G == 16;                    // the slab's x as float4s (c0 * 16 floats)
    float4 xsv = make_float4(0.f, 0.f, 0.f, 0.f);
    if (slab4) xsv = ld4f(x + 4 * ((size_t)c0 * 4 + min(tid, cn * 4 - 1)));
    const bool cb16 = hf == 8;
    uint4 cbv = make_uint4(0, 0, 0, 0);
    if (cb16) {
        const int ci = min(tid, 2 * K - 1);
        cbv = ld16((ci < K ? t.cb1l : t.cb1r) + (size_t)(ci < K ? ci : ci - K) * 8);
    }
    uint4 cbv2 = make_uint4(0, 0, 0, 0);
    if (TWO && cb16) {
        const int ci = min(tid, 2 * K2 - 1);
        cbv2 = ld16((ci < K2 ? t.cb2l : t.cb2r) + (size_t)(ci < K2 ? ci : ci - K2) * 8);
    }
    __builtin_amdgcn_sched_barrier(0);
    float4 xs4[4];
    if (x4ok) {
        const int n4 = ninner >> 2;
#pragma unroll
        for (int u = 0; u < 4; u++) xs4[u] = ld4f(x + 4 * (size_t)min(u * kFThreads + tid, n4 - 1));
    }
    // the index bytes last, unconditionally (a load under a branch is waited
    // for where it joins): 16 chunks from w0 on, the thread's own or, where the
    // row ends before, its last 16.  A row of fewer loads pq_spare and its
    // bytes one by one below (64 lanes' bytes lie in 64 lines, and a load takes
    // a clock for each: 1024 x 3200, 256 + 256 codes 24.3 us with byte loads
    // for every C that is not a multiple of 16, 11.2 so).
    __builtin_amdgcn_sched_barrier(0);
    const bool vec = C >= 16;
    const int w0 = min(c0 + 16 * q, max(C - 16, 0));
    const uint8_t* const spare = (const uint8_t*)&pq_spare;
    const uint8_t *const b1l = vec ? t.i1l : spare, *const b1r = vec ? t.i1r : spare;
    const uint8_t *const b2l = vec ? t.i2l : spare, *const b2r = vec ? t.i2r : spare;
    // level 2: 16 bytes a side, or 8 of packed 4-bit indices (from the even
    // chunk e0; a last piece of an odd C starts one behind w0, whose own index
    // is then another thread's)
    const int e0 = min(c0 + 16 * q, max(((C + 1) & ~1) - 16, 0));
    uint4 ivl[NR], ivr[NR], jvl[NR], jvr[NR];
#pragma unroll
    for (int h = 0; h < NR; h++) {
        const size_t rr = min(r0 + h * kFRows, M - 1), io = vec ? rr * C + w0 : 0;
        ivl[h] = ld16(b1l + io);
        ivr[h] = ld16(b1r + io);
        jvl[h] = jvr[h] = make_uint4(0, 0, 0, 0);
        if constexpr (P4) {
            const size_t po = vec ? rr * ((C + 1) >> 1) + (e0 >> 1) : 0;
            const u2a_t a = *(const u2a_t*)(b2l + po), b = *(const u2a_t*)(b2r + po);
            jvl[h] = make_uint4(a.x, a.y, 0, 0);
            jvr[h] = make_uint4(b.x, b.y, 0, 0);
        } else if constexpr (TWO) {
            jvl[h] = ld16(b2l + io);
            jvr[h] = ld16(b2r + io);
        }
    }
    PQ_TT(0);

    // codebooks and the slab's x into LDS; the slab's max|x| and max|codeword|
    // (fmaxf drops NaN, so what is not finite is flagged on its own: x below,
    // and for two levels the codewords here, which the three-kernel path
    // carries into the rows that use them)
    float mc = 0.f, ms = 0.f, mc2 = 0.f;
    bool nonfin = false;
    if (tid < 2 * K) {
        h8_t h;
        if (cb16) h = __builtin_bit_cast(h8_t, cbv);
        else {
            const uint16_t* cr = (tid < K ? t.cb1l : t.cb1r) + (size_t)(tid < K ? tid : tid - K) * hf;
#pragma unroll
            for (int i = 0; i < 8; i++) h[i] = i < hf ? __builtin_bit_cast(_Float16, cr[min(i, hf - 1)]) : (_Float16)0.f;
        }
        cbs[tid] = h;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            mc = fmaxf(mc, fabsf((float)h[i]));
            if (TWO) nonfin |= !(fabsf((float)h[i]) <= 65504.f);
        }
    }
    if (TWO && tid < 2 * K2) {
        h8_t h;
        if (cb16) h = __builtin_bit_cast(h8_t, cbv2);
        else {
            const uint16_t* cr = (tid < K2 ? t.cb2l : t.cb2r) + (size_t)(tid < K2 ? tid : tid - K2) * hf;
#pragma unroll
            for (int i = 0; i < 8; i++) h[i] = i < hf ? __builtin_bit_cast(_Float16, cr[min(i, hf - 1)]) : (_Float16)0.f;
        }
        cbs[2 * K + tid] = h;
        float m2 = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            m2 = fmaxf(m2, fabsf((float)h[i]));
            nonfin |= !(fabsf((float)h[i]) <= 65504.f);
        }
        mc2 = m2;
    }
    if (slab4) {
        if (tid < cn * 4) {
            ((float4*)(xsl + (tid >> 2) * kXS))[tid & 3] = xsv;
            ms = fmaxf(fmaxf(fabsf(xsv.x), fabsf(xsv.y)), fmaxf(fabsf(xsv.z), fabsf(xsv.w)));
        }
    } else {
        for (int i = tid; i < cn * 16; i += kFThreads) {
            const int cc = i >> 4, sd = (i >> 3) & 1, e = i & 7;
            const float v = e < hf ? x[inner_col(t, (c0 + cc) * G + sd * hf + e)] : 0.f;
            xsl[cc * kXS + sd * 8 + e] = v;
            ms = fmaxf(ms, fabsf(v));
        }
    }
    ms = wave_max_dpp(ms);
    mc = wave_max_dpp(mc);
    if (TWO) mc2 = wave_max_dpp(mc2);
    if (lane == 0) {
        red[wave] = ms;
        redc[wave] = mc;
        if (TWO) redc2[wave] = mc2;
    }
    __syncthreads();
    float smax = 0.f, cbmax = 0.f, cbmax2 = 0.f;
#pragma unroll
    for (int w = 0; w < kFThreads / 64; w++) {
        smax = fmaxf(smax, red[w]);
        cbmax = fmaxf(cbmax, redc[w]);
        if (TWO) cbmax2 = fmaxf(cbmax2, redc2[w]);
    }
    if (TWO) cbmax += cbmax2;
    // the tables carry 2^-ex, the slab's max|x| below 2^15
    int ex = 0;
    if (smax > 0.f) frexpf(smax, &ex);                     // smax < 2^ex
    ex = max(ex, kMinExp) - 15;

    // 2. tables
    slab_tables<KA, TWO>(K, K2, cbs, xsl, cn, wave, lane, ex, T, T2, cmax_s);
    PQ_TT(1);
    // max|x| over the inner columns (the skipping rule's reference) and sum|x|
    float mx = 0.f, sx = 0.f;
    float ox = 0.f, osc = 0.f;                             // thread j: outlier j's x and scale
    if (t.n_outlier > 0) {
        const int j = min(tid, t.n_outlier - 1);
        ox = x[t.ocols[j]];
        osc = f16_to_f32(t.oscale[j]);
    }
    if (x4ok) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const float a = fmaxf(fmaxf(fabsf(xs4[u].x), fabsf(xs4[u].y)), fmaxf(fabsf(xs4[u].z), fabsf(xs4[u].w)));
            const float b = (fabsf(xs4[u].x) + fabsf(xs4[u].y)) + (fabsf(xs4[u].z) + fabsf(xs4[u].w));
            mx = fmaxf(mx, a);
            sx += u * kFThreads + tid < ninner >> 2 ? b : 0.f;
            nonfin |= !(fabsf(xs4[u].x) <= 3.4e38f && fabsf(xs4[u].y) <= 3.4e38f && fabsf(xs4[u].z) <= 3.4e38f &&
                        fabsf(xs4[u].w) <= 3.4e38f);
        }
    } else {
        for (int j0 = 0; j0 < ninner; j0 += 16 * kFThreads) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) v[u] = x[inner_col(t, min(j0 + u * kFThreads + tid, ninner - 1))];
#pragma unroll
            for (int u = 0; u < 16; u++) {
                mx = fmaxf(mx, fabsf(v[u]));
                sx += j0 + u * kFThreads + tid < ninner ? fabsf(v[u]) : 0.f;
                nonfin |= !(fabsf(v[u]) <= 3.4e38f);
            }
        }
    }
    mx = wave_max_dpp(mx);
    sx = wave_sum_dpp(sx);
    __syncthreads();                                       // tables done; red[] read above
    if (lane == 0) {
        red[wave] = mx;
        redc[wave] = sx;
    }
    const bool nonfinite = __syncthreads_or(nonfin) != 0;
    
    float gmax = 0.f, gsum = 0.f;
#pragma unroll
    for (int w = 0; w < kFThreads / 64; w += 4) {
        gmax = fmaxf(fmaxf(gmax, fmaxf(red[w], red[w + 1])), fmaxf(red[w + 2], red[w + 3]));
        gsum += (redc[w] + redc[w + 1]) + (redc[w + 2] + redc[w + 3]);
    }
    // the slab's kept chunks as a mask, made by every wavefront (lane = chunk)
    bool keep = false;
    if (lane < cn) {
        const float cm = fmaxf(cmax_s[0][lane], cmax_s[1][lane]);
        keep = t.skip_mode == 1 ? (gmax > 0.f ? cm >= gmax * t.skip_val : true)
             : t.skip_mode == 2 ? (t.skip_val > 0.f ? cm > t.skip_val : true) : true;
    }
    const unsigned long long keepm = __ballot(keep);
    const unsigned long long full = cn == 64 ? ~0ull : ((1ull << cn) - 1);
    PQ_TT(2);

    // 2^qe maps 2 * max|cb| * sum|x| (a bound on |row sum|) to <= 2^50; the
    // same on every slab (cbmax, gsum and the flag are over the whole tensor,
    // summed in the same order), so either every slab adds or none does
    const float bound = 2.0f * cbmax * gsum;
    // (two levels: neither does an x so small that its fp16 parts, scaled by at
    // most 2^115, or the bound would lose bits)
    const bool off = nonfinite || !(bound <= 3.4e38f) ||
                     (TWO && ((S > 1 && !wsok) || (gmax > 0.f && gmax < 1e-30f)));
    bool fin[NR];
    float sum[NR];
    uint16_t rs_bits[NR];
    if (TWO && off) {
        // rows that the tables cannot serve: every slab's block takes its share
        // of the tile's rows whole (the tables' LDS is free now)
        const int per = (kFRows * NR + S - 1) / S, lo = min(sl * per, kFRows * NR), hi = min(lo + per, kFRows * NR);
        float* const dsum = T + ((C >> t.slab_sh) + 1) * ((16 << t.slab_sh) + kDPad);
        direct_rows<P4>(t, x, cbs, T, dsum, rt * (kFRows * NR), lo, hi, gmax, tid);
#pragma unroll
        for (int h = 0; h < NR; h++) {
            const int r = r0 + h * kFRows, i = (tid >> 1) + h * kFRows;
            fin[h] = q == 0 && r < M && i >= lo && i < hi;
            sum[h] = dsum[i];
            rs_bits[h] = t.row_scale[min(r, M - 1)];
        }
    } else {
#pragma unroll
        for (int h = 0; h < NR; h++) {
            const int r = r0 + h * kFRows;
            // 4. gather: the thread's 16 chunks, L then R per chunk (entries carry 2^-ex)
            float acc = 0.f;
            if (vec) {
                const uint32_t wl[4] = {ivl[h].x, ivl[h].y, ivl[h].z, ivl[h].w}, wr[4] = {ivr[h].x, ivr[h].y, ivr[h].z, ivr[h].w};
                uint32_t vl[4] = {jvl[h].x, jvl[h].y, jvl[h].z, jvl[h].w}, vr[4] = {jvr[h].x, jvr[h].y, jvr[h].z, jvr[h].w};
                if (P4 && w0 != e0) {                          // nibble j: chunk w0 + j
                    vl[1] = vl[1] << 4 | vl[0] >> 28; vl[0] <<= 4;
                    vr[1] = vr[1] << 4 | vr[0] >> 28; vr[0] <<= 4;
                }
                // entry sum of the j-th loaded chunk, tables at Tc (and T2c)
                auto term = [&](int j, const float* Tc, const float* T2c) {
                    const int il = (wl[j >> 2] >> (8 * (j & 3))) & 0xff, ir = (wr[j >> 2] >> (8 * (j & 3))) & 0xff;
                    float v = Tc[il] + Tc[K + ir];
                    if constexpr (TWO) {
                        const int jl = P4 ? (vl[j >> 3] >> (4 * (j & 7))) & 0xf : (vl[j >> 2] >> (8 * (j & 3))) & 0xff;
                        const int jr = P4 ? (vr[j >> 3] >> (4 * (j & 7))) & 0xf : (vr[j >> 2] >> (8 * (j & 3))) & 0xff;
                        v = v + (T2c[jl] + T2c[K2 + jr]);
                    }
                    return v;
                };
                const float* Tq = T + (size_t)(16 * q) * TS;
                const float* Tq2 = T2 + (size_t)(16 * q) * TS2;
                if (cn == CS && keepm == full) {
#pragma unroll
                    for (int j = 0; j < 16; j++) acc = acc + term(j, Tq + j * TS, Tq2 + j * TS2);
                } else if (cn == CS) {
#pragma unroll
                    for (int j = 0; j < 16; j++) {
                        const float val = term(j, Tq + j * TS, Tq2 + j * TS2);
                        acc = acc + (((keepm >> (16 * q + j)) & 1) ? val : 0.f);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 16; j++) {
                        // chunks of the other thread or slab are loaded and not added
                        const int c = w0 - c0 + j, cc = max(c, 0);
                        const float val = term(j, T + cc * TS, T2 + cc * TS2);
                        acc = acc + (c >= 16 * q && ((keepm >> cc) & 1) ? val : 0.f);
                    }
                }
            } else if (r < M) {
                const uint8_t* pl = t.i1l + (size_t)r * C + c0;
                const uint8_t* pr = t.i1r + (size_t)r * C + c0;
                const size_t l2s = TWO ? l2_stride(t) : 0;
                for (int c = 16 * q; c < min(16 * q + 16, cn); c++) {
                    const float* Tc = T + (size_t)c * TS;
                    float val = Tc[pl[c]] + Tc[K + pr[c]];
                    if constexpr (TWO) {
                        const float* Tc2 = T2 + (size_t)c * TS2;
                        val = val + (Tc2[l2_at(t, t.i2l + (size_t)r * l2s, c0 + c)] +
                                     Tc2[K2 + l2_at(t, t.i2r + (size_t)r * l2s, c0 + c)]);
                    }
                    acc = acc + (((keepm >> c) & 1) ? val : 0.f);
                }
            }
            // the row's two partials, lanes 2i, 2i+1
            acc += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, acc), 0xB1, 0xF, 0xF, false));
            PQ_TT(3);

            // 5. the rows' words
            const bool own = q == 0 && r < M;
            fin[h] = own;
            sum[h] = ldexpf(acc, ex);
            rs_bits[h] = t.row_scale[min(r, M - 1)];   // in flight with the atomic below
            if (S > 1 && off) {
                if (own) out[r] = __builtin_nanf("");
                fin[h] = false;
            }
            if (S > 1 && own && !off) {
                int eb = 0;
                if (bound > 0.f) frexpf(bound, &eb);               // bound < 2^eb
                const int qe = 50 - eb;
                const long long v = llrint((double)acc * ldexp(1.0, qe + ex));
                const unsigned long long add = (1ull << 58) + (unsigned long long)(v + (1ll << 50));
                const unsigned long long old =
                    __hip_atomic_fetch_add(&words[r], add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const unsigned long long tot = old + add;
                fin[h] = (tot >> 58) == (unsigned long long)S;
                if (fin[h]) {
                    const long long val = (long long)(tot & ((1ull << 58) - 1)) - (long long)S * (1ll << 50);
                    sum[h] = (float)((double)val * ldexp(1.0, -qe));
                    __hip_atomic_store(&words[r], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
    }
    PQ_TT(4);
    // outliers (pq_decode.c:1233-1421): int8-quantised dot for >= 32
    // outliers, fp32 otherwise
    const int no = t.n_outlier;
    const bool quant = no >= 32;
    float meta = 1.f;
    if (no > 0) {
        bool any = false;
#pragma unroll
        for (int h = 0; h < NR; h++) any |= fin[h];
        if (__syncthreads_or(any) == 0) return;
        // (the largest product by a reduction over the threads, one product each:
        // thread 0 walking 128 of them took 20 us)
        const float ov = ox * osc;
        if (quant) {
            const float m = wave_max_dpp(tid < no ? fabsf(ov) : 0.f);
            if (lane == 0) red[wave] = m;
        } else if (tid < no) {
            ox_s[tid] = ox;
            os_s[tid] = osc;
        }
        __syncthreads();
        if (quant) {
            float m = 0.f;
#pragma unroll
            for (int w = 0; w < kFThreads / 64; w++) m = fmaxf(m, red[w]);
            meta = m > 0.f ? m / 127.0f : 1.0f;
            if (tid < no) {
                const float sv = ov * (1.0f / meta);
                const int v = (int)(sv >= 0 ? sv + 0.5f : sv - 0.5f);
                qq_s[tid] = (int8_t)(v > 127 ? 127 : (v < -128 ? -128 : v));
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int h = 0; h < NR; h++) {
        if (!fin[h]) continue;
        const int r = r0 + h * kFRows;
        float y = sum[h] * f16_to_f32(rs_bits[h]);
        if (no > 0) {
            const int8_t* sdc = t.oside + (size_t)r * no;
            if (quant) {
                int32_t isum = 0;
#pragma unroll 8
                for (int j = 0; j < no; j++) isum += (int32_t)sdc[j] * (int32_t)qq_s[j];
                y = fmaf((float)isum, meta, y);
            } else {
#pragma unroll 8
                for (int j = 0; j < no; j++) y = fmaf((float)sdc[j] * os_s[j], ox_s[j], y);
            }
        }
        out[r] = y;
    }
    PQ_TT(5);
}

// ── top-K LM head (ib_pq_lm_head_topk, pq_decode.c:2259-2346) ─────────────
// Order key of a float, descending: smaller key = larger value.
__device__ __forceinline__ uint32_t desc_key(float v) {
    const uint32_t f = __float_as_uint(v);
    const uint32_t u = (f & 0x80000000u) ? ~f : (f | 0x80000000u);
    return ~u;
}

constexpr int kSelThreads = 1024;

// The K largest of v[0..M): radix select of the K-th key (4 passes of 8 bits;
// per-wavefront histograms, the bin search one wavefront-wide scan), then
// every element above it plus the first ties of the K-th key in index order;
// the selection ends sorted by row index.  One block.
__device__ void topk_radix(const float* __restrict__ v, int M, int K, int32_t* __restrict__ sel) {
    constexpr int NW = kSelThreads / 64;
    __shared__ int hist[NW][256];
    __shared__ int tot[256];
    __shared__ int tmp[1024];
    __shared__ uint32_t s_prefix, s_mask;
    __shared__ int s_kk, s_nless, s_neq, s_eqtot;
    __shared__ int wcnt[NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) { s_prefix = 0; s_mask = 0; s_kk = K; s_nless = 0; s_neq = 0; s_eqtot = 0; }
    for (int pass = 0; pass < 4; pass++) {
        const int shift = 24 - 8 * pass;
        for (int e = tid; e < NW * 256; e += kSelThreads) (&hist[0][0])[e] = 0;
        __syncthreads();
        const uint32_t prefix = s_prefix, mask = s_mask;
        for (int i = tid; i < M; i += kSelThreads) {
            const uint32_t d = desc_key(v[i]);
            if ((d & mask) == prefix) atomicAdd(&hist[wave][(d >> shift) & 255], 1);
        }
        __syncthreads();
        if (tid < 256) {
            int c = 0;
#pragma unroll
            for (int w = 0; w < NW; w++) c += hist[w][tid];
            tot[tid] = c;
        }
        __syncthreads();
        if (wave == 0) {
            // first bin b (<= 255) whose inclusive count reaches kk
            int c[4], sum = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) { c[j] = tot[4 * lane + j]; sum += c[j]; }
            int incl = sum;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int n = __shfl_up(incl, o, 64);
                if (lane >= o) incl += n;
            }
            const int excl = incl - sum, kk = s_kk;
            const bool last = lane == 63;
            if ((excl < kk && kk <= incl) || (last && incl < kk)) {
                int cum = excl, j = 0;
                for (; j < 3; j++) {
                    if (cum + c[j] >= kk) break;
                    cum += c[j];
                }
                s_kk = kk - cum;
                s_prefix = prefix | ((uint32_t)(4 * lane + j) << shift);
                s_mask = mask | (0xFFu << shift);
            }
        }
        __syncthreads();
    }
    const uint32_t kth = s_prefix;
    const int take_eq = s_kk;                     // ties of the K-th key to keep, lowest indices first
    for (int i = tid; i < M; i += kSelThreads) {
        const uint32_t d = desc_key(v[i]);
        if (d < kth) sel[atomicAdd(&s_nless, 1)] = i;
        else if (d == kth) atomicAdd(&s_eqtot, 1);
    }
    __syncthreads();
    if (s_eqtot <= take_eq) {
        for (int i = tid; i < M; i += kSelThreads)
            if (desc_key(v[i]) == kth) sel[(K - take_eq) + atomicAdd(&s_neq, 1)] = i;
    } else {
        // more ties than places: the lowest indices, in index order
        for (int base = 0; base < M; base += kSelThreads) {
            const int i = base + tid;
            const bool eq = i < M && desc_key(v[i]) == kth;
            const unsigned long long b = __ballot(eq);
            if (lane == 0) wcnt[wave] = __popcll(b);
            __syncthreads();
            int before = s_neq;
            for (int w = 0; w < wave; w++) before += wcnt[w];
            const int r = before + __popcll(b & ((1ull << lane) - 1ull));
            if (eq && r < take_eq) sel[(K - take_eq) + r] = i;
            __syncthreads();
            if (tid == 0) {
                int t = 0;
                for (int w = 0; w < NW; w++) t += wcnt[w];
                s_neq += t;
            }
            __syncthreads();
            if (s_neq >= take_eq) break;
        }
    }
    __syncthreads();
    // selection order = row index order (K <= 1024, distinct rows)
    __threadfence_block();
    for (int i = tid; i < K; i += kSelThreads) {
        const int r = sel[i];
        int rank = 0;
        for (int j = 0; j < K; j++) rank += sel[j] < r;
        tmp[rank] = r;
    }
    __syncthreads();
    for (int i = tid; i < K; i += kSelThreads) sel[i] = tmp[i];
}

__global__ __launch_bounds__(kSelThreads) void pq_topk_select(const float* __restrict__ v, int M, int K,
                                                              int32_t* __restrict__ sel) {
    topk_radix(v, M, K, sel);
}

// The same selection for K <= kPickK without histograms (logits crowd a few
// exponents, so the radix passes' LDS atomics pile up on a few bins: 44.8 us
// for 50 of 32000).  Each thread keeps the best of its share; the K-th best of
// those 1024 is a bound that at least K values reach and few others do, found
// bit by bit with ballots; the values within it (more than kSelThreads of
// them, as with many ties, take the radix passes) are ranked by (key, index)
// against each other.  One block, one read of v up to 32768 values: 13.4 us.
constexpr int kPickK = 256, kPickPer = 32;

__global__ __launch_bounds__(kSelThreads) void pq_topk_pick(const float* __restrict__ v, int M, int K,
                                                            int32_t* __restrict__ sel) {
    constexpr int NW = kSelThreads / 64;
    __shared__ __align__(16) int cnt[2][NW];
    __shared__ unsigned long long ck[kSelThreads];        // key, row
    __shared__ int pick[kPickK];
    __shared__ int nc_s;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) nc_s = 0;
    // v is a workspace array of whole 256-byte lines, so the last float4 may
    // hold values past M that no key is made of
    uint32_t key[kPickPer], best = 0xFFFFFFFFu;
    const int span = kPickPer * kSelThreads, n4 = (M + 3) >> 2;
    auto at = [&](int base, int u) { return base + 4 * ((u >> 2) * kSelThreads + tid) + (u & 3); };
    auto load = [&](int base) {
        float4 f[kPickPer / 4];
#pragma unroll
        for (int u = 0; u < kPickPer / 4; u++) f[u] = ((const float4*)v)[min(base / 4 + u * kSelThreads + tid, n4 - 1)];
#pragma unroll
        for (int u = 0; u < kPickPer; u++) {
            const float4 q = f[u >> 2];
            const float e = (u & 3) == 0 ? q.x : (u & 3) == 1 ? q.y : (u & 3) == 2 ? q.z : q.w;
            key[u] = at(base, u) < M ? desc_key(e) : 0xFFFFFFFFu;
        }
    };
    for (int base = 0; base < M; base += span) {
        load(base);
#pragma unroll
        for (int u = 0; u < kPickPer; u++) best = min(best, key[u]);
    }
    // smallest bound with at least K of the threads' best keys at or below it
    uint32_t p = 0;
    for (int bit = 31; bit >= 0; bit--) {
        const uint32_t trial = p + ((1u << bit) - 1u);
        const int c = __popcll(__ballot(best <= trial));
        if (lane == 0) cnt[bit & 1][wave] = c;
        __syncthreads();
        int n = 0;
#pragma unroll
        for (int w = 0; w < NW; w += 4) {
            const int4 q = *(const int4*)&cnt[bit & 1][w];
            n += q.x + q.y + q.z + q.w;
        }
        if (n < K) p += 1u << bit;
    }
    for (int base = 0; base < M; base += span) {
        if (M > span) load(base);
#pragma unroll
        for (int u = 0; u < kPickPer; u++) {
            const int i = at(base, u);
            if (i < M && key[u] <= p) {
                const int n = atomicAdd(&nc_s, 1);
                if (n < kSelThreads) ck[n] = ((unsigned long long)key[u] << 32) | (uint32_t)i;
            }
        }
    }
    __syncthreads();
    const int nc = nc_s;
    if (nc > kSelThreads) {
        topk_radix(v, M, K, sel);
        return;
    }
    // ranks, 8 lanes a candidate (their shares of the comparisons independent)
    const int sub = tid & 7;
    for (int b = 0; b < nc; b += kSelThreads / 8) {
        const int c = b + (tid >> 3);
        const unsigned long long k = ck[min(c, nc - 1)];
        int rank = 0;
#pragma unroll 4
        for (int j = sub; j < nc; j += 8) rank += ck[j] < k;
        rank = (int)group_sum_dpp<8>((float)rank);
        if (c < nc && rank < K && sub == 0) pick[rank] = (int)(uint32_t)k;
    }
    __syncthreads();
    for (int b = 0; b < K; b += kSelThreads / 8) {
        const int c = b + (tid >> 3), i = pick[min(c, K - 1)];
        int rank = 0;
#pragma unroll 4
        for (int j = sub; j < K; j += 8) rank += pick[j] < i;
        rank = (int)group_sum_dpp<8>((float)rank);
        if (c < K && sub == 0) sel[rank] = i;
    }
}

// Full-pyramid logits of the selected rows (ib_pq_matmul_fp32_subset,
// pq_decode.c:2145-2250): one block per row, a chunk per thread, the outlier
// sidecar in fp32.  Two dependent reads (indices, codewords) set its time, so
// a codeword of 8 halves is one 16-byte load and no thread has a second chunk
// up to 256 (one wavefront per row with 2-byte loads, 4 chunks a lane: 18.5 us
// for 50 rows of 256 chunks; 5.2 us).
__global__ __launch_bounds__(256) void pq_subset_rows(PqDev t, const float* __restrict__ x,
                                                      const int32_t* __restrict__ rows, int n,
                                                      float* __restrict__ out) {
    __shared__ float red[2][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = blockIdx.x;
    const int r = rows[i], C = t.C, G = t.G, hf = G / 2;
    const bool two = t.n_levels == 2;
    const size_t l2s = two ? l2_stride(t) : 0;
    const bool wide = hf == 8 && (((uintptr_t)t.cb1l | (uintptr_t)t.cb1r | (two ? (uintptr_t)t.cb2l | (uintptr_t)t.cb2r : 0)) & 15) == 0;
    float acc = 0.f;
    for (int c = tid; c < C; c += 256) {
        const uint16_t* e[4];
        e[0] = t.cb1l + (size_t)t.i1l[(size_t)r * C + c] * hf;
        e[1] = t.cb1r + (size_t)t.i1r[(size_t)r * C + c] * hf;
        e[2] = two ? t.cb2l + (size_t)l2_at(t, t.i2l + (size_t)r * l2s, c) * hf : e[0];
        e[3] = two ? t.cb2r + (size_t)l2_at(t, t.i2r + (size_t)r * l2s, c) * hf : e[1];
        if (wide) {
            uint4 w[4];
#pragma unroll
            for (int k = 0; k < 4; k++) w[k] = *(const uint4*)e[k];
            float xv[16];
#pragma unroll
            for (int j = 0; j < 16; j++) xv[j] = x[inner_col(t, c * 16 + j)];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                auto half = [&](int k) {
                    const uint32_t d[4] = {w[k].x, w[k].y, w[k].z, w[k].w};
                    return f16_to_f32((uint16_t)(d[j >> 1] >> (16 * (j & 1))));
                };
                acc = fmaf(half(0), xv[j], acc);
                acc = fmaf(half(1), xv[8 + j], acc);
                if (two) {
                    acc = fmaf(half(2), xv[j], acc);
                    acc = fmaf(half(3), xv[8 + j], acc);
                }
            }
            continue;
        }
        for (int j = 0; j < hf; j++) {
            const float xl = x[inner_col(t, c * G + j)], xr = x[inner_col(t, c * G + hf + j)];
            acc = fmaf(f16_to_f32(e[0][j]), xl, acc);
            acc = fmaf(f16_to_f32(e[1][j]), xr, acc);
            if (two) {
                acc = fmaf(f16_to_f32(e[2][j]), xl, acc);
                acc = fmaf(f16_to_f32(e[3][j]), xr, acc);
            }
        }
    }
    float o = 0.f;
    for (int j = tid; j < t.n_outlier; j += 256)
        o = fmaf((float)t.oside[(size_t)r * t.n_outlier + j] * f16_to_f32(t.oscale[j]), x[t.ocols[j]], o);
    acc = wave_sum(acc);
    o = wave_sum(o);
    if (lane == 0) {
        red[0][wave] = acc;
        red[1][wave] = o;
    }
    __syncthreads();
    if (tid == 0)
        out[i] = ((red[0][0] + red[0][1]) + (red[0][2] + red[0][3])) * f16_to_f32(t.row_scale[r]) +
                 ((red[1][0] + red[1][1]) + (red[1][2] + red[1][3]));
}

// Descending order of the refined logits (the reference's insertion sort:
// ties keep their selection order, here row order).  One block, K <= 1024.
__global__ __launch_bounds__(1024) void pq_topk_sort(const float* __restrict__ val, const int32_t* __restrict__ ids,
                                                     int K, float* __restrict__ out_v, int32_t* __restrict__ out_i) {
    for (int i = threadIdx.x; i < K; i += 1024) {
        const float v = val[i];
        int rank = 0;
        for (int j = 0; j < K; j++) {
            const float w = val[j];
            rank += (w > v) || (w == v && j < i);
        }
        out_v[rank] = v;
        out_i[rank] = ids[i];
    }
}

}  // namespace

void* ibh_workspace(size_t bytes);

typedef ibh_pq_tensor ibh_pq_tensor_abi;

// Workspace: both levels' tables for all chunks, the per-slab partial sums,
// then the chunk maxima, the chunk norms and the cluster bounds.
struct PqWs {
    size_t tab1, tab2, part, cmax, cnorm, c2max, need;
};

// front: the stamp and row words of a caller workspace come first
static int pq_geometry(const ibh_pq_tensor_abi* t, int* CS, int* nslabs, size_t* lds, PqWs* w, bool front = true) {
    const bool two = t->n_levels == 2;
    const int K2 = t->K_l2 > 0 ? t->K_l2 : t->K;
    int cs = 16;
    auto need = [&](int c) { return (size_t)c * 2 * t->K * 4 + (two ? (size_t)c * 2 * K2 * 4 : 0); };
    while (cs > 1 && need(cs) > 60 * 1024) cs >>= 1;
    if (need(cs) > 60 * 1024) return IBH_ERROR_PARAM;
    *CS = cs;
    *nslabs = (t->C + cs - 1) / cs;
    *lds = need(cs);
    auto al = [](size_t v) { return (v + 255) / 256 * 256; };
    w->tab1 = front ? kPqFront : 0;
    w->tab2 = w->tab1 + al((size_t)t->C * 2 * t->K * 4);
    w->part = w->tab2 + (two ? al((size_t)t->C * 2 * K2 * 4) : 0);
    w->cmax = w->part + al((size_t)(*nslabs) * t->M * sizeof(float));
    w->cnorm = w->cmax + al((size_t)t->C * sizeof(float));
    w->c2max = w->cnorm + al((size_t)t->C * 2 * sizeof(float));
    w->need = w->c2max + al((size_t)2 * (t->K + 1) * sizeof(float));
    return IBH_OK;
}

namespace {
// The stamp of a caller workspace and zero row words (a fill kernel, not a
// memset, so that a captured graph may hold it).
__global__ void pq_ws_init(unsigned long long* __restrict__ w) {
    const size_t n = kPqFront / 8;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        w[i] = i == 0 ? kPqStamp : (i == 1 ? (unsigned long long)(uintptr_t)w : 0ull);
}
}  // namespace

extern "C" int ibh_pq_workspace_init(void* ws, size_t ws_bytes, void* stream) {
    if (!ws || ws_bytes < kPqFront || ((uintptr_t)ws & 255)) {
        ibh_set_error("ibh_pq_workspace_init: need a 256-byte aligned workspace of >= %zu bytes", kPqFront);
        return IBH_ERROR_PARAM;
    }
    pq_ws_init<<<256, 256, 0, ibh_resolve_stream(stream)>>>((unsigned long long*)ws);
    IBH_CHECK_LAUNCH("ibh_pq_workspace_init");
    return IBH_OK;
}

int ibh_pq_errors(bool clear) {
    unsigned int v = 0;
    if (hipMemcpyFromSymbol(&v, HIP_SYMBOL(ibh_pq_err), sizeof(v)) != hipSuccess) return -1;
    if (clear && v) {
        const unsigned int z = 0;
        if (hipMemcpyToSymbol(HIP_SYMBOL(ibh_pq_err), &z, sizeof(z)) != hipSuccess) return -1;
    }
    return (int)v;
}

static size_t pq_ws_need(const ibh_pq_tensor_abi* t, bool front) {
    int cs, ns;
    size_t lds;
    PqWs w;
    return t && pq_geometry(t, &cs, &ns, &lds, &w, front) == IBH_OK ? w.need : 0;
}

extern "C" size_t ibh_pq_workspace_bytes(const ibh_pq_tensor_abi* t) { return pq_ws_need(t, true); }

namespace {
struct PqMode {
    int skip_mode = 1;        // see PqDev
    float skip_val = 0.01f;
    bool level2 = true;       // false: level 1 only
    bool q8 = false;
    bool l2skip = false;
    float l2_thr = 0.f;
    bool tq8 = false;         // tables quantised to int8 per (chunk, side) (q8lut)
};

// ib_pq_matmul_fp32_q8lut's table quantisation (build_q8_lut,
// pq_decode.c:2405-2449): per (chunk, side) of each level, sc = max|T|/127
// (1 if 0), q = (int)(T * (1/sc) +- 0.5) clamped to [-128, 127]; the tables
// are replaced by q * sc, the terms the reference's gather adds.  Block per
// chunk, grid.y = level.
__global__ __launch_bounds__(kThreads) void pq_tq8(float* __restrict__ tab1, float* __restrict__ tab2, int K) {
    __shared__ float red[kThreads / 64];
    __shared__ float s_sc;
    float* tab = (blockIdx.y ? tab2 : tab1) + (size_t)blockIdx.x * 2 * K;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int side = 0; side < 2; side++) {
        float* T = tab + side * K;
        float m = 0.f;
        for (int k = threadIdx.x; k < K; k += kThreads) m = fmaxf(m, fabsf(T[k]));
        m = wave_max(m);
        if (lane == 0) red[wave] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            float mm = 0.f;
            for (int w = 0; w < kThreads / 64; w++) mm = fmaxf(mm, red[w]);
            s_sc = mm > 0.f ? mm / 127.0f : 1.0f;
        }
        __syncthreads();
        const float sc = s_sc, inv = 1.0f / sc;
        for (int k = threadIdx.x; k < K; k += kThreads) {
            const float u = T[k] * inv;
            int q = (int)(u >= 0 ? u + 0.5f : u - 0.5f);
            q = q > 127 ? 127 : (q < -128 ? -128 : q);
            T[k] = (float)q * sc;
        }
        __syncthreads();
    }
}
}  // namespace

// lib_ws: `ws` is the library workspace (no stamp; the library's row words)
static int pq_run(const ibh_pq_tensor_abi* t, const float* x, float* out, void* ws, size_t ws_bytes, void* stream,
                  const PqMode& md, const char* who, bool lib_ws = false);

extern "C" int ibh_pq_matmul(const ibh_pq_tensor_abi* t, const float* x, float* out, void* ws, size_t ws_bytes,
                             void* stream) {
    return pq_run(t, x, out, ws, ws_bytes, stream, PqMode{}, "ibh_pq_matmul");
}

extern "C" int ibh_pq_matmul_streaming(const ibh_pq_tensor_abi* t, const float* x, float* out, void* ws,
                                       size_t ws_bytes, void* stream) {
    const ibh_pq_policy p{IBH_PQ_VARIANT_STREAMING, 0.f, 0.f};
    return ibh_pq_matmul_policy(t, x, out, &p, ws, ws_bytes, stream);
}

// ib_pq_matmul_fp32_q8lut (pq_decode.c:2451-2561): every chunk, tables in the
// matmul_impl order quantised to int8 per (chunk, side), gather, row scale,
// outliers.  Its level-2 tables hold K entries read through uint8 indices,
// so a level-2 tensor must have K_l2 == K (not 16-packed, not 2-byte).
extern "C" int ibh_pq_matmul_q8lut(const ibh_pq_tensor_abi* t, const float* x, float* out, void* ws,
                                   size_t ws_bytes, void* stream) {
    if (t && (t->G > 32 || (t->n_levels == 2 && ((t->K_l2 > 0 && t->K_l2 != t->K) || t->K == 16 ||
                                                   t->l2_idx_bytes == 2)))) {
        ibh_set_error("ibh_pq_matmul_q8lut: needs G <= 32 and, with two levels, K_l2 == K (uint8 indices)");
        return IBH_ERROR_PARAM;
    }
    PqMode md;
    md.skip_mode = 0;
    md.tq8 = true;
    return pq_run(t, x, out, ws, ws_bytes, stream, md, "ibh_pq_matmul_q8lut");
}

// ib_pq_session_matmul's dispatch on the tensor's policy (pq_decode.c:4468-4491).
extern "C" int ibh_pq_matmul_policy(const ibh_pq_tensor_abi* t, const float* x, float* out, const ibh_pq_policy* p,
                                    void* ws, size_t ws_bytes, void* stream) {
    if (!p) {
        ibh_set_error("ibh_pq_matmul_policy: null policy");
        return IBH_ERROR_PARAM;
    }
    if (t && t->G > 32) {
        ibh_set_error("ibh_pq_matmul_policy: G=%d > 32 (the reference's chunk buffers hold 16 per side)", t->G);
        return IBH_ERROR_PARAM;
    }
    PqMode md;
    md.skip_mode = 0;
    switch (p->variant) {
    case IBH_PQ_VARIANT_L1_ONLY:
        md.level2 = false;
        break;
    case IBH_PQ_VARIANT_L2SKIP:
        md.l2skip = true;
        md.l2_thr = p->skip_threshold;
        if (t && t->format == IBH_PQ_FORMAT_PYRAMID && t->K > 256) {
            ibh_set_error("ibh_pq_matmul_policy: pyramid L2SKIP supports K <= 256 (K=%d)", t->K);
            return IBH_ERROR_PARAM;
        }
        break;
    case IBH_PQ_VARIANT_SPARSE:
        md.skip_mode = 2;
        md.skip_val = p->act_threshold;
        break;
    case IBH_PQ_VARIANT_INT8:
        md.q8 = true;
        break;
    default:   // STREAMING, and the reference's default branch
        break;
    }
    return pq_run(t, x, out, ws, ws_bytes, stream, md, "ibh_pq_matmul_policy");
}

static int g_pq_fused = 1;

// Development switch (no counterpart in the reference): 0 sends every PQ
// matvec through the three-kernel path, 1 (default) lets eligible tensors
// run in one launch.
#ifdef IBH_PQ_TRACE
extern "C" int ibh_pq_trace_read(void* out) {
    return hipMemcpyFromSymbol(out, HIP_SYMBOL(ibh_pq_tt), sizeof(ibh_pq_tt)) == hipSuccess ? 0 : -1;
}
#endif

extern "C" int ibh_pq_set_fused(int on) {
    g_pq_fused = on != 0;
    return IBH_OK;
}

static int pq_run(const ibh_pq_tensor_abi* t, const float* x, float* out, void* ws, size_t ws_bytes, void* stream,
                  const PqMode& md, const char* who, bool lib_ws) {
    if (!t || !x || !out || t->M <= 0 || t->C <= 0 || t->G <= 0 || t->G % 2 || t->G > 64 || t->K <= 0 || t->K > 65536 ||
        !t->codebook_l1_l || !t->codebook_l1_r || !t->indices_l1_l || !t->indices_l1_r || !t->row_scale ||
        t->N != t->C * t->G + t->n_outlier || t->n_outlier < 0 || t->n_outlier > 1024 ||
        (t->n_outlier > 0 && (!t->outlier_cols || !t->outlier_sidecar || !t->outlier_scale || !t->inner_cols)) ||
        (t->n_levels == 2 && (!t->codebook_l2_l || !t->codebook_l2_r || !t->indices_l2_l || !t->indices_l2_r)) ||
        (t->n_levels != 1 && t->n_levels != 2)) {
        ibh_set_error("%s: invalid tensor", who);
        return IBH_ERROR_PARAM;
    }
    if (t->K > 256 && t->n_levels == 1) {
        // level-1 indices are uint8 (pq_decode.h:59-60)
        ibh_set_error("%s: K=%d exceeds uint8 level-1 indices", who, t->K);
        return IBH_ERROR_PARAM;
    }
    int CS, nslabs;
    size_t lds;
    PqWs w;
    const bool own_ws = ws != nullptr && !lib_ws;
    if (pq_geometry(t, &CS, &nslabs, &lds, &w, own_ws) != IBH_OK) {
        ibh_set_error("%s: codebooks too large for the LDS tables", who);
        return IBH_ERROR_PARAM;
    }
    if (!ws) {
        ws = ibh_workspace(w.need);
        ws_bytes = ws ? w.need : 0;
    }
    if (!ws || ws_bytes < w.need) {
        ibh_set_error("%s: workspace of %zu bytes needed", who, w.need);
        return IBH_ERROR_MEMORY;
    }
    const bool two = t->n_levels == 2 && md.level2;
    PqDev d;
    d.M = t->M; d.N = t->N; d.G = t->G; d.K = t->K; d.K2 = t->K_l2 > 0 ? t->K_l2 : t->K;
    d.n_levels = t->n_levels; d.n_outlier = t->n_outlier; d.C = t->C;
    d.skip_mode = md.skip_mode; d.skip_val = md.skip_val; d.q8 = md.q8;
    d.l2skip = two && md.l2skip && md.l2_thr > 0.f; d.l2_thr = md.l2_thr;
    d.pyramid = t->format == IBH_PQ_FORMAT_PYRAMID;
    d.l2_idx_bytes = t->l2_idx_bytes > 0 ? t->l2_idx_bytes : 1;
    d.cb1l = t->codebook_l1_l; d.cb1r = t->codebook_l1_r; d.cb2l = t->codebook_l2_l; d.cb2r = t->codebook_l2_r;
    d.i1l = t->indices_l1_l; d.i1r = t->indices_l1_r; d.i2l = t->indices_l2_l; d.i2r = t->indices_l2_r;
    d.row_scale = t->row_scale; d.ocols = t->outlier_cols; d.oside = t->outlier_sidecar;
    d.oscale = t->outlier_scale; d.inner = t->n_outlier > 0 ? t->inner_cols : nullptr;
    hipStream_t st = ibh_resolve_stream(stream);
    char* base = (char*)ws;
    float* tab1 = (float*)(base + w.tab1);
    float* tab2 = (float*)(base + w.tab2);
    float* part = (float*)(base + w.part);
    float* cmax = (float*)(base + w.cmax);
    float* cnorm = (float*)(base + w.cnorm);
    float* c2max = (float*)(base + w.c2max);
    d.cnorm = cnorm;
    d.c2max = c2max;
    // one launch for half-chunks of <= 8 columns and <= 256 codes a level with
    // byte or 4-bit level-2 indices (the scope of pq_fused); 2-byte indices,
    // the level-2 skip and the int8 tables take the three-kernel path below
    int tiles = (t->M + kFRows - 1) / kFRows;
    const int S = (t->C + kFCS - 1) / kFCS;
    const bool l2ok = !two || (!d.l2skip && d.l2_idx_bytes == 1 && d.K2 <= 256 && (CS == 8 || CS == 16));
    if (l2ok && !md.q8 && !md.tq8 && t->G <= 16 && t->K <= 256 && S <= kFMaxS && t->M <= kFMaxRows && g_pq_fused) {
        size_t flds = (size_t)kFCS * (2 * t->K + 4 + (two ? 2 * d.K2 + 4 : 0)) * sizeof(float);
        // direct_rows' x and sums (a block of 1024 threads has a CU to itself,
        // so more LDS costs no block its place)
        d.slab_sh = CS == 8 ? 3 : 4;
        const size_t dlds = ((size_t)(t->C / CS + 1) * (16 * CS + kDPad) + 2 * kFRows) * sizeof(float);
        if (two && dlds > flds) flds = dlds;
        unsigned long long* hdr = own_ws ? (unsigned long long*)ws : nullptr;
        unsigned long long* racc = own_ws ? hdr + 32 : nullptr;
        const bool ka = t->K % 32 == 0 && (!two || d.K2 % 32 == 0);
        const bool nr2 = tiles * S > 256;                  // more than one round of blocks
        if (nr2) tiles = (tiles + 1) / 2;
#define IBH_PF1(A_, L_, R_) do { \
        if (L_ > 1 && flds > 65536 && hipFuncSetAttribute((const void*)pq_fused<A_, L_, R_>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                                          (int)flds) != hipSuccess) { \
            ibh_set_error("%s: %zu bytes of LDS not available", who, flds); \
            return IBH_ERROR_INTERNAL; } \
        pq_fused<A_, L_, R_><<<tiles * S, kFThreads, flds, st>>>(d, x, out, S, racc, hdr); } while (0)
#define IBH_PF(A_, L_) do { if (nr2) IBH_PF1(A_, L_, 2); else IBH_PF1(A_, L_, 1); } while (0)
        if (two && d.K2 == 16) IBH_PF(false, 3);
        else if (two) { if (ka) IBH_PF(true, 2); else IBH_PF(false, 2); }
        else if (ka) IBH_PF(true, 1);
        else IBH_PF(false, 1);
#undef IBH_PF
#undef IBH_PF1
        IBH_CHECK_LAUNCH("ibh_pq_matmul (one launch)");
        return IBH_OK;
    }
    if (d.l2skip) {
        const int n_outer = d.pyramid ? t->K : 1;
        const int k_inner = d.pyramid ? d.K2 / t->K : d.K2;
        pq_c2max<<<n_outer, kThreads, 0, st>>>(d, c2max, n_outer, k_inner);
        IBH_CHECK_LAUNCH("ibh_pq_matmul (cluster bounds)");
    }
    if (two) pq_tables<true><<<t->C, kThreads, 0, st>>>(d, x, tab1, tab2, cmax, cnorm);
    else pq_tables<false><<<t->C, kThreads, 0, st>>>(d, x, tab1, tab2, cmax, cnorm);
    IBH_CHECK_LAUNCH("ibh_pq_matmul (tables)");
    if (md.tq8) {
        pq_tq8<<<dim3(t->C, two ? 2 : 1), kThreads, 0, st>>>(tab1, tab2, t->K);
        IBH_CHECK_LAUNCH("ibh_pq_matmul (table quantisation)");
    }
    dim3 grid((t->M + kRowsPerBlock - 1) / kRowsPerBlock, nslabs);
    if (two) pq_gather<true><<<grid, kThreads, lds, st>>>(d, tab1, tab2, cmax, part, CS);
    else pq_gather<false><<<grid, kThreads, lds, st>>>(d, tab1, tab2, cmax, part, CS);
    IBH_CHECK_LAUNCH("ibh_pq_matmul (gather)");
    pq_reduce<<<(t->M + kThreads - 1) / kThreads, kThreads, 0, st>>>(d, x, part, nslabs, out);
    IBH_CHECK_LAUNCH("ibh_pq_matmul (reduce)");
    return IBH_OK;
}

// Workspace of ibh_pq_lm_head_topk: the matvec's, then the coarse logits,
// the selected rows and their refined logits.
static size_t pq_topk_need(const ibh_pq_tensor_abi* t, int k_top, bool front) {
    const size_t base = pq_ws_need(t, front);
    if (!base || k_top <= 0) return 0;
    auto al = [](size_t v) { return (v + 255) / 256 * 256; };
    return base + al((size_t)t->M * 4) + 2 * al((size_t)k_top * 4);
}

extern "C" size_t ibh_pq_topk_workspace_bytes(const ibh_pq_tensor_abi* t, int k_top) {
    return pq_topk_need(t, k_top, true);
}

extern "C" int ibh_pq_lm_head_topk(const ibh_pq_tensor_abi* t, const float* x, int k_top, float* out_logits,
                                   int32_t* out_ids, void* ws, size_t ws_bytes, void* stream) {
    if (!t || !x || !out_logits || !out_ids || k_top <= 0 || k_top > t->M || k_top > 1024) {
        ibh_set_error("ibh_pq_lm_head_topk: invalid arguments (K_top=%d, M=%d; K_top <= 1024)", k_top, t ? t->M : 0);
        return IBH_ERROR_PARAM;
    }
    const bool lib_ws = ws == nullptr;
    const size_t need = pq_topk_need(t, k_top, !lib_ws);
    if (!need) {
        ibh_set_error("ibh_pq_lm_head_topk: invalid tensor");
        return IBH_ERROR_PARAM;
    }
    if (!ws) {
        ws = ibh_workspace(need);
        ws_bytes = ws ? need : 0;
    }
    if (!ws || ws_bytes < need) {
        ibh_set_error("ibh_pq_lm_head_topk: workspace of %zu bytes needed", need);
        return IBH_ERROR_MEMORY;
    }
    auto al = [](size_t v) { return (v + 255) / 256 * 256; };
    const size_t base = pq_ws_need(t, !lib_ws);
    float* coarse = (float*)((char*)ws + base);
    int32_t* sel = (int32_t*)((char*)coarse + al((size_t)t->M * 4));
    float* refined = (float*)((char*)sel + al((size_t)k_top * 4));
    hipStream_t st = ibh_resolve_stream(stream);
    // 1. level-1 logits of every row (ib_pq_matmul_fp32_l1_only)
    PqMode md;
    md.skip_mode = 0;
    md.level2 = false;
    int rc = pq_run(t, x, coarse, ws, base, stream, md, "ibh_pq_lm_head_topk", lib_ws);
    if (rc) return rc;
    // 2. the K largest, 3. their full-pyramid logits, 4. sorted
    if (k_top <= kPickK) pq_topk_pick<<<1, kSelThreads, 0, st>>>(coarse, t->M, k_top, sel);
    else pq_topk_select<<<1, kSelThreads, 0, st>>>(coarse, t->M, k_top, sel);
    IBH_CHECK_LAUNCH("ibh_pq_lm_head_topk (select)");
    PqDev d{};
    d.M = t->M; d.N = t->N; d.G = t->G; d.K = t->K; d.K2 = t->K_l2 > 0 ? t->K_l2 : t->K;
    d.n_levels = t->n_levels; d.n_outlier = t->n_outlier; d.C = t->C;
    d.l2_idx_bytes = t->l2_idx_bytes > 0 ? t->l2_idx_bytes : 1;
    d.cb1l = t->codebook_l1_l; d.cb1r = t->codebook_l1_r; d.cb2l = t->codebook_l2_l; d.cb2r = t->codebook_l2_r;
    d.i1l = t->indices_l1_l; d.i1r = t->indices_l1_r; d.i2l = t->indices_l2_l; d.i2r = t->indices_l2_r;
    d.row_scale = t->row_scale; d.ocols = t->outlier_cols; d.oside = t->outlier_sidecar;
    d.oscale = t->outlier_scale; d.inner = t->n_outlier > 0 ? t->inner_cols : nullptr;
    pq_subset_rows<<<k_top, 256, 0, st>>>(d, x, sel, k_top, refined);
    IBH_CHECK_LAUNCH("ibh_pq_lm_head_topk (refine)");
    pq_topk_sort<<<1, 1024, 0, st>>>(refined, sel, k_top, out_logits, out_ids);
    IBH_CHECK_LAUNCH("ibh_pq_lm_head_topk (sort)");
    return IBH_OK;
}

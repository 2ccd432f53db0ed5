// ibh_skinny.hip -- weights x a few columns (2 .. 32 activation vectors: the
// slots of a verify or prompt pass) on the int8 matrix cores, gfx950.
//
// A wavefront owns 16 rows and a range of a row's 128-column groups and
// streams its weights once, every load issued up front; the 16 (or 2 x 16)
// columns are the other operand of v_mfma_i32_16x16x64_i8, so D gives lane
// (column n = lane & 15, rows 4 (lane >> 4) .. +3) the exact int32 group sums,
// and everything behind them (scales, folds) is lane-local.  The row's groups
// are split over the KW wavefronts of a block; RT row tiles of a block share
// the staged columns.
#include "ibh_common.h"

using namespace ibh;

namespace {

typedef int i4_t __attribute__((ext_vector_type(4)));

// ── W4A8: int4 weights x int8 codes with 128-group scales ───────────────────
// (kernels/scalar.c:86-124: acc = acc + (float)isum * sa, both rounded;
// FUSED: kernels/avx2.c:331-343, acc = fma((float)isum, sa, acc)), groups in
// order, times the row scale: bit-exact.
//
// The phases add up rather than overlap, since every wavefront's loads are in
// flight at once (14336 x 4096, 16 columns, 13.0 us: 7.1 the weight loads
// alone, 1.4 the columns, 1.5 the contraction, 1.4 the fold, 1.6 that a load
// touches 16 rows x 64 bytes and not 4 x 256), so each is kept short.
//  - Columns: their codes are loaded ahead of the weights (loads return in
//    order), permuted to the nibble order of the weight operand and, XLDS,
//    staged in LDS in operand order for all row tiles of the block: a lane
//    finds its 32 bytes of a group with two conflict-free 16-byte reads.  Rows
//    too long for that take them from L2 straight into registers.
//  - The fold over groups is serial.  Two or three wavefronts per row (tall
//    matrices) hand the running sum on through LDS, the first folding as its
//    weights arrive; more of them (GATHER) put their sums in LDS over the codes
//    and a thread per (column, row) folds, its reads independent.
// Measured in a graph, before (4, 8 or 16 columns per pass, w4a8_mfma) and
// here: 14336 x 4096 at 8 / 16 / 32 columns 13.7 / 17.5 / 35.4 -> 12.5 / 13.0 /
// 17.2 us; 5632 x 2048 6.7 / 8.0 / 15.8 -> 5.8 / 6.2 / 8.2; 4096 x 4096 at 32
// columns 13.5 -> 9.8, 2048 x 2048 at 16 / 32 5.3 / 10.3 -> 4.6 / 6.8.
template <int KIND, bool FUSED, int NT, int MAXC, bool XLDS, bool GATHER>
__global__ __launch_bounds__(512) void w4a8_skinny(const BatchSet bs, const int8_t* __restrict__ qx,
                                                   const float* __restrict__ sa, int N, int B, int G, int KW,
                                                   int CPW, int SOFF) {
    extern __shared__ __align__(16) unsigned char smem[];
    const RowPick P = pick_rows(bs.rs);
    const int ys = (int)blockIdx.x >= bs.rs.b2 ? bs.ys[2] : ((int)blockIdx.x >= bs.rs.b1 ? bs.ys[1] : bs.ys[0]);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nw = blockDim.x >> 6, RT = nw / KW;
    const int rt = wave / KW, kw = wave - rt * KW;
    const int i = lane & 15, q = lane >> 4;
    const int row0 = (P.bid * RT + rt) * 16;
    const int g0 = kw * CPW, gn = max(0, min(CPW, G - g0));
    const size_t rb = (size_t)N / 2;
    uint4* xs = (uint4*)smem;                                         // XLDS: [G][NT][2][64]
    float* ss = (float*)(smem + SOFF);                                // [G][16 NT] group scales
    float* hand = ss + (size_t)G * 16 * NT;                           // [RT][NT][4][64] running sums

    // this lane's 32 codes of group g (clamped addresses: order() zeroes the
    // codes past the row's end and past B, behind the loads)
    auto codes = [&](int g, int nt, uint4& a, uint4& b) {
        const int8_t* p = qx + (size_t)min(16 * nt + i, B - 1) * N + min(128 * g + 32 * q, N - 32);
        a = *(const uint4*)p;
        b = *(const uint4*)(p + 16);
    };
    // codes in the order of the weight operand: even columns of each 8, then odd
    auto order = [&](int g, int nt, uint4& a, uint4& b) {
        const uint32_t on = 16 * nt + i < B && 128 * g + 32 * q < N ? 0xffffffffu : 0u;
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint32_t o[8];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            o[2 * e] = __builtin_amdgcn_perm(w[2 * e + 1], w[2 * e], 0x06040200u) & on;
            o[2 * e + 1] = __builtin_amdgcn_perm(w[2 * e + 1], w[2 * e], 0x07050301u) & on;
        }
        a = make_uint4(o[0], o[1], o[2], o[3]);
        b = make_uint4(o[4], o[5], o[6], o[7]);
    };

    // 1. codes (XLDS: this wavefront's share of all groups, 4 at a time ahead
    // of the weights; else its own first groups) and scales
    constexpr int XB = XLDS ? 4 : (MAXC + 1) / 2;                     // groups loaded before the weights
    uint4 xa[XB][NT], xb[XB][NT];
#pragma unroll
    for (int u = 0; u < XB; u++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
            codes(min(XLDS ? wave + nw * u : g0 + u, G - 1), nt, xa[u][nt], xb[u][nt]);
    const int nsc = G * 16 * NT;
    float sv[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int e = min((int)threadIdx.x + u * (int)blockDim.x, nsc - 1);
        sv[u] = sa[(size_t)min(e % (16 * NT), B - 1) * G + e / (16 * NT)];
    }
    // 2. every weight of the wavefront
    const uint8_t* wrow = P.W + (size_t)min(row0 + i, P.M - 1) * rb;
    uint4 seg[MAXC];
#pragma unroll
    for (int c = 0; c < MAXC; c++) {
        const size_t off = min((size_t)(g0 + min(c, max(gn - 1, 0))) * 64 + 16 * q, rb - 16);
        seg[c] = ld_stream16(wrow + off);
    }
    float rsc[4];
    uint32_t rsb[4];
#pragma unroll
    for (int r = 0; r < 4; r++) rsb[r] = scale_bits<KIND>(P.sc, min(row0 + 4 * q + r, P.M - 1));
    __builtin_amdgcn_sched_barrier(0);
    // 3. stage
    if constexpr (XLDS) {
#pragma unroll
        for (int u = 0; u < XB; u++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const int g = wave + nw * u;
                order(g, nt, xa[u][nt], xb[u][nt]);
                if (g < G) {
                    xs[((size_t)g * NT + nt) * 128 + lane] = xa[u][nt];
                    xs[((size_t)g * NT + nt) * 128 + 64 + lane] = xb[u][nt];
                }
            }
        for (int g = wave + nw * XB; g < G; g += nw)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                uint4 a, b;
                codes(g, nt, a, b);
                order(g, nt, a, b);
                xs[((size_t)g * NT + nt) * 128 + lane] = a;
                xs[((size_t)g * NT + nt) * 128 + 64 + lane] = b;
            }
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int e = (int)threadIdx.x + u * (int)blockDim.x;
        if (e < nsc) ss[e] = sv[u];
    }
    for (int e = (int)threadIdx.x + 2 * (int)blockDim.x; e < nsc; e += blockDim.x)
        ss[e] = sa[(size_t)min(e % (16 * NT), B - 1) * G + e / (16 * NT)];
    lds_only_barrier();

    // 4. group sums: kept as floats (exact: below 2^18)
    float f[MAXC][NT][4];
    auto group = [&](int c, const uint4& x0, const uint4& x1, float (&o)[4]) {
        const uint32_t w[4] = {seg[c].x, seg[c].y, seg[c].z, seg[c].w};
        uint32_t av[8];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t s = w[e] ^ 0x88888888u;
            av[2 * e] = (s << 4) & 0xf0f0f0f0u;
            av[2 * e + 1] = s & 0xf0f0f0f0u;
        }
        i4_t d = __builtin_amdgcn_mfma_i32_16x16x64_i8(i4_t{(int)av[0], (int)av[1], (int)av[2], (int)av[3]},
                                                       i4_t{(int)x0.x, (int)x0.y, (int)x0.z, (int)x0.w},
                                                       i4_t{0, 0, 0, 0}, 0, 0, 0);
        d = __builtin_amdgcn_mfma_i32_16x16x64_i8(i4_t{(int)av[4], (int)av[5], (int)av[6], (int)av[7]},
                                                  i4_t{(int)x1.x, (int)x1.y, (int)x1.z, (int)x1.w}, d, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; r++) o[r] = (float)(d[r] >> 4);
    };
    // (no branch on gn: a group past the wavefront's range is a repeat of the
    // last one, and its sums are not used)
    float acc[NT][4];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[nt][r] = 0.f;
    // acc over this wavefront's group c (a repeated group folds as sum * 0:
    // acc + (+-0) = acc, acc is never -0)
    auto fold = [&](int c, int nt, const float (&v)[4]) {
        const float sg = ss[min(g0 + c, G - 1) * 16 * NT + 16 * nt + i], s = c < gn ? sg : 0.f;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if constexpr (FUSED) acc[nt][r] = fmaf(v[r], s, acc[nt][r]);
            else acc[nt][r] = acc[nt][r] + v[r] * s;
        }
    };
    if (XLDS && !GATHER && kw == 0) {
        // the first wavefront of a row folds as its groups arrive
#pragma unroll
        for (int c = 0; c < MAXC; c++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const uint4* xg = xs + ((size_t)min(g0 + c, G - 1) * NT + nt) * 128 + lane;
                float v[4];
                group(c, xg[0], xg[64], v);
                fold(c, nt, v);
            }
    } else if constexpr (XLDS) {
#pragma unroll
        for (int c = 0; c < MAXC; c++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const uint4* xg = xs + ((size_t)min(g0 + c, G - 1) * NT + nt) * 128 + lane;
                group(c, xg[0], xg[64], f[c][nt]);
            }
    } else {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h) {
#pragma unroll
                for (int u = 0; u < XB; u++)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++) codes(min(g0 + XB + u, G - 1), nt, xa[u][nt], xb[u][nt]);
            }
#pragma unroll
            for (int u = 0; u < XB; u++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    const int c = XB * h + u;
                    if (c >= MAXC) continue;
                    order(min(g0 + c, G - 1), nt, xa[u][nt], xb[u][nt]);
                    group(c, xa[u][nt], xb[u][nt], f[c][nt]);
                }
        }
    }

    // 5. the serial fold
    if constexpr (GATHER) {
        // sums to LDS as [row tile][group][column][16 rows] (over the codes,
        // once every wavefront is done with them), then a thread per (column,
        // row): its reads do not depend on one another, only the chain does
        float* gs = (float*)smem;
        constexpr int NCOL = 16 * NT;
        __syncthreads();
#pragma unroll
        for (int c = 0; c < MAXC; c++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                if (c >= gn) continue;
                *(float4*)(gs + (((size_t)rt * G + g0 + c) * NCOL + 16 * nt + i) * 16 + 4 * q) =
                    float4{f[c][nt][0], f[c][nt][1], f[c][nt][2], f[c][nt][3]};
            }
        __syncthreads();
        for (int e = threadIdx.x; e < RT * NCOL * 16; e += blockDim.x) {
            const int r = e & 15, s = (e >> 4) % NCOL, t = e / (16 * NCOL);
            const float* p = gs + ((size_t)t * G * NCOL + s) * 16 + r;
            const float* ps = ss + s;
            float acc = 0.f;
#pragma unroll 8
            for (int g = 0; g < G; g++) {
                const float v = p[(size_t)g * NCOL * 16], sc = ps[g * NCOL];
                if constexpr (FUSED) acc = fmaf(v, sc, acc);
                else acc = acc + v * sc;
            }
            const int row = (P.bid * RT + t) * 16 + r;
            if (s < B && row < P.M) P.y[(size_t)s * ys + row] = acc * load_scale<KIND>(P.sc, row);
        }
        return;
    }
    // wavefront after wavefront
    for (int k = 0; k < KW; k++) {
        if (kw == k) {
            if (k) {
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[nt][r] = hand[((rt * NT + nt) * 4 + r) * 64 + lane];
#pragma unroll
                for (int c = 0; c < MAXC; c++)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++) fold(c, nt, f[c][nt]);
            }
            if (k + 1 < KW) {
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) hand[((rt * NT + nt) * 4 + r) * 64 + lane] = acc[nt][r];
            }
        }
        if (k + 1 < KW) lds_only_barrier();
    }
    if (kw != KW - 1) return;
#pragma unroll
    for (int r = 0; r < 4; r++) rsc[r] = scale_from_bits<KIND>(rsb[r]);
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        const int s = 16 * nt + i;
        if (s >= B) continue;
        float* o = P.y + (size_t)s * ys + row0 + 4 * q;
        const int left = P.M - (row0 + 4 * q);
        if (left >= 4 && ((uintptr_t)o & 15) == 0) {
            *(float4*)o = float4{acc[nt][0] * rsc[0], acc[nt][1] * rsc[1], acc[nt][2] * rsc[2], acc[nt][3] * rsc[3]};
        } else {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (r < left) o[r] = acc[nt][r] * rsc[r];
        }
    }
}

constexpr size_t kLds = 160 * 1024;

bool lds_ok(const void* fn, size_t bytes) {
    return bytes <= 65536 ||
           hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess;
}

}  // namespace

// 1-3 INT4 matrices x B coded columns (qx [B][N], sa [B][G]) -> d[i].out[b * ys
// + row], ys = d[i].M or (one matrix) M_stride.  Returns 1 if launched, 0 if
// the call is not taken (N % 32, unaligned operands, or the 16-row kernels of
// ibh_mfma.hip measure faster), < 0 on an error.
int ibh_launch_w4a8_batch(const MatDesc* d, int n, int kind, const int8_t* qx, const float* sa, int N, int B,
                          bool fused, hipStream_t st, int M_stride) {
    if (n < 1 || n > 3 || B < 2 || B > 32 || (M_stride && n > 1) || N % 32 || ((uintptr_t)qx & 15)) return 0;
    int T = 0;
    for (int i = 0; i < n; i++) {
        if ((uintptr_t)d[i].w & 15) return 0;
        T += (d[i].M + 15) / 16;
    }
    const int G = (N + 127) / 128, nt = B > 16 ? 2 : 1;
    // Row tiles per block: as many as make one block per CU, up to 4; from two
    // on the running sum is handed on (2 wavefronts per row where 16 groups
    // each reach), one takes the gather with up to 8 wavefronts of 4 groups.
    // Fewer columns than these stay with the 4- to 16-column kernels, which
    // stage nothing they do not need (measured crossings: tall matrices 5
    // columns, short rows 9, others 17).
    int rt = (T + 255) / 256;
    rt = rt > 4 ? 4 : rt;
    int KW = (G + 15) / 16 > 2 ? (G + 15) / 16 : 2;
    if (rt * KW > 8) rt = 8 / KW;
    if (rt < 1) return 0;
    const bool gather = rt == 1;
    if (gather) KW = (G + 3) / 4 < 8 ? (G + 3) / 4 : 8;
    if (B <= (!gather ? 4 : G <= 16 ? 8 : 16)) return 0;
    const int CPW = (G + KW - 1) / KW;
    KW = (G + CPW - 1) / CPW;
    auto soff_of = [&](bool x) {
        const size_t a = x ? (size_t)G * nt * 2048 : 0, b = gather ? (size_t)G * nt * 1024 : 0;
        return a > b ? a : b;
    };
    const size_t tail = (size_t)G * 16 * nt * 4 + (gather ? 0 : (size_t)rt * nt * 1024);
    const bool xlds = soff_of(true) + tail <= kLds;
    if (!xlds && (!gather || nt != 2 || CPW > 8 || soff_of(false) + tail > kLds)) return 0;
    const size_t lds = soff_of(xlds) + tail;
    const int soff = (int)soff_of(xlds);
    const BatchSet bs{make_rowset(d, n, 16 * rt),
                      {M_stride ? M_stride : d[0].M, d[n > 1 ? 1 : 0].M, d[n > 2 ? 2 : 0].M}};
    const int blocks = rowset_blocks(d, n, 16 * rt);
#define IBH_SK(K_, F_, T_, C_, X_, G_) do { \
        if (!lds_ok((const void*)w4a8_skinny<K_, F_, T_, C_, X_, G_>, lds)) return 0; \
        w4a8_skinny<K_, F_, T_, C_, X_, G_><<<blocks, 64 * rt * KW, lds, st>>>(bs, qx, sa, N, B, G, KW, CPW, soff); } while (0)
#define IBH_SKC(K_, F_, T_, X_, G_) do { if (CPW <= 4) IBH_SK(K_, F_, T_, 4, X_, G_); else if (CPW <= 8) IBH_SK(K_, F_, T_, 8, X_, G_); \
                                         else IBH_SK(K_, F_, T_, 16, X_, G_); } while (0)
#define IBH_SKX(K_, F_) do { if (!xlds) { if (CPW <= 4) IBH_SK(K_, F_, 2, 4, false, true); else IBH_SK(K_, F_, 2, 8, false, true); } \
                             else if (nt == 2) { if (gather) IBH_SKC(K_, F_, 2, true, true); else IBH_SKC(K_, F_, 2, true, false); } \
                             else { if (gather) IBH_SKC(K_, F_, 1, true, true); else IBH_SKC(K_, F_, 1, true, false); } } while (0)
#define IBH_SKF(K_) do { if (fused) IBH_SKX(K_, true); else IBH_SKX(K_, false); } while (0)
    if (kind == IBH_SCALE_F16) IBH_SKF(IBH_SCALE_F16); else IBH_SKF(IBH_SCALE_F32);
#undef IBH_SKF
#undef IBH_SKX
#undef IBH_SKC
#undef IBH_SK
    IBH_CHECK_LAUNCH("w4a8 batch");
    return 1;
}

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
// flight at once, so each is kept short.
//  - Loads: neighbouring lanes in different lines get one lane per clock from
//    L1, so weights and codes come as 128 contiguous bytes per 8 lanes and are
//    turned into operand order afterwards, the weights (8 rows x 128 bytes a
//    load, two groups a pair of loads) between lanes, the codes on their way
//    to LDS.  Loading both in operand order (16 rows x 64 bytes) took 13.1 us
//    instead of 11.7 at 14336 x 4096 with 16 columns, 10.0 instead of 7.9 at
//    4096 x 4096 with 32.
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
// here: 14336 x 4096 at 8 / 16 / 32 columns 13.7 / 17.5 / 35.4 -> 11.5 / 11.7 /
// 14.6 us; 5632 x 2048 6.7 / 8.0 / 15.8 -> 5.7 / 5.9 / 7.3; 4096 x 4096 at 16 /
// 32 columns 7.0 / 13.5 -> 6.0 / 7.9, 2048 x 2048 5.3 / 10.3 -> 4.6 / 6.0.

// Two loads of 8 rows x 128 bytes, lane 8 r + u holding 16-byte unit u of row r
// (a) or r + 8 (b): the lines of L1 are taken whole.  -> the operands of the two
// 64-byte groups, lane (i, k quarter q) holding unit q of row i.  A lane and its
// mirror in the 8 exchange the half that belongs to the other group, and one
// lane permutation (p0, p1: turn_lanes) orders each group.
__device__ __forceinline__ void turn_lanes(int lane, int& p0, int& p1) {
    const int i = lane & 15, q = lane >> 4, b = i >> 3;
    p0 = 4 * (8 * (i & 7) + (b ? 7 - q : q));
    p1 = 4 * (8 * (i & 7) + (b ? 4 + q : 3 - q));
}
__device__ __forceinline__ void turn_pair(const uint4 a, const uint4 b, int p0, int p1, uint4& x0, uint4& x1) {
    const uint32_t av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
    uint32_t o0[4], o1[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        // row_half_mirror into lanes 4 .. 7 of each 8, or into lanes 0 .. 3
        const int m0 = __builtin_amdgcn_update_dpp((int)av[e], (int)bv[e], 0x141, 0xF, 0xA, false);
        const int m1 = __builtin_amdgcn_update_dpp((int)bv[e], (int)av[e], 0x141, 0xF, 0x5, false);
        o0[e] = (uint32_t)__builtin_amdgcn_ds_bpermute(p0, m0);
        o1[e] = (uint32_t)__builtin_amdgcn_ds_bpermute(p1, m1);
    }
    x0 = make_uint4(o0[0], o0[1], o0[2], o0[3]);
    x1 = make_uint4(o1[0], o1[1], o1[2], o1[3]);
}

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
    // XLDS: unit lane & 7 of group g of slots (lane >> 3) (a) and + 8 (b), 128
    // contiguous bytes per 8 lanes
    auto codes8 = [&](int g, int nt, uint4& a, uint4& b) {
        const int8_t* p = qx + min(128 * g + 16 * (lane & 7), N - 16);
        a = *(const uint4*)(p + (size_t)min(16 * nt + (lane >> 3), B - 1) * N);
        b = *(const uint4*)(p + (size_t)min(16 * nt + 8 + (lane >> 3), B - 1) * N);
    };
    // ... and where the contraction's lane (column, k quarter u >> 1) finds it
    // as its half u & 1, conflict-free for both sides
    auto stage = [&](int g, int nt, int s, const uint4& v) {
        const int u = lane & 7;
        const uint32_t on = 16 * nt + s < B && 128 * g + 16 * u < N ? 0xffffffffu : 0u;
        xs[((size_t)g * NT + nt) * 128 + 64 * (u & 1) + 16 * (u >> 1) + (s ^ (2 * u))] =
            make_uint4(__builtin_amdgcn_perm(v.y, v.x, 0x06040200u) & on, __builtin_amdgcn_perm(v.y, v.x, 0x07050301u) & on,
                       __builtin_amdgcn_perm(v.w, v.z, 0x06040200u) & on, __builtin_amdgcn_perm(v.w, v.z, 0x07050301u) & on);
    };
    const int xl0 = 16 * q + (i ^ (4 * q)), xl1 = 64 + 16 * q + (i ^ (4 * q + 2));
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
        for (int nt = 0; nt < NT; nt++) {
            if constexpr (XLDS) codes8(min(wave + nw * u, G - 1), nt, xa[u][nt], xb[u][nt]);
            else codes(min(g0 + u, G - 1), nt, xa[u][nt], xb[u][nt]);
        }
    const int nsc = G * 16 * NT;
    float sv[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int e = min((int)threadIdx.x + u * (int)blockDim.x, nsc - 1);
        sv[u] = sa[(size_t)min(e % (16 * NT), B - 1) * G + e / (16 * NT)];
    }
    // 2. every weight of the wavefront, two groups per pair of loads
    uint4 seg[MAXC];
#pragma unroll
    for (int c = 0; c < MAXC; c += 2) {
        const size_t off = min((size_t)(g0 + min(c, max(gn - 1, 0))) * 64 + 16 * (lane & 7), rb - 16);
#pragma unroll
        for (int h = 0; h < 2; h++)
            seg[c + h] = ld_stream16(P.W + (size_t)min(row0 + 8 * h + (lane >> 3), P.M - 1) * rb + off);
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
                if (g < G) {
                    stage(g, nt, lane >> 3, xa[u][nt]);
                    stage(g, nt, 8 + (lane >> 3), xb[u][nt]);
                }
            }
        for (int g = wave + nw * XB; g < G; g += nw)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                uint4 a, b;
                codes8(g, nt, a, b);
                stage(g, nt, lane >> 3, a);
                stage(g, nt, 8 + (lane >> 3), b);
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
    int tp0, tp1;
    turn_lanes(lane, tp0, tp1);
    auto turn = [&](int c) {                                          // ahead of groups c and c + 1
        uint4 x0, x1;
        turn_pair(seg[c], seg[c + 1], tp0, tp1, x0, x1);
        seg[c] = x0;
        seg[c + 1] = x1;
    };
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
        for (int c = 0; c < MAXC; c++) {
            if (c % 2 == 0) turn(c);
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const uint4* xg = xs + ((size_t)min(g0 + c, G - 1) * NT + nt) * 128;
                float v[4];
                group(c, xg[xl0], xg[xl1], v);
                fold(c, nt, v);
            }
        }
    } else if constexpr (XLDS) {
#pragma unroll
        for (int c = 0; c < MAXC; c++) {
            if (c % 2 == 0) turn(c);
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const uint4* xg = xs + ((size_t)min(g0 + c, G - 1) * NT + nt) * 128;
                group(c, xg[xl0], xg[xl1], f[c][nt]);
            }
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
                    if (c % 2 == 0 && nt == 0) turn(c);
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

// ── INT8 rows x fp32 columns ────────────────────────────────────────────────
// (kernels/scalar.c:70-84, within fp32 tolerance: sums in another order.)
//
// x becomes four int8 digit planes per (column, 128-column group): Q =
// trunc(x * 2^(30 - e)), e the exponent of the group's max|x|, in balanced
// base-256 digits, so there is no second pass over x and an element is held to
// 2^-29 of the group's largest: exactly down to 2^-6 of it.  (Three planes, 2^-23
// of the largest, left elements that lie far below it fewer bits than an fp32
// product has, which shows in rows whose weights on the large channels are 0.)
// Each group's exact integer sum is rounded to fp32 once, scaled by the power of
// two and added.  The 8 wavefronts of a block split K (their sums meet in LDS,
// added in order).
//
// What bounds it is how its loads reach L1: neighbouring lanes in different
// lines get one lane per clock.  With every lane loading its own 16 weights and
// 16 floats of x in operand order (16 rows x 64 bytes an instruction), 4096 x
// 4096 at 2 / 8 / 16 / 32 columns took 9.5 / 12.5 / 17.8 / 24.6 us.  So 8
// neighbouring lanes load 128 contiguous bytes of a row of weights or of a
// column, and both go through the wavefront's own LDS (no barrier; 16-byte
// units swizzled to conflict-free) into the operands' order: x as digits, lane
// 8 s + p holding columns 32 e + 4 p of slot s, 8 slots a pass, read back as
// unit p = 4 m + q by lane (n, k quarter q) for MFMA m; the weights by the same
// units of 16 columns, two lane swaps then giving them x's order of columns.
// RT row tiles of a wavefront share its digits.
// Measured in a graph, one wavefront per row on the VALU (biased weights) and
// here, at 3 / 8 / 16 / 32 columns: 4096 x 4096 15.6 / 34 / 65 / 124 -> 9.5 / 9.7 /
// 11.7 / 18.2 us, 14336 x 4096 46 / 118 / 214 / 467 -> 23.5 / 24.5 / 30.1 / 41.7,
// 4096 x 1024 6.2 / 11.9 / 21.5 / 40 -> 4.7 / 4.7 / 6.1 / 8.2 (three planes 4 to 8
// % less).  Error against 64 bits relative to the outputs' norm: 5e-7 .. 1.1e-6
// -> 7e-8 .. 9e-8 (three planes 3.3e-7 .. 5.2e-7).
struct DigArgs {
    const int8_t* W;
    const void* sc;          // row scales
    const float* x;          // [B][N]
    float* y;
    int M, N, B, ys, G, CPW; // G: 128-column groups of a row, CPW of them per wavefront
};

constexpr int kDigWaves = 8, kDigPlanes = 4;
constexpr int kDigBytes = kDigPlanes * 1024;                   // digits of 8 slots x 128 columns
constexpr int kDigBits = 30;                                   // |Q| < 2^30
constexpr int kDigMinExp = -119;                               // 2^(e - 30) stays a (subnormal) number: exact below it

// max that lets a NaN through (v_maximum3_f32)
__device__ __forceinline__ float nmax(float a, float b) { return __builtin_elementwise_maximum(a, b); }

template <int CTRL>
__device__ __forceinline__ float dpp_nmax(float v) {
    return nmax(v, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false)));
}

// orders a wavefront's LDS writes before its reads (no wait: they run in order)
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Lane (i, k quarter q) of unit 4 m + q holds columns 64 m + 16 q + 4 d .. + 3 in
// dword d.  Swapping dword and quarter gives it columns 64 m + 16 j + 4 q in
// dword j, which is element 2 m + (j >> 1) of x's unit 4 (j & 1) + q.
__device__ __forceinline__ i4_t quarter_transpose(const uint4 w) {
    typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
    const u2_t a = __builtin_amdgcn_permlane32_swap(w.x, w.z, false, false);
    const u2_t b = __builtin_amdgcn_permlane32_swap(w.y, w.w, false, false);
    const u2_t c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    const u2_t d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    return i4_t{(int)c[0], (int)c[1], (int)d[0], (int)d[1]};
}

// Row tiles staged in LDS at a time: both, except where 4 passes' digits leave
// room for one (they take turns then).
constexpr int dig_row_bufs(int rt, int sh) { return rt == 2 && sh == 4 ? 1 : rt; }

// SH: passes of 8 slots.
template <int KIND, int RT, int SH>
__global__ __launch_bounds__(64 * kDigWaves) void int8_skinny(const DigArgs a) {
    constexpr int NT = (SH + 1) / 2;                           // column tiles
    constexpr int RING = 4, XR = SH <= 2 ? 2 : 1;   // groups of weights and of x in flight
    constexpr int RB = dig_row_bufs(RT, SH);
    constexpr int WB = (SH * (kDigBytes + 32) + RB * 2048) / 4;   // a wavefront's LDS, in floats
    static_assert(RT * NT * 256 <= WB, "the sums reuse the digits' LDS");
    extern __shared__ __align__(16) unsigned char smem[];
    const int N = a.N, B = a.B, M = a.M, G = a.G;
    const int tid = threadIdx.x, lane = tid & 63;
    const int kw = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, q = lane >> 4;
    const int row0 = (int)blockIdx.x * 16 * RT;
    const int g0 = kw * a.CPW, gn = max(0, min(a.CPW, G - g0));
    float* mine = (float*)smem + (size_t)kw * WB;
    uint4* ds = (uint4*)mine;                                  // [SH][4][64]
    uint4* wl = ds + SH * 64 * kDigPlanes;                     // [RB][16 rows][8 units]
    float* ss = (float*)(wl + RB * 128);                       // [SH][8] scales

    float4 xr[XR][SH][4];
    uint4 wr[RING][RT][2];
    // columns past a row's end re-read its last 16 (same group): they leave the
    // group's max as it is and meet zeroed weights
    auto xload = [&](int u, int g) {
        const int gc = min(g, G - 1);
#pragma unroll
        for (int h = 0; h < SH; h++) {
            const uint32_t o = (uint32_t)min(8 * h + (lane >> 3), B - 1) * (uint32_t)N;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int c = 128 * gc + 32 * e + 4 * (lane & 7);
                xr[u][h][e] = *(const float4*)((const char*)a.x + 4 * (o + (uint32_t)(c < N ? c : N - 16 + (c & 15))));
            }
        }
    };
    const int8_t* wb = a.W + (size_t)row0 * N;
    auto wload = [&](int u, int g) {
        const int gc = min(g, G - 1);
#pragma unroll
        for (int t = 0; t < RT; t++) {
#pragma unroll
            for (int m = 0; m < 2; m++) {
                const uint32_t o = (uint32_t)(min(row0 + 16 * t + 8 * m + (lane >> 3), M - 1) - row0) * (uint32_t)N;
                wr[u][t][m] = ld_stream16((const uint8_t*)wb + (o + (uint32_t)min(128 * gc + 16 * (lane & 7), N - 16)));
            }
        }
    };
#pragma unroll
    for (int u = 0; u < XR; u++) xload(u, g0 + u);
#pragma unroll
    for (int u = 0; u < RING; u++) wload(u, g0 + u);
    __builtin_amdgcn_sched_barrier(0);

    float acc[RT][NT][4];
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[t][nt][r] = 0.f;

    for (int c0 = 0; c0 < gn; c0 += RING) {
#pragma unroll
        for (int u = 0; u < RING; u++) {
            const int c = c0 + u, g = g0 + c;
            if (c >= gn) break;                                // wave-uniform
            // 1. digits of the group, 8 slots a pass, to LDS
#pragma unroll
            for (int h = 0; h < SH; h++) {
                float v[16];
                float mx = 0.f;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float4 f = xr[u % XR][h][e];
                    v[4 * e] = f.x; v[4 * e + 1] = f.y; v[4 * e + 2] = f.z; v[4 * e + 3] = f.w;
                }
#pragma unroll
                for (int e = 0; e < 16; e += 2) mx = nmax(nmax(mx, fabsf(v[e])), fabsf(v[e + 1]));
                // the eight lanes of a slot share the scale, and with it that
                // an element is not finite: the column's sums become NaN and
                // are formed again in fp32 below
                mx = dpp_nmax<0x141>(dpp_nmax<0x4E>(dpp_nmax<0xB1>(mx)));   // lane ^ 1, ^ 2, 7 - lane
                const int sh = kDigBits - max(__builtin_amdgcn_frexp_expf(mx), kDigMinExp);
                i4_t dg[kDigPlanes];
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    uint32_t b[4];                             // biased digits, least significant first
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        b[e] = (uint32_t)(int)__builtin_amdgcn_ldexpf(v[4 * d + e], sh) + 0x80808080u;
                    const uint32_t l01 = __builtin_amdgcn_perm(b[1], b[0], 0x05010400u);
                    const uint32_t l23 = __builtin_amdgcn_perm(b[3], b[2], 0x05010400u);
                    const uint32_t h01 = __builtin_amdgcn_perm(b[1], b[0], 0x07030602u);
                    const uint32_t h23 = __builtin_amdgcn_perm(b[3], b[2], 0x07030602u);
                    dg[0][d] = (int)(__builtin_amdgcn_perm(l23, l01, 0x05040100u) ^ 0x80808080u);
                    dg[1][d] = (int)(__builtin_amdgcn_perm(l23, l01, 0x07060302u) ^ 0x80808080u);
                    dg[2][d] = (int)(__builtin_amdgcn_perm(h23, h01, 0x05040100u) ^ 0x80808080u);
                    dg[3][d] = (int)(__builtin_amdgcn_perm(h23, h01, 0x07060302u) ^ 0x80808080u);
                }
                const int s = lane >> 3, at = s * 8 + ((lane & 7) ^ s ^ (h & 1));
#pragma unroll
                for (int p = 0; p < kDigPlanes; p++) *(i4_t*)(ds + (h * kDigPlanes + p) * 64 + at) = dg[p];
                if ((lane & 7) == 0) ss[8 * h + s] = mx < __builtin_inff() ? __builtin_amdgcn_ldexpf(1.0f, -sh) : __builtin_nanf("");
            }
            xload(u % XR, g + XR);
            // the wavefront's LDS operations run in order: reads see the writes
            // above them, later writes come after these reads
            i4_t av[RT][2];
#pragma unroll
            for (int t0 = 0; t0 < RT; t0 += RB) {
                if (t0) wave_fence();
#pragma unroll
                for (int t = t0; t < t0 + RB; t++)
#pragma unroll
                    for (int m = 0; m < 2; m++)
                        wl[(t - t0) * 128 + 64 * m + (lane & 56) + ((lane & 7) ^ (lane >> 3) ^ m)] = wr[u][t][m];
                if (t0 + RB == RT) wload(u, g + RING);
                wave_fence();
#pragma unroll
                for (int t = t0; t < t0 + RB; t++) {
#pragma unroll
                    for (int m = 0; m < 2; m++) {
                        const i4_t T = quarter_transpose(wl[(t - t0) * 128 + 8 * n + ((4 * m + q) ^ (n & 7) ^ (n >> 3))]);
                        av[t][0][2 * m] = T[0]; av[t][1][2 * m] = T[1];
                        av[t][0][2 * m + 1] = T[2]; av[t][1][2 * m + 1] = T[3];
                    }
                    if (128 * (g + 1) > N)                     // av[m][e]: columns 32 e + 16 m + 4 q
#pragma unroll
                        for (int e = 0; e < 8; e++)
                            if (128 * g + 16 * e >= N) av[t][e & 1][e >> 1] = 0;
                }
            }
            // 2. contraction and fold
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                // a last tile of 8 slots has them in both halves of its columns
                const int h = 2 * nt + 1 < SH ? 2 * nt + (n >> 3) : 2 * nt, s = n & 7;
                const uint4* src = ds + h * 64 * kDigPlanes + s * 8;
                const int sw = s ^ (h & 1);
                i4_t d[RT][kDigPlanes];
#pragma unroll
                for (int m = 0; m < 2; m++)
#pragma unroll
                    for (int p = 0; p < kDigPlanes; p++) {
                        const i4_t b = *(const i4_t*)(src + p * 64 + ((4 * m + q) ^ sw));
#pragma unroll
                        for (int t = 0; t < RT; t++)
                            d[t][p] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[t][m], b, m ? d[t][p] : i4_t{0, 0, 0, 0}, 0, 0, 0);
                    }
                const float sc = ss[8 * h + s];
#pragma unroll
                for (int t = 0; t < RT; t++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        // |d| <= 2^21, so two planes join exactly in int32;
                        // the low pair's carry moves up, so that one rounding
                        // of the high pair and one of the sum remain
                        const int lo = d[t][0][r] + (d[t][1][r] << 8), hi = d[t][2][r] + (d[t][3][r] << 8) + (lo >> 16);
                        acc[t][nt][r] = fmaf(fmaf((float)hi, 65536.f, (float)(lo & 0xffff)), sc, acc[t][nt][r]);
                    }
            }
            wave_fence();
        }
    }

    // 3. the wavefronts' sums, in order; thread -> (row fastest, column)
#pragma unroll
    for (int t = 0; t < RT; t++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int r = 0; r < 4; r++) mine[(t * NT + nt) * 256 + r * 64 + lane] = acc[t][nt][r];
    __syncthreads();
    for (int e = tid; e < RT * NT * 256; e += 64 * kDigWaves) {    // whole wavefronts
        const int rr = e & 15, col = (e >> 4) & 15, tile = e >> 8, t = tile / NT, nt = tile - t * NT;
        const int row = row0 + 16 * t + rr, s = 16 * nt + col;
        const bool live = row < M && s < B;
        const float* p = (const float*)smem + tile * 256 + (rr & 3) * 64 + (rr >> 2) * 16 + col;
        float y = 0.f;
#pragma unroll
        for (int k = 0; k < kDigWaves; k++) y += p[(size_t)k * WB];
        // a column that holds Inf or NaN: the sum in fp32, by the whole
        // wavefront, so that both come out where they do without digits
        for (unsigned long long bad = __ballot(live && !(fabsf(y) <= 3.4e38f)); bad; bad &= bad - 1) {
            const int l = __builtin_ctzll(bad);
            const int8_t* w = a.W + (size_t)__builtin_amdgcn_readlane(row, l) * N;
            const float* x = a.x + (size_t)__builtin_amdgcn_readlane(s, l) * N;
            float v = 0.f;
#pragma unroll 8
            for (int j = lane; j < N; j += 64) v = fmaf((float)w[j], x[j], v);
            v = wave_sum(v);
            if (lane == l) y = v;
        }
        if (live) a.y[(size_t)s * a.ys + row] = y * load_scale<KIND>(a.sc, row);
    }
}

// One column, or few beside a small matrix: a wavefront a row on the vector
// units, which take x in fp32 and have no digits to make.  A signed weight is
// the byte's float less 128: one operation more than the unsigned one, and none
// for a sum of x that takes the bias out again and would round at 128 times the
// largest x.  Bound by the L1 reads of x, made again for every row: 4096 x 4096
// at 1 / 2 columns 7.1 / 10.5 us with both forms.  All columns' loads are issued
// ahead of the products (with each column's in front of its own, 1000 x 4096 at
// 3 columns 5.8 us, 5.0 so).
template <int KIND, int B>
__global__ __launch_bounds__(256) void int8_rows(const DigArgs a) {
    const int lane = threadIdx.x & 63, row = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= a.M) return;
    const uint8_t* w = (const uint8_t*)a.W + (size_t)row * a.N;
    float acc[B];
#pragma unroll
    for (int b = 0; b < B; b++) acc[b] = 0.f;
    for (int j = 16 * lane; j < a.N; j += 16 * 64) {
        const uint4 q = ld_stream16(w + j);
        const uint32_t d[4] = {q.x ^ 0x80808080u, q.y ^ 0x80808080u, q.z ^ 0x80808080u, q.w ^ 0x80808080u};
        float f[16];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            f[4 * e] = ubyte<0>(d[e]) - 128.f;
            f[4 * e + 1] = ubyte<1>(d[e]) - 128.f;
            f[4 * e + 2] = ubyte<2>(d[e]) - 128.f;
            f[4 * e + 3] = ubyte<3>(d[e]) - 128.f;
        }
        float4 xv[B][4];                                       // every column's loads ahead of its products
#pragma unroll
        for (int b = 0; b < B; b++)
#pragma unroll
            for (int e = 0; e < 4; e++) xv[b][e] = ((const float4*)(a.x + (size_t)b * a.N + j))[e];
#pragma unroll
        for (int e = 0; e < 4; e++) {
#pragma unroll
            for (int b = 0; b < B; b++) {
                const float4 v = xv[b][e];
                acc[b] = fmaf(f[4 * e], v.x, acc[b]);
                acc[b] = fmaf(f[4 * e + 1], v.y, acc[b]);
                acc[b] = fmaf(f[4 * e + 2], v.z, acc[b]);
                acc[b] = fmaf(f[4 * e + 3], v.w, acc[b]);
            }
        }
    }
    const float scale = load_scale<KIND>(a.sc, row);
#pragma unroll
    for (int b = 0; b < B; b++) {
        const float v = wave_sum(acc[b]);
        if (lane == 0) a.y[(size_t)b * a.ys + row] = v * scale;
    }
}

// The most columns that stay with the 4- to 16-column kernels of ibh_mfma.hip,
// which stage nothing that they do not need, for rows of G groups in `blocks`
// blocks of rt row tiles.  Both sides measured in a graph at 256 to 32000 rows
// of 128 to 14336 columns (the sums are the same bits); there and here:
//  - at 4 columns every shape (14336 x 4096 10.0 and 11.5 us, 2048 x 2048 3.9
//    and 4.4), at 6 most are here (12.3 and 11.5, 4.5 and 4.4);
//  - rows of up to 7 groups give a block one or two wavefronts here: 1024 x 512
//    at 8 / 16 columns 3.4 / 3.8 and 4.2 / 4.5, 1024 x 768 3.5 / 3.9 and 3.9 /
//    4.0 (one group or eight: even at 5); 2 and 3 groups cross where the
//    other kernels need a second pass, 8192 x 256 at 8 / 9 3.4 / 6.0 and 3.8;
//  - 17 to 32 groups with one block per CU: the codes staged and the hand-on
//    show, 4096 x 4096 at 8 / 12 5.5 / 6.5 and 6.0 / 5.9, 8192 x 4096 at 8 / 10
//    / 12 7.6 / 8.4 / 8.9 and 8.8;
//  - blocks that fill their last round of the CUs badly: 9216 x 8192 (288
//    blocks) at 8 / 12 19.5 / 22.6 and 22.5, 20000 x 2048 at 8 8.4 and 9.6.
// Rows that end inside a group take a pass per 4 columns there.
int w4a8_stay(int N, int rt, int blocks) {
    const int G = N / 128, rounds = (blocks + 255) / 256;
    if (N % 128) return 4;
    if (G == 2 || G == 3) return 8;
    if (rounds > 1 && rt > 1 && 8 * blocks < 7 * 256 * rounds) {
        if (rt == 2) return rounds > 2 ? (G > 48 ? 8 : 4) : G <= 48 ? 8 : G < 64 ? 12 : 10;
        return G < 9 ? 4 : G < 12 ? 12 : 9;
    }
    if (rt == 1) return G > 3 && G < 8 ? 16 : (G > 8 && G < 12) || (G > 16 && G <= 32) ? 8 : 4;
    if (rt == 2) return G < 17 ? 4 : G < 24 ? 9 : G <= 32 ? 10 : G < 64 ? 4 : 5;
    if (rt == 3) return G > 16 && G <= 32 ? 8 : 4;
    return G > 8 && G <= 16 ? 8 : 4;
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
    int rt = (T + 255) / 256;
    rt = rt > 4 ? 4 : rt;
    int KW = (G + 15) / 16 > 2 ? (G + 15) / 16 : 2;
    if (rt * KW > 8) rt = 8 / KW;
    if (rt < 1) return 0;
    const bool gather = rt == 1;
    if (gather) KW = (G + 3) / 4 < 8 ? (G + 3) / 4 : 8;
    // (matrices of a joint launch are alone there, a launch each)
    if (B <= (n > 1 ? (gather && G > 16 && G <= 32 ? 8 : 4) : w4a8_stay(N, rt, (T + rt - 1) / rt))) return 0;
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

// INT8 rows x B fp32 columns (1 <= B <= 32).  Returns 1 if launched, 0 if the
// shape is not taken, < 0 on a launch error.
int ibh_launch_int8_skinny(float* out, const void* w, const void* sc, int kind, const float* x, int M, int N, int B,
                           int M_stride, hipStream_t st) {
    if (B < 1 || B > 32 || N % 16 || N < 16 || (((uintptr_t)w | (uintptr_t)x) & 15)) return 0;
    // offsets within a launch's columns and a block's rows are 32 bits
    if (N > 1 << 26) return 0;
    const int most = (1 << 30) / N;
    if (B > most) {
        for (int b = 0; b < B; b += most) {
            const int rc = ibh_launch_int8_skinny(out + (size_t)b * M_stride, w, sc, kind, x + (size_t)b * N, M, N,
                                                  B - b < most ? B - b : most, M_stride, st);
            if (rc <= 0) return rc;
        }
        return 1;
    }
    const int G = (N + 127) / 128, T = (M + 15) / 16;
    const DigArgs a{(const int8_t*)w, sc, x, out, M, N, B, M_stride, G, (G + kDigWaves - 1) / kDigWaves};
    // One column has no digits to share: 14336 x 4096 19.0 us here, 23.5 there.
    // Two cross at 2048 rows or 1024 columns (2048 x 8192 9.9 and 11.6, 4096 x
    // 4096 10.5 and 9.3, 14336 x 512 7.9 and 8.4), three and four where the
    // wavefront-a-row blocks pass one per CU (in a graph, 1000 rows of 4096 5.0
    // and 6.6 at three, 6.2 and 6.9 at four, of 14336 11.7 and 16.3, 15.5 and
    // 16.3; 1500 rows of 4096 8.2 and 6.7, 9.6 and 6.6); a few long rows at four
    // leave most CUs idle here (256 x 8192 11.9 and 10.7, 256 x 4096 6.0 and 6.4).
    if (B == 1 || (B == 2 && (M <= 2048 || N <= 1024)) || (B == 3 && M <= 1024) ||
        (B == 4 && M <= 1024 && (M > 256 || N <= 4096))) {
#define IBH_I8V(K_) do { const int g_ = (M + 3) / 4; \
        if (B == 1) int8_rows<K_, 1><<<g_, 256, 0, st>>>(a); else if (B == 2) int8_rows<K_, 2><<<g_, 256, 0, st>>>(a); \
        else if (B == 3) int8_rows<K_, 3><<<g_, 256, 0, st>>>(a); else int8_rows<K_, 4><<<g_, 256, 0, st>>>(a); } while (0)
        if (kind == IBH_SCALE_F16) IBH_I8V(IBH_SCALE_F16); else IBH_I8V(IBH_SCALE_F32);
#undef IBH_I8V
        if (hipGetLastError() == hipSuccess) return 1;
        ibh_set_error("int8 batch: launch failed");
        return -1;
    }
    // two row tiles share the digits where that still leaves a block per CU
    const int sh = (B + 7) / 8, rt = T > 256 ? 2 : 1;
    const int blocks = (T + rt - 1) / rt;
    const size_t lds = (size_t)kDigWaves * (sh * (kDigBytes + 32) + dig_row_bufs(rt, sh) * 2048);
#define IBH_I8L(K_, R_, H_) do { \
        if (!lds_ok((const void*)int8_skinny<K_, R_, H_>, lds)) return 0; \
        int8_skinny<K_, R_, H_><<<blocks, 64 * kDigWaves, lds, st>>>(a); } while (0)
#define IBH_I8R(K_, H_) do { if (rt == 2) IBH_I8L(K_, 2, H_); else IBH_I8L(K_, 1, H_); } while (0)
#define IBH_I8S(K_) do { if (sh == 1) IBH_I8R(K_, 1); else if (sh == 2) IBH_I8R(K_, 2); \
                         else if (sh == 3) IBH_I8R(K_, 3); else IBH_I8R(K_, 4); } while (0)
    if (kind == IBH_SCALE_F16) IBH_I8S(IBH_SCALE_F16); else IBH_I8S(IBH_SCALE_F32);
#undef IBH_I8S
#undef IBH_I8R
#undef IBH_I8L
    if (hipGetLastError() == hipSuccess) return 1;
    ibh_set_error("int8 batch: launch failed");
    return -1;
}

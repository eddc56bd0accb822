// q3t_att_int.h -- the exact causal attention of the tiled prefill on int8
// MFMA.
//
// An fp16 value is a whole multiple of 2^-24, so below 127 in magnitude it is
// four balanced base-256 digits (int8 planes p: v 2^24 = sum_p d_p 256^p).
// A dot product of such values is sum_g 256^g G_g with G_g the sum over the
// digit pairs a + b = g of int8 dot products: 16 v_mfma_i32_16x16x64_i8 per
// 64 terms, exact in int32, against 16 v_mfma_f64_16x16x4f64 of 66 clocks
// (the int8 ones take 18) and two conversions per operand element.  The seven
// G_g are put together in fp64 and rounded to fp32 once.  The f64 forms
// (k_att_scores, k_att_pv) add exact products in fp64, so the results are the
// same bits wherever both sums are exact (their terms and partial sums span 53
// bits or less), and otherwise unless an fp64 rounding lands on a tie of the
// fp32 one, about one in 2^28; so too the softmax's sums (below).  Per layer at 1,600 rows of the 0.6B shapes (16 heads): scores 151 -> 51
// us, P.V 153 -> 52 us; at 209 rows 21 -> 11 and 18 -> 10 us; the softmax that
// writes digits 27 -> 36 us and the split 15 us where k_att_q took 7.  2,048
// rows would be 31 us of MFMA time per kernel; the rest is the K / V / P tiles'
// path through LDS with two workgroups per CU.
//
// A value of 127 or more (or an infinity or NaN) in q, K or V has no four
// digits: k_att_split then writes the call's number to `wide`, and the
// kernels of that call run their f64 bodies.
#pragma once

#include "q3t_prefill.h"

namespace q3t {
namespace pf {

constexpr int kIntMaxPos = 4096;  // positions of the longest row the digit softmax holds in registers

// Balanced digits of v 2^24, plane p in byte p (v an fp16 value, |v| < 127).
__device__ __forceinline__ uint32_t digits4(float v) {
    const int x = (int) (v * 16777216.0f);
    return ((uint32_t) x + 0x00808080u) ^ 0x00808080u;
}

// Byte p of each of four words as one word (e0 lowest): a 4 x 4 byte transpose.
__device__ __forceinline__ void planes4(const uint32_t (&e)[4], uint32_t (&p)[4]) {
    const uint32_t lo01 = __builtin_amdgcn_perm(e[1], e[0], 0x05010400u);   // e0.0 e1.0 e0.1 e1.1
    const uint32_t lo23 = __builtin_amdgcn_perm(e[3], e[2], 0x05010400u);
    const uint32_t hi01 = __builtin_amdgcn_perm(e[1], e[0], 0x07030602u);   // e0.2 e1.2 e0.3 e1.3
    const uint32_t hi23 = __builtin_amdgcn_perm(e[3], e[2], 0x07030602u);
    p[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
    p[1] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
    p[2] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
    p[3] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
}

__device__ __forceinline__ bool has_digits(uint16_t h) { return (h & 0x7fffu) < 0x57f0u; }   // |v| < 127

struct AttInt {
    const float * qkv; int32_t qkv_stride;
    const float * q_norm; float eps;
    const float * rc, * rs;
    const uint16_t * kc, * vc;          // the layer's cache (fp16) [kv_head][n_ctx][128]
    int32_t n_ctx, n_head, n_kv_head, n, n_past, ls;
    uint16_t * Qh;                      // fp16 q rows [head][n][128] (for the f64 bodies)
    int8_t * Qd;                        // q digits [head][n][4 planes][128]
    int8_t * Kd;                        // K digits [kv_head][ls][4 planes][128]
    int8_t * Vd;                        // V digits [kv_head][4 planes][128 dims][ls]
    int32_t * wide; int32_t call;       // *wide == call: this call's values need the f64 bodies
};

// The operands of one call.  Workgroups 0 .. nq - 1 (nq = n * ceil(n_head / 4))
// are k_att_q with the digits beside the fp16 rows; the rest split 64 cached
// positions of one KV head each, K as it lies and V transposed through LDS
// (positions past the last are written as zeros).  Bound by the memory it moves.
__global__ __launch_bounds__(kBlock) void k_att_split(AttInt a) {
    __shared__ uint16_t vt[64 * (kHD + 2)];
    const int nhq = (a.n_head + 3) / 4, nq = a.n * nhq, b = blockIdx.x, t = threadIdx.x;
    if (b < nq) {
        const int row = b / nhq, h = (b % nhq) * 4 + (t >> 6), l = t & 63, pos = a.n_past + row;
        if (h >= a.n_head) return;
        const float * src = a.qkv + (size_t) row * a.qkv_stride + h * kHD;
        float x0 = src[l], x1 = src[64 + l];
        wave_norm_rope(x0, x1, a.q_norm, a.eps, a.rc + (size_t) pos * 64, a.rs + (size_t) pos * 64);
        const uint16_t h0 = f2h(x0), h1 = f2h(x1);
        uint16_t * dst = a.Qh + ((size_t) h * a.n + row) * kHD;
        dst[l] = h0;
        dst[64 + l] = h1;
        if (!has_digits(h0) || !has_digits(h1)) *a.wide = a.call;
        const uint32_t d0 = digits4(h2f(h0)), d1 = digits4(h2f(h1));
        int8_t * qd = a.Qd + ((size_t) h * a.n + row) * 4 * kHD;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            qd[p * kHD + l] = (int8_t) (d0 >> (8 * p));
            qd[p * kHD + 64 + l] = (int8_t) (d1 >> (8 * p));
        }
        return;
    }
    const int nt = a.ls / 64, g = (b - nq) / nt, j0 = (b - nq) % nt * 64, nkv = a.n_past + a.n;
    const uint16_t * kb = a.kc + ((size_t) g * a.n_ctx + j0) * kHD;
    const uint16_t * vb = a.vc + ((size_t) g * a.n_ctx + j0) * kHD;
    bool ok = true;
#pragma unroll
    for (int u = 0; u < 8; ++u) {                       // four dims of one position each
        const int c = t + u * kBlock, r = c >> 5, d = (c & 31) * 4;
        uint2 kv = make_uint2(0, 0), vv = make_uint2(0, 0);
        if (j0 + r < nkv) {
            kv = *(const uint2 *) (kb + (size_t) r * kHD + d);
            vv = *(const uint2 *) (vb + (size_t) r * kHD + d);
        }
        const uint16_t kh[4] = {(uint16_t) kv.x, (uint16_t) (kv.x >> 16), (uint16_t) kv.y, (uint16_t) (kv.y >> 16)};
        uint32_t e[4], pl[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) { ok = ok && has_digits(kh[m]); e[m] = digits4(h2f(kh[m])); }
        planes4(e, pl);
        uint32_t * dst = (uint32_t *) (a.Kd + ((size_t) g * a.ls + j0 + r) * 4 * kHD + d);
#pragma unroll
        for (int p = 0; p < 4; ++p) dst[p * (kHD / 4)] = pl[p];
        *(uint32_t *) (vt + r * (kHD + 2) + d) = vv.x;
        *(uint32_t *) (vt + r * (kHD + 2) + d + 2) = vv.y;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 8; ++u) {                       // four positions of one dim each
        const int c = t + u * kBlock, d = c >> 4, r = (c & 15) * 4;
        uint32_t e[4], pl[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const uint16_t h = vt[(r + m) * (kHD + 2) + d];
            ok = ok && has_digits(h);
            e[m] = digits4(h2f(h));
        }
        planes4(e, pl);
        int8_t * dst = a.Vd + ((size_t) g * 4 * kHD + d) * a.ls + j0 + r;
#pragma unroll
        for (int p = 0; p < 4; ++p) *(uint32_t *) (dst + (size_t) p * kHD * a.ls) = pl[p];
    }
    if (!ok) *a.wide = a.call;
}

// sum_g 256^g G_g, scaled by 2^-48.  Pairs of neighbours meet in int32 first:
// over 128 terms |G_3| <= 128 (2 * 128 * 127 + 2 * 128 * 128) and |G_2| <= 3 *
// 2^21, so G_2 + 256 G_3 stays below 2^31 (the others are smaller).
__device__ __forceinline__ float digits_sum128(const v4i (&g)[7], int e) {
    double s = (double) g[6][e];
    s = fma(s, 65536.0, (double) (g[4][e] + (g[5][e] << 8)));
    s = fma(s, 65536.0, (double) (g[2][e] + (g[3][e] << 8)));
    s = fma(s, 65536.0, (double) (g[0][e] + (g[1][e] << 8)));
    return (float) (s * 0x1p-48);
}

// k_att_scores on the digits: the same grid, tile pairing and masks.  Wave w
// owns rows 16w..16w+15 of a 64-row tile: lane (i = l%16, k = l/16) holds
// bytes 64 c + 16 k .. +15 of row 16w + i of every q plane as A and reads the
// same bytes of position 16 t4 + i from the staged K tile as B; accumulator
// element e is row 16w + 4k + e, position 16 t4 + i.
constexpr int kKD = 4 * kHD + 16;       // LDS row stride (bytes) of a staged K digit tile
__global__ __launch_bounds__(kAttT, 2) void k_att_scores_int(AttInt a, float scale, float * __restrict__ S) {
    __shared__ __align__(16) int8_t kt[2][kAT * kKD];
    static_assert(sizeof(kt) >= 2 * kAT * kKS * 2, "the f64 body's tiles fit");
    if (*a.wide == a.call) {
        att_scores_body(a.Qh, a.kc, a.n_ctx, a.n_head, a.n_kv_head, a.n, a.n_past, scale, S, a.ls, 0,
                        (uint16_t (*)[kAT * kKS]) kt);
        return;
    }
    const int n = a.n, n_past = a.n_past, ls = a.ls;
    const int h = blockIdx.x, tiles = (n + kAT - 1) / kAT, g = h / (a.n_head / a.n_kv_head), grp = blockIdx.z;
    const int t = threadIdx.x, w = t >> 6, l = t & 63, i = l & 15, k = l >> 4;
    const int8_t * kbase = a.Kd + (size_t) g * ls * 4 * kHD;
    const int y = blockIdx.y, Y = gridDim.y;
    const bool spread = 2 * Y + 1 == tiles;                     // middle tile's K steps dealt out
    for (int pass = 0; pass < (spread ? 3 : 2); ++pass) {
        const int tile = pass == 0 ? y : pass == 1 ? tiles - 1 - y : Y;
        if (pass == 1 && tile == y) break;
        const int row0 = tile * kAT, my_row = min(row0 + 16 * w + i, n - 1);
        const int lim_tile = n_past + min(row0 + kAT, n) - 1;
        if (lim_tile < 64 * grp) continue;
        const int nst = (lim_tile - 64 * grp) / (2 * kAT) + 1;
        const int st0 = pass == 2 ? y : 0, sd = pass == 2 ? Y : 1;
        if (st0 >= nst) continue;
        v4i qa[2][4];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int p = 0; p < 4; ++p)
                qa[c][p] = *(const v4i *) (a.Qd + (((size_t) h * n + my_row) * 4 + p) * kHD + 64 * c + 16 * k);
        // a K tile is 64 rows of 512 contiguous bytes: 8 chunks of 16 per thread
        v4i rk[8];
        auto fetch = [&](int j0) {
#pragma unroll
            for (int u = 0; u < 8; ++u)
                rk[u] = *(const v4i *) (kbase + (size_t) j0 * 4 * kHD + (size_t) (t + kAttT * u) * 16);
        };
        auto stash = [&](int buf) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int c = t + kAttT * u;
                *(v4i *) (&kt[buf][(c >> 5) * kKD + (c & 31) * 16]) = rk[u];
            }
        };
        fetch(2 * kAT * st0 + 64 * grp);
        stash(0);
        __syncthreads();
        for (int st = st0, it = 0; st < nst; st += sd, ++it) {
            const int buf = it & 1, j0 = 2 * kAT * st + 64 * grp;
            const bool more = st + sd < nst;
            if (more) fetch(j0 + 2 * kAT * sd);
#pragma unroll
            for (int t4 = 0; t4 < 4; ++t4) {
                v4i acc[7];
#pragma unroll
                for (int q = 0; q < 7; ++q) acc[q] = v4i{0, 0, 0, 0};
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    v4i kb[4];
#pragma unroll
                    for (int p = 0; p < 4; ++p)
                        kb[p] = *(const v4i *) (&kt[buf][(16 * t4 + i) * kKD + p * kHD + 64 * c + 16 * k]);
#pragma unroll
                    for (int pq = 0; pq < 4; ++pq)
#pragma unroll
                        for (int pk = 0; pk < 4; ++pk)
                            acc[pq + pk] = __builtin_amdgcn_mfma_i32_16x16x64_i8(qa[c][pq], kb[pk], acc[pq + pk], 0, 0, 0);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int row = row0 + 16 * w + 4 * k + e, j = j0 + 16 * t4 + i;
                    if (row < n && j <= n_past + row)
                        S[((size_t) h * n + row) * ls + j] = digits_sum128(acc, e) * scale;
                }
            }
            __asm__ volatile("" ::: "memory");
            if (more) stash(buf ^ 1);
            __syncthreads();
        }
    }
}

// One row held in registers, RQ groups of four consecutive positions per lane:
// softmax_row_reg with the probabilities' digits written over the row's own
// scores, [4 planes][ls] bytes (zeros from cnt to jend, the end of the last
// tile that k_att_pv_int reads).  The same exponentials in another order of the
// fp64 sum (there a lane has every 64th position): its last bits may differ,
// and the fp32 reciprocal where they meet a tie.
template <int RQ>
__device__ __forceinline__ void softmax_row_digits(float * sr, int cnt, int jend, int ls, int lane) {
    float4 v[RQ];
    float m = -INFINITY;
#pragma unroll
    for (int u = 0; u < RQ; ++u) {
        const int j = 4 * lane + 256 * u;
        v[u] = j < cnt ? *(const float4 *) (sr + j) : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
        if (j + 1 >= cnt) v[u].y = -INFINITY;
        if (j + 2 >= cnt) v[u].z = -INFINITY;
        if (j + 3 >= cnt) v[u].w = -INFINITY;
        m = fmaxf(m, fmaxf(fmaxf(v[u].x, v[u].y), fmaxf(v[u].z, v[u].w)));
    }
    const float mx = wave_max_f(m);
    double sum = 0.0;
#pragma unroll
    for (int u = 0; u < RQ; ++u) {
        const int j = 4 * lane + 256 * u;
        v[u].x = j < cnt ? expf_q3t(v[u].x - mx) : 0.0f;
        v[u].y = j + 1 < cnt ? expf_q3t(v[u].y - mx) : 0.0f;
        v[u].z = j + 2 < cnt ? expf_q3t(v[u].z - mx) : 0.0f;
        v[u].w = j + 3 < cnt ? expf_q3t(v[u].w - mx) : 0.0f;
        sum += (double) v[u].x; sum += (double) v[u].y; sum += (double) v[u].z; sum += (double) v[u].w;
    }
    const float inv = (float) (1.0 / wave_sum_d(sum));
    int8_t * pr = (int8_t *) sr;
#pragma unroll
    for (int u = 0; u < RQ; ++u) {
        const int j = 4 * lane + 256 * u;
        if (j >= jend) continue;
        const float e4[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
        uint32_t e[4], pl[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) e[q] = digits4(h2f(f2h(e4[q] * inv)));
        planes4(e, pl);
#pragma unroll
        for (int p = 0; p < 4; ++p) *(uint32_t *) (pr + (size_t) p * ls + j) = pl[p];
    }
}

// k_att_softmax with digit rows: grid (ceil(n / 4), n_head), one wave per row,
// rows of up to kIntMaxPos positions.
__global__ __launch_bounds__(kBlock) void k_att_softmax_int(AttInt a, float * S, uint16_t * __restrict__ P) {
    const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6), h = blockIdx.y;
    if (row >= a.n) return;                   // whole wave
    const size_t at = ((size_t) h * a.n + row) * a.ls;
    if (*a.wide == a.call) {
        att_softmax_row(S + at, P + at, a.n_past + row + 1, lane, 0);
        return;
    }
    const int cnt = a.n_past + row + 1, last = a.n_past + min(row / kAT * kAT + kAT, a.n) - 1;
    const int jend = (last / kAT + 1) * kAT;
    if (jend <= 256 * 4) softmax_row_digits<4>(S + at, cnt, jend, a.ls, lane);
    else if (jend <= 256 * 8) softmax_row_digits<8>(S + at, cnt, jend, a.ls, lane);
    else if (jend <= 256 * 10) softmax_row_digits<10>(S + at, cnt, jend, a.ls, lane);
    else softmax_row_digits<16>(S + at, cnt, jend, a.ls, lane);
}

// sum_g 256^g G_g 2^-48 of sums over any number of positions.
__device__ __forceinline__ float digits_sum(const v4i (&g)[7], int e) {
    double s = (double) g[6][e];
#pragma unroll
    for (int q = 5; q >= 0; --q) s = fma(s, 256.0, (double) g[q][e]);
    return (float) (s * 0x1p-48);
}

// k_att_pv on the digits: the same grid, tile pairing and dealt-out middle
// tile.  The wave's P rows come straight from memory (no other wave reads
// them), lane (i, k) holding positions 16 k .. +15 of its row of every plane;
// the V tile [4 planes][64 dims][64 positions] is staged in LDS, double-
// buffered.  A digit plane of P that is zero over the wave's 16 rows x 64
// positions is skipped: P below 2^-9 has two planes, below 1/2 three.
constexpr int kVDS = 64 + 16;           // LDS row stride (bytes) of a staged V digit row
__global__ __launch_bounds__(kAttT, 2) void k_att_pv_int(AttInt a, const int8_t * __restrict__ Pd,
                                                         const uint16_t * __restrict__ P, float * __restrict__ out,
                                                         int32_t out_stride) {
    __shared__ __align__(16) int8_t vt[2][4 * 64 * kVDS];
    static_assert(sizeof(vt) >= 2 * kAT * (kVS + kVN) * 2, "the f64 body's tiles fit");
    if (*a.wide == a.call) {
        uint16_t * lds = (uint16_t *) vt;
        att_pv_body(P, a.ls, a.vc, a.n_ctx, a.n_head, a.n_kv_head, a.n, a.n_past, out, out_stride, 0,
                    (uint16_t (*)[kAT * kVS]) lds, (uint16_t (*)[kAT * kVN]) (lds + 2 * kAT * kVS));
        return;
    }
    const int n = a.n, n_past = a.n_past, ls = a.ls;
    const int h = blockIdx.x, tiles = (n + kAT - 1) / kAT, g = h / (a.n_head / a.n_kv_head), grp = blockIdx.z;
    const int t = threadIdx.x, w = t >> 6, l = t & 63, i = l & 15, k = l >> 4;
    const int y = blockIdx.y, Y = gridDim.y;
    const int nrg = (2 * Y + 1 == tiles && y < 4) ? (4 - y + Y - 1) / Y : 0;
    for (int pass = 0; pass < 2 + nrg; ++pass) {
        const int rg = pass < 2 ? -1 : y + (pass - 2) * Y;
        const int tile = pass == 0 ? y : pass == 1 ? tiles - 1 - y : Y;
        if (pass == 1 && tile == y) continue;
        const int row0 = tile * kAT, prow = row0 + (rg < 0 ? 16 * w : 16 * rg);
        const int nst = (n_past + min(row0 + kAT, n) - 1) / kAT + 1;
        const int8_t * pr = Pd + ((size_t) h * n + min(prow + i, n - 1)) * ls * 4 + 16 * k;
        v4i rv[4], rp[4];
        auto fetch = [&](int j0) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                rp[p] = *(const v4i *) (pr + (size_t) p * ls + j0);
                rv[p] = *(const v4i *) (a.Vd + (((size_t) g * 4 + p) * kHD + 64 * grp + (t >> 2)) * ls + j0 + 16 * (t & 3));
            }
        };
        auto stash = [&](int buf) {
#pragma unroll
            for (int p = 0; p < 4; ++p) *(v4i *) (&vt[buf][(p * 64 + (t >> 2)) * kVDS + 16 * (t & 3)]) = rv[p];
        };
        v4i acc[4][7];
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int q = 0; q < 7; ++q) acc[b][q] = v4i{0, 0, 0, 0};
        auto mm = [&](int buf, int b, int dim, const v4i (&pa)[4], bool p2, bool p3) {
            v4i vb[4];
#pragma unroll
            for (int p = 0; p < 4; ++p) vb[p] = *(const v4i *) (&vt[buf][(p * 64 + dim + i) * kVDS + 16 * k]);
#pragma unroll
            for (int pp = 0; pp < 4; ++pp) {
                if ((pp == 2 && !p2) || (pp == 3 && !p3)) continue;
#pragma unroll
                for (int pv = 0; pv < 4; ++pv)
                    acc[b][pp + pv] = __builtin_amdgcn_mfma_i32_16x16x64_i8(pa[pp], vb[pv], acc[b][pp + pv], 0, 0, 0);
            }
        };
        fetch(0);
        stash(0);
        __syncthreads();
        for (int st = 0; st < nst; ++st) {
            const int buf = st & 1;
            const v4i pa[4] = {rp[0], rp[1], rp[2], rp[3]};
            if (st + 1 < nst) fetch((st + 1) * kAT);
            const bool p2 = __any((pa[2].x | pa[2].y | pa[2].z | pa[2].w) != 0);
            const bool p3 = __any((pa[3].x | pa[3].y | pa[3].z | pa[3].w) != 0);
            if (rg < 0) {
#pragma unroll
                for (int b = 0; b < 4; ++b) mm(buf, b, 16 * b, pa, p2, p3);
            } else {
                mm(buf, 0, 16 * w, pa, p2, p3);
            }
            __asm__ volatile("" ::: "memory");
            if (st + 1 < nst) stash(buf ^ 1);
            __syncthreads();
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if (rg >= 0 && b > 0) break;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = prow + 4 * k + e;
                if (row < n)
                    out[(size_t) row * out_stride + h * kHD + 64 * grp + 16 * (rg < 0 ? b : w) + i] = digits_sum(acc[b], e);
            }
        }
    }
}

}  // namespace pf
}  // namespace q3t

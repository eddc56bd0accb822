// The fast causal attention of the tiled F16 prefill: scores, softmax and P.V
// of one 64-row tile and head in one workgroup, on fp16 (bfloat16) MFMA with
// fp32 accumulation (the reference's F16 K.Q and V.P product class,
// src/tts_transformer.cpp:1474-1617 via ggml).  No score or probability goes
// to memory: as three kernels (scores, softmax, P.V) 2,049 rows took 158 us a
// layer, most of it the 537 MB of fp32 scores and 16-bit probabilities written
// and read back.
//   - The same numbers as those three kernels, bit for bit.  A score is its MFMA
//     chain over the head dims times the scale; the row's maximum over all its
//     positions comes first; exponentials are expf_q3t's; their fp64 sum runs
//     through 64 partial sums (position mod 64, tiles in order) and a tree of
//     neighbours, as a wave adds them one position a lane; a probability is the
//     exponential times the fp32 reciprocal, rounded to 16 bits once; P.V adds
//     32 positions an MFMA, in order.  So three sweeps over the row's K tiles
//     (maximum, sum, probabilities and P.V), each with its own K.Q MFMAs.
//   - Scores are computed transposed, S^T = K . Q^T (A = 16 positions, B = 16 q
//     rows), with A's row m of block h at position 32 grp + 8 (m / 4) + 4h + m % 4:
//     lane (i = l % 16, k = l / 16) then holds positions 32 grp + 8k .. +7 of q row
//     16w + i, which as 16-bit probabilities are the B operand of O^T = V^T . P^T
//     where they lie.
//   - Eight waves: both groups of four have the same 64 rows, group grp the
//     positions 32 grp .. +31 of every tile and the output dims 64 grp .. +63; the
//     groups exchange maxima, sums and, a 16-byte word a lane and tile, the
//     probabilities through LDS.  P.V runs a tile behind the probabilities, so that
//     its MFMAs stand beside the next tile's exponentials and a tile costs one
//     barrier.  K and V^T tiles are double-buffered (the first two sweeps hold two
//     K tiles a stage): 80 KB, two workgroups a CU, four waves a SIMD.
//   - Bound by the vector ALU: at 2,049 rows of 16 heads 131,000 of the 155,000
//     clocks that a CU is busy (two exponentials an element, 18 operations each, of
//     58 in all), and by the longest sweep, 33 tiles of 2.4 us on one CU, where
//     the kernel takes 82 us.  With 10 us for the operands: 92 us a layer (170 as
//     q rows, scores, softmax, P.V and rounding); 600 rows 30 (44), 200 rows 17 (29).
//     Loads two stages ahead, or the next tile's scores beside this tile's
//     exponentials, change nothing (83 to 85 us).
#pragma once

#include "q3t_prefill.h"

namespace q3t {
namespace pf {

// One 16x16x32 MFMA with fp32 accumulation on fp16 (or, bf, bfloat16)
// operands held as 16-bit patterns.
template <bool BF>
__device__ __forceinline__ f4v mfma_h32(const v4i & av, const v4i & bv, f4v c) {
    if constexpr (BF) {
        typedef __bf16 b8v __attribute__((ext_vector_type(8)));
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8v, av), __builtin_bit_cast(b8v, bv), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8v, av), __builtin_bit_cast(h8v, bv), c, 0, 0, 0);
    }
}

struct AttFlash {
    const float * qkv; int32_t qkv_stride;
    const float * q_norm; float eps;
    const float * rc, * rs;
    const uint16_t * kc, * vc;          // the layer's cache [kv_head][n_ctx][128]
    int32_t n_ctx, n_head, n_kv_head, n, n_past, bf;
    int32_t batch;                      // row tiles a head that one workgroup per CU takes
    uint16_t * Qh;                      // q rows [head][n][128]
    uint16_t * Vt;                      // V^T tiles [kv_head][ceil((n_past + n) / 64)][128 dims][64 positions]
};

// The operands of one call.  Workgroups 0 .. n * ceil(n_head / 4) - 1 are
// k_att_q's; the rest transpose 64 cached V rows of one kv head each (rows past
// the last position as zero).
__global__ __launch_bounds__(kBlock) void k_att_flash_in(AttFlash a) {
    __shared__ uint16_t vt[64 * (kHD + 2)];
    const int nhq = (a.n_head + 3) / 4, nq = a.n * nhq, b = blockIdx.x, t = threadIdx.x;
    if (b < nq) {
        att_q_rows(a.qkv, a.qkv_stride, a.q_norm, a.eps, a.rc, a.rs, a.n, a.n_past, a.n_head, a.Qh, a.bf, b / nhq,
                   b % nhq);
        return;
    }
    const int nkv = a.n_past + a.n, nt = (nkv + 63) / 64, g = (b - nq) / nt, tile = (b - nq) % nt, j0 = tile * 64;
    const uint16_t * vb = a.vc + ((size_t) g * a.n_ctx + j0) * kHD;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int c = t + u * kBlock, r = c >> 4, d = (c & 15) * 8;
        int4 v = make_int4(0, 0, 0, 0);
        if (j0 + r < nkv) v = *(const int4 *) (vb + (size_t) r * kHD + d);
        uint32_t * dst = (uint32_t *) (vt + r * (kHD + 2) + d);
        dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; dst[3] = v.w;
    }
    __syncthreads();
    uint16_t * out = a.Vt + ((size_t) g * nt + tile) * kHD * 64;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int c = t + u * kBlock, d = c >> 3, s = (c & 7) * 8;
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            w[e] = vt[(s + 2 * e) * (kHD + 2) + d] | (uint32_t) vt[(s + 2 * e + 1) * (kHD + 2) + d] << 16;
        *(int4 *) (out + (size_t) c * 8) = make_int4(w[0], w[1], w[2], w[3]);
    }
}

// p0 and p1 as 16-bit values of one word (round to nearest even)
template <bool BF>
__device__ __forceinline__ uint32_t pack_kv(float p0, float p1) {
    if constexpr (BF) {
        typedef __bf16 b2v __attribute__((ext_vector_type(2)));
        const b2v v = {(__bf16) p0, (__bf16) p1};
        return __builtin_bit_cast(uint32_t, v);
    } else {
        return f2h(p0) | (uint32_t) f2h(p1) << 16;
    }
}

// expf_q3t of four x <= 0 (or NaN), the same bits: the steps for large x are left
// out, and the rounded multiple k of ln 2 is taken from the low bits of k + 1.5 2^23
// (a sum that rounds as rintf does), which also give 2^k.  Four chains side by
// side: one alone waits on its own results with two waves a SIMD.
__device__ __forceinline__ f4v expf_neg(f4v x) {
    typedef uint32_t u4v __attribute__((ext_vector_type(4)));
    const f4v kb = x * 1.44269504088896341f + 12582912.0f, k = kb - 12582912.0f;
    f4v r = __builtin_elementwise_fma(-k, (f4v) 0.693145751953125f, x);
    r = __builtin_elementwise_fma(-k, (f4v) 1.428606765330187e-06f, r);
    f4v p = 1.98412698412698413e-4f;
    p = __builtin_elementwise_fma(p, r, (f4v) 1.38888888888888889e-3f);
    p = __builtin_elementwise_fma(p, r, (f4v) 8.33333333333333333e-3f);
    p = __builtin_elementwise_fma(p, r, (f4v) 4.16666666666666667e-2f);
    p = __builtin_elementwise_fma(p, r, (f4v) 1.66666666666666667e-1f);
    p = __builtin_elementwise_fma(p, r, (f4v) 0.5f);
    p = __builtin_elementwise_fma(p, r, (f4v) 1.0f);
    p = __builtin_elementwise_fma(p, r, (f4v) 1.0f);
    p *= __builtin_bit_cast(f4v, (__builtin_bit_cast(u4v, kb) << 23) + 0x3f800000u);
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = x[e] < -87.0f ? 0.0f : p[e];
    return p;
}

// The row tile that the y-th workgroup of a head takes.  The first `batch` take
// the longest sweeps, longest first, the next `batch` the next longest, shortest
// first, so that the two workgroups a CU holds at first are about equally long
// together on every CU; the rest longest first, so that short ones fill the end.
__host__ __device__ constexpr int flash_tile(int y, int tiles, int batch) {
    const int lo = tiles > 2 * batch ? tiles - 2 * batch : 0;
    return y < batch || y >= 2 * batch ? tiles - 1 - y : lo + y - batch;
}

constexpr int kFT = 512;               // threads of k_att_flash
constexpr int kFTile = kAT * kHD;      // halves of one K or V^T tile in LDS
constexpr int kFlashLds = 4 * kFTile + 2 * kFT * 8;   // halves: four tiles, two P tiles

// LDS: tiles 0 .. 3 of 16 KB.  A K tile is [position][dim] in 16-byte chunks,
// chunk c of position p at c ^ fk(p) with fk(p) = p % 4 + 4 ((p / 8) % 4): the 16
// positions that the lanes of a read take are 16 different chunks.  A V^T tile
// is [dim][position], chunk c of dim d at c ^ (d / 2) % 8.  Then two P tiles
// [w][grp][lane] of 16 bytes; the first also takes the groups' maxima and sums.
template <bool BF>
__device__ __forceinline__ void att_flash_body(const AttFlash & a, float scale, uint16_t * __restrict__ out,
                                               int32_t out_stride, uint16_t * __restrict__ lds) {
    const int h = blockIdx.x, tile = flash_tile(blockIdx.y, gridDim.y, a.batch), g = h / (a.n_head / a.n_kv_head);
    const int t = threadIdx.x, grp = __builtin_amdgcn_readfirstlane(t >> 8), w = (t >> 6) & 3;
    const int l = t & 63, i = l & 15, k = l >> 4;
    const int row0 = tile * kAT, row = row0 + 16 * w + i, lim = a.n_past + row;
    const int lim_tile = a.n_past + min(row0 + kAT, a.n) - 1, nst = lim_tile / kAT + 1, ns = (nst + 1) / 2;
    const int diag = a.n_past + row0 + 16 * w;      // from this position on a tile needs the mask
    const int nt = (a.n_past + a.n + 63) / 64;
    const int sp = t >> 4, sc = t & 15, sd = t >> 3, sv = t & 7;   // staging: K position, chunk; V^T dim, chunk
    const uint16_t * const kbase = a.kc + (size_t) g * a.n_ctx * kHD, * const vbase = a.Vt + (size_t) g * nt * kFTile;
    uint16_t * const kdst = lds + sp * kHD + ((sc ^ ((sp & 3) | ((sp >> 3) & 3) << 2)) << 3);
    uint16_t * const vdst = lds + sd * 64 + ((sv ^ ((sd >> 1) & 7)) << 3);
    v4i * const pt = (v4i *) (lds + 4 * kFTile);
    v4i qf[4];                                      // dims 32c + 8k .. +7 of the lane's row (rows past n: row n - 1)
#pragma unroll
    for (int c = 0; c < 4; ++c)
        qf[c] = *(const v4i *) (a.Qh + ((size_t) h * a.n + min(row, a.n - 1)) * kHD + 32 * c + 8 * k);
    // the q rows are here before the first tile's loads go out: a wait for them inside
    // the loop would wait for the loads of the next tile too
#pragma unroll
    for (int c = 0; c < 4; ++c) __asm__ volatile("" : "+v"(qf[c]));
    v4i rk[4], rv[2];
    auto fetch_k = [&](int st, int at) {            // K tile st (past the last one: the last one again, never used)
        const int j0 = min(st, nst - 1) * kAT;
#pragma unroll
        for (int u = 0; u < 2; ++u)
            rk[at + u] = *(const v4i *) (kbase + (uint32_t) (min(j0 + sp + 32 * u, lim_tile) * kHD + 8 * sc));
    };
    auto stash_k = [&](int region, int at) {
#pragma unroll
        for (int u = 0; u < 2; ++u) *(v4i *) (kdst + region * kFTile + 32 * u * kHD) = rk[at + u];
    };
    auto fetch_v = [&](int st) {
#pragma unroll
        for (int u = 0; u < 2; ++u) rv[u] = *(const v4i *) (vbase + (uint32_t) (st * kFTile + 8 * (t + kFT * u)));
    };
    // V of later tiles' rows is staged as zero: the probabilities here are zero, the values may be infinite
    auto keep = [&](int p) { return (p <= lim_tile ? 0xffff : 0) | (p + 1 <= lim_tile ? (int) 0xffff0000u : 0); };
    auto stash_v = [&](int st, int region) {
        const int p = st * kAT + 8 * sv;
        const v4i kv = {keep(p), keep(p + 2), keep(p + 4), keep(p + 6)};
#pragma unroll
        for (int u = 0; u < 2; ++u) *(v4i *) (vdst + region * kFTile + 64 * u * 64) = rv[u] & kv;
    };
    // scores (before the scale) of positions 64 st + 32 grp + 8k + 4b + r
    const uint16_t * const ks = lds + (32 * grp + 8 * (i >> 2) + (i & 3)) * kHD;
    auto scores = [&](int region, f4v (&s)[2]) {
#pragma unroll
        for (int b = 0; b < 2; ++b) s[b] = (f4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int b = 0; b < 2; ++b)
                s[b] = mfma_h32<BF>(*(const v4i *) (ks + region * kFTile + 4 * b * kHD + (((4 * c + k) ^ i) << 3)), qf[c], s[b]);
    };
    auto mask = [&](int st, f4v (&s)[2], float m) { // past the row's last position: m
        if (st * kAT + kAT - 1 <= diag) return;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) s[b][r] = st * kAT + 32 * grp + 8 * k + 4 * b + r > lim ? m : s[b][r];
    };
    // LDS stores (and the wait for their loads) stay behind the arithmetic before them
    auto fence = [&] {
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // One sweep over the K tiles in ns stages of two: stage q computes from regions 2 ((q0 + q) & 1) and
    // the next and fetches the stage after it, the last one the next sweep's first
    auto sweep = [&](int q0, auto && tile_fn) {
        for (int q = 0; q < ns; ++q) {
            const int next = q + 1 < ns ? 2 * (q + 1) : 0, buf = 2 * ((q0 + q) & 1);
            fetch_k(next, 0);
            fetch_k(next + 1, 2);
            tile_fn(2 * q, buf);
            if (2 * q + 1 < nst) tile_fn(2 * q + 1, buf + 1);
            fence();
            stash_k(buf ^ 2, 0);
            stash_k((buf ^ 2) + 1, 2);
            __syncthreads();
        }
    };
    fetch_k(0, 0);
    fetch_k(1, 2);
    stash_k(0, 0);
    stash_k(1, 2);
    __syncthreads();

    float mx = -INFINITY;                           // the row's largest score
    sweep(0, [&](int st, int region) {
        f4v s[2];
        scores(region, s);
        mask(st, s, -INFINITY);
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[b][r]);
    });
    float * const xf = (float *) pt;
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    xf[t] = mx;
    __syncthreads();
    mx = fmaxf(mx, xf[t ^ 256]) * scale;            // rounding keeps the order: the largest scaled score

    double sum[2][4];                               // of the row's exponentials, position mod 64
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[b][r] = 0.0;
    sweep(ns, [&](int st, int region) {
        f4v s[2];
        scores(region, s);
#pragma unroll
        for (int b = 0; b < 2; ++b) s[b] = expf_neg(s[b] * scale - mx);
        mask(st, s, 0.0f);
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[b][r] += (double) s[b][r];
    });
    double s0 = ((sum[0][0] + sum[0][1]) + (sum[0][2] + sum[0][3])) + ((sum[1][0] + sum[1][1]) + (sum[1][2] + sum[1][3]));
    s0 += __shfl_xor(s0, 16);
    s0 += __shfl_xor(s0, 32);
    double * const xd = (double *) pt;
    xd[t] = s0;
    __syncthreads();
    const float inv = (float) (1.0 / (s0 + xd[t ^ 256]));
    __syncthreads();

    // Probabilities of tile st and P.V of tile st - 1.  2 ns stages are behind, so tile 0 is in
    // region 0: K of tile st in region 2 (st & 1), its V^T in the one after.
    f4v o[4];                                       // dims 64 grp + 16b + 4k + r of the lane's row
#pragma unroll
    for (int b = 0; b < 4; ++b) o[b] = (f4v){0.f, 0.f, 0.f, 0.f};
    const uint16_t * const vs = lds + (64 * grp + i) * 64;
    auto pv = [&](int st) {
        const uint16_t * v = vs + (2 * (st & 1) + 1) * kFTile;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const v4i pb = pt[(st & 1) * kFT + (2 * w + c) * 64 + l];
#pragma unroll
            for (int b = 0; b < 4; ++b)
                o[b] = mfma_h32<BF>(*(const v4i *) (v + 16 * b * 64 + (((4 * c + k) ^ ((i >> 1) & 7)) << 3)), pb, o[b]);
        }
    };
    for (int st = 0; st < nst; ++st) {
        fetch_k(st + 1, 0);
        fetch_v(st);
        f4v s[2];
        scores(2 * (st & 1), s);
        if (st) pv(st - 1);
#pragma unroll
        for (int b = 0; b < 2; ++b) s[b] = expf_neg(s[b] * scale - mx) * inv;
        mask(st, s, 0.0f);
        const v4i pw = {(int) pack_kv<BF>(s[0][0], s[0][1]), (int) pack_kv<BF>(s[0][2], s[0][3]),
                        (int) pack_kv<BF>(s[1][0], s[1][1]), (int) pack_kv<BF>(s[1][2], s[1][3])};
        fence();
        pt[(st & 1) * kFT + (2 * w + grp) * 64 + l] = pw;
        stash_k(2 * ((st + 1) & 1), 0);
        stash_v(st, 2 * (st & 1) + 1);
        __syncthreads();
    }
    pv(nst - 1);
    if (row >= a.n) return;
#pragma unroll
    for (int b = 0; b < 4; ++b)
        *(uint2 *) (out + (size_t) row * out_stride + h * kHD + 64 * grp + 16 * b + 4 * k) =
            make_uint2(f2h(o[b][0]) | (uint32_t) f2h(o[b][1]) << 16, f2h(o[b][2]) | (uint32_t) f2h(o[b][3]) << 16);
}

// grid (n_head, ceil(n / 64)); out: the attention rows in fp16, as the output
// GEMM takes them.
__global__ __launch_bounds__(kFT, 4) void k_att_flash(AttFlash a, float scale, uint16_t * __restrict__ out,
                                                      int32_t out_stride) {
    __shared__ __align__(16) uint16_t lds[kFlashLds];
    if (a.bf) att_flash_body<true>(a, scale, out, out_stride, lds);
    else att_flash_body<false>(a, scale, out, out_stride, lds);
}

}  // namespace pf
}  // namespace q3t

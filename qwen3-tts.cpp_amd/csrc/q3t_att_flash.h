// The fast causal attention of the tiled F16 prefill: scores, softmax and P.V
// of one 64-row tile and head in one workgroup, on fp16 (bfloat16) MFMA with
// fp32 accumulation (the reference's F16 K.Q and V.P product class,
// src/tts_transformer.cpp:1474-1617 via ggml).  No score or probability goes
// to memory: as three kernels (scores, softmax, P.V) 2,049 rows took 158 us a
// layer, most of it the 537 MB of fp32 scores and 16-bit probabilities written
// and read back.
//   - Scores are computed transposed, S^T = K . Q^T (A = 16 positions, B = 16 q
//     rows), so lane (i = l % 16, k = l / 16) holds positions 16 t + 4k + r of
//     q row 16w + i: the row's maximum is one register sweep and two shuffles,
//     and the probabilities are the B operand of O^T = V^T . P^T where they
//     lie.  A contraction may take its positions in any order that both operands
//     share, so V^T holds the 32 positions of an MFMA in the order the scores
//     leave them (vt_pos) and one 16-byte LDS read is lane (i, k)'s A operand.
//   - Online softmax per row in powers of two: p = 2^(s c - m c), c = scale
//     log2(e), m the largest raw score so far (a finite lowest value before the
//     first tile, so that a row of -inf scores stays finite).  The accumulators
//     are rescaled only in a tile that raises a maximum.  p is rounded to 16 bits
//     unnormalised; the row's sum is one more MFMA row of ones over the same
//     rounded values, so their rounding leaves no bias; one division ends the row.
//   - Bound by LDS reads (32 KB a wave and tile) and the vector ALU (16
//     exponentials and their conversions a lane and tile), MFMAs a quarter of it.
//     Eight waves: one group of four takes the even 64-position tiles, one the
//     odd, both for the same 64 rows, and their parts of a row are joined at the
//     end; each group's K and V^T tiles are double-buffered (143 KB, one workgroup
//     a CU).  heads x tiles workgroups, longest sweeps dispatched first, so that
//     short ones fill the end.  2,049 rows: 47 us a layer and 10 us for the operands
//     (one group of four waves and two workgroups a CU: 76 us).
#pragma once

#include "q3t_prefill.h"

namespace q3t {
namespace pf {

constexpr int kVT = 64 + 8;      // LDS row stride (halves) of a V^T tile: conflict-free 16-byte reads

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

// Position (within a 64-position tile) at element s of a V^T row: MFMA s / 32
// takes element e of lane group k = (s / 8) % 4 from score block 2 (s / 32) + e / 4.
__device__ __forceinline__ int vt_pos(int s) {
    const int e = s & 7;
    return (s & 32) + 16 * (e >> 2) + 4 * ((s >> 3) & 3) + (e & 3);
}

struct AttFlash {
    const float * qkv; int32_t qkv_stride;
    const float * q_norm; float eps;
    const float * rc, * rs;
    const uint16_t * kc, * vc;          // the layer's cache [kv_head][n_ctx][128]
    int32_t n_ctx, n_head, n_kv_head, n, n_past, bf;
    uint16_t * Qh;                      // q rows [head][n][128]
    uint16_t * Vt;                      // V^T tiles [kv_head][ceil((n_past + n) / 64)][128 dims][64], order vt_pos
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
            w[e] = vt[vt_pos(s + 2 * e) * (kHD + 2) + d] | (uint32_t) vt[vt_pos(s + 2 * e + 1) * (kHD + 2) + d] << 16;
        *(int4 *) (out + (size_t) c * 8) = make_int4(w[0], w[1], w[2], w[3]);
    }
}

// p[0] and p[1] as 16-bit values of one word (round to nearest even)
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

// The largest of a value's four copies in lanes i, i + 16, i + 32, i + 48: a swap of
// 16-lane rows (of 32-lane halves) leaves a row beside its neighbour in two registers.
__device__ __forceinline__ float max_lane_groups(float x) {
    typedef unsigned int u2v __attribute__((ext_vector_type(2)));
    u2v s = __builtin_bit_cast(u2v, __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false));
    x = fmaxf(__uint_as_float(s.x), __uint_as_float(s.y));
    s = __builtin_bit_cast(u2v, __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false));
    return fmaxf(__uint_as_float(s.x), __uint_as_float(s.y));
}

constexpr int kFT = 512;         // threads of k_att_flash

template <bool BF>
__device__ __forceinline__ void att_flash_body(const AttFlash & a, float c2, uint16_t * __restrict__ out,
                                               int32_t out_stride, uint16_t * __restrict__ lds) {
    const int h = blockIdx.x, tile = gridDim.y - 1 - blockIdx.y, g = h / (a.n_head / a.n_kv_head);
    const int grp = threadIdx.x >> 8, t = threadIdx.x & 255, w = t >> 6, l = t & 63, i = l & 15, k = l >> 4;
    const int row0 = tile * kAT, row = row0 + 16 * w + i, lim = a.n_past + row;
    const int lim_tile = a.n_past + min(row0 + kAT, a.n) - 1, nst = lim_tile / kAT + 1, nit = (nst + 1) / 2;
    const int nt = (a.n_past + a.n + 63) / 64;
    const uint16_t * kbase = a.kc + (size_t) g * a.n_ctx * kHD + 8 * (t & 15);
    const uint16_t * vbase = a.Vt + (size_t) g * nt * kHD * 64 + 8 * t;
    uint16_t * const kt = lds + grp * 2 * kAT * kKS, * const vt = lds + 4 * kAT * kKS + grp * 2 * kHD * kVT;
    v4i qf[4];                                      // dims 32c + 8k .. +7 of the lane's row (rows past n: row n - 1)
#pragma unroll
    for (int c = 0; c < 4; ++c)
        qf[c] = *(const v4i *) (a.Qh + ((size_t) h * a.n + min(row, a.n - 1)) * kHD + 32 * c + 8 * k);
    // the q rows are here before the first tile's loads go out: a wait for them inside
    // the loop would wait for the loads of the next tile too
#pragma unroll
    for (int c = 0; c < 4; ++c) __asm__ volatile("" : "+v"(qf[c]));
    v4i rk[4], rv[4];
    auto fetch = [&](int st) {                      // tile st (st >= nst: the last one again, never used)
        const int j0 = min(st, nst - 1) * kAT;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            rk[u] = *(const v4i *) (kbase + (size_t) min(j0 + (t >> 4) + 16 * u, lim_tile) * kHD);
            rv[u] = *(const v4i *) (vbase + (size_t) j0 * kHD + 8 * 256 * u);
        }
    };
    // V of later tiles' rows is staged as zero: the probabilities here are zero, the values may be infinite
    auto keep = [&](int p) { return (p <= lim_tile ? 0xffff : 0) | (p + 1 <= lim_tile ? (int) 0xffff0000u : 0); };
    auto stash = [&](int st, int buf) {
        uint16_t * kd = kt + buf * kAT * kKS + (t >> 4) * kKS + 8 * (t & 15);
        uint16_t * vd = vt + buf * kHD * kVT + (t >> 3) * kVT + 8 * (t & 7);
        const int p = st * kAT + vt_pos(8 * (t & 7));
        const v4i kv = {keep(p), keep(p + 2), keep(p + 16), keep(p + 18)};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            *(v4i *) (kd + 16 * u * kKS) = rk[u];
            *(v4i *) (vd + 32 * u * kVT) = rv[u] & kv;
        }
    };
    constexpr int kOne = BF ? 0x3f803f80 : 0x3c003c00;
    const v4i ones = {kOne, kOne, kOne, kOne};
    f4v o[8], os = (f4v){0.f, 0.f, 0.f, 0.f};       // dims 16b + 4k + r of the lane's row; its sum in every element
#pragma unroll
    for (int b = 0; b < 8; ++b) o[b] = (f4v){0.f, 0.f, 0.f, 0.f};
    float m = -3.0e38f, mc = m * c2;
    fetch(grp);
    stash(grp, 0);
    __syncthreads();
    for (int it = 0; it < nit; ++it) {
        const int buf = it & 1, st = 2 * it + grp, j0 = st * kAT;
        const bool more = it + 1 < nit;
        if (more) fetch(st + 2);
        if (st < nst) {
            const uint16_t * ks = kt + buf * kAT * kKS + i * kKS + 8 * k;
            const uint16_t * vs = vt + buf * kHD * kVT + i * kVT + 8 * k;
            f4v s[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) s[b] = (f4v){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int b = 0; b < 4; ++b) s[b] = mfma_h32<BF>(*(const v4i *) (ks + 16 * b * kKS + 32 * c), qf[c], s[b]);
            if (j0 + kAT - 1 > a.n_past + row0 + 16 * w) {
#pragma unroll
                for (int b = 0; b < 4; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        s[b][r] = j0 + 16 * b + 4 * k + r > lim ? -INFINITY : s[b][r];
            }
            float mx = m;
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[b][r]);
            mx = max_lane_groups(mx);
            if (__any(mx > m)) {
                const float mn = mx * c2, al = __builtin_amdgcn_exp2f(mc - mn);
                m = mx;
                mc = mn;
                os *= al;
#pragma unroll
                for (int b = 0; b < 8; ++b) o[b] *= al;
            }
            uint32_t pw[8];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                float p[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) p[r] = __builtin_amdgcn_exp2f(fmaf(s[b][r], c2, -mc));
                pw[2 * b] = pack_kv<BF>(p[0], p[1]);
                pw[2 * b + 1] = pack_kv<BF>(p[2], p[3]);
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const v4i pb = {(int) pw[4 * c], (int) pw[4 * c + 1], (int) pw[4 * c + 2], (int) pw[4 * c + 3]};
                os = mfma_h32<BF>(ones, pb, os);
#pragma unroll
                for (int b = 0; b < 8; ++b)
                    o[b] = mfma_h32<BF>(*(const v4i *) (vs + 16 * b * kVT + 32 * c), pb, o[b]);
            }
        }
        // keep the LDS stores (and the wait for their loads) after this tile's MFMAs
        __asm__ volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (more) stash(st + 2, buf ^ 1);
        __syncthreads();
    }
    // the odd tiles' part of a row joins the even tiles'
    float * x = (float *) lds + t;
    if (grp) {
#pragma unroll
        for (int b = 0; b < 8; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) x[(4 * b + r) * 256] = o[b][r];
        x[32 * 256] = os[0];
        x[33 * 256] = mc;
    }
    __syncthreads();
    if (grp || row >= a.n) return;
    const float mo = x[33 * 256], mn = fmaxf(mc, mo);
    const float fa = __builtin_amdgcn_exp2f(mc - mn), fb = __builtin_amdgcn_exp2f(mo - mn);
    const float inv = 1.0f / (os[0] * fa + x[32 * 256] * fb);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (o[b][r] * fa + x[(4 * b + r) * 256] * fb) * inv;
        *(uint2 *) (out + (size_t) row * out_stride + h * kHD + 16 * b + 4 * k) =
            make_uint2(f2h(v[0]) | (uint32_t) f2h(v[1]) << 16, f2h(v[2]) | (uint32_t) f2h(v[3]) << 16);
    }
}

// grid (n_head, ceil(n / 64)); out: the attention rows in fp16, as the output
// GEMM takes them.  LDS: K tiles [group][buffer][position][dim], then V^T tiles
// [group][buffer][dim][position]; at the end the odd group's part of each row.
__global__ __launch_bounds__(kFT) void k_att_flash(AttFlash a, float c2, uint16_t * __restrict__ out,
                                                   int32_t out_stride) {
    __shared__ __align__(16) uint16_t lds[4 * (kAT * kKS + kHD * kVT)];
    if (a.bf) att_flash_body<true>(a, c2, out, out_stride, lds);
    else att_flash_body<false>(a, c2, out, out_stride, lds);
}

}  // namespace pf
}  // namespace q3t

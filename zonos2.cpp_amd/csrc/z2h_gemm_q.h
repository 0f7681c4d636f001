// z2h_gemm_q.h — MFMA GEMMs of the Q8_0 and Q6_K matmuls of wide passes (prefill chunks, mixed passes,
// large MoE batches: mul_mat / mul_mat_id over a whole batch, src/zonos2-graph.cpp:107-111, 175,
// 179-185, 222-231). Same tiling as k_gemm_q4k: a block owns four 16-row groups (DUAL: of gate and the
// same four of up), one per wave, x GT = 16 TS token or route rows, reads each weight unit once for all GT rows
// and stages the activations in LDS one 256-column superblock at a time, double-buffered. A weight
// unit's registers are refilled with the next superblock's bytes as soon as they are unpacked, so the
// weight stream runs one superblock ahead without a second register set. A row's result is the GEMVs'
// bits: the same exact block sums, the same fp32 operations in the same order.
//
// What bounds them is not memory but the fp32 fold the format asks for: every (row, token, block) sum
// is scaled and added by itself.
//   k_gemm_q80   per 32-column block t = t + (dw * dx) * (float) dot, and the 8 blocks' t into the row
//                sum. dot is an int8 product; dw * dx (f16 x f16, exact in fp32) comes off the vector
//                unit: it is an f16 product with the token's scales masked to one block (so the matrix's scales
//                must be finite; the host sees to that: masking them too took 4% of the kernel), and the
//                conversion, the multiply by dot and the add stay per output.
//   k_gemm_q6k   x = (d * dx) * (float) sum_g sc_g * dot_g per superblock. The scale times the 6-bit
//                value, sc * (w - 32), is formed once per weight and split as 64 * hi + lo (both int8),
//                so two int8 products accumulate the whole superblock's integer sum exactly.
//
// Measured against the GEMVs' repeated 8- and 16-row passes: 1500 rows, top-4 of 32 experts (2048 x
// 1536), Q8_0: gate/up 387 -> 180 us, down 223 -> 103; 1024 rows, Q6_K: 311 -> 132 and 177 -> 75. Q8_0's
// dots as f16 products of converted int8 values (no conversion of the sums) cost the same vector
// operations in operand conversions: 240 and 138 us.
#pragma once
#include "z2h_gemm.h"

namespace z2d {

constexpr int GQ_QP = 256 + 16;          // LDS pitch of a row's int8 superblock (bytes): 68 dwords, so the 8-byte reads of
                                         // 16 rows x 2 k-slices (half a wave) fall in distinct banks
constexpr int GQ_DP = 8;                 // LDS halves of a row's 8 Q8_0 block scales

// ------------------------------------------------------------------ Q8_0 x Q8_0
// One superblock of GT = 16 TS rows: TS x 16 B of values and up to two block scales per thread; in LDS
// [GT][GQ_QP] bytes and f16 scales [GT][GQ_DP] (the scales are f16-rounded by the encoding).
template <int TS>
struct GqQ80 {
    u32x4 v[TS];
    float d[(TS + 1) / 2];
    const int8_t * pv[TS];           // the thread's items of superblock 0
    const float * pd[(TS + 1) / 2];
};
template <int TS>
__device__ __forceinline__ void gq_rows_q80(GqQ80<TS> & st, const ActBuf & act, int K, const int * s_row) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < TS; ++j) {
        const int i = tid + 256 * j;
        st.pv[j] = act.q + (int64_t) s_row[i >> 4] * K + (i & 15) * 16;
    }
#pragma unroll
    for (int j = 0; j < (TS + 1) / 2; ++j) {
        const int i = min(tid + 256 * j, 128 * TS - 1);
        st.pd[j] = act.d32 + (int64_t) s_row[i >> 3] * (K / 32) + (i & 7);
    }
}

template <int TS>
__device__ __forceinline__ void gq_load_q80(GqQ80<TS> & st, int sb) {
#pragma unroll
    for (int j = 0; j < TS; ++j) st.v[j] = *(const u32x4 *) (st.pv[j] + sb * 256);
#pragma unroll
    for (int j = 0; j < (TS + 1) / 2; ++j) st.d[j] = st.pd[j][sb * 8];
}
template <int TS>
__device__ __forceinline__ void gq_store_q80(const GqQ80<TS> & st, int8_t * sq, uint16_t * sd) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < TS; ++j) {
        const int i = tid + 256 * j;
        *(u32x4 *) (sq + (i >> 4) * GQ_QP + (i & 15) * 16) = st.v[j];
    }
#pragma unroll
    for (int j = 0; j < (TS + 1) / 2; ++j) {
        const int i = tid + 256 * j;
        if (i < 128 * TS) sd[i] = f2h(st.d[j]);
    }
}

__host__ __device__ constexpr size_t gemm_q80_buf(int ts) { return (size_t) 16 * ts * (GQ_QP + 2 * GQ_DP); }
__host__ __device__ inline size_t gemm_q80_lds(int ts) { return 2 * gemm_q80_buf(ts) + 3 * 16 * ts * 4; }

// grid: x = blocks of four groups, y = tile slots; 256 threads
template <bool DUAL, int TS>
__global__ void __launch_bounds__(256, 2) k_gemm_q80(GemmArgs a) {
    constexpr int NG = DUAL ? 2 : 1, GT = 16 * TS, BUF = (int) gemm_q80_buf(TS);
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int * s_row = (int *) (smem + 2 * BUF), * s_out = s_row + GT;
    int e, c0, nt;
    if (!gemm_tile<GT>(a, blockIdx.y, e, c0, nt)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), K = a.nsb * 256;
    gemm_rows<GT>(a, e, c0, nt, s_row, s_out);
    // the wave's units (a wave past the last group repeats it and stores nothing)
    const uint4 * w[NG];
    int grp[NG];
#pragma unroll
    for (int x = 0; x < NG; ++x) {
        grp[x] = blockIdx.x * 4 + wave;
        w[x] = (const uint4 *) ((DUAL ? a.w[x] : a.w[0]) + (int64_t) __builtin_amdgcn_readfirstlane(e) * a.mat_bytes + (size_t) min(grp[x], a.tiles - 1) * a.nsb * 4352);
    }
    uint4 raw[NG][4], hd[NG];
#pragma unroll
    for (int x = 0; x < NG; ++x) {
#pragma unroll
        for (int c = 0; c < 4; ++c) raw[x][c] = w[x][c * 64 + lane];
        hd[x] = w[x][256 + (lane & 15)];
    }
    lds_sync();                                                      // s_row
    GqQ80<TS> st;
    gq_rows_q80<TS>(st, a.act, K, s_row);
    gq_load_q80<TS>(st, 0);
    gq_store_q80<TS>(st, (int8_t *) smem, (uint16_t *) (smem + GT * GQ_QP));
    lds_sync();
    float acc[NG][TS][4] = {};
    const v4f_t zf = {0.0f, 0.0f, 0.0f, 0.0f};
    const v4i_t zi = {0, 0, 0, 0};
    const int q = lane >> 4;
    // the lane's operand slots of the scale product: k = 4q + i is block 4q + i (q < 2; idle above)
    const uint32_t m0 = q == 0 ? ~0u : 0u, m1 = q == 1 ? ~0u : 0u;
    const uint32_t msk[4] = {m0 & 0xffffu, m0 & 0xffff0000u, m1 & 0xffffu, m1 & 0xffff0000u};
    for (int sb = 0; sb < a.nsb; ++sb) {
        const int8_t * sq = (const int8_t *) (smem + (sb & 1) * BUF);
        const uint16_t * sd = (const uint16_t *) (sq + GT * GQ_QP);
        char * nb = smem + ((sb + 1) & 1) * BUF;
        const int nx = min(sb + 1, a.nsb - 1);                       // (the last superblock re-reads itself)
        gq_load_q80<TS>(st, nx);
        v4h_t dw[NG];
#pragma unroll
        for (int x = 0; x < NG; ++x) {
            const uint2 h = make_uint2((hd[x].x & m0) | (hd[x].z & m1), (hd[x].y & m0) | (hd[x].w & m1));
            dw[x] = __builtin_bit_cast(v4h_t, h);
            hd[x] = w[x][(size_t) nx * 272 + 256 + (lane & 15)];
        }
        uint2 dx[TS];
#pragma unroll
        for (int ts = 0; ts < TS; ++ts) dx[ts] = *(const uint2 *) (sd + (ts * 16 + (lane & 15)) * GQ_DP + 4 * (q & 1));
        // block b + 1's activations are read ahead of block b's products; the fences (the empty asm pins
        // each sum's order, the barrier the rest) keep the compiler from forming all eight blocks'
        // operands and products at once, which spills
        auto load_a = [&](int b, long (&A)[TS]) {
#pragma unroll
            for (int ts = 0; ts < TS; ++ts) A[ts] = *(const long *) (sq + (ts * 16 + (lane & 15)) * GQ_QP + 32 * b + 8 * q);
        };
        v4f_t t[NG][TS];
        long A[2][TS];
        load_a(0, A[0]);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            if (b < 7) load_a(b + 1, A[(b + 1) & 1]);
            long B[NG];
#pragma unroll
            for (int x = 0; x < NG; ++x) {
                const uint4 v = raw[x][b >> 1];
                B[x] = (b & 1) ? (long) (((uint64_t) v.w << 32) | v.z) : (long) (((uint64_t) v.y << 32) | v.x);
            }
            const uint32_t mb = msk[2 * (b >> 2) + (b & 1)];
#pragma unroll
            for (int ts = 0; ts < TS; ++ts) {
                const v4h_t Ad = __builtin_bit_cast(v4h_t, (b & 2) ? make_uint2(0u, dx[ts].y & mb) : make_uint2(dx[ts].x & mb, 0u));
#pragma unroll
                for (int x = 0; x < NG; ++x) {
                    const v4i_t c = __builtin_amdgcn_mfma_i32_16x16x32_i8(A[b & 1][ts], B[x], zi, 0, 0, 0);
                    const v4f_t s = __builtin_amdgcn_mfma_f32_16x16x16f16(Ad, dw[x], zf, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) t[x][ts][i] = b == 0 ? s[i] * (float) c[i] : t[x][ts][i] + s[i] * (float) c[i];
                }
            }
            if (b & 1)
#pragma unroll
                for (int x = 0; x < NG; ++x) raw[x][b >> 1] = w[x][(size_t) nx * 272 + (b >> 1) * 64 + lane];
#pragma unroll
            for (int x = 0; x < NG; ++x)
#pragma unroll
                for (int ts = 0; ts < TS; ++ts) asm volatile("" : "+v"(t[x][ts]));
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int x = 0; x < NG; ++x)
#pragma unroll
            for (int ts = 0; ts < TS; ++ts)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[x][ts][i] = acc[x][ts][i] + t[x][ts][i];
        gq_store_q80<TS>(st, (int8_t *) nb, (uint16_t *) (nb + GT * GQ_QP));
        lds_sync();
    }
    gemm_store<DUAL, NG, TS>(a, acc, grp, lane, nt, s_out);
}

// ------------------------------------------------------------------ Q6_K x Q8_K
template <int TS>
struct GqQ6K {
    u32x4 v[TS];
    float dx;
    const int8_t * pv[TS];           // the thread's items of superblock 0
    const float * pd;
};
template <int TS>
__device__ __forceinline__ void gq_rows_q6k(GqQ6K<TS> & st, const ActBuf & act, int K, const int * s_row) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < TS; ++j) {
        const int i = tid + 256 * j;
        st.pv[j] = act.q + (int64_t) s_row[i >> 4] * K + (i & 15) * 16;
    }
    st.pd = act.d256 + (int64_t) s_row[tid & (16 * TS - 1)] * (K / 256);
}

template <int TS>
__device__ __forceinline__ void gq_load_q6k(GqQ6K<TS> & st, int sb) {
#pragma unroll
    for (int j = 0; j < TS; ++j) st.v[j] = *(const u32x4 *) (st.pv[j] + sb * 256);
    st.dx = st.pd[sb];
}
template <int TS>
__device__ __forceinline__ void gq_store_q6k(const GqQ6K<TS> & st, int8_t * sq, float * sdx) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < TS; ++j) {
        const int i = tid + 256 * j;
        *(u32x4 *) (sq + (i >> 4) * GQ_QP + (i & 15) * 16) = st.v[j];
    }
    if (tid < 16 * TS) sdx[tid] = st.dx;
}

// eight 6-bit values w (low nibbles of four in L's even nibbles, of the next four in its odd ones, the
// high bits in hb) times the scale: 4 sc (w - 32) in 16 bits (|.| <= 2^14); its high byte is the part hi
// and its low byte / 4 the part lo of sc (w - 32) = 64 hi + lo.
__device__ __forceinline__ void gq_prep_q6k(uint32_t L, uint32_t hb, int sc, v4i_t & hi, v4i_t & lo, int at) {
    const uint32_t b[2] = {(L & 0x0f0f0f0fu) | ((hb << 4) & 0x30303030u), ((L >> 4) & 0x0f0f0f0fu) | ((hb << 2) & 0x30303030u)};
    const unsigned short s4 = (unsigned short) (4 * sc), off = (unsigned short) (-128 * sc);
    const u16x2_t S = {s4, s4}, O = {off, off};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const u16x2_t w01 = __builtin_bit_cast(u16x2_t, __builtin_amdgcn_perm(0u, b[h], 0x0c010c00u));
        const u16x2_t w23 = __builtin_bit_cast(u16x2_t, __builtin_amdgcn_perm(0u, b[h], 0x0c030c02u));
        const uint32_t v01 = __builtin_bit_cast(uint32_t, (u16x2_t) (w01 * S + O)), v23 = __builtin_bit_cast(uint32_t, (u16x2_t) (w23 * S + O));
        hi[at + h] = (int) __builtin_amdgcn_perm(v23, v01, 0x07050301u);
        lo[at + h] = (int) ((__builtin_amdgcn_perm(v23, v01, 0x06040200u) >> 2) & 0x3f3f3f3fu);
    }
}

__host__ __device__ constexpr size_t gemm_q6k_buf(int ts) { return (size_t) 16 * ts * (GQ_QP + 4); }
__host__ __device__ inline size_t gemm_q6k_lds(int ts) { return 2 * gemm_q6k_buf(ts) + 3 * 16 * ts * 4; }

template <bool DUAL, int TS>
__global__ void __launch_bounds__(256, 2) k_gemm_q6k(GemmArgs a) {
    constexpr int NG = DUAL ? 2 : 1, GT = 16 * TS, BUF = (int) gemm_q6k_buf(TS);
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int * s_row = (int *) (smem + 2 * BUF), * s_out = s_row + GT;
    int e, c0, nt;
    if (!gemm_tile<GT>(a, blockIdx.y, e, c0, nt)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), K = a.nsb * 256;
    gemm_rows<GT>(a, e, c0, nt, s_row, s_out);
    const uint4 * w[NG];
    int grp[NG];
#pragma unroll
    for (int x = 0; x < NG; ++x) {
        grp[x] = blockIdx.x * 4 + wave;
        w[x] = (const uint4 *) ((DUAL ? a.w[x] : a.w[0]) + (int64_t) __builtin_amdgcn_readfirstlane(e) * a.mat_bytes + (size_t) min(grp[x], a.tiles - 1) * a.nsb * 3360);
    }
    uint4 raw[NG][3], hd[NG];
    uint32_t dr[NG];
#pragma unroll
    for (int x = 0; x < NG; ++x) {
#pragma unroll
        for (int c = 0; c < 3; ++c) raw[x][c] = w[x][c * 64 + lane];
        hd[x] = w[x][192 + (lane & 15)];
        dr[x] = ((const uint32_t *) (w[x] + 208))[(lane & 15) >> 1];
    }
    lds_sync();                                                      // s_row
    GqQ6K<TS> st;
    gq_rows_q6k<TS>(st, a.act, K, s_row);
    gq_load_q6k<TS>(st, 0);
    gq_store_q6k<TS>(st, (int8_t *) smem, (float *) (smem + GT * GQ_QP));
    lds_sync();
    float acc[NG][TS][4] = {};
    const int q = lane >> 4, par8 = 8 * (lane >> 5);
    for (int sb = 0; sb < a.nsb; ++sb) {
        const int8_t * sq = (const int8_t *) (smem + (sb & 1) * BUF);
        const float * sdx = (const float *) (sq + GT * GQ_QP);
        char * nb = smem + ((sb + 1) & 1) * BUF;
        const int nx = min(sb + 1, a.nsb - 1);                       // (the last superblock re-reads itself)
        const size_t no = (size_t) nx * 210;
        gq_load_q6k<TS>(st, nx);
        float d[NG];
        v4i_t ch[NG][TS], cl[NG][TS];
#pragma unroll
        for (int x = 0; x < NG; ++x) {
            d[x] = h2f((dr[x] >> (16 * (lane & 1))) & 0xffffu);
            dr[x] = ((const uint32_t *) (w[x] + no + 208))[(lane & 15) >> 1];
#pragma unroll
            for (int ts = 0; ts < TS; ++ts) ch[x][ts] = cl[x][ts] = (v4i_t) {0, 0, 0, 0};
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {                                // columns 64 s .. 64 s + 63
            v4i_t bh[NG], bl[NG];
#pragma unroll
            for (int x = 0; x < NG; ++x) {
                const uint4 l4 = raw[x][s >> 1];
                const uint32_t H = s == 0 ? raw[x][2].x : s == 1 ? raw[x][2].y : s == 2 ? raw[x][2].z : raw[x][2].w;
                const uint32_t sw = (s == 0 ? hd[x].x : s == 1 ? hd[x].y : s == 2 ? hd[x].z : hd[x].w) >> par8;
                gq_prep_q6k((s & 1) ? l4.z : l4.x, H, (int) (int8_t) (sw & 0xffu), bh[x], bl[x], 0);
                gq_prep_q6k((s & 1) ? l4.w : l4.y, H >> 4, (int) (int8_t) ((sw >> 16) & 0xffu), bh[x], bl[x], 2);
                if (s & 1) raw[x][s >> 1] = w[x][no + (s >> 1) * 64 + lane];
                if (s == 3) { raw[x][2] = w[x][no + 128 + lane]; hd[x] = w[x][no + 192 + (lane & 15)]; }
            }
#pragma unroll
            for (int ts = 0; ts < TS; ++ts) {
                const int8_t * ap = sq + (ts * 16 + (lane & 15)) * GQ_QP + 8 * q + 64 * s;
                const uint2 lo = *(const uint2 *) ap, hi = *(const uint2 *) (ap + 32);
                const v4i_t A = {(int) lo.x, (int) lo.y, (int) hi.x, (int) hi.y};
#pragma unroll
                for (int x = 0; x < NG; ++x) {
                    ch[x][ts] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, bh[x], ch[x][ts], 0, 0, 0);
                    cl[x][ts] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, bl[x], cl[x][ts], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int ts = 0; ts < TS; ++ts) {
            const v4f_t dx = *(const v4f_t *) (sdx + ts * 16 + 4 * q);
#pragma unroll
            for (int x = 0; x < NG; ++x)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[x][ts][i] = acc[x][ts][i] + (d[x] * dx[i]) * (float) ((ch[x][ts][i] << 6) + cl[x][ts][i]);
        }
        gq_store_q6k<TS>(st, (int8_t *) nb, (float *) (nb + GT * GQ_QP));
        lds_sync();
    }
    gemm_store<DUAL, NG, TS>(a, acc, grp, lane, nt, s_out);
}

} // namespace z2d

// z2h_gemm.h — MFMA GEMMs for the passes with many rows per weight tile: prefill chunks and mixed
// prefill + decode passes (mul_mat / mul_mat_id over a whole batch, src/zonos2-graph.cpp:107-111,
// 175, 179-185, 222-231). A block owns a tile of output rows x GT token (or route) rows and reads
// each weight byte of its rows once for all GT rows; the activations of the tile are staged in LDS
// one 256-column superblock at a time (double-buffered, the next superblock's loads in flight during
// the current one's products). Grouped launches (experts) take their tiles from the route grouping
// (k_route_sort's offsets and permutation): tile slots are numbered expert by expert, ceil(routes /
// GT) per expert, and blocks whose slot is past the last tile exit.
//
//   k_gemm_q4k   Q4_K weights (m16 layout) x Q8_K activations on int8 MFMA (v_mfma_i32_32x32x32_i8).
//                A Q4_K sub-block's 6-bit scale sc is split as 8 * (sc >> 3) + (sc & 7); the weights'
//                4-bit values times each part stay below 106, so two int8 products over the whole
//                superblock give sum_j sc_j * dot_j = 8 * hi + lo exactly, with no per-sub-block
//                scaling of MFMA results. The min term sum_g m_g * bsum_g (bsum = the activation's
//                sums of 16, g's min that of its sub-block) is one f16 MFMA on exact operands, exact
//                in fp32. Per superblock: acc = fma(dx, fma(d, isum, -dmin * msum), acc), the
//                fold of the Q4_K GEMVs, so a row's result is the same bits at any batch width.
//   k_gemm_f16   F16 weights (t64 layout) x f16 activations on v_mfma_f32_16x16x32_f16, fp32
//                accumulation; the weight fragments stream straight from HBM into a register ring of
//                32-column steps. Decode widths run on its narrow shape, or on k_gemm_f16_few.
#pragma once
#include "z2h_kernels.h"

namespace z2d {


typedef _Float16 v4h_t __attribute__((ext_vector_type(4)));
typedef _Float16 v8h_t __attribute__((ext_vector_type(8)));
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

struct GemmArgs {
    const uint8_t * w[2];              // DUAL: gate, up (same layout); else w[0]
    int64_t mat_bytes;                 // per-expert stride of a matrix
    int nsb, rows, tiles;              // K = 256 * nsb; output rows; 16-row groups (m16) / 64-row tiles (t64)
    int grouped, n_tok, k, E, act_by_route;
    const int32_t * r_off, * r_perm;   // grouped: route offsets by expert [E+1], routes in expert order
    ActBuf act;
    float * out; int out_ld;           // out[row-index][rows]; row-index = token (dense) or route
    int epi; float cap; const float * route_w;
};

// Block tiles of GT rows in a launch (grid y): dense ceil(n_tok / GT); grouped at most
// ceil(routes / GT) + E.
__host__ __device__ inline int gemm_slots(int grouped, int n_tok, int k, int E, int GT) {
    return grouped ? (n_tok * k + GT - 1) / GT + E : (n_tok + GT - 1) / GT;
}

// The block's tile of up to GT rows: dense rows [c0, c0 + nt), or routes [c0, c0 + nt) of expert e
// in expert order. Every wave computes the same answer (no LDS); false for slots past the last tile.
template <int GT>
__device__ __forceinline__ bool gemm_tile(const GemmArgs & a, int slot, int & e, int & c0, int & nt) {
    e = 0;
    if (!a.grouped) {
        c0 = slot * GT;
        nt = min(GT, a.n_tok - c0);
        return nt > 0;
    }
    const int lane = threadIdx.x & 63;
    int base = 0;
    for (int e0 = 0; e0 < a.E; e0 += 64) {
        const int ee = e0 + lane;
        const int cnt = ee < a.E ? a.r_off[ee + 1] - a.r_off[ee] : 0;
        const int nte = (cnt + GT - 1) / GT;
        const int incl = wave_scan_incl(nte, lane);
        const int tot = __builtin_amdgcn_readlane(incl, 63);
        if (slot < base + tot) {
            const uint64_t hit = __ballot(slot < base + incl);
            const int l = (int) __ffsll((unsigned long long) hit) - 1;
            e = e0 + l;
            const int first = base + __builtin_amdgcn_readlane(incl, l) - __builtin_amdgcn_readlane(nte, l);
            c0 = (slot - first) * GT;
            nt = min(GT, __builtin_amdgcn_readlane(cnt, l) - c0);
            return true;
        }
        base += tot;
    }
    return false;
}

// Tile rows -> activation rows (s_row, the last valid row repeated past nt), output row indices (s_out) and,
// behind those, the rows' route weights (EPI_ROUTE_W): 3 GT words of LDS.
template <int GT>
__device__ __forceinline__ void gemm_rows(const GemmArgs & a, int e, int c0, int nt, int * s_row, int * s_out) {
    const int tid = threadIdx.x;
    if (tid < GT) {
        const int t = min(tid, nt - 1);
        const int it = a.grouped ? a.r_perm[a.r_off[e] + c0 + t] : c0 + t;
        s_out[tid] = it;
        s_row[tid] = a.grouped && !a.act_by_route ? it / a.k : it;
        ((float *) s_out)[GT + tid] = a.epi == EPI_ROUTE_W ? a.route_w[it] : 0.0f;
    }
}

// rw: the row's route weight
__device__ __forceinline__ float gemm_epi(const GemmArgs & a, float y, float rw) {
    if (a.epi == EPI_SOFTCAP) return z_softcap(y, a.cap);
    if (a.epi == EPI_ROUTE_W) return y * rw;
    return y;
}

// Store a wave's sums: acc[x][ts][i] is token 16 ts + 4 (lane / 16) + i of the block tile by row lane % 16
// of 16-row group grp[x] (DUAL: x = 0 gate, 1 up, SwiGLU).
template <bool DUAL, int NG, int TS>
__device__ __forceinline__ void gemm_store(const GemmArgs & a, const float (&acc)[NG][TS][4], const int (&grp)[NG], int lane,
                                           int nt, const int * s_out) {
    constexpr int GT = 16 * TS;
#pragma unroll
    for (int ts = 0; ts < TS; ++ts) {
        const int t0 = ts * 16 + 4 * (lane >> 4);
        const v4i_t oi = *(const v4i_t *) (s_out + t0);
        const v4f_t rw = *(const v4f_t *) ((const float *) s_out + GT + t0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (t0 + i >= nt) continue;
            float * o = a.out + (int64_t) oi[i] * a.out_ld;
#pragma unroll
            for (int x = 0; x < (DUAL ? 1 : NG); ++x) {
                const int row = grp[x] * 16 + (lane & 15);
                if (grp[x] >= a.tiles || row >= a.rows) continue;
                if constexpr (DUAL) o[row] = acc[1][ts][i] * z_silu(acc[0][ts][i]);
                else o[row] = gemm_epi(a, acc[x][ts][i], rw[i]);
            }
        }
    }
}

// ------------------------------------------------------------------ Q4_K x Q8_K
// A block owns 128 weight rows (DUAL: 64 of gate and the same 64 of up), 32 per wave, x GT = 32 TS
// token rows. The wave's 32 rows are one B operand of v_mfma_i32_32x32x32_i8: lane l has row l % 32
// (16-row group (l / 16) & 1; DUAL: gate, up) and columns 32 j + 16 h .. + 15 of sub-block j, h = l / 32.
//
// Bounded by issue, not by memory (82% of the L2 reads hit): the vector unit (the weights' unpacking, 22
// instructions per sub-block, and the fp32 fold, 5 per output) and the matrix unit are busy 57% and 32%
// of the time. So the unpacking of sub-block j + 1 sits between the products of sub-block j (the group
// barriers), 32 x 32 products take half the LDS reads and min-term products of 16 x 16 ones, the min term
// takes the sums of 16 as they are, the staging has no address arithmetic, and a SwiGLU is formed once per output
// by splitting the tokens over the gate and up lanes. A tile of up to 32 rows takes one product per sub-block.
// Measured: 2088 rows, top-4 of 32, 2048 x 1536: gate/up 201 -> 167 us, down 129 -> 96; QKV 58 -> 48, W_o 46 ->
// 38; 1024 rows 115 -> 95, 71 -> 54, 32 -> 27, 23 -> 19. Tiles of 96 and 128 rows (2 waves per SIMD still; 128
// spills) 179 and 250 us for gate/up, of 32 rows only 178 (three waves per SIMD, twice the L2 reads).
constexpr int Q4_SP = 12;                // LDS pitch (dwords) of a row's 16 f16 sums: 16 rows' 16-byte reads
                                         // fall in distinct banks
typedef int v16i_t __attribute__((ext_vector_type(16)));
typedef float v16f_t __attribute__((ext_vector_type(16)));

constexpr int Q4_T = 64;                 // token (route) rows per block tile: one or two products of 32
// One superblock of 32 S activation rows: values [32 S][256 B], a row's 16-byte chunk c at slot c ^ (row % 16)
// (16 rows' reads of one chunk fall in distinct banks), the 16 sums of 16 as f16 (|sum| <= 2032, exact)
// [32 S][Q4_SP], the scales [32 S].
constexpr int q4_buf(int S) { return 32 * S * (256 + 4 * Q4_SP + 4); }
constexpr size_t gemm_q4k_lds = 2 * q4_buf(2) + 3 * Q4_T * 4;

// A thread's share of a superblock: 16-byte items of values, pairs of sums, one scale, at 32-bit byte
// offsets (the host keeps rows x K below 2^32) from the superblock's uniform base: no address arithmetic.
template <int S>
struct Q4Stage {
    uint32_t ov[2 * S], os[S], od;
    u32x4 v[2 * S];
    uint32_t s[S];
    float dx;
};
template <int S>
__device__ __forceinline__ void q4_rows(Q4Stage<S> & st, int K, const int * s_row) {
    const uint32_t tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < 2 * S; ++j) st.ov[j] = (uint32_t) s_row[16 * j + (tid >> 4)] * (uint32_t) K + (tid & 15) * 16;
#pragma unroll
    for (int j = 0; j < S; ++j) st.os[j] = (uint32_t) s_row[32 * j + (tid >> 3)] * (uint32_t) (K / 8) + (tid & 7) * 4;
    st.od = (uint32_t) s_row[tid & (32 * S - 1)] * (uint32_t) (K / 64);
}
template <int S>
__device__ __forceinline__ void q4_load(Q4Stage<S> & st, const ActBuf & act, int sb) {
    const uint8_t * q = (const uint8_t *) act.q + (size_t) sb * 256, * bs = (const uint8_t *) act.bs + (size_t) sb * 32,
                  * d = (const uint8_t *) act.d256 + (size_t) sb * 4;
#pragma unroll
    for (int j = 0; j < 2 * S; ++j) st.v[j] = *(const u32x4 *) (q + st.ov[j]);
#pragma unroll
    for (int j = 0; j < S; ++j) st.s[j] = *(const uint32_t *) (bs + st.os[j]);
    st.dx = *(const float *) (d + st.od);
}
template <int S>
__device__ __forceinline__ void q4_store(const Q4Stage<S> & st, char * buf) {
    const int tid = threadIdx.x, c = (tid & 15) ^ (tid >> 4);         // (row % 16 = tid / 16)
    uint32_t * ss = (uint32_t *) (buf + 32 * S * 256);
    float * sdx = (float *) (ss + 32 * S * Q4_SP);
#pragma unroll
    for (int j = 0; j < 2 * S; ++j) *(u32x4 *) (buf + (16 * j + (tid >> 4)) * 256 + c * 16) = st.v[j];
#pragma unroll
    for (int j = 0; j < S; ++j) {
        const _Float16 lo = (_Float16) (int16_t) (st.s[j] & 0xffffu), hi = (_Float16) (int16_t) (st.s[j] >> 16);
        ss[(32 * j + (tid >> 3)) * Q4_SP + (tid & 7)] = (uint32_t) __builtin_bit_cast(uint16_t, lo) | ((uint32_t) __builtin_bit_cast(uint16_t, hi) << 16);
    }
    sdx[tid & (32 * S - 1)] = st.dx;                                   // (several threads store the same value)
}

__device__ __forceinline__ uint32_t gm_mul_bytes(uint32_t x, uint32_t s) {
    // four byte lanes (each <= 15) times s <= 7: two 16-bit products per half, no carry across bytes
    const u16x2_t r = __builtin_bit_cast(u16x2_t, x) * (u16x2_t) {(unsigned short) s, (unsigned short) s};
    return __builtin_bit_cast(uint32_t, r);
}

// The B operands of sub-block j for the lane's row and column half: its 16 weight values times the high and
// the low part of the sub-block's scale (sc03, sc47: the row's 8 scales). raw[2 c + e]: chunk c of the m16
// unit's k-slice 2 h + e.
struct Q4B { v4i_t hi, lo; };
__device__ __forceinline__ Q4B q4_prep(const u32x4 (&raw)[4], uint32_t sc03, uint32_t sc47, int j) {
    const int p = j >> 1;                                            // sub-blocks 2p (low nibbles) and 2p + 1
    const u32x4 & r0 = raw[2 * (p >> 1)], & r1 = raw[2 * (p >> 1) + 1];
    const uint32_t w[4] = {(p & 1) ? r0.z : r0.x, (p & 1) ? r0.w : r0.y, (p & 1) ? r1.z : r1.x, (p & 1) ? r1.w : r1.y};
    const uint32_t sc = (j < 4 ? sc03 : sc47) >> (8 * (j & 3)), sh = (sc >> 3) & 7u, sl = sc & 7u;
    Q4B b;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t v = ((j & 1) ? w[i] >> 4 : w[i]) & 0x0f0f0f0fu;
        b.hi[i] = (int) gm_mul_bytes(v, sh);
        b.lo[i] = (int) gm_mul_bytes(v, sl);
    }
    return b;
}

// One block tile of up to 32 S rows.
template <bool DUAL, int S>
__device__ __forceinline__ void q4_block(const GemmArgs & a, char * smem, const int * s_row, const int * s_out, int nt,
                                         int grp, const u32x4 * wl, const u32x4 * wh, u32x4 (&raw)[4], u32x4 & hd) {
    constexpr int BUF = q4_buf(S);
    const int tid = threadIdx.x, lane = tid & 63, K = a.nsb * 256, h = lane >> 5, x = (lane >> 4) & 1;
    Q4Stage<S> st;
    q4_rows(st, K, s_row);
    q4_load(st, a.act, 0);
    q4_store(st, smem);
    lds_sync();
    float acc[S][16] = {};
    for (int sb = 0; sb < a.nsb; ++sb) {
        const char * buf = smem + (sb & 1) * BUF;
        char * nb = smem + ((sb + 1) & 1) * BUF;
        const int nx = min(sb + 1, a.nsb - 1);                       // (the last superblock re-reads itself)
        q4_load(st, a.act, nx);
        // the row's 6-bit scales / mins of sub-blocks 0-3 and 4-7 (GGUF K-quant packing), d, dmin; the lane's
        // 8 sums of the min term belong to sub-blocks 4h .. 4h + 3
        const uint32_t sc03 = hd.y & 0x3f3f3f3fu, sc47 = (hd.w & 0x0f0f0f0fu) | ((hd.y >> 2) & 0x30303030u);
        const uint32_t mm = h ? ((hd.w >> 4) & 0x0f0f0f0fu) | ((hd.z >> 2) & 0x30303030u) : hd.z & 0x3f3f3f3fu;
        const float d = h2f(hd.x & 0xffffu), dmin = h2f(hd.x >> 16);
        v16i_t ch[S], cl[S];
#pragma unroll
        for (int ts = 0; ts < S; ++ts) ch[ts] = cl[ts] = (v16i_t) {};
        // sub-block j + 1's operands are read and unpacked between sub-block j's products
        auto load_a = [&](int j, v4i_t (&A)[S]) {
#pragma unroll
            for (int ts = 0; ts < S; ++ts)
                A[ts] = *(const v4i_t *) (buf + (ts * 32 + (lane & 31)) * 256 + (((2 * j + h) ^ (lane & 15)) << 4));
        };
        v4i_t A[2][S];
        Q4B B[2];
        load_a(0, A[0]);
        B[0] = q4_prep(raw, sc03, sc47, 0);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (j < 7) {
                load_a(j + 1, A[(j + 1) & 1]);
                B[(j + 1) & 1] = q4_prep(raw, sc03, sc47, j + 1);
            }
            if (j == 3) { raw[0] = wl[(size_t) nx * 144]; raw[1] = wl[(size_t) nx * 144 + 16]; hd = wh[(size_t) nx * 144]; }
            if (j == 7) { raw[2] = wl[(size_t) nx * 144 + 64]; raw[3] = wl[(size_t) nx * 144 + 80]; }
#pragma unroll
            for (int ts = 0; ts < S; ++ts) {
                ch[ts] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[j & 1][ts], B[j & 1].hi, ch[ts], 0, 0, 0);
                cl[ts] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[j & 1][ts], B[j & 1].lo, cl[ts], 0, 0, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, S, 0);    // LDS reads
#pragma unroll
            for (int i = 0; i < 2 * S; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);     // MFMA
                __builtin_amdgcn_sched_group_barrier(0x2, 10 / S, 0);   // VALU
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        v8h_t bm;
#pragma unroll
        for (int i = 0; i < 4; ++i) bm[2 * i] = bm[2 * i + 1] = (_Float16) (float) ((mm >> (8 * i)) & 0xffu);
#pragma unroll
        for (int ts = 0; ts < S; ++ts) {
            const uint32_t * sp = (const uint32_t *) (buf + 32 * S * 256) + (ts * 32 + (lane & 31)) * Q4_SP + 4 * h;
            const float * dxp = (const float *) (buf + 32 * S * (256 + 4 * Q4_SP)) + ts * 32 + 4 * h;
            const v16f_t M = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(const v8h_t *) sp, bm, (v16f_t) {}, 0, 0, 0);
#pragma unroll
            for (int i4 = 0; i4 < 4; ++i4) {
                const v4f_t dx = *(const v4f_t *) (dxp + 8 * i4);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // the Q4_K unit value and fold of m16_unit / m16_fold (same operations)
                    const int c = 4 * i4 + i;
                    const float f = (float) ((ch[ts][c] << 3) + cl[ts][c]);
                    acc[ts][c] = __builtin_fmaf(dx[i], __builtin_fmaf(d, f, -(dmin * M[c])), acc[ts][c]);
                }
            }
        }
        q4_store(st, nb);
        lds_sync();
    }
    const int row = grp * 16 + (lane & 15);
    const bool st_ok = grp < a.tiles && row < a.rows;
#pragma unroll
    for (int i8 = 0; i8 < 4 * S; ++i8) {
        const int ts = i8 >> 2, i4 = i8 & 3, t0 = ts * 32 + 8 * i4 + 4 * h;
        if (32 * ts >= nt) break;                                    // (uniform)
        if constexpr (DUAL) {
            // lanes x = 0 hold gate, the lanes 16 above the same rows of up: one swap leaves the gates of
            // tokens i (x = 0) and i + 1 (x = 1) in one register and their ups in the other
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                const auto sw = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, acc[ts][4 * i4 + i]),
                                                                 __builtin_bit_cast(unsigned, acc[ts][4 * i4 + i + 1]), false, false);
                const unsigned gb = sw[0], ub = sw[1];
                const float y = __builtin_bit_cast(float, ub) * z_silu(__builtin_bit_cast(float, gb));
                if (st_ok && t0 + i + x < nt) a.out[(int64_t) s_out[t0 + i + x] * a.out_ld + row] = y;
            }
        } else {
            const v4i_t oi = *(const v4i_t *) (s_out + t0);
            const v4f_t rw = *(const v4f_t *) ((const float *) s_out + Q4_T + t0);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (st_ok && t0 + i < nt) a.out[(int64_t) oi[i] * a.out_ld + row] = gemm_epi(a, acc[ts][4 * i4 + i], rw[i]);
        }
    }
}

// grid: x = blocks of eight 16-row groups (DUAL: four of gate and of up), y = tile slots. 256 threads;
// dynamic LDS gemm_q4k_lds.
template <bool DUAL>
__global__ void __launch_bounds__(256, 2) k_gemm_q4k(GemmArgs a) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    int * s_row = (int *) (smem + 2 * q4_buf(2)), * s_out = s_row + Q4_T;
    int e, c0, nt;
    if (!gemm_tile<Q4_T>(a, blockIdx.y, e, c0, nt)) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), x = (lane >> 4) & 1;
    // the lane's 16-row group (lanes past the last group read group 0 and store nothing) and its first unit
    const int grp = DUAL ? blockIdx.x * 4 + wave : (blockIdx.x * 4 + wave) * 2 + x;
    const u32x4 * w = (const u32x4 *) ((DUAL && x ? a.w[1] : a.w[0]) + (int64_t) e * a.mat_bytes + (size_t) (grp < a.tiles ? grp : 0) * a.nsb * 2304);
    const u32x4 * wl = w + 32 * (lane >> 5) + (lane & 15), * wh = w + 128 + (lane & 15);
    u32x4 raw[4] = {wl[0], wl[16], wl[64], wl[80]}, hd = wh[0];
    gemm_rows<Q4_T>(a, e, c0, nt, s_row, s_out);
    lds_sync();
    if (__builtin_amdgcn_readfirstlane(nt) > 32) q4_block<DUAL, 2>(a, smem, s_row, s_out, nt, grp, wl, wh, raw, hd);
    else q4_block<DUAL, 1>(a, smem, s_row, s_out, nt, grp, wl, wh, raw, hd);
}

// ------------------------------------------------------------------ F16 x f16
// Every F16 matmul but a dense one of few rows (k_gemm_f16_few) runs on this kernel, in two shapes: wide (passes of more than 64 rows: tiles of 64
// token rows, each wave 64 output rows; DUAL 32 rows of gate and up) and narrow (decode widths: tiles
// of 16 token rows, each wave 16 output rows; DUAL 16 of gate and up). A row's output is the same
// chain of v_mfma_f32_16x16x32_f16 products over its 32-column steps in order in both shapes, so it
// does not depend on the width of the pass. grid: x = row blocks of 4 waves, y = tile slots; 256
// threads; dynamic LDS gemm_f16_lds(TS).
//   NG: 16-row sub-groups per wave (DUAL: NG / 2 of gate, then the same rows of up)
//   TS: 16-row token tiles per block tile (GT = 16 * TS token rows). The wide shape is bounded by the weight reads of
//   a compute unit (64 rows per tile: 16 KB per 32-column step of a block, four steps in flight per wave); TS = 8
//   halves them per product, its rows staged 128 columns at a time.
constexpr int gm_f16_steps(int ts) { return ts >= 8 ? 4 : 8; }       // 32-column steps per staged chunk
constexpr int gm_f16_hp(int ts) { return 32 * gm_f16_steps(ts) + 8; } // LDS pitch of a row's chunk (halves)
template <int TS>
struct GmF16 { u32x4 v[TS * gm_f16_steps(TS) / 8]; };                // half of one chunk's staging

// half h of chunk c of GT = 16 TS f16 activation rows
template <int TS>
__device__ __forceinline__ void gm_load_f16(GmF16<TS> & st, const ActBuf & act, int K, int c, int h, const int * s_row) {
    constexpr int N = TS * gm_f16_steps(TS) / 8, RU = 4 * gm_f16_steps(TS);   // items per thread and half; 16-byte items per row
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = 256 * N * h + tid + 256 * j, r = i / RU, u = i % RU;
        st.v[j] = *(const u32x4 *) (act.h + (int64_t) s_row[r] * K + c * (8 * RU) + u * 8);
    }
}
template <int TS>
__device__ __forceinline__ void gm_store_f16(const GmF16<TS> & st, int h, uint16_t * sh) {
    constexpr int N = TS * gm_f16_steps(TS) / 8, RU = 4 * gm_f16_steps(TS);
    const int tid = threadIdx.x;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const int i = 256 * N * h + tid + 256 * j, r = i / RU, u = i % RU;
        *(u32x4 *) (sh + r * gm_f16_hp(TS) + u * 8) = st.v[j];
    }
}

__host__ __device__ inline size_t gemm_f16_lds(int ts) { return 2 * (size_t) (16 * ts) * gm_f16_hp(ts) * 2 + 3 * (16 * ts) * 4; }

template <bool DUAL, int NG, int TS>
__global__ void __launch_bounds__(256, 2) k_gemm_f16(GemmArgs a) {
    constexpr int CS = gm_f16_steps(TS), HP = gm_f16_hp(TS), GT = 16 * TS, BUF = GT * HP;   // BUF in halves
    constexpr int RING = TS >= 8 ? 2 : NG >= 4 ? 4 : 8;              // 32-column weight steps in flight
    constexpr int RPW = DUAL ? 8 * NG : 16 * NG;                     // output rows per wave
    extern __shared__ __attribute__((aligned(16))) char smem[];
    uint16_t * sh0 = (uint16_t *) smem;
    int * s_row = (int *) (smem + 2 * BUF * 2), * s_out = s_row + GT;
    int e, c0, nt;
    if (!gemm_tile<GT>(a, blockIdx.y, e, c0, nt)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, K = a.nsb * 256;
    gemm_rows<GT>(a, e, c0, nt, s_row, s_out);
    const int r0 = RPW * (blockIdx.x * 4 + wave);
    const bool has = r0 < a.rows;
    const int tile = has ? r0 / 64 : 0, sg0 = (r0 % 64) / 16;
    const uint8_t * base[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        // sub-group g: DUAL gate (g < NG / 2) or up rows r0 + 16 (g % (NG / 2)); else rows r0 + 16 g
        const uint8_t * wm = DUAL ? a.w[g / (NG / 2)] : a.w[0];
        const int sg = sg0 + (DUAL ? g % (NG / 2) : g);
        base[g] = wm + (int64_t) e * a.mat_bytes + ((size_t) tile * a.nsb * 32 * 64 + 16 * sg + (lane & 15)) * 16;
    }
    const int q = lane >> 4, nsteps = a.nsb * 8;
    // weight step kk (32 columns): chunk 4 * (kk % 8) + q of superblock kk / 8 (t64 layout)
    auto load_step = [&](int kk, u32x4 (&b)[NG]) {
        const size_t off = ((size_t) (kk >> 3) * 32 + 4 * (kk & 7) + q) * 64 * 16;
#pragma unroll
        for (int g = 0; g < NG; ++g) b[g] = *(const u32x4 *) (base[g] + off);
    };
    u32x4 ring[RING][NG];
#pragma unroll
    for (int j = 0; j < RING; ++j)
        if (has && j < nsteps) load_step(j, ring[j]);
    lds_sync();                                                      // s_row
    GmF16<TS> st;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        gm_load_f16<TS>(st, a.act, K, 0, h, s_row);
        gm_store_f16<TS>(st, h, sh0);
    }
    lds_sync();
    v4f_t acc[NG][TS];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int ts = 0; ts < TS; ++ts) acc[g][ts] = (v4f_t) {0.0f, 0.0f, 0.0f, 0.0f};
    const int nch = nsteps / CS;
    const bool tall = __builtin_amdgcn_readfirstlane(nt) > GT / 2;   // (TS 8: the upper half of the tile has rows)
    for (int ck = 0; ck < nch; ++ck) {
        // the next chunk's rows go into the other buffer (free: every wave passed the barrier
        // after its last reads) in two halves, so only half of them occupy registers at a time
        const uint16_t * sh = sh0 + (ck & 1) * BUF;
        uint16_t * nb = sh0 + ((ck + 1) & 1) * BUF;
        const bool more = ck + 1 < nch;
#pragma unroll
        for (int kb = 0; kb < CS; ++kb) {
            if (more && kb == 0) gm_load_f16<TS>(st, a.act, K, ck + 1, 0, s_row);
            if (more && kb == (CS == 4 ? 2 : 3)) { gm_store_f16<TS>(st, 0, nb); gm_load_f16<TS>(st, a.act, K, ck + 1, 1, s_row); }
            if (more && CS == 8 && kb == 6) gm_store_f16<TS>(st, 1, nb);
            if (has) {
                const int kk = ck * CS + kb;
                u32x4 (&b)[NG] = ring[kb % RING];                    // = kk % RING: RING divides CS
                auto mul = [&](int ts) {
                    const v8h_t A = *(const v8h_t *) (sh + (ts * 16 + (lane & 15)) * HP + 32 * kb + 8 * q);
#pragma unroll
                    for (int g = 0; g < NG; ++g)
                        acc[g][ts] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, __builtin_bit_cast(v8h_t, b[g]), acc[g][ts], 0, 0, 0);
                };
                constexpr int T1 = TS >= 8 ? TS / 2 : TS;
#pragma unroll
                for (int ts = 0; ts < T1; ++ts) mul(ts);
                if (T1 < TS && tall) {
#pragma unroll
                    for (int ts = T1; ts < TS; ++ts) mul(ts);
                }
                if (kk + RING < nsteps) load_step(kk + RING, b);
            }
        }
        if (more && CS == 4) gm_store_f16<TS>(st, 1, nb);
        lds_sync();
    }
    if (!has) return;
#pragma unroll
    for (int ts = 0; ts < TS; ++ts)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int t = ts * 16 + 4 * q + i;
            if (t >= nt) continue;
            const int it = s_out[t];
            float * o = a.out + (int64_t) it * a.out_ld;
            if (DUAL) {
#pragma unroll
                for (int g = 0; g < NG / 2; ++g) {
                    const int row = r0 + 16 * g + (lane & 15);
                    if (row < a.rows) o[row] = acc[g + NG / 2][ts][i] * z_silu(acc[g][ts][i]);
                }
            } else {
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    const int row = r0 + 16 * g + (lane & 15);
                    if (row < a.rows) o[row] = gemm_epi(a, acc[g][ts][i], ((const float *) s_out)[GT + t]);
                }
            }
        }
}

// Dense F16 matmuls of few rows (decode widths, the output head): a block owns 16 G weight rows and up to 64
// token rows, 16 per wave. Bounded by HBM latency and bytes in flight: one wave streaming its 16 rows (the narrow
// k_gemm_f16: 145 blocks for the 9225-row head) keeps 8 KB in flight; here the block's 256 threads request
// the rows' whole K range, in phases of 1024 columns through LDS with two phases in registers, so that 2048
// columns are in flight at once from every block. Each wave then runs k_gemm_f16's chain of 32-column
// products for its tokens: same bits. Head of 9225 x 2048, G = 1: one row 20.7 -> 11.1 us (cold 34 -> 13), 40 rows
// 37 -> 26, 64 rows 39 -> 35. More rows are bounded by the reads of the token rows, 256 KB per block, from L2;
// G = 2 halves them: 40 rows 23, 64 rows 29.
constexpr int FEW_SB = 4;                // superblocks per phase
constexpr int FEW_LD = FEW_SB * 2;       // 16-byte items per thread, phase and group: 32 FEW_SB chunks x 16 rows
template <int G>
__global__ void __launch_bounds__(256) k_gemm_f16_few(GemmArgs a) {
    __shared__ __attribute__((aligned(16))) u32x4 s_w[G][FEW_SB * 32 * 16];   // [group][chunk][row]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, q = lane >> 4, K = a.nsb * 256;
    const int r0 = 16 * G * blockIdx.x, t0 = 64 * blockIdx.y + 16 * wave, nt = min(16, a.n_tok - t0);
    // (64-row weight tiles hold whole groups, so a block's last group exists)
    const u32x4 * w = (const u32x4 *) a.w[0] + (size_t) (r0 / 64) * a.nsb * 32 * 64 + r0 % 64 + (tid & 15);
    const int nch = a.nsb * 32, steps = a.nsb * 8;
    auto load_w = [&](u32x4 (&v)[G * FEW_LD], int ph) {              // (chunks past the row repeat the last)
#pragma unroll
        for (int j = 0; j < FEW_LD; ++j)
#pragma unroll
            for (int g = 0; g < G; ++g) v[G * j + g] = w[(size_t) min(ph * FEW_SB * 32 + 16 * j + (tid >> 4), nch - 1) * 64 + 16 * g];
    };
    auto store_w = [&](const u32x4 (&v)[G * FEW_LD]) {
#pragma unroll
        for (int j = 0; j < FEW_LD; ++j)
#pragma unroll
            for (int g = 0; g < G; ++g) s_w[g][(16 * j + (tid >> 4)) * 16 + (tid & 15)] = v[G * j + g];
    };
    // the wave's token rows (rows past the last repeat it; a wave without rows only stages)
    const uint16_t * x = a.act.h + (int64_t) (nt > 0 ? t0 + min(lane & 15, nt - 1) : 0) * K + 8 * q;
    constexpr int RING = 8;
    u32x4 A[RING], v[2][G * FEW_LD];
    load_w(v[0], 0);
    if (nt > 0)
#pragma unroll
        for (int j = 0; j < RING; ++j) A[j] = *(const u32x4 *) (x + 32 * j);   // (steps >= 8)
    load_w(v[1], 1);
    v4f_t acc[G];
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = (v4f_t) {0.0f, 0.0f, 0.0f, 0.0f};
    auto phase = [&](u32x4 (&cur)[G * FEW_LD], int ph) {
        if (ph) lds_sync();                                          // the last phase is read
        store_w(cur);
        load_w(cur, ph + 2);
        lds_sync();
        if (nt <= 0) return;
        const int n = min(FEW_SB, a.nsb - ph * FEW_SB);
        for (int sb = 0; sb < n; ++sb) {
            const int k0 = (ph * FEW_SB + sb) * 8;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const v8h_t B = __builtin_bit_cast(v8h_t, s_w[g][(4 * (sb * 8 + j) + q) * 16 + (lane & 15)]);
                    acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h_t, A[j]), B, acc[g], 0, 0, 0);
                }
                A[j] = *(const u32x4 *) (x + 32 * min(k0 + j + RING, steps - 1));
            }
        }
    };
    for (int ph = 0; ph * FEW_SB < a.nsb; ph += 2) {
        phase(v[0], ph);
        if ((ph + 1) * FEW_SB < a.nsb) phase(v[1], ph + 1);
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const int row = r0 + 16 * g + (lane & 15);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (4 * q + i < nt && row < a.rows) a.out[(int64_t) (t0 + 4 * q + i) * a.out_ld + row] = gemm_epi(a, acc[g][i], 0.0f);
    }
}

} // namespace z2d

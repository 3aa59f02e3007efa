// A few tokens of Q4_K / Q6_K weights on the int8 matrix cores, bit-exact with the matvec.
//
// v_mfma_i32_16x16x32_i8 multiplies 32 elements of 16 rows with 16 tokens: a Q4_K sub-block, or two Q6_K
// sub-blocks one at a time (the other half's activations zero). Its exact int32 dots are weighted by the
// sub-block scales and added per super-block (a lane holds one row, so the scales are its own), the mins (Q4_K) and
// the offset 32 of the quants (Q6_K) come from one f16 matrix instruction against the activations' 16-element
// sums (exact integers below 2^24), and the f32 combine is the matvec's, super-blocks in order.
//
// Each wave takes one super-block of 16 MT rows and requests all it needs of it at once; the eight waves of a workgroup
// (four, or two, where a row has no more super-blocks) take as many super-blocks side by side and hand their terms
// through LDS to the threads that add them in order. What bounds it: the weights' stream and its latency (22016 x 2048
// Q4_K, 7 tokens: a wave waits 47 % of its time for data, the VALU is busy in 22 % of the cycles); the VALU work of a
// super-block is about 115 instructions per 16 rows whatever the tokens, up to 16, where the 8-token matvec spends 245
// per token and 64 units. 22016 x 2048 Q4_K (25 MB), 8 tokens, with the quantiser's launch: 33.5 -> 11.2 us; 2048 x 2048
// 13.0 -> 7.6; Q6_K 2048 x 11008 40.0 -> 19.6.
#include "sdy_device.h"
#include "sdy_internal.h"
#include "sdy_quant_dev.h"
#include "sdy_shim.h"

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct SbArgs {
    const uint8_t *p[5];  // planes (quant_kernels.hip), or the tiled copy's (blk, grow0)
    int T, nb;            // 64-element units and super-blocks per row
    int blk;              // records [row / 32][record][row % 32]; row r is row grow0 + r there
    long grow0;
    long row0, n_rows;
    const uint8_t *xq;    // Q8_K rows, nb blocks of 292 bytes,
    SdyGemmExp e;         // or the GEMM's expansion of them
    int n_tok;
    float *out;
    long out_stride;
    const float *bias, *resid;
    int swiglu;
};

SDY_DEV __amdgpu_buffer_rsrc_t rsrc(const uint8_t *p) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, -1, 0x00020000);
}
SDY_DEV u32x2 bload8(__amdgpu_buffer_rsrc_t r, uint32_t v, int s) {
    const auto x = __builtin_amdgcn_raw_buffer_load_b64(r, v, s, 0);
    return u32x2{(uint32_t)x[0], (uint32_t)x[1]};
}
SDY_DEV long as_long(u32x2 v) { return __builtin_bit_cast(long, v); }

// Hides where the sums come from: the compiler keeps one multiply-add per product (it would add the products of two
// sub-blocks at once, in three instructions).
SDY_DEV void opaque(i32x4 &v) { __asm__ volatile("" : "+v"(v)); }

// KS: waves, super-blocks of a round. by: the workgroup's row tile
template <int WT, int MT, int KS, bool EXP>
SDY_DEV void sb_body(const SbArgs &g, int by, float (*terms)[KS][MT * 256]) {
    constexpr bool Q4 = WT == SDY_Q4_K;
    constexpr int OUT = MT * 256, NTH = 64 * KS;  // outputs of the workgroup, threads
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long rt = (long)by * (16 * MT);
    const int t0 = (int)blockIdx.x * 16, nb = g.nb;

    // The lane's rows n of each row tile: byte offsets of their records, and from one unit's (super-block's) to the
    // next's. The k-slots 8 q .. 8 q + 7 of a 32-element half unit are bytes 8 (q % 2) .. of plane q / 2.
    uint32_t vu[MT], vs[MT];
    const int us = g.blk ? 512 : 16;
    const uint32_t qo = (q >> 1 ? (uint32_t)(g.p[1] - g.p[0]) : 0u) + 8u * (uint32_t)(q & 1);
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const long ri = rt + 16 * m + n, rc = g.row0 + (ri < g.n_rows ? ri : g.n_rows - 1);
        const uint32_t R = (uint32_t)(g.grow0 + rc);
        vu[m] = g.blk ? ((R >> 5) * (uint32_t)g.T * 32u + (R & 31u)) * 16u : (uint32_t)rc * (uint32_t)g.T * 16u;
        vs[m] = g.blk ? ((R >> 5) * (uint32_t)nb * 32u + (R & 31u)) : (uint32_t)rc * (uint32_t)nb;
    }
    const int ss = g.blk ? 32 : 1;  // super-block records from one to the next
    const __amdgpu_buffer_rsrc_t r0 = rsrc(g.p[0]), r2 = rsrc(g.p[2]), r3 = rsrc(g.p[3]), r4 = rsrc(g.p[4]),
                                 rx = rsrc(EXP ? (const uint8_t *)g.e.y8 : g.xq), ry = rsrc((const uint8_t *)g.e.yd), rb = rsrc((const uint8_t *)g.e.bs16);
    // token n's row for the products, tokens 4 q + i for the scales of the results
    constexpr uint32_t XB = EXP ? 256u : 292u, YB = EXP ? 4u : 292u;
    auto tok_sb = [&](int t) { return (uint32_t)(t0 + t < g.n_tok ? t0 + t : g.n_tok - 1) * (uint32_t)nb; };
    const uint32_t va = tok_sb(n) * XB, vb = tok_sb(n) * 32u;
    uint32_t vy[4];
#pragma unroll
    for (int i = 0; i < 4; i++) vy[i] = tok_sb(4 * q + i) * YB;

    struct Regs {
        u32x2 w[MT][4], hb[Q4 ? 1 : MT][4];
        u32x4 sc[MT];
        uint32_t d[Q4 ? 1 : MT];
        u32x2 a[8], bs;
        float yd[4];
    };
    auto load = [&](int sb, Regs &r) {
        const int xb = sb * (int)XB;
#pragma unroll
        for (int i = 0; i < 4; i++)
            r.yd[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(EXP ? ry : rx, vy[i], sb * (int)YB, 0));
        r.bs = EXP ? bload8(rb, vb + 8u * (uint32_t)q, sb * 32) : bload8(rx, va + 8u * (uint32_t)q, xb + 260);
#pragma unroll
        for (int j = 0; j < 8; j++) r.a[j] = bload8(rx, va + 8u * (uint32_t)q, xb + (EXP ? 0 : 4) + 32 * j);
#pragma unroll
        for (int m = 0; m < MT; m++) {
            r.sc[m] = __builtin_amdgcn_raw_buffer_load_b128(Q4 ? r2 : r3, vs[m] * 16u, sb * ss * 16, 0);
            if constexpr (!Q4) r.d[m] = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r4, vs[m] * 2u, sb * ss * 2, 0);
#pragma unroll
            for (int u = 0; u < 4; u++) {
                r.w[m][u] = bload8(r0, vu[m] + qo, (4 * sb + u) * us);
                if constexpr (!Q4) r.hb[m][u] = bload8(r2, vu[m] + 8u * (uint32_t)(q & 1), (4 * sb + u) * us);
            }
        }
    };
    // the super-block's f32 terms of the lane's outputs (token 4 q + i, row n), as the matvec forms them
    auto compute = [&](const Regs &r, float *dst) {
        f16x4 bsf;
        if constexpr (EXP) {
            bsf = __builtin_bit_cast(f16x4, r.bs);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) bsf[e] = (_Float16)(float)(int16_t)(r.bs[e >> 1] >> (16 * (e & 1)));
        }
#pragma unroll
        for (int m = 0; m < MT; m++) {
            i32x4 isum = {};
            f16x4 gw;  // the weights of the lane's 16-element groups 4 q .. 4 q + 3 in the sums' product
            float t[4];
            if constexpr (Q4) {
                const uint32_t A = r.sc[m].y, B = r.sc[m].z, C = r.sc[m].w;
                const uint32_t s[2] = {A & 0x3F3F3F3Fu, (C & 0x0F0F0F0Fu) | ((A >> 2) & 0x30303030u)};
                const uint32_t mn[2] = {B & 0x3F3F3F3Fu, ((C >> 4) & 0x0F0F0F0Fu) | ((B >> 2) & 0x30303030u)};
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const u32x2 w = r.w[m][u];
#pragma unroll
                    for (int hi = 0; hi < 2; hi++) {
                        const int j = 2 * u + hi;
                        const i32x4 p = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                            as_long(r.a[j]), as_long((hi ? w >> 4u : w) & 0x0F0F0F0Fu), i32x4{}, 0, 0, 0);
                        const int sc = (int)((s[j >> 2] >> (8 * (j & 3))) & 255u);
#pragma unroll
                        for (int i = 0; i < 4; i++) isum[i] += __mul24(sc, p[i]);  // |p| <= 32 * 15 * 128
                        opaque(isum);
                    }
                }
                const uint32_t mq = (q & 2 ? mn[1] : mn[0]) >> (16 * (q & 1));  // sub-blocks 2 q and 2 q + 1
                gw[0] = gw[1] = (_Float16)(float)(mq & 255u);
                gw[2] = gw[3] = (_Float16)(float)((mq >> 8) & 255u);
                const f32x4 msum = __builtin_amdgcn_mfma_f32_16x16x16f16(bsf, gw, f32x4{}, 0, 0, 0);
                const float d = sdy_h2f((uint16_t)(r.sc[m].x & 0xFFFFu)), dmin = sdy_h2f((uint16_t)(r.sc[m].x >> 16));
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float dall = r.yd[i] * d, dmn = r.yd[i] * dmin;
                    const float t1 = dall * (float)isum[i], t2 = dmn * msum[i];
                    t[i] = t1 - t2;
                }
            } else {
                const uint32_t lo = q < 2 ? ~0u : 0u;  // the first 16 elements' lanes
                const unsigned hs = q < 2 ? 0u : 2u;   // planes N0 / N1: high bits 0, 4 / 2, 6 of HB
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const u32x2 w = r.w[m][u], hb = r.hb[m][u] >> hs;
#pragma unroll
                    for (int hi = 0; hi < 2; hi++) {
                        const u32x2 e = hi ? ((w >> 4u) & 0x0F0F0F0Fu) | (hb & 0x30303030u)
                                           : (w & 0x0F0F0F0Fu) | ((hb & 0x03030303u) << 4u);
                        const uint32_t scw = (u == 0 ? r.sc[m].x : u == 1 ? r.sc[m].y : u == 2 ? r.sc[m].z : r.sc[m].w) >> (16 * hi);
                        const u32x2 a = r.a[2 * u + hi];
                        const i32x4 p0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(as_long(a & lo), as_long(e), i32x4{}, 0, 0, 0);
                        const i32x4 p1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(as_long(a & ~lo), as_long(e), i32x4{}, 0, 0, 0);
                        const int s0 = (int)(int8_t)(scw & 255u), s1 = (int)(int8_t)((scw >> 8) & 255u);
#pragma unroll
                        for (int i = 0; i < 4; i++) isum[i] += __mul24(s0, p0[i]);  // |p| <= 16 * 63 * 128
                        opaque(isum);
#pragma unroll
                        for (int i = 0; i < 4; i++) isum[i] += __mul24(s1, p1[i]);
                        opaque(isum);
                    }
                }
                const uint32_t sq = q == 0 ? r.sc[m].x : q == 1 ? r.sc[m].y : q == 2 ? r.sc[m].z : r.sc[m].w;
#pragma unroll
                for (int e = 0; e < 4; e++) gw[e] = (_Float16)(float)(int8_t)((sq >> (8 * e)) & 255u);
                // sum of sc * bsum: the 32 that each quant is stored above its value
                const f32x4 off = __builtin_amdgcn_mfma_f32_16x16x16f16(bsf, gw, f32x4{}, 0, 0, 0);
                const float d = sdy_h2f((uint16_t)r.d[m]);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float ydd = r.yd[i] * d;
                    t[i] = ydd * (float)(isum[i] - 32 * (int)off[i]);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) dst[(4 * m + i) * 64 + lane] = t[i];
        }
    };

    constexpr int NO = (OUT + NTH - 1) / NTH;  // outputs per thread: o = tid + NTH j
    float acc[NO];
#pragma unroll
    for (int j = 0; j < NO; j++) acc[j] = 0.0f;
    Regs R[2];
    const int nr = (nb + KS - 1) / KS;
    auto has = [&](int rd) { return rd * KS + wave < nb; };  // (waves past the last super-block only add)
    if (has(0)) load(wave, R[0]);
    auto round = [&](int rd, const Regs &cur, Regs &nxt, int z) {
        if (has(rd + 1)) load((rd + 1) * KS + wave, nxt);
        if (has(rd)) compute(cur, &terms[z][wave][0]);
        __syncthreads();  // (a buffer is written again two rounds on, past the next round's barrier)
        const int left = nb - rd * KS;
#pragma unroll
        for (int j = 0; j < NO; j++) {
            const int o = tid + NTH * j < OUT ? tid + NTH * j : 0;
            float v[KS];
#pragma unroll
            for (int k = 0; k < KS; k++) v[k] = terms[z][k][o];
#pragma unroll
            for (int k = 0; k < KS; k++)
                if (k < left) acc[j] = acc[j] + v[k];
        }
    };
    for (int rd = 0; rd < nr; rd += 2) {
        round(rd, R[0], R[1], 0);
        if (rd + 1 < nr) round(rd + 1, R[1], R[0], 1);
    }
    // output o: row tile o / 256, token 4 (o / 16 % 4) + o / 64 % 4, row o % 16
    const uint32_t etab = sdy_expf_tab_lane(lane);
#pragma unroll
    for (int j = 0; j < NO; j++) {
        const int o = tid + NTH * j;
        const int tok = t0 + 4 * ((o >> 4) & 3) + ((o >> 6) & 3);
        const long ri = rt + 16 * (o >> 8) + (o & 15), row = g.row0 + ri;
        const bool on = o < OUT && tok < g.n_tok && ri < g.n_rows;
        float v = acc[j];
        if (g.swiglu) {  // the pair's up row is in the next lane
            const float up = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));
            v = sdy_silu_mul1_reg(v, up, etab);
            if (on && !(o & 1)) g.out[(size_t)tok * g.out_stride + (ri >> 1)] = v;
        } else if (on) {
            const size_t at = (size_t)tok * g.out_stride + row;
            if (g.bias) v = v + g.bias[row];
            if (g.resid) v = g.resid[at] + v;
            g.out[at] = v;
        }
    }
}

template <int WT, int MT, int KS, bool EXP>
__global__ __launch_bounds__(64 * KS, 2) void k_mm_superblocks(SbArgs g) {
    __shared__ float terms[2][KS][MT * 256];
    sb_body<WT, MT, KS, EXP>(g, (int)blockIdx.y, terms);
}

// Two matrices, Q4_K and Q6_K, on the same activations in one launch: row tiles [0, gy1) of the grid multiply g1, the rest
// g2.
template <int KS>
__global__ __launch_bounds__(64 * KS, 2) void k_mm_superblocks_pair(SbArgs g1, SbArgs g2, int gy1) {
    __shared__ float terms[2][KS][256];
    if ((int)blockIdx.y < gy1) sb_body<SDY_Q4_K, 1, KS, true>(g1, (int)blockIdx.y, terms);
    else sb_body<SDY_Q6_K, 1, KS, true>(g2, (int)blockIdx.y - gy1, terms);
}

template <int WT, int MT, int KS, bool EXP>
int launch_ks(const SbArgs &g, hipStream_t st) {
    SDY_NOTE_KERNEL((k_mm_superblocks<WT, MT, KS, EXP>));
    hipLaunchKernelGGL((k_mm_superblocks<WT, MT, KS, EXP>),
                       dim3((unsigned)((g.n_tok + 15) / 16), (unsigned)((g.n_rows + 16 * MT - 1) / (16 * MT))), dim3(64 * KS), 0, st, g);
    return sdy_check_launch("matvec (super-block MFMA)");
}

// As many waves to a workgroup as rows have super-blocks, up to eight: the others would only hold their places (1024 x 33786
// Q4_K, 3 tokens: 12.9 us with eight, 10.9 with four, where the 8-token matvec took 12.6).
template <int WT, int MT, bool EXP>
int launch_sb(const SbArgs &g, hipStream_t st) {
    if (g.nb <= 2) return launch_ks<WT, MT, 2, EXP>(g, st);
    return g.nb <= 4 ? launch_ks<WT, MT, 4, EXP>(g, st) : launch_ks<WT, MT, 8, EXP>(g, st);
}

// The kernel's arguments of one call; 1 when its 32-bit offsets do not reach every byte of the matrix or the activations.
template <bool EXP>
int sb_args(const sdy_mat *m, const sdy_mv_args *a, const SdyGemmExp *e, SbArgs &g) {
    const int nb = m->n_in / 256;
    const size_t lim = 0xFFFFFFFFu;
    const long n_rows = a->row1 - a->row0;
    if (m->bytes >= lim || m->gbytes >= lim || (size_t)nb * 292 * a->n_tok >= lim || (!EXP && ((uintptr_t)a->xq & 3)) ||
        (n_rows + 15) / 16 > 65535)
        return 1;
    g = SbArgs{};
    for (int i = 0; i < 5; i++) g.p[i] = (const uint8_t *)m->base + m->plane_off[i];
    if (m->gbase) {
        size_t off[5];
        sdy_gemm_layout_planes(m->type, m->n_in, m->grows, off);
        for (int i = 0; i < 5; i++) g.p[i] = (const uint8_t *)m->gbase + off[i];
        g.blk = 1;
        g.grow0 = m->grow0;
    }
    g.T = m->n_units;
    g.nb = nb;
    g.row0 = a->row0;
    g.n_rows = n_rows;
    if (EXP) g.e = *e;
    else g.xq = (const uint8_t *)a->xq;
    g.n_tok = a->n_tok;
    g.out = a->out;
    g.out_stride = a->out_stride;
    g.bias = a->bias;
    g.resid = a->resid;
    g.swiglu = a->epilogue == SDY_EPI_SWIGLU;
    return 0;
}

template <bool EXP>
int run_sb(const sdy_mat *m, const sdy_mv_args *a, const SdyGemmExp *e, hipStream_t st) {
    SbArgs g;
    if (int rc = sb_args<EXP>(m, a, e, g)) return rc;
    // Two row tiles to a wave, sharing the activations' loads: Q4_K when one each gives every CU more than two
    // workgroups (22016 x 2048, 8 tokens: 11.2 us against 13.2; 2048 x 4096: 10.0 against 8.4), Q6_K, whose registers then
    // leave two waves to a SIMD, only with several token tiles (2048 x 11008, 64 tokens: 31.6 against 37.0; 151936 x
    // 2048, 8 tokens: 104 against 84)
    const long tiles = (g.n_rows + 15) / 16 * ((g.n_tok + 15) / 16);
    if (m->type == SDY_Q6_K)
        return g.n_tok > 16 && tiles >= 512 ? launch_sb<SDY_Q6_K, 2, EXP>(g, st) : launch_sb<SDY_Q6_K, 1, EXP>(g, st);
    return tiles > 512 ? launch_sb<SDY_Q4_K, 2, EXP>(g, st) : launch_sb<SDY_Q4_K, 1, EXP>(g, st);
}

}  // namespace

// The tokens of a->xq through rows [a->row0, a->row1) of m (Q4_K, Q6_K), with the bits of sdy_matvec. Returns 1,
// launching nothing, when the kernel's 32-bit offsets do not reach every byte of the matrix or the activations.
extern "C" int sdy_mm_superblocks(const sdy_mat *m, const sdy_mv_args *a, sdy_stream s) {
    return run_sb<false>(m, a, nullptr, (hipStream_t)s);
}

// The same from the GEMM's expansion of the activations.
int sdy_mm_superblocks_exp(const sdy_mat *m, const sdy_mv_args *a, const SdyGemmExp *e, sdy_stream s) {
    return run_sb<true>(m, a, e, (hipStream_t)s);
}

// A Q4_K and a Q6_K matrix of one or two super-blocks to a row in one launch, from one expansion.
int sdy_mm_superblocks_exp2(const sdy_mat *m1, const sdy_mv_args *a1, const sdy_mat *m2, const sdy_mv_args *a2,
                            const SdyGemmExp *e, sdy_stream s) {
    SbArgs g1, g2;
    if (m1->type != SDY_Q4_K || m2->type != SDY_Q6_K || m1->n_in > 512 || sb_args<true>(m1, a1, e, g1) || sb_args<true>(m2, a2, e, g2))
        return 1;
    const long gy1 = (g1.n_rows + 15) / 16, gy2 = (g2.n_rows + 15) / 16;
    if (gy1 + gy2 > 65535) return 1;
    SDY_NOTE_KERNEL(k_mm_superblocks_pair<2>);
    hipLaunchKernelGGL(k_mm_superblocks_pair<2>, dim3((unsigned)((g1.n_tok + 15) / 16), (unsigned)(gy1 + gy2)), dim3(128), 0,
                       (hipStream_t)s, g1, g2, (int)gy1);
    return sdy_check_launch("gemm2 (super-block MFMA)");
}

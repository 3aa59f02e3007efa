// Prompt GEMM of Q4_K / Q6_K weights on the int8 matrix cores, bit-exact with the reference's integer-dot path
// (csrc/quant.c:191-235, csrc/quant.h:84-91; the reference's 4-token micro-kernels csrc/quant_avx2.c:290-385 give
// the same bits as its one-token dots).
//
// v_mfma_i32_32x32x32_i8 multiplies a 32-element Q4_K sub-block of 32 rows with 32 tokens (Q6_K, whose sub-blocks
// have 16 elements: v_mfma_i32_32x32x16_i8). A lane holds one row of the 32 x 32 products, so a sub-block's scale
// is the lane's own: one 24-bit multiply-add per product sums them over the super-block, exactly, for every block
// the formats can hold. The Q4_K mins and the Q6_K quants' offset 32 are one f16 matrix instruction against the
// activations' 16-element sums (exact integers below 2^24), the f32 scale products an f32 outer product (one
// rounding, the VALU multiply's; a zero product may be +0 where the multiply gives -0, which no sum keeps), and
// the combine is the reference's expression, super-blocks in order.
//
// What bounds it: VALU work and the waits between it. Per super-block and 32 x 32 outputs Q4_K takes 304 VALU
// instructions (128 multiply-adds, 96 of the combine) and the f32 outer product's 64 cycles, Q6_K 524, or 424 where a
// wave unpacks the weights once for two token tiles; the matrix cores' 290 and 540 cycles run beside them. With three
// or more waves to a SIMD (22016 x 2048 Q4_K, 512 tokens) the VALU is busy in 74 % of the cycles; with two, a wave's
// waits show (151936 x 2048 Q6_K, 64 tokens, two token tiles to a wave: 51 %; 2048 x 11008 Q6_K, 203 tokens, 448 tiles
// split over four waves each: 40 %). The weights dequantised to f16 (sc * q, one fragment, two for the scales of real
// Q6_K files) summed whole super-blocks on the matrix cores with fewer VALU instructions, but its registers and LDS left
// two waves to a SIMD that waited for each other. With the quantiser's launch, f16 form -> this: 22016 x 2048 Q4_K, 512
// tokens 90.7 -> 81.2 us (568 TFLOP/s), 128 tokens 40.4 -> 29.0; 2048 x 11008 Q6_K, 203 tokens 69.1 -> 42.1, 64 tokens
// 66.3 -> 31.6 (on mm_superblocks.hip); 151936 x 2048 Q6_K, 32 tokens 110 -> 79, 64 tokens 121 -> 113. Q6_K on the
// largest grids is slower than on the f16 form: 22016 x 2048, 512 tokens 109 -> 113, 22016 x 4096 196 -> 216.
#include <stdlib.h>

#include <type_traits>

#include "sdy_device.h"
#include "sdy_internal.h"
#include "sdy_quant_dev.h"
#include "sdy_shim.h"

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct GemmArgs {
    const uint8_t *p[5];  // planes (quant_kernels.hip), or the tiled copy's (blk, grow0)
    int n_in, T, nb;      // elements, 64-element units and super-blocks per row
    int blk;              // records [row / 32][record][row % 32]; row r is row grow0 + r there
    long grow0;
    long row0, n_rows;    // rows row0 .. row0 + n_rows
    SdyGemmExp e;         // the activations' expansion
    int n_tok;
    float *out;
    long out_stride;
    const float *bias, *resid;
    int swiglu;
    // grouped (grp_tile set): group e (a routed expert) multiplies weight rows row0 + e * grp_rows + [0, n_rows) with
    // rows grp_tok[e] .. grp_tok[e + 1] - 1 on token tiles grp_tile[e] .. grp_tile[e + 1] - 1 of the grid; row t reads
    // expansion row act_row[t] and writes output row out_row[t] (either may be null: t)
    const int *grp_tile, *grp_tok, *out_row, *act_row;
    long grp_rows;
    int n_grp;
};

SDY_DEV __amdgpu_buffer_rsrc_t rsrc(const void *p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, -1, 0x00020000);
}
SDY_DEV long as_long(u32x2 v) { return __builtin_bit_cast(long, v); }
SDY_DEV u32x2 bload8(__amdgpu_buffer_rsrc_t r, uint32_t v, int s) {
    const auto x = __builtin_amdgcn_raw_buffer_load_b64(r, v, s, 0);
    return u32x2{(uint32_t)x[0], (uint32_t)x[1]};
}

template <int RW, int KS, int NT>
constexpr size_t gemm_lds_bytes() { return 2 * (size_t)(32 * NT * 292 * KS) + (KS > 1 ? RW * KS * 16 * 64 * 4 : 0); }

// A workgroup of RW * KS waves computes 32 RW rows x 32 NT tokens; a wave owns a row tile and, with KS > 1, every KS-th
// super-block: its f32 terms go through LDS to the tile's waves, each adding up a part of the outputs over the KS
// super-blocks in order. The activations are shared through LDS in stages of KS super-blocks, requested a stage ahead
// into registers, 16-byte chunk c of a token's 256 at slot c ^ (token % 16) (16 tokens' reads of one chunk then hit all
// 64 banks once). The weights go straight to registers, each lane (row lr, k-half h) loading its own records, and
// are reloaded for the next stage as they are used: from the tiled copy a load instruction reads runs of 512
// bytes. The workgroup's place in the grid is (bx, by) of (gx, gy): a pair launch gives each matrix a part of one grid.
// ALT, another way to the weights. Q4_K: planes too far apart for a lane to reach both by a 32-bit offset, by 64-bit
// addresses. Q6_K: the planes, where a lane's 8 bytes of a unit are half of a 16-byte record in a cache line per row: it
// loads a whole record of every second unit, and the two lanes of a row swap halves.
template <int WT, int RW, int KS, int NT, bool ALT>
SDY_DEV void gemm_body(const GemmArgs &g, int bx, int by, int gx, int gy, uint8_t *lds) {
    constexpr bool Q4 = WT == SDY_Q4_K;
    static_assert(NT == 1 || KS == 1, "token tiles share a wave's weights only where it has the row tile to itself");
    constexpr int BM = 32 * RW, BN = 32 * NT, NTH = 64 * RW * KS;
    constexpr int NA = BN * 16 * KS / NTH;             // 16-byte chunks of activations per thread and stage
    constexpr int NS = (BN * 2 * KS + NTH - 1) / NTH;  // of their 16-element sums
    constexpr int NY = (BN * KS + NTH - 1) / NTH;      // and scales
    static_assert(BN * 16 * KS % NTH == 0, "whole chunks per thread");
    constexpr int OFF_B = BN * 256 * KS, OFF_Y = OFF_B + BN * 32 * KS, STAGE = OFF_Y + BN * 4 * KS;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, lr = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = wave % KS, rw = wave / KS;
    // token tiles of a row tile on one XCD (workgroups are dealt to the 8 XCDs in turn)
    const long n_tt = gx, n_rt = gy, L = (long)by * n_tt + bx;
    long rti, tti;
    if (L < n_rt / 8 * 8 * n_tt) {
        const long gq = L / (8 * n_tt), w = L - gq * 8 * n_tt;
        rti = gq * 8 + (w & 7);
        tti = w >> 3;
    } else {
        const long w = L - n_rt / 8 * 8 * n_tt;
        rti = n_rt / 8 * 8 + w / n_tt;
        tti = w % n_tt;
    }
    int t0 = (int)tti * BN, t_end = g.n_tok;
    long row0 = g.row0;
    if (g.grp_tile) {
        // the group of this token tile: the last e with grp_tile[e] <= tti (empty groups share their successor's
        // start, so the last one is the group that owns the tile)
        if (tti >= g.grp_tile[g.n_grp]) return;  // past the routed tokens (uniform over the workgroup)
        int lo = 0, hi = g.n_grp - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (g.grp_tile[mid] <= (int)tti) lo = mid;
            else hi = mid - 1;
        }
        t0 = g.grp_tok[lo] + ((int)tti - g.grp_tile[lo]) * BN;
        t_end = g.grp_tok[lo + 1];
        row0 += (long)lo * g.grp_rows;
    }
    const int nb = g.nb, T = g.T, ns = (nb + KS - 1) / KS;

    // Weights: buffers from the first record of the wave's rows (of its first tile of 32 in the copy), the lane's
    // offsets from there, and a unit's (super-block's) scalar one.
    const long rt = rti * BM + 32 * rw, ri = rt + lr;
    const long rfirst = row0 + (rt < g.n_rows ? rt : g.n_rows - 1), rc = row0 + (ri < g.n_rows ? ri : g.n_rows - 1);
    const long t32 = (g.grow0 + rfirst) >> 5;
    const size_t ub = g.blk ? (size_t)t32 * T * 32 : (size_t)rfirst * T, sb0 = g.blk ? (size_t)t32 * nb * 32 : (size_t)rfirst * nb;
    const uint32_t dt = (uint32_t)(((g.grow0 + rc) >> 5) - t32), r32 = (uint32_t)(g.grow0 + rc) & 31u, dr = (uint32_t)(rc - rfirst);
    const uint32_t vu = (g.blk ? dt * (uint32_t)T * 32u + r32 : dr * (uint32_t)T) * 16u;
    const uint32_t vs = g.blk ? dt * (uint32_t)nb * 32u + r32 : dr * (uint32_t)nb;
    const int us = g.blk ? 512 : 16, ss = g.blk ? 32 : 1;
    const __amdgpu_buffer_rsrc_t r0 = rsrc(g.p[0] + ub * 16), r1 = rsrc(g.p[1] + ub * 16),
                                 r2 = rsrc(g.p[2] + (Q4 ? sb0 : ub) * 16), r3 = rsrc(g.p[3] + sb0 * 16), r4 = rsrc(g.p[4] + sb0 * 2);
    // (Q4_K: lane half h reads plane h; Q6_K: bytes 8 h .. of each plane's record, ALT: the record of unit 2 p + h)
    const uint32_t vq = vu + (Q4 ? (h ? (uint32_t)(g.p[1] - g.p[0]) : 0u) : (ALT ? (uint32_t)us : 8u) * (uint32_t)h);
    const uint8_t *const vfar = (h ? g.p[1] : g.p[0]) + ub * 16 + vu;
    u32x4 w4[Q4 ? 4 : 1], sc;
    u32x4 w6[Q4 ? 1 : 2][3];  // of units 2 p and 2 p + 1, eight bytes of each (ALT: as loaded, before the swap)
    uint32_t d6 = 0;
    auto sb_of = [&](int s) { return s * KS + ks < nb ? s * KS + ks : nb - 1; };  // (past the end: not added)
    auto load_u = [&](int s, int u) {
        const int so = (4 * sb_of(s) + u) * us;
        if constexpr (Q4 && ALT) {
            w4[u] = *reinterpret_cast<const u32x4 *>(vfar + so);
        } else if constexpr (Q4) {
            w4[u] = __builtin_amdgcn_raw_buffer_load_b128(r0, vq, so, 0);
        } else if constexpr (ALT) {
            if (u & 1) {
                const int sp = so - us;
                w6[u >> 1][0] = __builtin_amdgcn_raw_buffer_load_b128(r0, vq, sp, 0);
                w6[u >> 1][1] = __builtin_amdgcn_raw_buffer_load_b128(r1, vq, sp, 0);
                w6[u >> 1][2] = __builtin_amdgcn_raw_buffer_load_b128(r2, vq, sp, 0);
            }
        } else {
            const u32x2 x[3] = {bload8(r0, vq, so), bload8(r1, vq, so), bload8(r2, vq, so)};
#pragma unroll
            for (int i = 0; i < 3; i++) {
                w6[u >> 1][i][2 * (u & 1)] = x[i][0];
                w6[u >> 1][i][2 * (u & 1) + 1] = x[i][1];
            }
        }
    };
    auto load_s = [&](int s) {
        sc = __builtin_amdgcn_raw_buffer_load_b128(Q4 ? r2 : r3, vs * 16u, sb_of(s) * ss * 16, 0);
        if constexpr (!Q4) d6 = (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r4, vs * 2u, sb_of(s) * ss * 2, 0);
    };
    // Activations: this thread's chunks of a stage, of fixed tokens, super-block of the stage and place in it.
    const __amdgpu_buffer_rsrc_t ry = rsrc(g.e.y8), rb = rsrc(g.e.bs16), rd = rsrc(g.e.yd);
    auto act_of = [&](int t) {
        const int r = t0 + t < t_end ? t0 + t : t_end - 1;
        return (uint32_t)(g.act_row ? g.act_row[r] : r);
    };
    const int ac = tid % 16, ak = tid / 16 % KS, at0 = tid / (16 * KS), bk = tid / 2 % KS, yk = tid % KS;
    constexpr int AS = NTH / (16 * KS);  // tokens between a thread's chunks
    // (fewer sums and scales than threads: the threads past them repeat one, with the same values)
    auto bt = [&](int i) { return (tid + NTH * i) / (2 * KS) % BN; };
    auto yt = [&](int i) { return (tid + NTH * i) / KS % BN; };
    uint32_t ao[NA], bo[NS], yo[NY];
#pragma unroll
    for (int i = 0; i < NA; i++) ao[i] = act_of(at0 + AS * i) * (uint32_t)g.n_in + 16u * (uint32_t)ac;
#pragma unroll
    for (int i = 0; i < NS; i++) bo[i] = act_of(bt(i)) * (uint32_t)nb * 32u + 16u * (uint32_t)(tid & 1);
#pragma unroll
    for (int i = 0; i < NY; i++) yo[i] = act_of(yt(i)) * (uint32_t)nb * 4u;
    u32x4 av[NA], bv[NS];
    uint32_t yv[NY];
    auto load_a = [&](int s) {
        auto blk = [&](int k) { return s * KS + k < nb ? s * KS + k : nb - 1; };
#pragma unroll
        for (int i = 0; i < NA; i++) av[i] = __builtin_amdgcn_raw_buffer_load_b128(ry, ao[i] + 256u * (uint32_t)blk(ak), 0, 0);
#pragma unroll
        for (int i = 0; i < NS; i++) bv[i] = __builtin_amdgcn_raw_buffer_load_b128(rb, bo[i] + 32u * (uint32_t)blk(bk), 0, 0);
#pragma unroll
        for (int i = 0; i < NY; i++) yv[i] = __builtin_amdgcn_raw_buffer_load_b32(rd, yo[i] + 4u * (uint32_t)blk(yk), 0, 0);
    };
    auto store_a = [&](uint8_t *buf) {
#pragma unroll
        for (int i = 0; i < NA; i++) {
            const int t = at0 + AS * i;
            *reinterpret_cast<u32x4 *>(buf + (ak * BN + t) * 256 + 16 * (ac ^ (t & 15))) = av[i];
        }
#pragma unroll
        for (int i = 0; i < NS; i++) *reinterpret_cast<u32x4 *>(buf + OFF_B + (bk * BN + bt(i)) * 32 + 16 * (tid & 1)) = bv[i];
#pragma unroll
        for (int i = 0; i < NY; i++) *reinterpret_cast<uint32_t *>(buf + OFF_Y + (yk * BN + yt(i)) * 4) = yv[i];
    };

    constexpr int NF = 16 / KS;  // the outputs a wave adds up: registers NF ks .. of the tile's 16
    float acc[NT][NF];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int i = 0; i < NF; i++) acc[nt][i] = 0.0f;
    float *xch = reinterpret_cast<float *>(lds + 2 * STAGE);
    // isum[nt] += scale(j) * products (j, nt), j = 0 .. n - 1, each issued a step ahead of its use
    auto sums = [&](auto issue, auto scale, auto n, i32x16 isum[NT]) {
        i32x16 p[2];
        issue(0, 0, p[0]);
#pragma unroll
        for (int k = 0; k < n() * NT; k++) {
            if (k + 1 < n() * NT) issue((k + 1) / NT, (k + 1) % NT, p[(k + 1) & 1]);
            const int f = scale(k / NT), nt = k % NT;
#pragma unroll
            for (int i = 0; i < 16; i++) isum[nt][i] += __mul24(f, p[k & 1][i]);  // |p| <= 32 * 15 * 128 or 16 * 63 * 128
            // hide where the sums come from: the compiler then keeps one multiply-add per product (it would add
            // the products of two sub-blocks at once, in three instructions and with both products' registers)
            __asm__ volatile("" : "+v"(isum[nt]));
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // the wave's super-block of stage s, and its weights' reload for the next stage
    auto compute = [&](int s, const uint8_t *buf) {
        const uint8_t *ab = buf + (ks * BN + lr) * 256;
        i32x16 isum[NT] = {};
        f16x8 gw;  // the mins (Q4_K) or -32 times the scales (Q6_K) of the lane's 16-element groups 8 h .. 8 h + 7
        float dl;  // d, and for Q4_K dmin in lane half 1
        auto group_sums = [&](int nt, const f16x8 &w) {
            const f16x8 bs = *reinterpret_cast<const f16x8 *>(buf + OFF_B + (ks * BN + 32 * nt + lr) * 32 + 16 * h);
            return __builtin_amdgcn_mfma_f32_32x32x16_f16(bs, w, f32x16{}, 0, 0, 0);
        };
        if constexpr (Q4) {
            // 6-bit scales and mins of the 8 sub-blocks as bytes (csrc/quant.h:72-80)
            const uint32_t A = sc.y, B = sc.z, C = sc.w;
            const uint32_t sw[2] = {A & 0x3F3F3F3Fu, (C & 0x0F0F0F0Fu) | ((A >> 2) & 0x30303030u)};
            const uint32_t mw = h ? ((C >> 4) & 0x0F0F0F0Fu) | ((B >> 2) & 0x30303030u) : B & 0x3F3F3F3Fu;
            dl = sdy_h2f((uint16_t)(h ? sc.x >> 16 : sc.x & 0xFFFFu));
#pragma unroll
            for (int e = 0; e < 8; e++) gw[e] = (_Float16)(float)((mw >> (8 * (e >> 1))) & 255u);
            load_s(s + 1);
            i32x4 wf;
            auto issue = [&](int j, int nt, i32x16 &p) {  // sub-block j: the low or high nibbles of unit j / 2, 16 to a lane half
                if (nt == 0) {
                    const u32x4 w = w4[j >> 1];
                    wf = __builtin_bit_cast(i32x4, ((j & 1) ? w >> 4u : w) & 0x0F0F0F0Fu);
                    if (j & 1) load_u(s + 1, j >> 1);
                }
                const i32x4 a = *reinterpret_cast<const i32x4 *>(ab + 32 * 256 * nt + 16 * ((2 * j + h) ^ (lr & 15)));
                p = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, wf, i32x16{}, 0, 0, 0);
            };
            sums(issue, [&](int j) { return (int)((sw[j >> 2] >> (8 * (j & 3))) & 255u); }, std::integral_constant<int, 8>{}, isum);
        } else {
            const u32x4 scv = sc;
            dl = sdy_h2f((uint16_t)d6);
            const uint32_t g0 = h ? scv.z : scv.x, g1 = h ? scv.w : scv.y;
#pragma unroll
            for (int e = 0; e < 8; e++) gw[e] = (_Float16)(-32.0f * (float)(int8_t)(((e < 4 ? g0 : g1) >> (8 * (e & 3))) & 255u));
            load_s(s + 1);
            // the sums begin with what the 32 in every quant adds to them: exact, multiples of 32 below 2^27
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const f32x16 off = group_sums(nt, gw);
#pragma unroll
                for (int i = 0; i < 16; i++) isum[nt][i] = (int)off[i];
            }
            long wf;
            auto issue = [&](int j, int nt, i32x16 &p) {  // sub-block j = 4 u + k: elements 16 k .. of unit u, stored 32 too high
                const int u = j >> 2, k = j & 3;
                if (nt == 0) {
                    if constexpr (ALT) {
                        if (k == 0 && !(u & 1)) {  // dwords 2, 3 of the first lane's unit for 0, 1 of the second's
#pragma unroll
                            for (int i = 0; i < 3; i++)
#pragma unroll
                                for (int e = 0; e < 2; e++) {
                                    const auto x = __builtin_amdgcn_permlane32_swap(w6[u >> 1][i][e], w6[u >> 1][i][e + 2], false, false);
                                    w6[u >> 1][i][e] = x[0];
                                    w6[u >> 1][i][e + 2] = x[1];
                                }
                        }
                    }
                    auto unit = [&](int i) { return u & 1 ? u32x2{w6[u >> 1][i][2], w6[u >> 1][i][3]} : u32x2{w6[u >> 1][i][0], w6[u >> 1][i][1]}; };
                    const u32x2 nn = unit(k & 1), hb = unit(2);
                    const u32x2 lo = (k & 2) ? (nn >> 4u) & 0x0F0F0F0Fu : nn & 0x0F0F0F0Fu;
                    const u32x2 hi = k == 0 ? (hb & 0x03030303u) << 4u : k == 1 ? (hb & 0x0C0C0C0Cu) << 2u
                                     : k == 2 ? hb & 0x30303030u : (hb >> 2u) & 0x30303030u;
                    wf = as_long(lo | hi);
                    if (k == 3) load_u(s + 1, u);
                }
                const long a = *reinterpret_cast<const long *>(ab + 32 * 256 * nt + 16 * (j ^ (lr & 15)) + 8 * h);
                p = __builtin_amdgcn_mfma_i32_32x32x16_i8(a, wf, i32x16{}, 0, 0, 0);
            };
            sums(issue, [&](int j) { return (int)(int8_t)((scv[j >> 2] >> (8 * (j & 3))) & 255u); }, std::integral_constant<int, 16>{}, isum);
        }
        float *xw = xch + (size_t)wave * (16 * 64) + lane;
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const float yd = *reinterpret_cast<const float *>(buf + OFF_Y + (ks * BN + 32 * nt + lr) * 4);
            f32x16 off;
            if constexpr (Q4) off = group_sums(nt, gw);
            // yd d in registers 0 .. 15 and (Q4_K) yd dmin in 16 .. 31: block b takes its factors from lane half b
            const f32x32 sd = __builtin_amdgcn_mfma_f32_32x32x1f32(yd, dl, f32x32{}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 16; i++) {
                float term;
                if constexpr (Q4) {
                    const float t1 = sd[i] * (float)isum[nt][i], t2 = sd[16 + i] * off[i];
                    term = t1 - t2;
                } else {
                    term = sd[i] * (float)isum[nt][i];
                }
                if constexpr (KS == 1) acc[nt][i] = acc[nt][i] + term;
                else xw[i * 64] = term;
            }
        }
    };
    // orders LDS only: the weights in flight stay in flight
    auto barrier = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    load_a(0);
    load_s(0);
#pragma unroll
    for (int u = 0; u < 4; u++) load_u(0, u);
    store_a(lds);
    barrier();
    for (int s = 0; s < ns; s++) {
        load_a(s + 1);  // (past the last stage the loads are clamped, their values not used)
        compute(s, lds + (s & 1) * STAGE);
        store_a(lds + ((s + 1) & 1) * STAGE);
        barrier();
        if constexpr (KS > 1) {
            const float *xr = xch + (size_t)(rw * KS) * (16 * 64) + NF * ks * 64 + lane;
            const int left = nb - s * KS;
            float v[KS][NF];
#pragma unroll
            for (int k = 0; k < KS; k++)
#pragma unroll
                for (int i = 0; i < NF; i++) v[k][i] = xr[k * (16 * 64) + i * 64];
#pragma unroll
            for (int k = 0; k < KS; k++)
#pragma unroll
                for (int i = 0; i < NF; i++) acc[0][i] = k < left ? acc[0][i] + v[k][i] : acc[0][i];
            barrier();  // the terms are read before the next stage's overwrite them
        }
    }
    // register f of the tile's 16 (this wave's: NF ks + i) holds token 8 (f / 4) + 4 h + f % 4, row lr. The residuals and
    // output rows are requested before the first store.
    const uint32_t etab = sdy_expf_tab_lane(lane);
    const bool on_row = ri < g.n_rows;
    const long row = g.grp_tile ? ri : g.row0 + ri;
    const float bias = g.bias && on_row ? g.bias[row] : 0.0f;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        int orow[NF];
        bool on[NF];
#pragma unroll
        for (int i = 0; i < NF; i++) {
            const int f = NF * ks + i, t = t0 + 32 * nt + 8 * (f >> 2) + 4 * h + (f & 3), tc = t < t_end ? t : t_end - 1;
            on[i] = on_row && t < t_end;
            orow[i] = g.out_row ? g.out_row[tc] : tc;
        }
        if (g.swiglu) {  // the pair's up row is in the next lane
#pragma unroll
            for (int i = 0; i < NF; i++) {
                const float up = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, acc[nt][i]), 0xB1, 0xF, 0xF, false));
                const float v = sdy_silu_mul1_reg(acc[nt][i], up, etab);
                if (on[i] && !(lr & 1)) g.out[(size_t)orow[i] * g.out_stride + (ri >> 1)] = v;
            }
            continue;
        }
        float rv[NF];
#pragma unroll
        for (int i = 0; i < NF; i++) rv[i] = g.resid && on[i] ? g.resid[(size_t)orow[i] * g.out_stride + row] : 0.0f;
#pragma unroll
        for (int i = 0; i < NF; i++) {
            float v = acc[nt][i];
            if (g.bias) v = v + bias;
            if (g.resid) v = rv[i] + v;
            if (on[i]) g.out[(size_t)orow[i] * g.out_stride + row] = v;
        }
    }
}

template <int WT, int RW, int KS, int NT, bool ALT>
__global__ __launch_bounds__(64 * RW * KS, NT == 1 ? 3 : 2) void k_gemm(GemmArgs g) {
    extern __shared__ __align__(16) uint8_t lds[];
    gemm_body<WT, RW, KS, NT, ALT>(g, (int)blockIdx.x, (int)blockIdx.y, (int)gridDim.x, (int)gridDim.y, lds);
}

// Two GEMMs on the same activations in one launch (a layer's q|k and a v of another type): row tiles [0, gy1) of
// the grid multiply g1, the rest g2.
template <int WT1, int WT2, int RW, int KS>
__global__ __launch_bounds__(64 * RW * KS, 3) void k_gemm_pair(GemmArgs g1, GemmArgs g2, int gy1) {
    extern __shared__ __align__(16) uint8_t lds[];
    if ((int)blockIdx.y < gy1) gemm_body<WT1, RW, KS, 1, false>(g1, (int)blockIdx.x, (int)blockIdx.y, (int)gridDim.x, gy1, lds);
    else gemm_body<WT2, RW, KS, 1, false>(g2, (int)blockIdx.x, (int)blockIdx.y - gy1, (int)gridDim.x, (int)gridDim.y - gy1, lds);
}

// Q8_K rows -> the GEMM's expansion: int8 values, f32 scales and f16 sums in planes of their own (exact: |bsum| <=
// 2032). One thread per 16 values of a super-block (n_sb = n_tok * nb super-blocks in a row); 256 threads.
__global__ __launch_bounds__(256) void k_gemm_prep(const uint8_t *__restrict__ xq, long n_sb, SdyGemmExp e) {
    const long i = blockIdx.x * 256L + threadIdx.x, sbg = i >> 4;
    const int part = (int)(i & 15);
    if (sbg >= n_sb) return;
    const uint8_t *blk = xq + sbg * 292;
    const uint32_t *q = reinterpret_cast<const uint32_t *>(blk + 4 + 16 * part);
    *reinterpret_cast<u32x4 *>(e.y8 + sbg * 256 + 16 * part) = u32x4{q[0], q[1], q[2], q[3]};
    e.bs16[sbg * 16 + part] = (_Float16)(float)reinterpret_cast<const int16_t *>(blk + 260)[part];
    if (part == 0) e.yd[sbg] = *reinterpret_cast<const float *>(blk);
}

// What sdy_mat's gemm_ok says of a K-quant matrix: flags a row super-block whose 127 * sum |sc * q| reaches 2^24 or
// (Q6_K) whose |sc * (q - 32)| exceeds 2048. (The GEMM multiplies either exactly.) One thread per (row,
// super-block) of rows [0, n_rows) of the planes.
template <int WT>
__global__ void k_gemm_check(GemmArgs g, int *bad) {
    const long gid = blockIdx.x * (long)blockDim.x + threadIdx.x;
    const long row = gid / g.nb;
    const int sb = (int)(gid - row * g.nb);
    if (row >= g.n_rows) return;
    long sum = 0;
    int over = 0;
    if constexpr (WT == SDY_Q4_K) {
        const uint8_t *hd = g.p[2] + ((size_t)row * g.nb + sb) * 16 + 4;
        for (int u = 0; u < 4; u++)
            for (int half = 0; half < 2; half++) {
                const uint8_t *qp = g.p[half] + ((size_t)row * g.T + 4 * sb + u) * 16;
                const int j0 = 2 * u, j1 = 2 * u + 1;
                const int s0 = j0 < 4 ? hd[j0] & 63 : (hd[j0 + 4] & 15) | ((hd[j0 - 4] >> 6) << 4);
                const int s1 = j1 < 4 ? hd[j1] & 63 : (hd[j1 + 4] & 15) | ((hd[j1 - 4] >> 6) << 4);
                for (int i = 0; i < 16; i++) sum += (long)s0 * (qp[i] & 15) + (long)s1 * (qp[i] >> 4);
            }
    } else {
        const int8_t *scs = reinterpret_cast<const int8_t *>(g.p[3] + ((size_t)row * g.nb + sb) * 16);
        for (int u = 0; u < 4; u++) {
            const size_t ou = ((size_t)row * g.T + 4 * sb + u) * 16;
            for (int e = 0; e < 64; e++) {
                const int lo = e < 32 ? (g.p[e < 16 ? 0 : 1][ou + (e & 15)] & 15) : (g.p[e < 48 ? 0 : 1][ou + (e & 15)] >> 4);
                const int hi = (g.p[2][ou + (e & 15)] >> (2 * (e >> 4))) & 3;
                const int w = scs[4 * u + (e >> 4)] * ((lo | (hi << 4)) - 32);
                const int aw = w < 0 ? -w : w;
                if (aw > 2048) over = 1;
                sum += aw;
            }
        }
    }
    if (over || 127 * sum >= (1L << 24)) atomicOr(bad, 1);
}

}  // namespace

// =============================================================================== host

// The planes of the tiled copy of a matrix of `rows` rows (tiles of 32 rows: records [tile][unit][32], the
// K-quants' per-super-block records [tile][super-block][32]): offsets, sizes, and each plane's records per row and
// record bytes. Returns the copy's bytes, 0 for types without one.
static size_t gemm_layout_planes(int type, int n_in, long rows, size_t off[5], size_t sz[5], int nrec[5], int rsz[5]) {
    const int T = (n_in + 63) / 64, nb = n_in / 256;
    static const int bytes[5][5] = {
        {16, 16, 16, 0, 0}, {16, 16, 16, 16, 2}, {16, 16, 16, 16, 4}, {16, 16, 0, 0, 4}, {16, 16, 8, 0, 4}};
    int k;  // row of the table
    switch (type) {
    case SDY_Q4_K: k = 0; break;
    case SDY_Q6_K: k = 1; break;
    case SDY_Q8_0: k = 2; break;
    case SDY_Q4_0: k = 3; break;
    case SDY_Q5_0: k = 4; break;
    default: return 0;
    }
    const size_t tiles = (size_t)(rows + 31) / 32;
    size_t o = 0;
    for (int i = 0; i < 5; i++) {
        rsz[i] = bytes[k][i];
        nrec[i] = (k == 0 && i == 2) || (k == 1 && i >= 3) ? nb : T;
        sz[i] = tiles * nrec[i] * 32 * rsz[i];
        off[i] = o;
        o += (sz[i] + 255) & ~(size_t)255;
    }
    return o;
}

extern "C" size_t sdy_gemm_layout_planes(int type, int n_in, long rows, size_t off[5]) {
    size_t sz[5];
    int nrec[5], rsz[5];
    return gemm_layout_planes(type, n_in, rows, off, sz, nrec, rsz);
}

// The kernel arguments of m; with its tiled copy when it has one and `layout` is set.
static GemmArgs gemm_args(const sdy_mat *m, bool layout = false) {
    GemmArgs g;
    memset(&g, 0, sizeof(g));
    for (int i = 0; i < 5; i++) g.p[i] = (const uint8_t *)m->base + m->plane_off[i];
    g.n_in = m->n_in;
    g.T = m->n_units;
    g.nb = m->n_in / 256;
    g.n_rows = m->n_rows;
    if (layout && m->gbase) {
        size_t off[5];
        sdy_gemm_layout_planes(m->type, m->n_in, m->grows, off);
        for (int i = 0; i < 5; i++) g.p[i] = (const uint8_t *)m->gbase + off[i];
        g.blk = 1;
        g.grow0 = m->grow0;
    }
    return g;
}

// Plane record r = row * n_rec + j (rs bytes: 16, 8, 4 or 2) into the tiled copy: [row / 32][j][row % 32].
__global__ __launch_bounds__(256) void k_gemm_layout(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst,
                                                     long n_rows, int n_rec, int rs) {
    const long i = blockIdx.x * 256L + threadIdx.x;
    if (i >= n_rows * (long)n_rec) return;
    const long row = i / n_rec;
    const int j = (int)(i - row * n_rec);
    const size_t o = (((size_t)(row >> 5) * n_rec + j) * 32 + (row & 31)) * rs;
    const uint8_t *r = src + (size_t)i * rs;
    if (rs == 16) *reinterpret_cast<uint4 *>(dst + o) = *reinterpret_cast<const uint4 *>(r);
    else if (rs == 8) *reinterpret_cast<uint2 *>(dst + o) = *reinterpret_cast<const uint2 *>(r);
    else if (rs == 4) *reinterpret_cast<uint32_t *>(dst + o) = *reinterpret_cast<const uint32_t *>(r);
    else *reinterpret_cast<uint16_t *>(dst + o) = *reinterpret_cast<const uint16_t *>(r);
}

// whether m can have a tiled copy: a quantised matrix in device memory (the kernels that multiply many
// tokens read one in host memory in place)
static bool gemm_layout_ok(const sdy_mat *m) {
    if (!m || !m->base || m->hbase) return false;
    if (m->type == SDY_Q4_K || m->type == SDY_Q6_K) return m->gemm_ok != 0;
    return m->type == SDY_Q8_0 || m->type == SDY_Q4_0 || m->type == SDY_Q5_0;
}

extern "C" size_t sdy_mat_gemm_layout_bytes(const sdy_mat *m) {
    if (!gemm_layout_ok(m) || m->gbase) return 0;
    size_t off[5];
    return sdy_gemm_layout_planes(m->type, m->n_in, m->n_rows, off);
}

extern "C" int sdy_mat_gemm_layout(sdy_mat *m, sdy_stream s) {
    if (!gemm_layout_ok(m)) return 0;
    if (m->grow0 != 0 || (m->gbase && m->grows != m->n_rows))
        return sdy_fail(-1, "gemm_layout: made for a whole matrix, not a row view");
    size_t off[5], sz[5];
    int nrec[5], rsz[5];
    const size_t bytes = gemm_layout_planes(m->type, m->n_in, m->n_rows, off, sz, nrec, rsz);
    int rc;
    if (!m->gbase) {
        if ((rc = sdy_malloc(&m->gbase, bytes))) return rc;
        m->gbytes = bytes;
        m->grows = m->n_rows;
        // the padding rows of the last tile: zero (never read: the kernels clamp their rows)
        if ((rc = sdy_memset(m->gbase, 0, bytes, s))) return rc;
    }
    for (int i = 0; i < 5; i++) {
        if (!sz[i]) continue;
        const long total = m->n_rows * (long)nrec[i];
        SDY_NOTE_KERNEL(k_gemm_layout);
        hipLaunchKernelGGL(k_gemm_layout, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)s,
                           (const uint8_t *)m->base + m->plane_off[i], (uint8_t *)m->gbase + off[i], m->n_rows,
                           nrec[i], rsz[i]);
        if ((rc = sdy_check_launch("gemm_layout"))) return rc;
    }
    return 0;
}

// Flags (bad = 1) rows [r0, r0 + n) of m with a block of gemm_ok 2. Synchronous.
extern "C" int sdy_gemm_check_rows_async(const sdy_mat *m, long r0, long n, int *bad_dev, sdy_stream s) {
    if ((m->type != SDY_Q4_K && m->type != SDY_Q6_K) || m->hbase) return 0;  // (host memory: unchecked)
    sdy_mat v = sdy_mat_rows(m, r0, n);
    GemmArgs g = gemm_args(&v);
    const long total = n * (long)g.nb;
    dim3 grid((unsigned)((total + 255) / 256));
    if (m->type == SDY_Q4_K) hipLaunchKernelGGL(k_gemm_check<SDY_Q4_K>, grid, dim3(256), 0, (hipStream_t)s, g, bad_dev);
    else hipLaunchKernelGGL(k_gemm_check<SDY_Q6_K>, grid, dim3(256), 0, (hipStream_t)s, g, bad_dev);
    return sdy_check_launch("gemm_check");
}

extern "C" int sdy_gemm_check_rows(const sdy_mat *m, long r0, long n, int *bad_host, sdy_stream s) {
    *bad_host = 1;
    if ((m->type != SDY_Q4_K && m->type != SDY_Q6_K) || m->hbase) return 0;
    sdy_mat v = sdy_mat_rows(m, r0, n);
    GemmArgs g = gemm_args(&v);
    int *bad = nullptr, rc;
    if ((rc = sdy_malloc((void **)&bad, sizeof(int)))) return rc;
    if ((rc = sdy_memset(bad, 0, sizeof(int), s))) {
        sdy_free(bad);
        return rc;
    }
    const long total = n * (long)g.nb;
    dim3 grid((unsigned)((total + 255) / 256));
    if (m->type == SDY_Q4_K) hipLaunchKernelGGL(k_gemm_check<SDY_Q4_K>, grid, dim3(256), 0, (hipStream_t)s, g, bad);
    else hipLaunchKernelGGL(k_gemm_check<SDY_Q6_K>, grid, dim3(256), 0, (hipStream_t)s, g, bad);
    if (!(rc = sdy_check_launch("gemm_check")) && !(rc = sdy_d2h(bad_host, bad, sizeof(int), s))) rc = sdy_sync(s);
    sdy_free(bad);
    return rc;
}

extern "C" size_t sdy_gemm_ws_bytes(int n_tok, int n_in) {
    const size_t nb = (size_t)n_in / 256;
    return (size_t)n_tok * n_in + (size_t)n_tok * nb * 4 + (size_t)n_tok * nb * 32 + 3 * 256;
}

extern "C" int sdy_gemm_ok(const sdy_mat *m, int n_tok) {
    return (m->type == SDY_Q4_K || m->type == SDY_Q6_K) && m->gemm_ok && n_tok >= 2 &&
           (size_t)m->n_rows * m->n_units * 16 < 0xFFFFFFFFu;
}

// A Q4_K lane reaches both quant planes by one 32-bit offset from its row tile in the first, but where a plane ends just
// short of 4 GiB (the most sdy_gemm_ok takes): the ALT form.
static bool gemm_far(const GemmArgs &g) { return (size_t)(g.p[1] - g.p[0]) + (size_t)g.T * 4096 > 0xFFFFFFFFu; }

template <int WT, int RW, int KS, int NT = 1, bool ALT = false>
static int launch_gemm(const GemmArgs &g, unsigned tok_tiles, hipStream_t st) {
    constexpr size_t lds = gemm_lds_bytes<RW, KS, NT>();
    static size_t granted = 0;
    if (int rc = sdy_lds_limit((const void *)k_gemm<WT, RW, KS, NT, ALT>, lds, &granted)) return rc;
    SDY_NOTE_KERNEL((k_gemm<WT, RW, KS, NT, ALT>));
    hipLaunchKernelGGL((k_gemm<WT, RW, KS, NT, ALT>), dim3((tok_tiles + NT - 1) / NT, (unsigned)((g.n_rows + 32 * RW - 1) / (32 * RW))),
                       dim3(64 * RW * KS), lds, st, g);
    return sdy_check_launch("gemm");
}

// The forms of the GEMM: the 16 x 16 tiles of mm_superblocks.hip (0); 32 x 32 tiles, a tile's super-blocks over four waves
// (4), two (2) or one (1); and one wave to two token tiles (12), which unpacks the weights once for 64 tokens with two
// waves to a SIMD instead of three. All give the same bits, so they are chosen by size and by whether the weights come
// from the tiled copy. By the 32 x 32 tiles: four waves while these alone are fewer than two to a CU, two up to eight, one
// beyond (Q4_K 2048 x 2048, 130 tokens: 11.8, 13.6, 17.3 us; 512 tokens: 21.2, 18.5, 19.1; 22016 x 2048, 64 tokens: 27.0,
// 20.8, 22.6; 128 tokens: 47.4, 33.4, 29.0; with the quantiser's launch). Beside that (rows x inputs, without it):
// - Small grids: the 16 x 16 tiles, up to 2.5 to a CU and up to 16 tokens on more rows (Q4_K 2560 x 2048, 64 tokens: 10.0
//   against 11.4, 128 tokens 12.7 against 11.8; 22016 x 2048, 16 tokens 12.2 against 16.1).
// - Rows too short to split (Q4_K to two super-blocks, Q6_K to three): the 16 x 16 tiles further, then two waves, then one
//   (Q6_K 4096 x 768, 64 tokens: 6.3 us, with four waves 8.4; 8192 x 768, 96 tokens: one wave 10.4, two 10.9; 4096 x 256, 96 tokens:
//   5.5, two waves 6.7; Q4_K 4096 x 512, 96 tokens: 5.5, two 6.0; Q6_K 8192 x 512, 160 tokens: two 9.7, one 11.2, 256: 12.7, 11.8).
// - Q6_K on large grids: two token tiles, half the unpacking of 6 bits (32768 x 2048, 512 tokens: 183 -> 160 us; 256: 95 -> 85),
//   from four workgroups to a CU, six on shorter rows (147456 x 1024, 128 tokens: 110 -> 106; 22016 x 768, 512 tokens 55.0
//   against 59.9), where the last pair of tiles is whole or one of several (65536 x 2048, 96 tokens: 72 against 84). Q4_K's
//   nibbles cost less than the third wave (22016 x 2048, 512 tokens: 70.4 against 83.9).
// - From the planes, where a wave's load of 32 rows' units meets as many cache lines: two token tiles as soon as they
//   fill the chip (22016 x 2048, 512 tokens: Q6_K 176 -> 131 us, with whole records loaded 120; Q4_K 107 -> 89), two waves
//   before (Q4_K 22016 x 8192, 96 tokens: 111 -> 82).
static int gemm_form(const sdy_mat *m, long n_rows, int n_tok) {
    const int nb = m->n_in / 256;
    const bool q4 = m->type == SDY_Q4_K, tiled = m->gbase != nullptr, few = nb <= (q4 ? 2 : tiled ? 3 : 4);
    const long t16 = (n_rows + 15) / 16 * ((n_tok + 15) / 16), t32 = (n_rows + 31) / 32 * ((n_tok + 31) / 32);
    const long wide = (n_rows + 127) / 128 * ((n_tok + 63) / 64);
    const long line = few ? (nb == 1 ? (q4 ? 3072 : 2560) : q4 ? 1408 : 1024) : tiled ? 640 : 512;
    // (host memory: a row's token tiles read it together only where they run on one XCD, not as 16 x 16 tiles)
    if (m->hbase ? n_tok <= 16 : t16 <= line || (n_tok <= 16 && t16 <= (q4 && (tiled || few) ? 4096 : 1024))) return 0;
    if (few && (tiled || q4 || t32 < 2048)) {
        const long two = nb == 2 && (tiled || q4) ? (tiled ? 1536 : 2048) : q4 ? 1024 : 513;
        return t32 < two ? 2 : 1;
    }
    if (!tiled) return t32 < 512 ? 4 : t32 < (q4 ? 4096 : 2048) ? 2 : 12;
    const int tt = (n_tok + 31) / 32;
    if (!q4 && (wide >= 1536 ? nb >= 4 : wide >= 1024 && nb >= 6) && (tt % 2 == 0 || tt > 8)) return 12;
    return t32 < 512 ? 4 : t32 < 2048 ? 2 : 1;
}

template <int WT, bool ALT>
static int launch_form(const GemmArgs &g, int form, unsigned tok_tiles, hipStream_t st) {
    if (form == 12) return launch_gemm<WT, 4, 1, 2, ALT>(g, tok_tiles, st);
    if (form == 4) return launch_gemm<WT, 2, 4, 1, ALT>(g, tok_tiles, st);
    return form == 2 ? launch_gemm<WT, 2, 2, 1, ALT>(g, tok_tiles, st) : launch_gemm<WT, 4, 1, 1, ALT>(g, tok_tiles, st);
}

template <int WT>
static int gemm_type(const GemmArgs &g, const sdy_mat *m, const sdy_mv_args *a, hipStream_t st) {
    // SARDYNE_GEMM_VARIANT picks one form (tests and tuning): 11, 12, 13: one, two, four waves; 14: 16 x 16 tiles; 15: two
    // token tiles. Default: by shape
    const char *ev = getenv("SARDYNE_GEMM_VARIANT");
    const int variant = ev ? atoi(ev) : 0;
    static const int forms[] = {1, 2, 4, 0, 12};
    int form = variant >= 11 && variant <= 15 ? forms[variant - 11] : gemm_form(m, g.n_rows, g.n_tok);
    const unsigned tt = (unsigned)((g.n_tok + 31) / 32);
    if (form == 0) {
        const int rc = sdy_mm_superblocks_exp(m, a, &g.e, (sdy_stream)st);
        if (rc <= 0) return rc;
        form = 4;
    }
    if (WT == SDY_Q6_K && !g.blk) return launch_form<WT, WT == SDY_Q6_K>(g, form, tt, st);
    return launch_form<WT, false>(g, form, tt, st);
}

// The activations' expansion of one call in ws: made unless ws_ready.
static int gemm_expand(const sdy_mv_args *a, int rows, int n_in, void *ws, SdyGemmExp &e, hipStream_t st) {
    e = sdy_gemm_exp(ws, rows, n_in);
    if (a->ws_ready) return 0;
    const long n_sb = (long)rows * (n_in / 256);
    SDY_NOTE_KERNEL(k_gemm_prep);
    hipLaunchKernelGGL(k_gemm_prep, dim3((unsigned)((n_sb * 16 + 255) / 256)), dim3(256), 0, st, (const uint8_t *)a->xq, n_sb, e);
    return sdy_check_launch("gemm_prep");
}

// The checks and kernel arguments of one sdy_gemm call; the activations' expansion is made first
// unless ws_ready. *empty: an empty row range (nothing to launch).
static int gemm_setup(const sdy_mat *m, const sdy_mv_args *a, void *ws, hipStream_t st, GemmArgs &g, bool *empty) {
    *empty = false;
    if (!sdy_gemm_ok(m, a->n_tok)) return sdy_fail(-1, "gemm: matrix not eligible (type %d)", m->type);
    if (a->row0 < 0 || a->row1 > m->n_rows || a->row0 > a->row1)
        return sdy_fail(-1, "gemm rows [%ld, %ld) outside %ld", a->row0, a->row1, m->n_rows);
    if (a->epilogue == SDY_EPI_SWIGLU && (((a->row1 - a->row0) | a->row0) & 1 || a->bias || a->resid))
        return sdy_fail(-1, "gemm: the SwiGLU epilogue needs an even row range from an even row, no bias, no residual");
    if (a->row0 == a->row1) {
        *empty = true;
        return 0;
    }
    g = gemm_args(m, true);
    if (int rc = gemm_expand(a, a->n_tok, g.n_in, ws, g.e, st)) return rc;
    g.row0 = a->row0;
    g.n_rows = a->row1 - a->row0;
    g.n_tok = a->n_tok;
    g.out = a->out;
    g.out_stride = a->out_stride;
    g.bias = a->bias;
    g.resid = a->resid;
    g.swiglu = a->epilogue == SDY_EPI_SWIGLU;
    // with a row range the outputs are indexed by row - row0 only for SwiGLU (as in the matvec)
    return 0;
}

// out[t][row] for rows [a->row0, a->row1) and a->n_tok tokens of Q8_K activations a->xq; ws:
// sdy_gemm_ws_bytes(n_tok, n_in) bytes of device scratch.
extern "C" int sdy_gemm(const sdy_mat *m, const sdy_mv_args *a, void *ws, sdy_stream s) {
    hipStream_t st = (hipStream_t)s;
    GemmArgs g;
    bool empty;
    if (int rc = gemm_setup(m, a, ws, st, g, &empty)) return rc;
    if (empty) return 0;
    if (m->type == SDY_Q4_K && gemm_far(g)) return launch_gemm<SDY_Q4_K, 4, 1, 1, true>(g, (unsigned)((g.n_tok + 31) / 32), st);
    return m->type == SDY_Q4_K ? gemm_type<SDY_Q4_K>(g, m, a, st) : gemm_type<SDY_Q6_K>(g, m, a, st);
}

template <int RW, int KS>
static int launch_gemm_pair(const GemmArgs &g1, const GemmArgs &g2, hipStream_t st) {
    constexpr size_t lds = gemm_lds_bytes<RW, KS, 1>();
    static size_t granted = 0;
    if (int rc = sdy_lds_limit((const void *)k_gemm_pair<SDY_Q4_K, SDY_Q6_K, RW, KS>, lds, &granted)) return rc;
    const int gy1 = (int)((g1.n_rows + 32 * RW - 1) / (32 * RW)), gy2 = (int)((g2.n_rows + 32 * RW - 1) / (32 * RW));
    SDY_NOTE_KERNEL((k_gemm_pair<SDY_Q4_K, SDY_Q6_K, RW, KS>));
    hipLaunchKernelGGL((k_gemm_pair<SDY_Q4_K, SDY_Q6_K, RW, KS>), dim3((unsigned)((g1.n_tok + 31) / 32), (unsigned)(gy1 + gy2)),
                       dim3(64 * RW * KS), lds, st, g1, g2, gy1);
    return sdy_check_launch("gemm2");
}

// Two GEMMs over the same activations (a layer's q|k and its v): one launch, on the forms of four waves or two (rows of one
// or two super-blocks: the 16 x 16 tiles), when the first matrix is Q4_K and the second Q6_K and neither would fill the GPU
// by itself; otherwise, or with SARDYNE_GEMM_VARIANT set, two sdy_gemm calls. The same bits either way.
extern "C" int sdy_gemm2(const sdy_mat *m1, const sdy_mv_args *a1, const sdy_mat *m2, const sdy_mv_args *a2, void *ws,
                         sdy_stream s) {
    hipStream_t st = (hipStream_t)s;
    if (a2->xq != a1->xq || a2->n_tok != a1->n_tok || m2->n_in != m1->n_in)
        return sdy_fail(-1, "gemm2: the two GEMMs must read the same activation rows");
    const long rows = (a1->row1 - a1->row0) + (a2->row1 - a2->row0), tiles = (rows + 31) / 32 * ((a1->n_tok + 31) / 32);
    const bool pair = m1->type == SDY_Q4_K && m2->type == SDY_Q6_K && !getenv("SARDYNE_GEMM_VARIANT") &&
                      a1->row1 > a1->row0 && a2->row1 > a2->row0 && tiles < 2048;
    sdy_mv_args b = *a2;
    b.ws_ready = 1;  // the expansion the first call makes (or finds)
    if (!pair) {
        if (int rc = sdy_gemm(m1, a1, ws, s)) return rc;
        return sdy_gemm(m2, &b, ws, s);
    }
    GemmArgs g1, g2;
    bool e1, e2;
    if (int rc = gemm_setup(m1, a1, ws, st, g1, &e1)) return rc;  // (both ranges non-empty here)
    if (int rc = gemm_setup(m2, &b, ws, st, g2, &e2)) return rc;
    if (gemm_far(g1)) {
        sdy_mv_args a = *a1;
        a.ws_ready = 1;
        if (int rc = sdy_gemm(m1, &a, ws, s)) return rc;
        return sdy_gemm(m2, &b, ws, s);
    }
    // (384 + 128 rows x 256, 64 tokens: 3.5 us, four waves to a tile 7.4; 768 + 256 x 512: 3.8 against 6.6)
    if (g1.nb <= 2 && (rows + 30) / 16 * ((a1->n_tok + 15) / 16) <= 1408) {
        const int rc = sdy_mm_superblocks_exp2(m1, a1, m2, &b, &g1.e, s);
        if (rc <= 0) return rc;
    }
    return tiles < 512 ? launch_gemm_pair<2, 4>(g1, g2, st) : launch_gemm_pair<2, 2>(g1, g2, st);
}

extern "C" int sdy_gemm_grouped_tile(void) { return 32; }

extern "C" int sdy_gemm_grouped(const sdy_mat *m, long grp_rows, int n_grp, const int *grp_tok, const int *grp_tile,
                                const int *out_row, const int *act_row, int n_act, const sdy_mv_args *a, void *ws,
                                sdy_stream s) {
    hipStream_t st = (hipStream_t)s;
    const int n_tok = a->n_tok;
    if (n_tok <= 0) return 0;
    if (!((m->type == SDY_Q4_K || m->type == SDY_Q6_K) && m->gemm_ok &&
          (size_t)m->n_rows * m->n_units * 16 < 0xFFFFFFFFu))
        return sdy_fail(-1, "gemm_grouped: matrix not eligible (type %d)", m->type);
    if (n_grp < 1 || grp_rows < 1 || (long)n_grp * grp_rows > m->n_rows)
        return sdy_fail(-1, "gemm_grouped: %d groups of %ld rows in %ld rows", n_grp, grp_rows, m->n_rows);
    if (a->bias || a->resid || (a->epilogue == SDY_EPI_SWIGLU && (grp_rows & 1)))
        return sdy_fail(-1, "gemm_grouped: no bias or residual; the SwiGLU epilogue needs an even row count per group");
    if (act_row && (!a->ws_ready || n_act < 1))
        return sdy_fail(-1, "gemm_grouped: activation rows by index read an expansion of n_act >= 1 rows that the "
                            "caller made (ws_ready)");
    GemmArgs g = gemm_args(m, true);
    if (int rc = gemm_expand(a, act_row ? n_act : n_tok, g.n_in, ws, g.e, st)) return rc;
    g.row0 = 0;
    g.n_rows = grp_rows;
    g.n_tok = n_tok;
    g.out = a->out;
    g.out_stride = a->out_stride;
    g.bias = a->bias;
    g.resid = a->resid;
    g.swiglu = a->epilogue == SDY_EPI_SWIGLU;
    g.grp_tile = grp_tile;
    g.grp_tok = grp_tok;
    g.out_row = out_row;
    g.act_row = act_row;
    g.grp_rows = grp_rows;
    g.n_grp = n_grp;
    // token tiles: at most one partial tile per group beyond the full ones (the grid's extra workgroups return at once)
    const unsigned tok_tiles = (unsigned)((n_tok + 31) / 32 + n_grp - 1);
    if (m->type == SDY_Q4_K && gemm_far(g)) return launch_gemm<SDY_Q4_K, 4, 1, 1, true>(g, tok_tiles, st);
    const char *ev = getenv("SARDYNE_GEMM_VARIANT");
    const int v = ev ? atoi(ev) : 0;
    // One wave to a row tile; from the planes, whose loads take longer, two where rows have eight super-blocks for them (128
    // groups of 1536 rows x 2048, 512 tokens: Q4_K 71 -> 62 us, Q6_K 107 -> 99; 32 tokens 28 -> 19 and 37 -> 24)
    const int form = v ? (v == 12 ? 2 : v == 13 ? 4 : 1) : !g.blk && !m->hbase && g.nb >= 8 ? 2 : 1;
    if (m->type == SDY_Q4_K) return launch_form<SDY_Q4_K, false>(g, form, tok_tiles, st);
    return g.blk ? launch_form<SDY_Q6_K, false>(g, form, tok_tiles, st) : launch_form<SDY_Q6_K, true>(g, form, tok_tiles, st);
}

// Several tokens of Q8_0 / Q4_0 / Q5_0 weights on the int8 matrix cores.
//
// A 32-element block contributes (float)isum * (dw * dx), isum the exact int32 dot of its quants with the
// token's Q8_0 quants (csrc/quant.c:148-189). v_mfma_i32_32x32x32_i8 multiplies one block of 32 rows
// with 32 tokens: its K = 32 is the block, so its result is isum itself. The scale products dw * dx of the
// tile are an outer product: one f16 matrix instruction with the two scales in its first k-slot and zeros
// in the others (exact: a product of two 11-bit significands in f32, subnormal scales included). The
// sum over blocks is one conversion and one fma per block and output, in f32.
//
// What bounds it: per 32 x 32 x 32 products the VALU's 32 instructions take 128 cycles, beside them the matrix
// cores' two instructions 64. (The f32 outer product on v_mfma_f32_32x32x1 does not run beside VALU work.) At
// 22016 x 2048 and 512 tokens, 46 GFLOP: 2213 us on the 8-token matvec before, 121 us now, the VALU busy in 50 % of
// the cycles; a wave waits 27 % of its time for data and barriers, 21 % for its turn to issue, at two waves per SIMD.
// Up to 32 tokens it is the weights' stream, a stage's latency per 128 inputs of a wave: 22016 x 2048 (46 MB) with 8
// tokens 32.1 -> 16.2 us, 11008 x 2048 62 -> 29.5, 2048 x 2048 15.2 -> 12.3.
#include <hip/hip_runtime.h>

#include "sdy_device.h"
#include "sdy_internal.h"
#include "sdy_quant_dev.h"
#include "sdy_shim.h"

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

struct MmArgs {
    const uint8_t *p[5];  // planes (quant_kernels.hip), or the tiled copy's (blk, grow0)
    int nb, T;            // 32-element blocks and 64-element units per row
    int blk;              // records [row / 32][unit][row % 32] instead of [row][unit]; row r is row grow0 + r there
    long grow0;
    long row0, n_rows;
    const uint8_t *xq;    // Q8_0 rows, nb blocks of 34 bytes (2-byte aligned)
    uint32_t xoff;        // bytes from xq (4-byte aligned) to the first row: 0 or 2
    int n_tok;
    float *out;
    long out_stride;
    const float *bias, *resid;
    int swiglu;
};

SDY_DEV __amdgpu_buffer_rsrc_t rsrc(const uint8_t *p) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, (short)0, -1, 0x00020000);
}

// The int8 quants of a lane's half block (k-half h) from its 16 raw bytes: Q4_0 q - 8 and Q5_0 q - 16,
// q the low nibbles for h = 0, the high ones for h = 1 (Q5_0: and bits 16 h .. 16 h + 15 of qh).
// q - z per byte: ((q | 0x80) - z) ^ 0x80 borrows from no other byte.
template <int WT>
SDY_DEV i32x4 quants(u32x4 raw, uint32_t qh, int h) {
    if constexpr (WT == SDY_Q8_0) {
        return __builtin_bit_cast(i32x4, raw);
    } else {
        constexpr uint32_t Z = WT == SDY_Q4_0 ? 0x08080808u : 0x10101010u;
        u32x4 v = (raw >> (unsigned)(4 * h)) & 0x0F0F0F0Fu;
        if constexpr (WT == SDY_Q5_0) {
            const uint32_t q = qh >> (16 * h);
            v |= u32x4{sdy_spread4(q), sdy_spread4(q >> 4), sdy_spread4(q >> 8), sdy_spread4(q >> 12)};
        }
        return __builtin_bit_cast(i32x4, ((v | 0x80808080u) - Z) ^ 0x80808080u);
    }
}

// A workgroup of RW * KS waves computes 32 RW rows x 32 NT tokens; a wave owns 32 rows and all the
// tokens and, with KS > 1, every KS-th group of 4 blocks (the KS partial sums are added through
// LDS at the end: for few tokens the waves of a matrix' rows would otherwise be too few to keep HBM
// busy). The weights go straight to registers, each lane (row lr, k-half h) loading its own 16-byte
// records: from the tiled copy a load instruction reads two runs of 512 bytes, from the row-major planes 64
// records of 16 bytes (the fallback where there is no copy). The activations are shared through
// LDS in stages of 4 KS blocks, requested a stage ahead, 16-byte chunk c of token t at slot
// c ^ (t / 2 % 8): the 16 tokens of a quarter of the wave's read of one chunk then hit all 64 banks once (a
// row is 32 banks or a multiple of it; with t % 8 the reads took 1.6 times as long). Blocks past the row's end
// are read from its last ones and count with scale 0.
template <int WT, int RW, int KS, int NT>
__global__ __launch_bounds__(64 * RW * KS, 2) void k_mm_blocks(MmArgs g) {
    constexpr int NTH = 64 * RW * KS, NB = 4;  // threads, a wave's blocks of a stage
    constexpr int BM = 32 * RW, BN = 32 * NT, SB = NB * KS;  // rows, tokens, blocks of a stage
    constexpr bool Q8 = WT == SDY_Q8_0;
    constexpr int NA = BN * 2 * SB / NTH;                   // activation chunks per thread
    static_assert(BN * 2 * SB % NTH == 0 && (BN * SB % NTH == 0 || BN * SB < NTH), "whole chunks per thread");
    constexpr int NX = (BN * SB + NTH - 1) / NTH;
    constexpr int OFF_X = BN * 2 * SB * 16, STAGE = OFF_X + 2 * BN * SB * 4;
    constexpr int RED = KS > 1 ? RW * KS * NT * 16 * 64 * 4 : 0;
    __shared__ __align__(16) uint8_t lds[2 * STAGE > RED ? 2 * STAGE : RED];
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, lr = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = wave % KS, rw = wave / KS;
    // token tiles of a row tile on one XCD (workgroups are dealt to the 8 XCDs in turn)
    const long n_tt = gridDim.x, n_rt = gridDim.y, L = (long)blockIdx.y * n_tt + blockIdx.x;
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
    const int t0 = (int)tti * BN;
    const int nb = g.nb, T = g.T, ns = (nb + SB - 1) / SB;

    // the lane's row: its first record, and the records from one unit to the next
    const long ri = rti * BM + 32 * rw + lr, row = g.row0 + ri;
    const long rc = g.row0 + (ri < g.n_rows ? ri : g.n_rows - 1);
    const uint32_t R = (uint32_t)(g.grow0 + rc);
    const uint32_t rec0 = g.blk ? (R >> 5) * (uint32_t)T * 32u + (R & 31u) : (uint32_t)rc * (uint32_t)T;
    const uint32_t us = g.blk ? 32u : 1u;
    const uint32_t ho[2] = {Q8 && h ? (uint32_t)(g.p[1] - g.p[0]) : 0u, Q8 && h ? (uint32_t)(g.p[3] - g.p[2]) : 0u};
    // the wave's NB blocks of the next WS stages, each reloaded WS stages ahead as it is multiplied (two where
    // the registers allow it: with one wave per SIMD a stage is shorter than a round trip to memory)
    constexpr int WS = NT == 2 ? 1 : 2;
    u32x4 wq[WS][NB];
    uint32_t wd[WS][NB / 2];
    uint2 wh[WS][WT == SDY_Q5_0 ? NB / 2 : 1];
    // buffer loads: the lane's offsets are fixed, a unit's is scalar
    const __amdgpu_buffer_rsrc_t r0 = rsrc(g.p[0]), r1 = rsrc(Q8 ? g.p[2] : g.p[1]), rd = rsrc(g.p[4]), rh = rsrc(g.p[2]);
    const uint32_t vq[2] = {ho[0] + rec0 * 16u, ho[1] + rec0 * 16u}, vd = rec0 * 4u;
    auto unit_of = [&](int s, int j) {  // records to the wave's unit j (blocks 2j, 2j + 1) of stage s
        const int u = (s * SB + NB * ks) / 2 + j;
        return (u < T ? u : T - 1) * (int)us;
    };
    auto load_wq = [&](int s, int z, int b) {
        wq[z][b] = __builtin_amdgcn_raw_buffer_load_b128((b & 1) ? r1 : r0, vq[b & 1], unit_of(s, b >> 1) * 16, 0);
    };
    auto load_wd = [&](int s, int z, int j) {
        wd[z][j] = __builtin_amdgcn_raw_buffer_load_b32(rd, vd, unit_of(s, j) * 4, 0);
        if constexpr (WT == SDY_Q5_0) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(rh, 2 * vd, unit_of(s, j) * 8, 0);
            wh[z][j] = make_uint2(v[0], v[1]);
        }
    };
    // this thread's share of a stage's activations: its chunk and block do not change
    const int ac = tid % (2 * SB), xblk = tid % SB, at0 = tid / (2 * SB), xt0 = tid / SB % BN;
    constexpr int AS = NTH / 2 / SB, XS = NTH / SB;  // tokens between a thread's chunks
    // (fewer scales than threads: the threads past them repeat one, with the same value)
    const uint32_t arow = (uint32_t)nb * 34u;
    auto tok_of = [&](int t) { return (uint32_t)(t0 + t < g.n_tok ? t0 + t : g.n_tok - 1); };
    uint32_t ao[NA], xo[NX];
#pragma unroll
    for (int i = 0; i < NA; i++) ao[i] = tok_of(at0 + AS * i) * arow + g.xoff + 2u + 16u * (uint32_t)(tid & 1);
#pragma unroll
    for (int i = 0; i < NX; i++) xo[i] = tok_of(xt0 + XS * i) * arow + g.xoff;
    // A block's quants start at a multiple of 2 bytes: the 16 bytes at a are read as 4 dwords from a rounded
    // down to 4 and the last 2 bytes, and shifted into place as they go to LDS (a 16-byte load at 2 bytes'
    // alignment is served lane by lane).
    u32x4 av[NA];
    uint16_t al[NA], xv[NX];
    uint32_t ash = 0;
    auto load_a = [&](int s) {
        const int b0 = s * SB;
        const uint32_t ab = 34u * (uint32_t)(b0 + (ac >> 1) < nb ? b0 + (ac >> 1) : nb - 1);
        const uint32_t xb = 34u * (uint32_t)(b0 + xblk < nb ? b0 + xblk : nb - 1);
#pragma unroll
        for (int i = 0; i < NA; i++) {
            const uint32_t o = ao[i] + ab;
            av[i] = *reinterpret_cast<const u32x4 *>(g.xq + (o & ~3u));
            al[i] = *reinterpret_cast<const uint16_t *>(g.xq + (o + 14u));
        }
        ash = ab;
#pragma unroll
        for (int i = 0; i < NX; i++) xv[i] = *reinterpret_cast<const uint16_t *>(g.xq + (xo[i] + xb));
    };
    auto store_a = [&](int s, uint8_t *buf) {
#pragma unroll
        for (int i = 0; i < NA; i++) {
            const int t = at0 + AS * i;
            const uint32_t sh = 8u * ((ao[i] + ash) & 2u);
            const u32x4 v = av[i];
            const u32x4 w = {__builtin_amdgcn_alignbit(v.y, v.x, sh), __builtin_amdgcn_alignbit(v.z, v.y, sh),
                             __builtin_amdgcn_alignbit(v.w, v.z, sh), __builtin_amdgcn_alignbit((uint32_t)al[i], v.w, sh)};
            *reinterpret_cast<u32x4 *>(buf + 16 * (at0 * 2 * SB + AS * 2 * SB * i + (ac ^ (t >> 1 & 7)))) = w;
        }
        uint32_t *xl = reinterpret_cast<uint32_t *>(buf + OFF_X) + xblk * BN + xt0;
#pragma unroll
        for (int i = 0; i < NX; i++) {
            xl[XS * i] = s * SB + xblk < nb ? xv[i] : 0u;
            xl[BN * SB + XS * i] = 0u;
        }
    };

    float acc[NT][16];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[nt][i] = 0.0f;
    // The work of a stage in steps of two products of 32 x 32 outputs and their scales: a block of two
    // token tiles, or two blocks of one. A step's products are issued before the previous step's are
    // folded into the sums, so that the matrix cores and the VALU work side by side, and its activation
    // fragments are read a step ahead.
    constexpr int NST = NT == 2 ? NB : NB / 2, BP = NT == 2 ? 1 : 2;  // steps, blocks of one
    struct Frag {
        i32x4 a[2];
        uint32_t x[2];  // the tokens' scales in k-slot 0 (lane half 1: zeros)
    };
    auto read_f = [&](const uint8_t *buf, int st, Frag &f) {
        const uint32_t *xl = reinterpret_cast<const uint32_t *>(buf + OFF_X) + (NB * ks + BP * st) * BN + lr + h * (BN * SB);
#pragma unroll
        for (int j = 0; j < 2; j++) {
            f.x[j] = xl[NT == 2 ? 32 * j : BN * j];
            const int c = 2 * (NB * ks + BP * st + (NT == 2 ? 0 : j)) + h, t = lr + (NT == 2 ? 32 * j : 0);
            f.a[j] = *reinterpret_cast<const i32x4 *>(buf + (t * 2 * SB + (c ^ (lr >> 1 & 7))) * 16);
        }
    };
    i32x16 prod[2];
    f32x16 scale[2][2];
    const uint32_t hmask = h ? 0u : 0xFFFFu;
    auto slot0 = [](uint32_t v) { return __builtin_bit_cast(f16x4, u32x2{v, 0u}); };
    // the products j of step st of stage s (weight set z), and the reload of its weights for stage s + WS
    auto issue = [&](int s, int z, int st, int j, const Frag &f, f32x16 &sc) {
        const int b = BP * st + (NT == 2 ? 0 : j);
        const uint32_t d = (b & 1) ? wd[z][b >> 1] >> 16 : wd[z][b >> 1];
        // (a block past the row's end: scale 0)
        sc = __builtin_amdgcn_mfma_f32_32x32x8f16(slot0(f.x[j]), slot0(d & (s * SB + NB * ks + b < nb ? hmask : 0u)), f32x16{}, 0, 0, 0);
        const uint32_t qh = WT == SDY_Q5_0 ? ((b & 1) ? wh[z][b >> 1].y : wh[z][b >> 1].x) : 0u;
        prod[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.a[j], quants<WT>(wq[z][b], qh, h), i32x16{}, 0, 0, 0);
        if (NT == 1 || j == 1) load_wq(s + WS, z, b);
        if (j == 1 && (b & 1)) load_wd(s + WS, z, b >> 1);
    };
    // The sums in two levels (the blocks of two stages, then those sums): the rounding error of a row of 64 blocks
    // is half of one chain's. Against 64 bits (relative, with the KS split): 7.29e-8 at 2048 inputs, 7.78e-8 at 4096,
    // 9.3e-8 at 11008 (64 tokens; 1.08e-7 from 256, on two waves); the one-token kernel, a tree up to 4096 inputs where
    // 64 units divide among the lanes and a chain elsewhere: 7.16e-8, 7.66e-8 and 2.41e-7 (1.0e-7 at 1536, 1.5e-7 at
    // 4000). So against the tree it is 2 to 3 % more (at most 5 % by the partial sums' sizes), against the chain half
    // or less.
    float part[NT][16];
    auto fold = [&](int j, const f32x16 &sc, bool first) {
        const int t = NT == 2 ? j : 0;
#pragma unroll
        for (int i = 0; i < 16; i++)
            part[t][i] = first ? (float)prod[j][i] * sc[i] : __builtin_fmaf((float)prod[j][i], sc[i], part[t][i]);
    };
    auto add_part = [&](int t) {
#pragma unroll
        for (int i = 0; i < 16; i++) acc[t][i] += part[t][i];
    };
    // orders LDS only: the weights in flight stay in flight
    auto barrier = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    Frag F[2];
    load_a(0);
#pragma unroll
    for (int z = 0; z < WS; z++) {
#pragma unroll
        for (int b = 0; b < NB; b++) load_wq(z, z, b);
#pragma unroll
        for (int j = 0; j < NB / 2; j++) load_wd(z, z, j);
    }
    store_a(0, lds);
    barrier();
    read_f(lds, 0, F[0]);
    issue(0, 0, 0, 0, F[0], scale[0][0]);
    issue(0, 0, 0, 1, F[0], scale[0][1]);
    // A step folds the previous step's products as it issues its own into their registers. (Past the last
    // stage the loads are clamped and the scales zero.)
    static_assert(NST % 2 == 0, "the steps' buffers alternate over the stages");
    auto stage = [&](int s, int z) {
        uint8_t *buf = lds + z * STAGE, *nbuf = lds + (1 - z) * STAGE;
        load_a(s + 1);
        read_f(buf, 1, F[1]);
#pragma unroll
        for (int st = 1; st <= NST; st++) {
            const int p = st & 1;  // the parity of this step's buffers
            const bool last = st == NST;
            if (last) {  // the next stage's first step
                store_a(s + 1, nbuf);
                barrier();
                read_f(nbuf, 0, F[0]);
            } else if (st + 1 < NST) {
                read_f(buf, st + 1, F[1 - p]);
            }
            __builtin_amdgcn_sched_barrier(0);
            const int is = last ? s + 1 : s, iz = (last ? 1 - z : z) % WS, ist = last ? 0 : st;
            const bool first = z == 0 && st == 1, end = z == 1 && last;  // of the two stages
            fold(0, scale[1 - p][0], first);
            if (NT == 2 && end) add_part(0);
            issue(is, iz, ist, 0, F[p], scale[p][0]);
            __builtin_amdgcn_sched_barrier(0);
            fold(1, scale[1 - p][1], NT == 2 && first);
            if (end) add_part(NT - 1);
            issue(is, iz, ist, 1, F[p], scale[p][1]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int s = 0; s < ns; s += 2) {
        stage(s, 0);
        stage(s + 1, 1);
    }
    if constexpr (KS > 1) {  // the partial sums of the waves: 0 + 1, or (0 + 1) + (2 + 3)
        float *red = reinterpret_cast<float *>(lds);
        constexpr int TILE = NT * 16 * 64;
        float *mine = red + wave * TILE + lane;
        if (ks > 0) {
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
#pragma unroll
                for (int i = 0; i < 16; i++) mine[(nt * 16 + i) * 64] = acc[nt][i];
        }
        __syncthreads();
        if (ks > 0) return;
        static_assert(KS == 2 || KS == 4, "the order of the sums");
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const float *v = mine + (nt * 16 + i) * 64;
                acc[nt][i] += v[TILE];
                if constexpr (KS == 4) acc[nt][i] += v[2 * TILE] + v[3 * TILE];
            }
    }
    // lane (lr, h) holds row ri and, in register i, token 8 (i / 4) + 4 h + i % 4 of each token tile
    const uint32_t etab = sdy_expf_tab_lane(lane);
    const int tok0 = t0 + 4 * h;
    if (g.swiglu) {  // the pair's up row is in the next lane
        float *o = g.out + (size_t)tok0 * g.out_stride + (ri >> 1);
        const bool on = ri < g.n_rows && !(lr & 1);
#pragma unroll
        for (int nt = 0; nt < NT; nt++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int t = 32 * nt + 8 * (i >> 2) + (i & 3);
                const float v = acc[nt][i];
                const float up = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));
                const float y = sdy_silu_mul1_reg(v, up, etab);
                if (on && tok0 + t < g.n_tok) o[t * g.out_stride] = y;
            }
        return;
    }
    if (ri >= g.n_rows) return;
    const float bias = g.bias ? g.bias[row] : 0.0f;
    float rv[NT][16];
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = tok0 + 32 * nt + 8 * (i >> 2) + (i & 3);
            rv[nt][i] = g.resid ? g.resid[(size_t)(t < g.n_tok ? t : g.n_tok - 1) * g.out_stride + row] : 0.0f;
        }
    float *o = g.out + (size_t)tok0 * g.out_stride + row;
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int t = 32 * nt + 8 * (i >> 2) + (i & 3);
            float v = acc[nt][i];
            if (g.bias) v = v + bias;
            if (g.resid) v = rv[nt][i] + v;
            if (tok0 + t < g.n_tok) o[t * g.out_stride] = v;
        }
}

}  // namespace

template <int WT, int RW, int KS, int NT>
static int launch_mm(const MmArgs &g, hipStream_t st) {
    constexpr int BM = 32 * RW, BN = 32 * NT;
    SDY_NOTE_KERNEL((k_mm_blocks<WT, RW, KS, NT>));
    hipLaunchKernelGGL((k_mm_blocks<WT, RW, KS, NT>),
                       dim3((unsigned)((g.n_tok + BN - 1) / BN), (unsigned)((g.n_rows + BM - 1) / BM)), dim3(64 * RW * KS), 0, st, g);
    return sdy_check_launch("matvec (block MFMA)");
}

template <int WT>
static int mm_type(const MmArgs &g, long mat_rows, hipStream_t st) {
    // The split of a row's blocks over KS waves sets the order of its sum, so it is chosen by the row length, the
    // tokens and the matrix' rows: a row's result does not depend on how many rows a call computes. Two waves for rows of
    // up to 2048 inputs, four for longer ones (11008 x 2048, 32 tokens: 31.7 us against 41.6 with two), whose error against
    // 64 bits then is 2 to 3 % above the one-token kernel's at 4096 (see fold; the four sums added one by one: 1 %
    // more). Two again where the rows alone are waves enough: from 256 tokens above 4096 inputs (72 against 80 us), and on
    // more rows than 256 tiles of 32, one to a CU, of 33 to 63 units of 64 inputs, where the four also idle through most of
    // a row's last stage of 16 blocks (Q8_0, 5 tokens: 121872 x 2080 60 against 95 us, the matvec 67; 16000 x 3072 16.3
    // against 17.6, but 8000 x 3072 14.7 against 13.0; 64 tokens, 16000 x 2080 19 against 31). The one-token kernel is a chain there (error 1.15e-7,
    // 1.24e-7 and 1.34e-7 at 2080, 2560 and 3072 inputs, here 7.5e-8, 7.6e-8 and 7.8e-8); of 64 units it is the tree, which
    // two waves miss by 8 %.
    if (g.nb <= 64 || (g.T < 64 && mat_rows > 8192) || (g.nb > 128 && g.n_tok >= 256)) {
        // Tiles of 128 rows x 64 tokens where that leaves work for most CUs (22016 x 2048, 512 tokens: 121 us against
        // 155 with 64 x 32), else 64 x 32 (2048 x 2048, 512 tokens: 20.5 against 25.3).
        const bool wide = g.n_tok > 32 && ((g.n_tok + 63) / 64) * ((g.n_rows + 127) / 128) >= 160;
        return wide ? launch_mm<WT, 4, 2, 2>(g, st) : launch_mm<WT, 2, 2, 1>(g, st);
    }
    return g.n_tok > 64 ? launch_mm<WT, 2, 4, 1>(g, st) : launch_mm<WT, 1, 4, 1>(g, st);
}

// The tokens of a->xq through rows [a->row0, a->row1) of m (Q8_0, Q4_0, Q5_0), as sdy_matvec. Returns 1, launching
// nothing, when the kernel's 32-bit offsets do not reach every byte of the matrix or the activations, a grid's 65535
// row tiles every row of the matrix, or the rows are not 2-byte aligned.
extern "C" int sdy_mm_blocks(const sdy_mat *m, const sdy_mv_args *a, sdy_stream s) {
    const size_t row_bytes = (size_t)(m->n_in / 32) * 34, lim = 0xFFFFFFFFu;
    if (m->bytes >= lim || m->gbytes >= lim || row_bytes * a->n_tok >= lim || ((uintptr_t)a->xq & 1) || m->n_rows > 65535L * 32)
        return 1;
    MmArgs g = {};
    for (int i = 0; i < 5; i++) g.p[i] = (const uint8_t *)m->base + m->plane_off[i];
    if (m->gbase) {
        size_t off[5];
        sdy_gemm_layout_planes(m->type, m->n_in, m->grows, off);
        for (int i = 0; i < 5; i++) g.p[i] = (const uint8_t *)m->gbase + off[i];
        g.blk = 1;
        g.grow0 = m->grow0;
    }
    g.nb = m->n_in / 32;
    g.T = m->n_units;
    g.row0 = a->row0;
    g.n_rows = a->row1 - a->row0;
    g.xoff = (uint32_t)((uintptr_t)a->xq & 3);
    g.xq = (const uint8_t *)a->xq - g.xoff;
    g.n_tok = a->n_tok;
    g.out = a->out;
    g.out_stride = a->out_stride;
    g.bias = a->bias;
    g.resid = a->resid;
    g.swiglu = a->epilogue == SDY_EPI_SWIGLU;
    hipStream_t st = (hipStream_t)s;
    switch (m->type) {
    case SDY_Q8_0: return mm_type<SDY_Q8_0>(g, m->n_rows, st);
    case SDY_Q4_0: return mm_type<SDY_Q4_0>(g, m->n_rows, st);
    default: return mm_type<SDY_Q5_0>(g, m->n_rows, st);
    }
}

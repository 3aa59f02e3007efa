// Prefill attention in flash form on the bf16 matrix cores with f32's precision (within tolerance of the reference, not
// its bits; the reference's own arithmetic is sdy_attention in attn_kernels.hip).
//
// For each prompt token t and query head, the reference (csrc/ops.c:405-414, called per token from
// csrc/model_llama.c:619-647) takes the scores s_j = q.k_j / sqrt(head_dim) over the positions
// j < n_kv0 + t, one softmax over them and the weighted sum of the V rows. Here:
//
//   k_attn_flash<HD, KT, MS>  grid (ceil(n_tok / 32), n_head), 512 threads: one workgroup per 32
//   consecutive queries of one head (the blocks with the most keys first, a head's blocks on one XCD),
//   its eight waves sharing the key tiles of 32 positions (wave w: tiles w, w + 8, ...). Per tile a wave
//   computes S^T = K Q^T (keys as rows, so a lane holds its own query's 16 scores of the tile), masks the
//   positions at or past each query's causal limit, and keeps the running maximum m, the sum l of
//   exp(s - m) and O^T = V^T P (HD / 32 tiles of 32 dims), rescaled by exp(m_old - m_new) when m grows.
//   The waves' (m, l, O) are then merged through LDS in wave order:
//   out = sum_w O_w exp(m_w - M) / sum_w l_w exp(m_w - M), M = max_w m_w.
//
// Every f32 operand is the exact sum of three bf16 (an f16 cache's of two), each at most 2^-8 of the one before, and a
// product the sum of the six (five) greatest of their bf16 products, added in f32 by v_mfma_f32_32x32x16_bf16: 192
// matrix-core cycles per 32 x 32 x 16 where v_mfma_f32_32x32x2_f32 takes 512 and lets no VALU work run beside it. Left
// out are two products of at most about 2^-25 of the whole each and less, together at most 2^-24 (found: 2^-24.01), as
// much as one rounding of an f32 product. The error against 64 bits is the f32 form's or less (512 tokens over 1024 cached positions, 32 heads of 128: 3.9e-7 against 4.7e-7): there are fewer
// sums to round. The queries' fragments sit in LDS; K's and V's are made in registers, 3.5 VALU instructions per
// element. What bounds it: latency at two waves per SIMD (256 registers; the VALU busy in 37 % of the cycles, a
// wave ready but not issuing 44 % of its time, waiting for data 26 %), the splits (450 of the tile's 730 VALU
// instructions) and the keys' stream from L2. The 512 tokens above, f32 cache: 129 -> 82 us (10.7 GFLOP), f16 129 -> 70;
// 301 tokens, 32 heads: 34 -> 24; 77 tokens over 3000 positions, 16 heads, f16: 123 -> 64. The XCD order is 6 us of the
// first. Two blocks of queries per wave, sharing the splits and the stream: f32 spills (100 us), f16 76, and half the
// workgroups for the shorter prompts (22 -> 32 us).
//
// Each sum has a fixed order (no float atomics), so the results are deterministic. They differ
// from the reference's in rounding: f32 products summed in the matrix core's order, tile-relative
// exponentials.
#include <type_traits>

#include "sdy_attn_dev.h"
#include "sdy_device.h"
#include "sdy_internal.h"
#include "sdy_ops.h"
#include "sdy_shim.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int QB = 32;  // queries per workgroup (the MFMA's 32 columns)
constexpr int KB = 32;  // positions per key tile (the MFMA's 32 rows)
constexpr int FW = 8;   // waves per workgroup

struct FlashArgs {
    const float *q;          // rotated queries [n_tok][q_stride], head h at h * HD
    long q_stride;
    const void *k_cache, *v_cache;  // [n_kv_head][max_seq][HD] of the element type KT
    long head_stride;        // max_seq * HD
    int n_head, n_kv_head, n_tok, n_kv0;  // token t attends to positions < n_kv0 + t
    float scale;             // 1 / sqrt(HD)
    float *out;              // [n_tok][out_stride], head h at h * HD
    long out_stride;
};

// LDS: the block's queries, as fragments [3][32][HD + 8] bf16 or as f32 [2][32][QS] (element (query q, dim
// half * HD/2 + s) at [half][q][s]), then, after the key tiles, the merge area: the waves' O dims, 1/MS of them at a time, as
// [FW][32][OS], their m, l as [2][FW][32] and whether their sums hold as [FW] (HD 128: 134 KB for MS 1, one workgroup per CU;
// 68 KB for MS 2, two).
template <int HD, int MS>
struct FlashLds {
    static constexpr int HH = HD / 2, QS = HH + 4, OS = HD / MS + 1;
    static constexpr size_t q_floats = 2 * 32 * QS;
    static constexpr size_t merge_floats = (size_t)FW * 32 * OS + 2 * FW * 32 + FW;
    static constexpr size_t bytes = 4 * (q_floats > merge_floats ? q_floats : merge_floats);
};

// Four consecutive elements of a buffer resource at byte offset o (zeros past its end)
template <class KT>
SDY_DEV sdy_f32x4 ld4_buf(__amdgpu_buffer_rsrc_t r, uint32_t o) {
    if constexpr (std::is_same<KT, float>::value) {
        return __builtin_bit_cast(sdy_f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0));
    } else {
        const auto u = __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0);
        return sdy_f32x4{sdy_h2f((uint16_t)(u[0] & 0xFFFFu)), sdy_h2f((uint16_t)((uint32_t)u[0] >> 16)),
                         sdy_h2f((uint16_t)(u[1] & 0xFFFFu)), sdy_h2f((uint16_t)((uint32_t)u[1] >> 16))};
    }
}

// ND consecutive elements of a V row (the lane's dims ND * (lane % 32) + dt, dt < ND)
template <int ND, class KT>
struct VLoad;
template <class KT>
struct VLoad<4, KT> {
    using T = sdy_f32x4;
    SDY_DEV static T ld(__amdgpu_buffer_rsrc_t r, uint32_t o) { return ld4_buf<KT>(r, o); }
    SDY_DEV static float at(const T &v, int j) { return v[j]; }
};
template <class KT>
struct VLoad<2, KT> {
    using T = float2;
    SDY_DEV static T ld(__amdgpu_buffer_rsrc_t r, uint32_t o) {
        if constexpr (std::is_same<KT, float>::value) {
            const auto u = __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0);
            return make_float2(__uint_as_float(u[0]), __uint_as_float(u[1]));
        } else {
            const uint32_t u = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0);
            return make_float2(sdy_h2f((uint16_t)(u & 0xFFFFu)), sdy_h2f((uint16_t)(u >> 16)));
        }
    }
    SDY_DEV static float at(const T &v, int j) { return j ? v.y : v.x; }
};

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Eight f32 as NP bf16 fragments that add up to them: each the rest's nearest bf16 (8 bits and a sign), so three hold
// the 24 bits of an f32 and two the 11 bits of an f16.
template <int NP>
struct Frag {
    u32x4 p[NP];
    SDY_DEV void set(const float x[8]) {
        // the rests as exact two-term dots with (-1, 0) and (0, -1) (not left as constants: the compiler would choose
        // an inline one, whose halves the instruction's definition leaves open)
        uint32_t lo = 0x0000BF80u, hi = 0xBF800000u;
        __asm__("" : "+s"(lo), "+s"(hi));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
            for (int k = 0; k < NP; k++) {
                const bf16x2 u = __builtin_convertvector(f32x2{a, b}, bf16x2);
                p[k][i] = __builtin_bit_cast(uint32_t, u);
                a = __builtin_amdgcn_fdot2_f32_bf16(u, __builtin_bit_cast(bf16x2, lo), a, false);
                b = __builtin_amdgcn_fdot2_f32_bf16(u, __builtin_bit_cast(bf16x2, hi), b, false);
            }
        }
    }
};

// c + A B in f32 from the fragments, least products first. Those left out are together at most 2^-24 of |a b|.
template <int NA>
SDY_DEV f32x16 mfma_split(const Frag<NA> &a, const Frag<3> &b, f32x16 c) {
#pragma unroll
    for (int n = 2; n >= 0; n--)
#pragma unroll
        for (int k = NA - 1; k >= 0; k--)
            if (n - k >= 0)
                c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a.p[k]), __builtin_bit_cast(bf16x8, b.p[n - k]), c, 0, 0, 0);
    return c;
}

// One block. SPLIT: the products on the bf16 matrix cores, from fragments; else on the f32 ones. Returns, the same for
// all threads, whether (SPLIT) the fragments may not have held the values; nothing is written then: some sum is infinite or
// NaN, or is so small (below 2^-90, but not 0) that a whole column of values may be below 2^-110, whose last fragments bf16
// does not hold. (A column of nothing but values below 2^-134, half of bf16's least, counts as zeros.)
template <int HD, class KT, int MS, bool SPLIT>
SDY_DEV bool flash_block(const FlashArgs &a, float *lds) {
    using LY = FlashLds<HD, MS>;
    constexpr int HH = HD / 2, ND = HD / 32, NK = std::is_same<KT, float>::value ? 3 : 2, QP = HD + 8;
    using VL = VLoad<ND, KT>;
    const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, ql = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // a head's blocks on one XCD (workgroups are dealt to the 8 XCDs in turn), whose L2 then holds the keys and values
    // of its own heads only; the blocks with the most keys first
    int qb = (int)blockIdx.x, h = (int)blockIdx.y;
    if (a.n_head % 8 == 0) {
        const int L = h * (int)gridDim.x + qb, n = a.n_head / 8, i = L >> 3;
        qb = i / n;
        h = (L & 7) * n + i - qb * n;
    }
    qb = (int)gridDim.x - 1 - qb;
    const int g = h / (a.n_head / a.n_kv_head);
    const int q0 = qb * QB;
    const int t_last = q0 + QB < a.n_tok ? q0 + QB - 1 : a.n_tok - 1;
    const int n_kv_max = a.n_kv0 + t_last;  // positions of the block's last query
    const int n_kt = (n_kv_max + KB - 1) / KB;

    uint16_t *qf = reinterpret_cast<uint16_t *>(lds);  // SPLIT: the fragments [3][32][QP]
    for (int i = tid; SPLIT && i < QB * HD / 8; i += 64 * FW) {
        const int q = i / (HD / 8), d = 8 * (i - q * (HD / 8));
        const int t = q0 + q < a.n_tok ? q0 + q : a.n_tok - 1;
        const float4 *src = reinterpret_cast<const float4 *>(a.q + (size_t)t * a.q_stride + (size_t)h * HD + d);
        const float4 v0 = src[0], v1 = src[1];
        const float v[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        Frag<3> f;
        f.set(v);
#pragma unroll
        for (int k = 0; k < 3; k++) *reinterpret_cast<u32x4 *>(qf + (k * 32 + q) * QP + d) = f.p[k];
    }
    for (int i = tid; !SPLIT && i < QB * HD / 4; i += 64 * FW) {
        const int q = i / (HD / 4), d = 4 * (i - q * (HD / 4));
        const int t = q0 + q < a.n_tok ? q0 + q : a.n_tok - 1;
        const float4 v = *reinterpret_cast<const float4 *>(a.q + (size_t)t * a.q_stride + (size_t)h * HD + d);
        const int part = d / HH, s = d - part * HH;
        *reinterpret_cast<float4 *>(lds + (part * 32 + q) * LY::QS + s) = v;
    }
    __syncthreads();

    const int t = q0 + ql;
    const int lim = t < a.n_tok ? a.n_kv0 + t : 0;  // this lane's query sees positions < lim
    const KT *kb = (const KT *)a.k_cache + (size_t)g * a.head_stride;
    const KT *vb = (const KT *)a.v_cache + (size_t)g * a.head_stride;
    constexpr uint32_t RB = HD * (uint32_t)sizeof(KT);  // bytes of a row
    const uint32_t vk = (uint32_t)ql * RB + hh * HH * (uint32_t)sizeof(KT), vo = 4 * hh * RB + ND * ql * (uint32_t)sizeof(KT);
    uint32_t qo = SPLIT ? (uint32_t)(ql * QP + hh * HH) : (uint32_t)((hh * 32 + ql) * LY::QS);
    f32x16 o[ND];
#pragma unroll
    for (int dt = 0; dt < ND; dt++) o[dt] = f32x16{};
    float m_run = -INFINITY, l_run = 0.0f;
    for (int kt = wave; kt < n_kt; kt += FW) {
        const int k0 = kt * KB;
        // K: lane (key ql of the tile, dims hh * HH ...); V of the PV step r: key
        // 8 (r / 4) + 4 hh + r % 4 of the tile (the key of the lane's score register r), dims
        // ND * ql ... Positions past the block's last one read as zeros (the resource ends there) and are masked below.
        // A scalar offset is left out of the resource's bound, so each 8 V rows have a resource of their own.
        const int rows = n_kv_max - k0 < KB ? n_kv_max - k0 : KB;
        auto rows_from = [&](const KT *base, int r) {
            return __builtin_amdgcn_make_buffer_rsrc((void *)(base + (size_t)(k0 + r) * HD), (short)0,
                                                     (rows > r ? rows - r : 0) * (int)RB, 0x00020000);
        };
        const __amdgpu_buffer_rsrc_t rk = rows_from(kb, 0), rv[4] = {rows_from(vb, 0), rows_from(vb, 8), rows_from(vb, 16), rows_from(vb, 24)};
        sdy_f32x4 kv[HH / 4];
#pragma unroll
        for (int i = 0; i < HH / 4; i++) kv[i] = ld4_buf<KT>(rk, vk + 4 * i * (uint32_t)sizeof(KT));
        typename VL::T vv[16];
        auto load_v = [&]() {
#pragma unroll
            for (int r = 0; r < 16; r++) vv[r] = VL::ld(rv[r >> 2], vo + (r & 3) * RB);
        };
        if constexpr (SPLIT) load_v();
        // S^T[key][query] = sum over dims of K[key][d] Q[query][d]: step (i, j) pairs dim 4i + j
        // (lanes 0-31) with dim HH + 4i + j (lanes 32-63)
        f32x16 s = f32x16{};
        __asm__ volatile("" : "+v"(qo));  // the queries are read again for each tile: they would fill the registers
        if constexpr (SPLIT) {  // step i: dims 8 i .. of each half
#pragma unroll
            for (int i = 0; i < HH / 8; i++) {
                Frag<3> q;
#pragma unroll
                for (int k = 0; k < 3; k++) q.p[k] = *reinterpret_cast<const u32x4 *>(qf + k * 32 * QP + qo + 8 * i);
                const float x[8] = {kv[2 * i][0], kv[2 * i][1], kv[2 * i][2], kv[2 * i][3],
                                    kv[2 * i + 1][0], kv[2 * i + 1][1], kv[2 * i + 1][2], kv[2 * i + 1][3]};
                Frag<NK> k;
                k.set(x);
                s = mfma_split(k, q, s);
            }
        } else
#pragma unroll
        for (int i = 0; i < HH / 4; i++) {
            const sdy_f32x4 qv = *reinterpret_cast<const sdy_f32x4 *>(lds + qo + 4 * i);
#pragma unroll
            for (int j = 0; j < 4; j++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[i][j], qv[j], s, 0, 0, 0);
        }
        if constexpr (!SPLIT) {  // (with K's registers free: the second form is not to cost the first any)
            __builtin_amdgcn_sched_barrier(0);
            load_v();
        }
        // scores of the lane's query (register r: key 8 (r / 4) + 4 hh + r % 4), running maximum
        // and sum; the other half of the tile's keys is in lane ^ 32
        float p[16];
        float mt = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r++) p[r] = s[r] * a.scale;
        if (k0 + KB > a.n_kv0 + q0) {  // some query does not see all of the tile
#pragma unroll
            for (int r = 0; r < 16; r++) p[r] = k0 + 8 * (r >> 2) + 4 * hh + (r & 3) < lim ? p[r] : -INFINITY;
        }
#pragma unroll
        for (int r = 0; r < 16; r++) mt = fmaxf(mt, p[r]);
        mt = fmaxf(mt, __shfl_xor(mt, 32));
        const float m_new = fmaxf(m_run, mt);
        const float mu = m_new == -INFINITY ? 0.0f : m_new;  // no key yet: every term is 0
        float ls = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            p[r] = __expf(p[r] - mu);
            ls += p[r];
        }
        ls += __shfl_xor(ls, 32);
        const float corr = __expf(m_run - mu);
        l_run = l_run * corr + ls;
        m_run = m_new;
#pragma unroll
        for (int dt = 0; dt < ND; dt++)
#pragma unroll
            for (int e = 0; e < 16; e++) o[dt][e] = o[dt][e] * corr;
        // O^T[dim][query] += V^T[dim][key] P[key][query] over the tile's keys: SPLIT 16 per step (score registers
        // 8 u .. of both lane halves), else two
        if constexpr (SPLIT) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                Frag<3> pf;
                pf.set(p + 8 * u);
#pragma unroll
                for (int dt = 0; dt < ND; dt++) {
                    float x[8];
#pragma unroll
                    for (int e = 0; e < 8; e++) x[e] = VL::at(vv[8 * u + e], dt);
                    Frag<NK> v;
                    v.set(x);
                    o[dt] = mfma_split(v, pf, o[dt]);
                }
            }
        } else
#pragma unroll
        for (int r = 0; r < 16; r++)
#pragma unroll
            for (int dt = 0; dt < ND; dt++)
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(VL::at(vv[r], dt), p[r], o[dt], 0, 0, 0);
    }

    bool unfit = false;
    if constexpr (SPLIT) {
        float z = 0.0f * l_run;  // NaN from an infinity or a NaN on
        uint32_t least = ~0u;    // the least |o| but 0, its bits shifted and less one
#pragma unroll
        for (int dt = 0; dt < ND; dt++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                z = __builtin_fmaf(0.0f, o[dt][e], z);
                const uint32_t u = (__float_as_uint(o[dt][e]) << 1) - 1;
                least = u < least ? u : least;
            }
        unfit = __ballot(z != z || least < (127u - 90u) << 24) != 0;
    }
    // merge of the waves' partials in wave order (the Q^T area is reused), in MS parts of the dims:
    // part x holds the O columns dt in [x NDH, (x + 1) NDH), dims ND * row + dt, at NDH * row + dt - x NDH
    constexpr int NDH = ND / MS;
    float *ml = lds + (size_t)FW * 32 * LY::OS;  // m [FW][32], then l [FW][32]
#pragma unroll
    for (int x = 0; x < MS; x++) {
        __syncthreads();
        float *om = lds + (size_t)wave * 32 * LY::OS;
#pragma unroll
        for (int dt = x * NDH; dt < (x + 1) * NDH; dt++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int row = 8 * (r >> 2) + 4 * hh + (r & 3);  // D row: dim ND * row + dt
                om[ql * LY::OS + NDH * row + dt - x * NDH] = o[dt][r];
            }
        if (x == 0 && hh == 0) {
            ml[wave * 32 + ql] = m_run;
            ml[FW * 32 + wave * 32 + ql] = l_run;
        }
        int *const fl = reinterpret_cast<int *>(ml + 2 * FW * 32);
        if (SPLIT && x == 0 && lane == 0) fl[wave] = unfit;
        __syncthreads();
        if (SPLIT && x == 0) {  // (the other form's queries do not reach the flags)
            static_assert(LY::q_floats <= (size_t)FW * 32 * LY::OS, "the flags outlive the queries' writes");
            int any = 0;
#pragma unroll
            for (int w = 0; w < FW; w++) any |= fl[w];
            if (__builtin_amdgcn_readfirstlane(any)) return true;
        }
        for (int i = tid; i < QB * (HD / MS); i += 64 * FW) {
            const int q = i / (HD / MS), dl = i - q * (HD / MS);
            if (q0 + q >= a.n_tok) continue;
            const int d = ND * (dl / NDH) + x * NDH + dl % NDH;
            float M = -INFINITY;
#pragma unroll
            for (int w = 0; w < FW; w++) M = fmaxf(M, ml[w * 32 + q]);
            float ls = 0.0f, os = 0.0f;
#pragma unroll
            for (int w = 0; w < FW; w++) {
                const float e = __expf(ml[w * 32 + q] - M);  // a wave without keys: m = -inf, e = 0
                ls += ml[FW * 32 + w * 32 + q] * e;
                os += lds[((size_t)w * 32 + q) * LY::OS + dl] * e;
            }
            a.out[(size_t)(q0 + q) * a.out_stride + (size_t)h * HD + d] = os / ls;
        }
    }
    return false;
}

template <int HD, class KT, int MS>
__global__ __launch_bounds__(64 * FW) void k_attn_flash(FlashArgs a) {
    extern __shared__ __align__(16) float lds[];
    // (an infinity's fragments are NaN, so a block that met one, or a value beyond bf16's largest, is computed again; so is
    // one with a column of values too small for theirs)
    if (flash_block<HD, KT, MS, true>(a, lds)) flash_block<HD, KT, MS, false>(a, lds);
}

template <int HD, class KT, int MS>
int launch_flash(const FlashArgs &A, hipStream_t st) {
    static size_t granted = 0;
    const void *fn = (const void *)k_attn_flash<HD, KT, MS>;
    int rc = sdy_lds_limit(fn, FlashLds<HD, MS>::bytes, &granted);
    if (rc) return rc;
    SDY_NOTE_KERNEL((k_attn_flash<HD, KT, MS>));
    hipLaunchKernelGGL((k_attn_flash<HD, KT, MS>), dim3((unsigned)((A.n_tok + QB - 1) / QB), (unsigned)A.n_head),
                       dim3(64 * FW), (FlashLds<HD, MS>::bytes), st, A);
    return sdy_check_launch("attn_flash");
}

// The merge in two parts (two workgroups per CU) when the grid has more workgroups than the GPU
// has CUs: the 30B-A3B's 32 heads x 16 blocks, 36.0 -> 34.2 ms for its 1024-token prefill; the 3B's
// 16 x 16 fill the CUs once, and a second merge round only costs (53.8k against 53.4k tok/s).
template <int HD, class KT>
int launch_flash_ms(const FlashArgs &A, hipStream_t st) {
    int n_cu = 0;
    size_t mem = 0;
    if (sdy_device_info(&n_cu, &mem) || n_cu <= 0) n_cu = 256;
    const long wgs = (long)((A.n_tok + QB - 1) / QB) * A.n_head;
    return wgs > n_cu ? launch_flash<HD, KT, 2>(A, st) : launch_flash<HD, KT, 1>(A, st);
}

template <int HD>
int launch_flash_kv(const FlashArgs &A, int kv_type, hipStream_t st) {
    return kv_type == SDY_KV_F16 ? launch_flash_ms<HD, uint16_t>(A, st) : launch_flash_ms<HD, float>(A, st);
}

}  // namespace

extern "C" int sdy_attention_flash_ok(int n_head, int n_kv_head, int hd) {
    return (hd == 64 || hd == 128) && n_head > 0 && n_kv_head > 0 && n_head % n_kv_head == 0;
}

extern "C" int sdy_attention_flash(const float *q, const void *k_cache, const void *v_cache, int kv_type, int n_tok,
                                   int n_head, int n_kv_head, int hd, int n_kv0, long head_stride, long q_stride,
                                   float *out, long out_stride, sdy_stream s) {
    if (n_tok <= 0) return 0;
    if (!sdy_attention_flash_ok(n_head, n_kv_head, hd))
        return sdy_fail(-1, "attention_flash: head_dim 64 or 128 and n_head a multiple of n_kv_head (got %d, %d, %d)",
                        hd, n_head, n_kv_head);
    if (kv_type != SDY_KV_F32 && kv_type != SDY_KV_F16) return sdy_fail(-1, "attention_flash: KV type %d", kv_type);
    if (n_kv0 < 1) return sdy_fail(-1, "attention_flash: the first token needs a position (n_kv0 %d)", n_kv0);
    if ((q_stride | out_stride) & 3 || (uintptr_t)q & 15)
        return sdy_fail(-1, "attention_flash: q rows (and strides) aligned to 16 bytes");
    FlashArgs A;
    A.q = q;
    A.q_stride = q_stride;
    A.k_cache = k_cache;
    A.v_cache = v_cache;
    A.head_stride = head_stride;
    A.n_head = n_head;
    A.n_kv_head = n_kv_head;
    A.n_tok = n_tok;
    A.n_kv0 = n_kv0;
    A.scale = 1.0f / sqrtf((float)hd);
    A.out = out;
    A.out_stride = out_stride;
    hipStream_t st = (hipStream_t)s;
    return hd == 64 ? launch_flash_kv<64>(A, kv_type, st) : launch_flash_kv<128>(A, kv_type, st);
}

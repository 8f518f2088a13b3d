// Prefill attention with the keys of one 32-row query block split over the waves of a
// workgroup: the kernel of launches whose query blocks are too few to fill the chip, of
// head_dim 64 and of un-rotated keys.
//
// What bounds such a launch is the serial chain of one wave (operand reads, QK^T, softmax,
// PV, one tile after the other), not the matrix cores or memory: with a tile stream shared
// by 4 waves of 32 rows each, 37 rows of 12 heads over 2037 keys ran 24 workgroups of 32
// tiles in turn (43 us) and left three waves of four without rows. Here one workgroup is
// one 32-row block of one head; its KW waves take every KW-th key tile, each through LDS
// of its own, so no wave waits for another before the end, where the partial (max, sum,
// output) of the waves are merged through LDS. The cost is KW times fewer rows per K / V
// byte read, which is why launches with many query blocks keep the shared stream.
//
//  * A tile is 8 KB of K and 8 KB of V (32 keys at head_dim 128, 64 at 64), one slot of
//    each per wave. A slot is refilled as soon as its operand reads have landed, so the
//    next K tile loads under this tile's softmax and PV, the next V tile under the next
//    QK^T and softmax.
//  * ROTK: keys come un-rotated; a lane holds the pairs (d, d + head_dim / 2) of its key
//    row in two operand fragments, so RoPE is applied in registers between the LDS read
//    and the MFMA.
//  * Softmax: the running max is the accumulator's start value, row sums are over the
//    bf16-rounded p. At head_dim 128 over rotated keys (calls that with more rows run the
//    pipelined kernel) the max is raised only past 2^8, as there. Otherwise every new max raises
//    it: the largest p of a wave is then exactly 1, where rounding it, the heaviest weight of a
//    row, made up to 3 % of the error of rows over 1000 keys and more (N(0, 1), 14/2 heads, 1259
//    rows behind 1112, relative error against 64 bits: 0.00335 raised past 2^8, 0.00325 always,
//    0.00330 register-staged), for up to 6 % of the time there (14/2 heads, 2410 rows 26.6 ->
//    28.1 us; 28/4 heads, RoPE inside, 524 rows 18.6 -> 19.2).
//  * At head_dim 128 over rotated keys Q is multiplied by log2(e) / sqrt(head_dim) before its
//    bf16 rounding;
//    otherwise the scores are (one multiplication each), so that a query that needs no
//    rotation enters the MFMAs unrounded, and so do the low-frequency pairs of one that
//    does, which the rotation hardly moves (12/2 heads, 1000 rows behind 24, relative error
//    against 64 bits: 0.00305 with Q scaled, 0.00298 with the scores; 0.00298 register-staged).
#pragma once
#include "attn_pipe.hpp"
#include "common.hpp"

#include <type_traits>
#include <utility>

namespace efm {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

struct PrefillArgs {
    const bf16_t* q;
    const bf16_t* k;
    const bf16_t* v;
    bf16_t* o;
    int S, L, Hq, Hkv;
    int q_sn, q_sh, k_sn, k_sh, v_sn, v_sh;
    int o_sn, o_sh;
    int causal;
    int rope_q, rope_k;
    int q_pos_off, k_pos_off;
    float sm_scale_log2;
    RopeTable rope;
};

union Pack8 {
    bf16x8_t v;
    uint4 u;
    uint32_t w[4];
};

constexpr float kP2Lazy = 8.0f;

// Sum of the two bf16 halves of `w` added to acc (fp32).
__device__ __forceinline__ float add_bf16_pair(uint32_t w, float acc) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w),
                                           __builtin_bit_cast(bf16x2_t, 0x3f803f80u), acc, false);
}

// LDS tile layout for rows of HD bf16 (attn_pipe.hpp's swizzles; 128-byte rows at HD 64):
// the 16 rows that an operand read phase touches land in distinct bank groups.
template <int HD>
struct SplitTile {
    static constexpr int kKeys = HD == 128 ? 32 : 64;
    static constexpr int kRow = HD * 2;             // bytes per row
    static constexpr int kChunks = kRow / 16;       // 16-byte chunks per row
    static constexpr int kRows = 1024 / kRow;       // rows per 1 KB wave load
    static constexpr int kBytes = kKeys * kRow;     // 8 KB
    static constexpr int kLoads = kBytes / 1024;    // wave loads per operand tile
    __device__ static __forceinline__ int k_swz(int row) { return HD == 128 ? (row & 15) : ((row >> 1) & 7); }
    __device__ static __forceinline__ int v_swz(int row) { return HD == 128 ? ((row & 3) << 2) : (((row >> 1) & 1) << 2); }
};

// Grid of the split kernel, late (heavy) query blocks first. Workgroups go to the 8 XCDs
// round-robin by linear index, so with 8 x G workgroups per grid row (1, 2, 4 or 8 KV heads
// of G query heads) an XCD takes the query heads of one KV head, and 8 / Hkv query blocks of
// each are in a row: its L2 streams one head's K and V and no other's (28/4 heads, 64 rows
// over 8064 keys: 56 -> 43 us). Other head counts: one grid row per query block.
struct SplitGrid {
    int group;       // query heads per KV head
    int hkv_log2;    // log2 of the KV heads, or -1: grid x is the query head
    static bool by_xcd(int Hkv) { return Hkv <= 8 && (Hkv & (Hkv - 1)) == 0; }
    static SplitGrid of(int Hq, int Hkv) {
        int lg = 0;
        while ((1 << lg) < Hkv) ++lg;
        return SplitGrid{Hq / Hkv, by_xcd(Hkv) ? lg : -1};
    }
    static dim3 dims(int nqt, int Hq, int Hkv) {
        if (!by_xcd(Hkv)) return dim3(Hq, nqt);
        const int per = 8 / Hkv;
        return dim3(8 * (Hq / Hkv), (nqt + per - 1) / per);
    }
};

template <int HD, int KW, bool ROTK>
__global__ __launch_bounds__(KW * 64, 2) void prefill_attn_split_kernel(PrefillArgs a, SplitGrid sg, int nqt) {
    typedef SplitTile<HD> T;
    constexpr int KT = T::kKeys, NH = KT / 32, KS = HD / 16, DT = HD / 32, NL = T::kLoads, KB = KT / 16;
    constexpr int SLOT = 2 * T::kBytes;
    constexpr bool SCALE_Q = HD == 128 && !ROTK;
    const float sc = SCALE_Q ? 1.f : a.sm_scale_log2;             // scores to log2 units
    constexpr float lazy = SCALE_Q ? kP2Lazy : 0.f;
    constexpr int CPR = HD / 4;                      // float4 chunks per output row
    static_assert(KW >= (ROTK ? 4 : 2) && NL == 8 && 32 * HD * 4 <= SLOT, "tile geometry");
    __shared__ __align__(1024) unsigned char smem[KW * SLOT];
    __shared__ float ml[2][KW][32];
    // frequencies and Q fragments; KW 2 takes no RoPE and shares no Q, so that four workgroups
    // fit a CU
    constexpr bool SHARE = KW >= 4;
    const bool rope_q = ROTK || a.rope_q;
    __shared__ __align__(16) float sfreq[SHARE ? HD / 2 : 4];
    __shared__ __align__(16) unsigned char qfrag[SHARE ? KS * 1024 : 16];

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;
    const int ql = lane % 32, hh = lane / 32;
    int qt, head, kvh;
    if (sg.hkv_log2 >= 0) {
        const int x = (int)blockIdx.x;
        kvh = x & ((1 << sg.hkv_log2) - 1);
        head = kvh * sg.group + (x >> 3);
        qt = nqt - 1 - (((int)blockIdx.y << (3 - sg.hkv_log2)) + ((x & 7) >> sg.hkv_log2));
        if (qt < 0) return;
    } else {
        head = (int)blockIdx.x;
        kvh = head / sg.group;
        qt = nqt - 1 - (int)blockIdx.y;
    }
    const int q0 = qt * 32, qi = q0 + ql;
    const int diag = a.L - a.S;
    const int kv_end = a.causal ? min(a.L, min(a.S - 1, q0 + 31) + diag + 1) : a.L;
    const int ntiles = (kv_end + KT - 1) / KT;

    const char* kbase = reinterpret_cast<const char*>(a.k + (size_t)kvh * a.k_sh);
    const char* vbase = reinterpret_cast<const char*>(a.v + (size_t)kvh * a.v_sh);
    unsigned char* const kslot = smem + wave * SLOT;
    unsigned char* const vslot = kslot + T::kBytes;
    // wave load i of an operand tile: rows i * kRows + lane / kChunks; the lane fetches the
    // chunk that belongs at its place under the swizzle
    const int pr = lane / T::kChunks, pc = lane % T::kChunks;
    auto issue = [&](const char* base, int sn, int k0, unsigned char* slot, auto is_v) {
        const char* t0 = base + (size_t)k0 * sn * 2;
        const bool whole = k0 + KT <= a.L;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int row = i * T::kRows + pr;
            const int c = pc ^ (decltype(is_v)::value ? T::v_swz(row) : T::k_swz(row));
            // rows past the end read the last row
            const int r = whole ? row : min(row, a.L - 1 - k0);
            __builtin_amdgcn_global_load_lds(static_cast<const void*>(t0 + (uint32_t)((r * sn + c * 8) * 2)),
                                             (__attribute__((address_space(3))) void*)(slot + i * 1024), 16, 0, 0);
        }
    };
    auto issue_k = [&](int t) { issue(kbase, a.k_sn, t * KT, kslot, std::false_type{}); };
    auto issue_v = [&](int t) { issue(vbase, a.v_sn, t * KT, vslot, std::true_type{}); };

    // ---- Q (B operand) of this lane's row, d = ks*16 + hh*8 + e, requested first. A wave loads,
    // rotates and rounds RE of a lane's 8 values in each of one pair of fragments (ks, ks + KS /
    // 2), and the waves exchange the fragments through LDS: the loads, and with RoPE the sines
    // and cosines (sincosf, some 60 instructions a pair), are shared out (12/2 heads, 1000 rows
    // behind 24, RoPE inside: 27.8 us where each wave rotates all of them, 24.4 shared).
    constexpr int RE = SHARE ? KS * 4 / KW : 8;
    typedef uint32_t rot_t __attribute__((ext_vector_type(RE / 2)));
    const int rk = wave * RE / 8, re = wave * RE % 8, rd = rk * 16 + hh * 8 + re;
    uint4 qraw[KS];
    rot_t r0{}, r1{};
    float freq = 0.f;
    {
        const bool qv = qi < a.S;
        const bf16_t* qp = a.q + (size_t)(qv ? qi : 0) * a.q_sn + (size_t)head * a.q_sh;
        if constexpr (SHARE) {
            if (rope_q && tid < HD / 2) freq = a.rope.inv_freq[tid];
            if (qv) {
                r0 = *reinterpret_cast<const rot_t*>(qp + rd);
                r1 = *reinterpret_cast<const rot_t*>(qp + rd + HD / 2);
            }
        } else {
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                qraw[ks] = qv ? *reinterpret_cast<const uint4*>(qp + ks * 16 + hh * 8) : make_uint4(0, 0, 0, 0);
        }
    }
    if (wave < ntiles) {
        issue_k(wave);
        issue_v(wave);
    }
    bf16x8_t qf[KS];
    if constexpr (SHARE) {
        if (rope_q) {
            if (tid < HD / 2) sfreq[tid] = freq;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        auto prepare = [&](float& x0, float& x1, int d) {
            if (rope_q) {
                float sn, cs;
                sincosf((float)(qi + a.q_pos_off) * sfreq[d], &sn, &cs);
                const float y0 = x0 * cs - x1 * sn;
                x1 = x1 * cs + x0 * sn;
                x0 = y0;
            }
            if constexpr (SCALE_Q) {
                x0 *= a.sm_scale_log2;
                x1 *= a.sm_scale_log2;
            }
        };
#pragma unroll
        for (int e = 0; e < RE; e += 2) {
            float x0 = __uint_as_float(r0[e / 2] << 16), x1 = __uint_as_float(r0[e / 2] & 0xffff0000u);
            float y0 = __uint_as_float(r1[e / 2] << 16), y1 = __uint_as_float(r1[e / 2] & 0xffff0000u);
            prepare(x0, y0, rd + e);
            prepare(x1, y1, rd + e + 1);
            r0[e / 2] = pack_bf16x2(x0, x1);
            r1[e / 2] = pack_bf16x2(y0, y1);
        }
        // fragment ks of lane l at 16 (64 ks + l)
        unsigned char* const dst = qfrag + rk * 1024 + lane * 16 + re * 2;
        *reinterpret_cast<rot_t*>(dst) = r0;
        *reinterpret_cast<rot_t*>(dst + KS * 512) = r1;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const uint32_t ra =
            (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)qfrag) + lane * 16;
        [&]<int... I>(std::integer_sequence<int, I...>) {
            (attn_pipe::read_b128<I * 1024>(qf[I], ra), ...);
        }(std::make_integer_sequence<int, KS>{});
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(qf[ks]));
    } else {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            float x[8];
            unpack8(qraw[ks], x);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] *= SCALE_Q ? a.sm_scale_log2 : 1.f;
            Pack8 pk;
            pk.u = pack8(x);
            qf[ks] = pk.v;
        }
    }

    f32x16_t oacc[DT];
#pragma unroll
    for (int tt = 0; tt < DT; ++tt)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[tt][e] = 0.f;
    // running row max of the scores (-inf until the wave meets a key that the row sees); the
    // accumulators start at -m_run (0 while it is -inf)
    float m_run = -INFINITY, l_run = 0.f;

    const uint32_t lk = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)kslot);
    uint32_t ka[KS], va[DT];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ka[ks] = lk + (uint32_t)(ql * T::kRow + (((ks * 2 + hh) ^ T::k_swz(ql)) << 4));
    {
        // V^T operand (ds_read_b64_tr_b16, see attn_pipe.hpp): row 4 (g / 2) + j / 4 of the
        // 8-key step, d = 32 tt + 16 (g % 2) + 4 (j % 4)
        const int g = lane >> 4, j = lane & 15, row = (g >> 1) * 4 + (j >> 2);
#pragma unroll
        for (int tt = 0; tt < DT; ++tt) {
            const int d = tt * 32 + 16 * (g & 1) + 4 * (j & 3);
            va[tt] = lk + (uint32_t)(T::kBytes + row * T::kRow + (((d >> 3) ^ T::v_swz(row)) << 4) + ((d & 7) << 1));
        }
    }
    typedef short s4_t __attribute__((ext_vector_type(4)));

    for (int kt = wave; kt < ntiles; kt += KW) {
        const bool more = kt + KW < ntiles;
        const int kb0 = kt * KT;
        attn_pipe::vm_wait<NL>();   // K has landed; the V tile's loads may be in flight
        asm volatile("" ::: "memory");
        bf16x8_t kf[NH][KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            attn_pipe::read_b128<0>(kf[0][ks], ka[ks]);
            if constexpr (NH == 2) attn_pipe::read_b128<32 * T::kRow>(kf[1][ks], ka[ks]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(kf[h][ks]));
        if (more) issue_k(kt + KW);
        if constexpr (ROTK) {
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                const float pos = (float)(kb0 + h * 32 + ql + a.k_pos_off);
#pragma unroll
                for (int ks = 0; ks < KS / 2; ++ks) {
                    Pack8 lo, hi;
                    lo.v = kf[h][ks];
                    hi.v = kf[h][ks + KS / 2];
                    float x0[8], x1[8];
                    unpack8(lo.u, x0);
                    unpack8(hi.u, x1);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        float sn, cs;
                        sincos_reduced(pos * sfreq[ks * 16 + hh * 8 + e], &sn, &cs);
                        const float y0 = x0[e] * cs - x1[e] * sn;
                        const float y1 = x1[e] * cs + x0[e] * sn;
                        x0[e] = y0;
                        x1[e] = y1;
                    }
                    lo.u = pack8(x0);
                    hi.u = pack8(x1);
                    kf[h][ks] = lo.v;
                    kf[h][ks + KS / 2] = hi.v;
                }
            }
        }
        // ---- S^T - m (element e of s[h]: key kb0 + 32 h + (e/4)*8 + hh*4 + e%4, row qi)
        const float start = (m_run == -INFINITY) ? 0.f : -m_run;
        f32x16_t s[NH];
#pragma unroll
        for (int h = 0; h < NH; ++h) {
#pragma unroll
            for (int e = 0; e < 16; ++e) s[h][e] = start;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                s[h] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[h][ks], qf[ks], s[h], 0, 0, 0);
        }
        // ---- V^T operand reads go out under the softmax
        if (more) attn_pipe::vm_wait<NL>();
        else attn_pipe::vm_wait<0>();
        asm volatile("" ::: "memory");
        s4_t vf[KB][DT][2];
#pragma unroll
        for (int tt = 0; tt < DT; ++tt) {
            attn_pipe::read_tr16<0>(vf[0][tt][0], va[tt]);
            attn_pipe::read_tr16<8 * T::kRow>(vf[0][tt][1], va[tt]);
            attn_pipe::read_tr16<16 * T::kRow>(vf[1][tt][0], va[tt]);
            attn_pipe::read_tr16<24 * T::kRow>(vf[1][tt][1], va[tt]);
            if constexpr (KB == 4) {
                attn_pipe::read_tr16<32 * T::kRow>(vf[KB - 2][tt][0], va[tt]);
                attn_pipe::read_tr16<40 * T::kRow>(vf[KB - 2][tt][1], va[tt]);
                attn_pipe::read_tr16<48 * T::kRow>(vf[KB - 1][tt][0], va[tt]);
                attn_pipe::read_tr16<56 * T::kRow>(vf[KB - 1][tt][1], va[tt]);
            }
        }
        // ---- online softmax
        if (kb0 + KT > kv_end || (a.causal && kb0 + KT - 1 > q0 + diag)) {
            const int lim = a.causal ? min(kv_end, qi + diag + 1) : kv_end;
#pragma unroll
            for (int h = 0; h < NH; ++h)
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    s[h][e] = (kb0 + h * 32 + (e / 4) * 8 + hh * 4 + (e % 4) < lim) ? s[h][e] : -INFINITY;
        }
        float mloc = s[0][0];
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int e = 0; e < 16; ++e) mloc = fmaxf(mloc, s[h][e]);
        {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mloc), __float_as_uint(mloc), false, false);
            mloc = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));   // tile max - m_run (or raw before)
        }
        if (__any(m_run == -INFINITY || mloc > lazy)) {
            asm volatile("" ::: "memory");
            // a row may see none of its wave's first tiles: its max stays -inf, its p are 0
            const float m_new = fmaxf(m_run, mloc - start);
            const float alpha = (m_run == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((m_run - m_new) * sc);
            const float shift = (m_new == -INFINITY) ? 0.f : m_new + start;
            l_run *= alpha;
#pragma unroll
            for (int tt = 0; tt < DT; ++tt)
#pragma unroll
                for (int e = 0; e < 16; ++e) oacc[tt][e] *= alpha;
#pragma unroll
            for (int h = 0; h < NH; ++h)
#pragma unroll
                for (int e = 0; e < 16; ++e) s[h][e] -= shift;
            m_run = m_new;
        }
        Pack8 pb[KB];
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            float p[16];
#pragma unroll
            for (int e = 0; e < 16; ++e) p[e] = __builtin_amdgcn_exp2f(s[h][e] * sc);
            pb[2 * h].u = pack8(&p[0]);
            pb[2 * h + 1].u = pack8(&p[8]);
        }
        float psum = 0.f;
#pragma unroll
        for (int b = 0; b < KB; ++b) {
            psum = add_bf16_pair(pb[b].u.x, psum);
            psum = add_bf16_pair(pb[b].u.y, psum);
            psum = add_bf16_pair(pb[b].u.z, psum);
            psum = add_bf16_pair(pb[b].u.w, psum);
        }
        {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(psum), __float_as_uint(psum), false, false);
            l_run += __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
        }
        // ---- O^T += V^T . P^T
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int tt = 0; tt < DT; ++tt) asm volatile("" : "+v"(vf[kb][tt][0]), "+v"(vf[kb][tt][1]));
        if (more) issue_v(kt + KW);
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            if (kb == 2 && kb0 + 32 >= kv_end) break;   // no row of the block sees keys 32..63
#pragma unroll
            for (int tt = 0; tt < DT; ++tt) {
                union {
                    s4_t h[2];
                    bf16x8_t v;
                } vv;
                vv.h[0] = vf[kb][tt][0];
                vv.h[1] = vf[kb][tt][1];
                oacc[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vv.v, pb[kb].v, oacc[tt], 0, 0, 0);
            }
        }
    }

    // ---- merge: every wave leaves its outputs in its own slot (float4 chunk c of row r at
    // c ^ (r & 15): distinct bank groups for the writes, a row per lane, and the reads, a
    // row per 16 or 32 lanes), then each thread combines whole chunks
    {
        float4* part = reinterpret_cast<float4*>(kslot);
#pragma unroll
        for (int tt = 0; tt < DT; ++tt)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                part[ql * CPR + ((tt * 8 + g * 2 + hh) ^ (ql & 15))] =
                    make_float4(oacc[tt][g * 4], oacc[tt][g * 4 + 1], oacc[tt][g * 4 + 2], oacc[tt][g * 4 + 3]);
        if (hh == 0) {
            ml[0][wave][ql] = m_run;
            ml[1][wave][ql] = l_run;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 32 * CPR / (KW * 64); ++i) {
        const int idx = tid + i * KW * 64;
        const int r = idx / CPR, c = idx % CPR;
        float m = ml[0][0][r];
#pragma unroll
        for (int w = 1; w < KW; ++w) m = fmaxf(m, ml[0][w][r]);
        float l = 0.f;
        float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < KW; ++w) {
            // a row whose visible scores are all -inf has no weight in any wave (SCALE_Q calls
            // with more rows run the pipelined kernel, which makes such rows NaN)
            const float x = !SCALE_Q && m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((ml[0][w][r] - m) * sc);
            const float4 v = reinterpret_cast<const float4*>(smem + w * SLOT)[r * CPR + (c ^ (r & 15))];
            l += x * ml[1][w][r];
            acc.x += x * v.x;
            acc.y += x * v.y;
            acc.z += x * v.z;
            acc.w += x * v.w;
        }
        if (q0 + r < a.S) {
            const float inv = (l > 0.f) ? 1.f / l : 0.f;
            uint2 w;
            w.x = pack_bf16x2(acc.x * inv, acc.y * inv);
            w.y = pack_bf16x2(acc.z * inv, acc.w * inv);
            *reinterpret_cast<uint2*>(a.o + (size_t)(q0 + r) * a.o_sn + (size_t)head * a.o_sh + c * 4) = w;
        }
    }
}

}  // namespace efm

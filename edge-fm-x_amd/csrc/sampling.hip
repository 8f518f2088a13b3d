// Temperature / top-p sampling of one fp32 logits row (the non-greedy branch of
// SamplerLayer::forward_sampling, src/layers/sampler.cu:251-298, widened with top-p).
//
// Definition (exact; every mass is an integer so the result is reproducible bit for bit):
//   m    = max_i l_i;  e_i = expf((l_i - m) / T);  w_i = rint(e_i * 2^44)  (uint64)
//   W    = sum_i w_i
//   nucleus = every i when top_p >= 1, else { i : e_i >= tau } where tau is the largest
//          fp32 value with sum_{e_j >= tau} w_j >= max(1, ceil(top_p * W)) (in double)
//   x    = Philox4x32-10(counter = (off_lo, off_hi, 0, 0), key = (seed_lo, seed_hi)).x
//   r    = floor(N * (x >> 8) / 2^24), N = nucleus mass
//   token = the smallest nucleus index i whose inclusive nucleus prefix mass exceeds r.
// e_i <= 1, so w_i <= 2^44 and every sum fits in 64 bits for V < 2^20.
//
// The row is split into blocks of 1024 logits, one 256-thread workgroup each, and the
// passes are separate launches (the launch boundary is the grid-wide barrier):
//   1. block maxima (workgroup 0 also clears the workspace accumulators)
//   2. m from the block maxima; the mass histogram of the top digit of the key of e
//      (device-scope integer atomics: exact and order independent)
//   3-4. each workgroup replays the digit choice of the previous passes from the
//      histograms, then histograms the next digit of the keys that share the chosen prefix
//   5. tau is fixed; every block writes its nucleus mass, and the last block to finish
//      scans the block masses, finds the block holding r and scans its elements.
// With top_p >= 1 passes 2-4 are skipped (tau = 0).
// The key is e's bit pattern (positive fp32 values order like theirs) less that of 2^-45: a
// smaller e has no mass and 1 is the largest, so it has 29 bits, three digits of 10. What
// bounds a call is its launches, 4 to 5 us each, and not the 0.6 MB of logits: with bytes as
// digits (6 launches) and a pass for the total mass (the first histogram's sum) 151936 logits
// took 31.0 us with top_p 0.9 and 14.1 without, now 25.3 and 10.1; 8192 25.0 / 11.1, now 20.7
// / 8.4 (graph replay).
#include "common.hpp"

namespace efm {

constexpr int kSampleThreads = 256;
constexpr int kSamplePer = 4;                                  // logits per thread
constexpr int kSampleBlock = kSampleThreads * kSamplePer;      // logits per workgroup
constexpr int kSampleMaxVocab = 1 << 20;
constexpr int kSampleMaxBlocks = kSampleMaxVocab / kSampleBlock;
constexpr int kSampleDigits = 3, kSampleDigitBits = 10, kSampleBins = 1 << kSampleDigitBits;
constexpr uint32_t kSampleKey0 = (127u - 45u) << 23;           // bits of 2^-45
static_assert(kSampleBins == 4 * kSampleThreads, "a thread scans 4 bins");

// Device workspace of one sampler call (efm_sampler_top_p_workspace_bytes).
struct SampleWs {
    float bmax[kSampleMaxBlocks];
    unsigned long long bmass[kSampleMaxBlocks];
    unsigned long long hist[kSampleDigits][kSampleBins];   // mass by digit
    uint32_t counter;
};

struct SampleArgs {
    const float* logits;
    int V;
    float temperature;
    float top_p;
    uint64_t seed;
    uint64_t offset;
    const int32_t* d_offset;   // optional device-resident addend to `offset`
    int32_t* token_out;
    SampleWs* ws;
    int nblocks;
};

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as easy as
// 1, 2, 3", SC'11): ten rounds of two 32x32->64 multiplies with a Weyl key schedule.
__device__ __forceinline__ uint32_t philox_x0(uint64_t counter, uint64_t key) {
    uint32_t c0 = (uint32_t)counter, c1 = (uint32_t)(counter >> 32), c2 = 0u, c3 = 0u;
    uint32_t k0 = (uint32_t)key, k1 = (uint32_t)(key >> 32);
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t n0 = (uint32_t)(p1 >> 32) ^ c1 ^ k0;
        const uint32_t n2 = (uint32_t)(p0 >> 32) ^ c3 ^ k1;
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return c0;
}

__device__ __forceinline__ float sample_e(float l, float m, float T) { return expf((l - m) / T); }

__device__ __forceinline__ uint64_t sample_w(float e) {
    return (uint64_t)__builtin_rint((double)e * 17592186044416.0);   // 2^44
}

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// Inclusive prefix sum over the 64 lanes of a wave.
__device__ __forceinline__ uint64_t wave_scan_u64(uint64_t v, int lane) {
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const uint64_t o = __shfl_up(v, off, kWave);
        if (lane >= off) v += o;
    }
    return v;
}

// Block-wide reductions of a 256-thread workgroup (4 waves) through LDS.
__device__ __forceinline__ float block_max_f(float v, float* red) {
    v = wave_max(v);
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = v;
    __syncthreads();
    float m = red[0];
#pragma unroll
    for (int w = 1; w < kSampleThreads / kWave; ++w) m = fmaxf(m, red[w]);
    return m;
}

__device__ __forceinline__ uint64_t block_sum_u64(uint64_t v, unsigned long long* red) {
    v = wave_sum_u64(v);
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = v;
    __syncthreads();
    uint64_t s = 0;
#pragma unroll
    for (int w = 0; w < kSampleThreads / kWave; ++w) s += red[w];
    return s;
}

// Exclusive prefix (in thread order) and total of a per-thread value.
__device__ __forceinline__ uint64_t block_scan_u64(uint64_t v, unsigned long long* red, uint64_t* total) {
    const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
    const uint64_t incl = wave_scan_u64(v, lane);
    if (lane == kWave - 1) red[wid] = incl;
    __syncthreads();
    uint64_t before = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kSampleThreads / kWave; ++w) {
        const uint64_t t = red[w];
        if (w < wid) before += t;
        tot += t;
    }
    *total = tot;
    return before + incl - v;
}

// The logits of this workgroup: element k of thread t is index base + t + 256 k.
__device__ __forceinline__ void load_block(const SampleArgs& a, float (&l)[kSamplePer], bool (&ok)[kSamplePer]) {
    const int base = blockIdx.x * kSampleBlock + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kSamplePer; ++k) {
        const int i = base + k * kSampleThreads;
        ok[k] = i < a.V;
        l[k] = ok[k] ? a.logits[i] : -INFINITY;
    }
}

// Global maximum from the block maxima (identical in every workgroup).
__device__ __forceinline__ float global_max(const SampleArgs& a, float* red) {
    float m = -INFINITY;
    for (int b = threadIdx.x; b < a.nblocks; b += kSampleThreads) m = fmaxf(m, a.ws->bmax[b]);
    return block_max_f(m, red);
}

// Replays the digit choices of passes [0, npass): returns the chosen key prefix. Every
// workgroup computes the same values. Thread t owns the bins 1023-4t .. 1020-4t (descending).
__device__ uint32_t select_prefix(const SampleArgs& a, int npass, unsigned long long* red, unsigned long long* s_sel) {
    uint64_t h[kSampleDigits][4];
#pragma unroll
    for (int p = 0; p < kSampleDigits; ++p)
#pragma unroll
        for (int k = 0; k < 4; ++k)
            h[p][k] = p < npass ? a.ws->hist[p][kSampleBins - 1 - 4 * (int)threadIdx.x - k] : 0ull;
    if (threadIdx.x < 2) s_sel[threadIdx.x] = 0ull;
    uint64_t rem = 0;
    uint32_t prefix = 0u;
#pragma unroll
    for (int p = 0; p < kSampleDigits; ++p) {
        if (p >= npass) break;
        const uint64_t own = h[p][0] + h[p][1] + h[p][2] + h[p][3];
        uint64_t W;
        const uint64_t excl = block_scan_u64(own, red, &W);
        if (p == 0) {   // the first histogram holds all of the mass
            rem = (uint64_t)ceil((double)a.top_p * (double)W);
            if (rem < 1) rem = 1;
            if (rem > W) rem = W;
        }
        // exactly one thread's bins hold the rem-th unit of mass
        if (excl < rem && rem <= excl + own) {
            uint64_t acc = excl;
            bool found = false;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (!found && rem <= acc + h[p][k]) {
                    s_sel[0] = (unsigned long long)(kSampleBins - 1 - 4 * (int)threadIdx.x - k);
                    s_sel[1] = rem - acc;
                    found = true;
                }
                acc += h[p][k];
            }
        }
        __syncthreads();
        prefix |= (uint32_t)s_sel[0] << (kSampleDigitBits * (kSampleDigits - 1 - p));
        rem = s_sel[1];
        __syncthreads();
    }
    return prefix;
}

// pass 1: block maxima; workgroup 0 clears the accumulators the later passes add into
__global__ void __launch_bounds__(kSampleThreads) sample_max_kernel(SampleArgs a) {
    __shared__ float red[kSampleThreads / kWave];
    float l[kSamplePer];
    bool ok[kSamplePer];
    load_block(a, l, ok);
    float m = l[0];
#pragma unroll
    for (int k = 1; k < kSamplePer; ++k) m = fmaxf(m, l[k]);
    m = block_max_f(m, red);
    if (threadIdx.x == 0) a.ws->bmax[blockIdx.x] = m;
    if (blockIdx.x == 0) {
        unsigned long long* h = &a.ws->hist[0][0];
        for (int i = threadIdx.x; i < kSampleDigits * kSampleBins; i += kSampleThreads) h[i] = 0ull;
        if (threadIdx.x == 0) a.ws->counter = 0u;
    }
}

// passes 2-4: histograms digit npass of the keys under the prefix chosen so far.
__global__ void __launch_bounds__(kSampleThreads) sample_hist_kernel(SampleArgs a, int npass) {
    __shared__ float red[kSampleThreads / kWave];
    __shared__ unsigned long long redu[kSampleThreads / kWave];
    __shared__ unsigned long long s_hist[kSampleBins];
    __shared__ unsigned long long s_sel[2];
    float l[kSamplePer];
    bool ok[kSamplePer];
    load_block(a, l, ok);
#pragma unroll
    for (int k = 0; k < 4; ++k) s_hist[threadIdx.x + k * kSampleThreads] = 0ull;
    const float m = global_max(a, red);
    const float T = a.temperature;
    const uint32_t prefix = npass > 0 ? select_prefix(a, npass, redu, s_sel) : 0u;
    const int shift = kSampleDigitBits * (kSampleDigits - 1 - npass);
    const uint32_t mask = 0xffffffffu << (shift + kSampleDigitBits);
    __syncthreads();   // s_hist is clear
#pragma unroll
    for (int k = 0; k < kSamplePer; ++k) {
        if (!ok[k]) continue;
        const float e = sample_e(l[k], m, T);
        const uint64_t w = sample_w(e);
        const uint32_t key = __float_as_uint(e) - kSampleKey0;
        if (w != 0 && (npass == 0 || (key & mask) == prefix))
            atomicAdd(&s_hist[(key >> shift) & (kSampleBins - 1)], (unsigned long long)w);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int d = threadIdx.x + k * kSampleThreads;
        const unsigned long long hv = s_hist[d];
        if (hv != 0ull) __hip_atomic_fetch_add(&a.ws->hist[npass][d], hv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// pass 5: nucleus mass per block; the last block to finish locates r.
__global__ void __launch_bounds__(kSampleThreads) sample_locate_kernel(SampleArgs a) {
    __shared__ float red[kSampleThreads / kWave];
    __shared__ unsigned long long redu[kSampleThreads / kWave];
    __shared__ unsigned long long s_sel[2];
    __shared__ uint32_t s_last;
    __shared__ int s_block;
    __shared__ unsigned long long s_base;
    float l[kSamplePer];
    bool ok[kSamplePer];
    load_block(a, l, ok);
    const float m = global_max(a, red);
    const float T = a.temperature;
    const uint32_t tau_key = (a.top_p < 1.0f) ? kSampleKey0 + select_prefix(a, kSampleDigits, redu, s_sel) : 0u;
    uint64_t own = 0;
#pragma unroll
    for (int k = 0; k < kSamplePer; ++k) {
        if (!ok[k]) continue;
        const float e = sample_e(l[k], m, T);
        if (__float_as_uint(e) >= tau_key) own += sample_w(e);
    }
    own = block_sum_u64(own, redu);
    if (threadIdx.x == 0) {
        // publish the block mass, wait for that atomic to return (it is then performed
        // where every XCD's atomics meet), then count in: no cache flush needed, and the
        // last block reads every mass with agent-scope atomic loads
        const uint64_t old =
            __hip_atomic_exchange(&a.ws->bmass[blockIdx.x], own, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" : : "v"(old) : "memory");
        const uint32_t prev = __hip_atomic_fetch_add(&a.ws->counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = (prev == (uint32_t)a.nblocks - 1) ? 1u : 0u;
        s_block = 0;   // no block holds r where the logits have no mass (NaN)
        s_base = 0ull;
    }
    __syncthreads();
    if (!s_last) return;

    // last block: N, r, the block that holds r (blocks in index order) ...
    const int per = (a.nblocks + kSampleThreads - 1) / kSampleThreads;   // <= 4
    const int b0 = threadIdx.x * per;
    uint64_t bm[4] = {0ull, 0ull, 0ull, 0ull}, mine = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (k < per && b0 + k < a.nblocks)
            bm[k] = __hip_atomic_load(&a.ws->bmass[b0 + k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        mine += bm[k];
    }
    uint64_t N;
    const uint64_t excl = block_scan_u64(mine, redu, &N);
    uint64_t off = a.offset;
    if (a.d_offset != nullptr) off += (uint64_t)(uint32_t)a.d_offset[0];
    const uint64_t bits = philox_x0(off, a.seed) >> 8;
    const uint64_t r = (__umul64hi(N, bits) << 40) | ((N * bits) >> 24);
    if (mine != 0 && excl <= r && r < excl + mine) {
        uint64_t acc = excl;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (acc <= r && r < acc + bm[k]) {
                s_block = b0 + k;
                s_base = acc;
            }
            acc += bm[k];
        }
    }
    __syncthreads();
    // ... then the element: thread t covers indices [4t, 4t + 4) of that block
    const int blk = s_block;
    const int i0 = blk * kSampleBlock + threadIdx.x * kSamplePer;
    uint64_t w4[kSamplePer], tm = 0;
#pragma unroll
    for (int k = 0; k < kSamplePer; ++k) {
        const int i = i0 + k;
        w4[k] = 0;
        if (i < a.V) {
            const float e = sample_e(a.logits[i], m, T);
            if (__float_as_uint(e) >= tau_key) w4[k] = sample_w(e);
        }
        tm += w4[k];
    }
    uint64_t btot;
    const uint64_t ex = s_base + block_scan_u64(tm, redu, &btot);
    if (tm != 0 && ex <= r && r < ex + tm) {
        uint64_t acc = ex;
        int tok = i0 + kSamplePer - 1;
#pragma unroll
        for (int k = 0; k < kSamplePer; ++k) {
            acc += w4[k];
            if (acc > r) {
                tok = i0 + k;
                break;
            }
        }
        a.token_out[0] = tok;
    }
    if (threadIdx.x == 0) a.ws->counter = 0u;
}

}  // namespace efm

using namespace efm;

extern "C" size_t efm_sampler_top_p_workspace_bytes(int64_t vocab) {
    (void)vocab;
    return (sizeof(SampleWs) + 255) & ~(size_t)255;
}

extern "C" int efm_sampler_top_p(int64_t vocab, const float* logits, float temperature, float top_p, uint64_t seed,
                                 uint64_t offset, const int32_t* d_offset, int32_t* token_out, void* workspace,
                                 size_t workspace_bytes, hipStream_t stream) {
    if (logits == nullptr || token_out == nullptr)
        return set_error(EFM_ERR_INVALID_ARGUMENT, "sampler_top_p: null pointer");
    if (vocab <= 0 || vocab >= kSampleMaxVocab)   // V < 2^20 keeps W = sum w_i < 2^64
        return set_error(EFM_ERR_INVALID_ARGUMENT, "sampler_top_p: vocab %lld outside [1, %d)", (long long)vocab,
                         kSampleMaxVocab);
    if (!(temperature >= 1e-6f) || !(temperature < INFINITY))
        return set_error(EFM_ERR_INVALID_ARGUMENT,
                         "sampler_top_p: temperature must be finite and >= 1e-6 (below that sampling is greedy)");
    if (!(top_p > 0.0f))
        return set_error(EFM_ERR_INVALID_ARGUMENT, "sampler_top_p: top_p must be > 0");
    if (workspace == nullptr || workspace_bytes < sizeof(SampleWs))
        return set_error(EFM_ERR_WORKSPACE, "sampler_top_p: workspace of %zu bytes required", sizeof(SampleWs));
    const int nb = (int)((vocab + kSampleBlock - 1) / kSampleBlock);
    SampleArgs a{logits, (int)vocab, temperature, top_p, seed, offset, d_offset, token_out,
                 static_cast<SampleWs*>(workspace), nb};
    hipLaunchKernelGGL(sample_max_kernel, dim3(nb), dim3(kSampleThreads), 0, stream, a);
    for (int p = 0; top_p < 1.0f && p < kSampleDigits; ++p)
        hipLaunchKernelGGL(sample_hist_kernel, dim3(nb), dim3(kSampleThreads), 0, stream, a, p);
    hipLaunchKernelGGL(sample_locate_kernel, dim3(nb), dim3(kSampleThreads), 0, stream, a);
    return check_launch("sampler_top_p");
}

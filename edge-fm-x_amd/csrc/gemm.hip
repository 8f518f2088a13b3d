// Prefill projections on the gfx950 matrix cores: C[M, N] = A[M, K] . B[N, K]^T in
// bf16 with fp32 accumulation (v_mfma_f32_32x32x16_bf16, 16x16x32 in the tall kernel). A
// holds activations (one row per token) and B the weights in their [out, in] layout, so both
// operands are K-contiguous and feed the MFMA lanes with 16-byte loads.
//
//  * K % 64 == 0 (every Qwen2.5 projection), kernels fed by global_load_lds DMA into
//    XOR-swizzled LDS rings, operand reads software-pipelined against the MFMAs and a
//    grouped tile order per XCD:
//      - the tall kernel: 256 x 256 or 192 x 256 tiles, one 4-wave workgroup per CU;
//      - the pipelined kernel: 128 x 128 (128 x 64, 64 x 64) tiles, two 4-wave
//        workgroups per CU (few tiles), plus its split-K form.
//    A cost model (rounds of resident workgroups) picks between them.
//  * The same K, few rows or few tiles: the K-split kernel, whose four waves take a quarter
//    of K each over 32 x 32 to 64 x 64 tiles.
//  * Other K: a register-staged kernel with a padded LDS row pitch (40 bf16).
//  * Epilogues: bf16 (+bias, the cuBLASLt BIAS epilogue), fp32, and SwiGLU, where the
//    B tile interleaves 32-row blocks of up and gate weights so that each lane holds u
//    and g of the same output element: out = bf16(silu(bf16(g)) * bf16(u)).
//  * Every kernel sums each output's keys 16 at a time in increasing order, so results
//    are bit-identical across kernels and tile shapes (K-split and split-K aside, which add
//    the sums of contiguous ranges of K in order).
#include "common.hpp"

#include <algorithm>
#include <type_traits>
#include <utility>
#include <cstdlib>

namespace efm {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

enum { GEPI_BF16 = 0, GEPI_F32 = 1, GEPI_SWIGLU = 2, GEPI_PARTIAL = 3 };

constexpr int kGemmThreads = 256;
constexpr int kBK = 32;
constexpr int kPitch = kBK + 8;  // LDS row pitch in bf16

template <int BM, int BN, int EPI>
__global__ __launch_bounds__(kGemmThreads) void gemm_bf16_kernel(const bf16_t* __restrict__ A,
                                                                 const bf16_t* __restrict__ B,
                                                                 const bf16_t* __restrict__ bias, void* __restrict__ Cout,
                                                                 int M, int N, int K, int ldc) {
    constexpr int WM = BM / 2, WN = BN / 2;        // wave tile
    constexpr int TM = WM / 32, TN = WN / 32;      // MFMA tiles per wave
    constexpr int ACH = BM * kBK / 8;              // 16-byte chunks per A slab
    constexpr int BCH = BN * kBK / 8;
    constexpr int AL = (ACH + kGemmThreads - 1) / kGemmThreads;
    constexpr int BL = (BCH + kGemmThreads - 1) / kGemmThreads;
    static_assert(TM >= 1 && TN >= 1, "tile too small");
    static_assert(EPI != GEPI_SWIGLU || TN % 2 == 0, "SwiGLU needs paired N tiles");

    __shared__ __align__(16) bf16_t As[2][BM * kPitch];
    __shared__ __align__(16) bf16_t Bs[2][BN * kPitch];

    const int tid = threadIdx.x;
    const int wave = tid / kWave, lane = tid % kWave;
    const int wm = wave / 2, wn = wave % 2;
    const int m0 = blockIdx.x * BM;
    // For SwiGLU the output tile is BN/2 columns wide; B rows interleave 32-row blocks
    // of up (even blocks) and gate (odd blocks) weights.
    const int n0 = (EPI == GEPI_SWIGLU) ? blockIdx.y * (BN / 2) : blockIdx.y * BN;

    auto b_row = [&](int r) -> int {
        if (EPI == GEPI_SWIGLU) {
            const int blk = r / 32;
            const int col = n0 + (blk / 2) * 32 + (r % 32);
            return (col < N) ? ((blk % 2 == 0) ? col : N + col) : -1;
        }
        const int n = n0 + r;
        return (n < N) ? n : -1;
    };

    uint4 ra[AL], rb[BL];
    auto gload = [&](int k0) {
#pragma unroll
        for (int i = 0; i < AL; ++i) {
            const int c = tid + i * kGemmThreads;
            const int r = c / (kBK / 8), kc = c % (kBK / 8);
            ra[i] = (c < ACH && m0 + r < M) ? *reinterpret_cast<const uint4*>(A + (size_t)(m0 + r) * K + k0 + kc * 8)
                                            : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < BL; ++i) {
            const int c = tid + i * kGemmThreads;
            const int r = c / (kBK / 8), kc = c % (kBK / 8);
            const int br = (c < BCH) ? b_row(r) : -1;
            rb[i] = (br >= 0) ? load_stream16(B + (size_t)br * K + k0 + kc * 8) : make_uint4(0, 0, 0, 0);
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int i = 0; i < AL; ++i) {
            const int c = tid + i * kGemmThreads;
            if (c < ACH) {
                const int r = c / (kBK / 8), kc = c % (kBK / 8);
                *reinterpret_cast<uint4*>(&As[buf][r * kPitch + kc * 8]) = ra[i];
            }
        }
#pragma unroll
        for (int i = 0; i < BL; ++i) {
            const int c = tid + i * kGemmThreads;
            if (c < BCH) {
                const int r = c / (kBK / 8), kc = c % (kBK / 8);
                *reinterpret_cast<uint4*>(&Bs[buf][r * kPitch + kc * 8]) = rb[i];
            }
        }
    };

    f32x16_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    const int nk = K / kBK;
    gload(0);
    lstore(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) gload((kt + 1) * kBK);
#pragma unroll
        for (int ks = 0; ks < kBK / 16; ++ks) {
            bf16x8_t af[TM], bfr[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int r = wm * WM + i * 32 + (lane % 32);
                af[i] = *reinterpret_cast<const bf16x8_t*>(&As[buf][r * kPitch + ks * 16 + (lane / 32) * 8]);
            }
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int r = wn * WN + j * 32 + (lane % 32);
                bfr[j] = *reinterpret_cast<const bf16x8_t*>(&Bs[buf][r * kPitch + ks * 16 + (lane / 32) * 8]);
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) {
            lstore(buf ^ 1);
        }
        __syncthreads();
    }

    // Epilogue. Accumulator element e of tile (i, j): row = (e/4)*8 + (lane/32)*4 + e%4,
    // column = lane % 32 within the 32 x 32 tile.
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int row = m0 + wm * WM + i * 32 + (e / 4) * 8 + (lane / 32) * 4 + (e % 4);
            if (row >= M) continue;
            if (EPI == GEPI_SWIGLU) {
#pragma unroll
                for (int j = 0; j < TN; j += 2) {
                    const int col = n0 + ((wn * WN + j * 32) / 64) * 32 + (lane % 32);
                    if (col < N) {
                        const float u = round_bf16(acc[i][j][e]);
                        const float g = round_bf16(acc[i][j + 1][e]);
                        const float o = silu_f32(g) * u;
                        reinterpret_cast<bf16_t*>(Cout)[(size_t)row * ldc + col] = (bf16_t)f32_to_bf16(o);
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int col = n0 + wn * WN + j * 32 + (lane % 32);
                    if (col >= N) continue;
                    float v = acc[i][j][e];
                    if (bias != nullptr) v += bf16_to_f32(bias[col]);
                    if (EPI == GEPI_F32) reinterpret_cast<float*>(Cout)[(size_t)row * ldc + col] = v;
                    else reinterpret_cast<bf16_t*>(Cout)[(size_t)row * ldc + col] = (bf16_t)f32_to_bf16(v);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------
// Pipelined variant for K % 64 == 0: K slabs of 64 stream global -> LDS with
// global_load_lds (no staging registers) into an S-deep ring, so S - 1 slabs are in
// flight while the matrix cores work on one. Each wave's 1 KB DMA load covers 8 rows x 128
// bytes; lane l fetches chunk (l % 8) ^ pipe_swz(row) of its row, so the ring holds an
// XOR-swizzled layout and the 32-row MFMA operand reads spread over the LDS banks. The
// operand reads are issued as ds_read_b128 with explicit waits: each wave waits for its
// own DMA loads of the slab (vmcnt, counted exactly: every wave issues LPW loads per slab)
// and a workgroup barrier makes all waves' loads visible. Tiles are assigned XCD by XCD
// (dispatch is round-robin over the 8 XCDs), so workgroups that share weight columns
// share an L2.
// ---------------------------------------------------------------------------------
// Tile order within one XCD's contiguous range of tile indices: groups of kGroupM row
// tiles are walked column by column, so the workgroups resident on an XCD at one time
// cover a kGroupM x (resident / kGroupM) block of output tiles and share its A and B
// slabs in that XCD's L2 (walking M first, as a plain index split does, re-reads a fresh
// A slab for every tile once M spans many tiles).
constexpr int kGroupM = 8;
__device__ __forceinline__ void tile_of(int t, int mt, int nt, int& tm, int& tn) {
    const int in_group = kGroupM * nt;
    const int first = (t / in_group) * kGroupM;
    const int gm = min(mt - first, kGroupM);
    const int r = t % in_group;
    tm = first + r % gm;
    tn = r / gm;
}

// LDS swizzles. gfx950's LDS has 64 four-byte banks and serves a ds_read_b128 sixteen
// lanes at a time: the 16 rows an MFMA operand read touches at once must land in 16
// distinct 16-byte bank groups. With 128-byte rows (8 chunks) two rows fill the 256-byte
// bank period, so rows of equal parity need distinct chunks: (row / 2) % 8, with the
// parity folded into bit 2 so that any 8 consecutive rows also differ.
__device__ __forceinline__ int pipe_swz(int row) { return ((row >> 1) ^ ((row & 1) << 2)) & 7; }

constexpr int kPBK = 64;            // K per slab
constexpr int kPRow = kPBK * 2;     // bytes per operand row in LDS

template <int N>
__device__ __forceinline__ void vm_wait() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Waits until at most `slabs` slabs of LPW loads are in flight (the counter holds 63: past
// that the wait is for fewer).
constexpr int vm_count(int loads) { return loads < 63 ? loads : 63; }
template <int LPW>
__device__ __forceinline__ void vm_wait_slabs(int slabs) {
    switch (slabs) {
        case 0: vm_wait<0>(); break;
        case 1: vm_wait<vm_count(1 * LPW)>(); break;
        case 2: vm_wait<vm_count(2 * LPW)>(); break;
        case 3: vm_wait<vm_count(3 * LPW)>(); break;
        case 4: vm_wait<vm_count(4 * LPW)>(); break;
        case 5: vm_wait<vm_count(5 * LPW)>(); break;
        default: vm_wait<vm_count(6 * LPW)>(); break;
    }
}

template <int BM, int BN, int S, int EPI>
__global__ __launch_bounds__(kGemmThreads) void gemm_pipe_kernel(const bf16_t* __restrict__ A,
                                                                 const bf16_t* __restrict__ B,
                                                                 const bf16_t* __restrict__ bias,
                                                                 void* __restrict__ Cout, int M, int N, int K, int ldc,
                                                                 int mt, int nt, int ksplit, int kt_per) {
    constexpr int WM = BM / 2, WN = BN / 2;
    constexpr int TM = WM / 32, TN = WN / 32;
    constexpr int STAGE = (BM + BN) * kPRow;
    constexpr int QA = BM / 8, QB = BN / 8;  // 1 KB wave loads per operand per slab
    constexpr int LPW = (QA + QB) / 4;       // wave loads per wave per slab
    static_assert((QA + QB) % 4 == 0 && S >= 2 && S <= 8 && (S - 2) * LPW <= 63, "bad pipeline shape");
    static_assert(EPI != GEPI_SWIGLU || TN % 2 == 0, "SwiGLU needs paired N tiles");
    __shared__ __align__(1024) unsigned char smem[S * STAGE];

    // split-K (GEPI_PARTIAL): work unit t covers K slice t / (mt * nt), slabs
    // [slice * kt_per, (slice + 1) * kt_per), and writes fp32 partial sums
    const int T = mt * nt * ksplit;
    const int per = (T + 7) / 8;
    const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (t >= T) return;
    const int slice = t / (mt * nt);
    int tm, tn;
    tile_of(t % (mt * nt), mt, nt, tm, tn);
    const int kt0 = slice * kt_per;
    const int m0 = tm * BM;
    const int n0 = (EPI == GEPI_SWIGLU) ? tn * (BN / 2) : tn * BN;

    const int tid = threadIdx.x;
    const int wave = tid / kWave, lane = tid % kWave;
    const int wm = wave / 2, wn = wave % 2;
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)smem);

    auto b_row = [&](int r) -> int {
        if (EPI == GEPI_SWIGLU) {
            const int blk = r / 32;
            const int col = n0 + (blk / 2) * 32 + (r % 32);
            return (col < N) ? ((blk % 2 == 0) ? col : N + col) : -1;
        }
        const int n = n0 + r;
        return (n < N) ? n : -1;
    };

    auto issue = [&](int kk, int slot) {
        const int k0 = (kt0 + kk) * kPBK;
        const int rr = lane >> 3, cs = lane & 7;
#pragma unroll
        for (int i = 0; i < LPW; ++i) {
            const int q = wave + i * 4;
            const bf16_t* src;
            if (q < QA) {
                const int row = min(m0 + q * 8 + rr, M - 1);
                src = A + (size_t)row * K + k0 + ((cs ^ pipe_swz(q * 8 + rr)) << 3);
            } else {
                int br = b_row((q - QA) * 8 + rr);
                if (br < 0) br = 0;
                src = B + (size_t)br * K + k0 + ((cs ^ pipe_swz(q * 8 + rr)) << 3);
            }
            __builtin_amdgcn_global_load_lds(
                static_cast<const void*>(src),
                (__attribute__((address_space(3))) void*)(smem + slot * STAGE + q * 1024), 16, 0, 0);
        }
    };

    f32x16_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    // Operand reads of one 16-key step: TM A fragments and TN B fragments (ds_read_b128).
    auto read_step = [&](uint32_t base, int ks, bf16x8_t (&af)[TM], bf16x8_t (&bfr)[TN]) {
        const int c = ks * 2 + (lane >> 5);
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int r = wm * WM + i * 32 + (lane & 31);
            const uint32_t addr = base + (uint32_t)(r * kPRow + ((c ^ pipe_swz(r)) << 4));
            asm volatile("ds_read_b128 %0, %1" : "=v"(af[i]) : "v"(addr) : "memory");
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int r = wn * WN + j * 32 + (lane & 31);
            const uint32_t addr = base + (uint32_t)(BM * kPRow + r * kPRow + ((c ^ pipe_swz(r)) << 4));
            asm volatile("ds_read_b128 %0, %1" : "=v"(bfr[j]) : "v"(addr) : "memory");
        }
    };
    // Software pipeline over the slab's four 16-key steps: the reads of step ks + 2 are
    // issued behind the MFMAs of step ks, so LDS latency hides behind matrix work within
    // the wave. The fragments come from inline-asm reads the compiler cannot track: each
    // step waits for its own reads (lgkmcnt = the reads issued after them), then passes
    // its fragments through an asm "write" so that no MFMA is scheduled above the wait.
    auto compute = [&](int slot) {
        const uint32_t base = lds0 + (uint32_t)(slot * STAGE);
        constexpr int KSN = kPBK / 16;
        constexpr int RPS = TM + TN;   // reads per step
        static_assert(RPS <= 15, "lgkmcnt holds at most 15 outstanding reads");
        bf16x8_t af[KSN][TM], bfr[KSN][TN];
        read_step(base, 0, af[0], bfr[0]);
        read_step(base, 1, af[1], bfr[1]);
#pragma unroll
        for (int ks = 0; ks < KSN; ++ks) {
            if (ks + 1 < KSN) asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(RPS) : "memory");
            else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int i = 0; i < TM; ++i) asm volatile("" : "+v"(af[ks][i]));
#pragma unroll
            for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(bfr[ks][j]));
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[ks][i], bfr[ks][j], acc[i][j], 0, 0, 0);
            if (ks + 2 < KSN) read_step(base, ks + 2, af[ks + 2], bfr[ks + 2]);
        }
    };

    const int nk = min(K / kPBK, kt0 + kt_per) - kt0;
    const int pre = min(S - 1, nk);
    for (int p = 0; p < pre; ++p) issue(p, p);
    for (int kt = 0; kt < nk; ++kt) {
        // Own DMA loads of slab kt have landed in LDS; the bare barrier (no fence, which
        // would drain every slab in flight) then orders them before all waves' reads, and
        // all waves' reads of slot (kt - 1) % S before it is refilled below.
        vm_wait_slabs<LPW>(min(S - 2, nk - 1 - kt));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (kt + S - 1 < nk) issue(kt + S - 1, (kt + S - 1) % S);
        compute(kt % S);
    }

    // Epilogue. Accumulator element e of tile (i, j): row = (e/4)*8 + (lane/32)*4 + e%4,
    // column = lane % 32 within the 32 x 32 tile.
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int row = m0 + wm * WM + i * 32 + (e / 4) * 8 + (lane / 32) * 4 + (e % 4);
            if (row >= M) continue;
            if (EPI == GEPI_SWIGLU) {
#pragma unroll
                for (int j = 0; j < TN; j += 2) {
                    const int col = n0 + ((wn * WN + j * 32) / 64) * 32 + (lane % 32);
                    if (col < N) {
                        const float u = round_bf16(acc[i][j][e]);
                        const float g = round_bf16(acc[i][j + 1][e]);
                        const float o = silu_f32(g) * u;
                        reinterpret_cast<bf16_t*>(Cout)[(size_t)row * ldc + col] = (bf16_t)f32_to_bf16(o);
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    const int col = n0 + wn * WN + j * 32 + (lane % 32);
                    if (col >= N) continue;
                    float v = acc[i][j][e];
                    if (EPI == GEPI_PARTIAL) {
                        reinterpret_cast<float*>(Cout)[((size_t)slice * M + row) * N + col] = v;
                        continue;
                    }
                    if (bias != nullptr) v += bf16_to_f32(bias[col]);
                    if (EPI == GEPI_F32) reinterpret_cast<float*>(Cout)[(size_t)row * ldc + col] = v;
                    else reinterpret_cast<bf16_t*>(Cout)[(size_t)row * ldc + col] = (bf16_t)f32_to_bf16(v);
                }
            }
        }
    }
}

template <int OFF>
__device__ __forceinline__ bf16x8_t ds_read16(uint32_t addr) {
    bf16x8_t d;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(d) : "v"(addr), "n"(OFF) : "memory");
    return d;
}

template <int N>
__device__ __forceinline__ void lgkm_wait() {
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}

// ---------------------------------------------------------------------------------
// Tall kernel (launches that fill the chip): 256 x 256 (192 x 256) tiles, one workgroup per
// CU, four waves, one per SIMD, each owning a 128 x 128 (96 x 128) block of 16 x 16 MFMA
// tiles in 256 (192) accumulator registers.
//  * What bounds it is the card's power: on zero operands the same launches run at 1.6-1.7
//    PF/s, on N(0, 1) ones at 1.3-1.4, and removing the DMA or the operand reads changes the
//    rate through what they consume. So the layout moves as little as it can: a 128 x 128
//    block reads two thirds of the LDS bytes per MFMA of a 128 x 64 one, rows of 64 keys
//    are whole 128-byte lines, buffer loads carry 32-bit offsets, and the 16 x 16 x 32 MFMA
//    sustains 1.97 PF/s on random operands where the 32 x 32 x 16 one sustains 1.65 (2 waves
//    a SIMD; the two give the same bits).
//  * 64-key operand slabs (32 KB) in a ring of five slots, A and B in turn. Step 0 of slab s
//    runs with its second half's operand reads and the loads of A(s + 2); then one barrier
//    (slab s is in registers everywhere, slab s + 1 has landed), and step 1 runs with the
//    first reads of slab s + 1 and the loads of B(s + 2) into the slot that A(s) has left.
//  * The weight rows are the MFMA's first operand: a lane ends with four consecutive columns
//    of one row. SwiGLU interleaves 16-row blocks of up and gate weights.
//  Measured against the 8-wave 32 x 32 x 16 kernel over 32-key stages that it replaces (us):
//  4096 x 3584 -> 2 x 18944 SwiGLU 1103 -> 855 (1.30 PF/s), 4096 x 18944 -> 3584 515 -> 436,
//  4096 x 3584 -> 4608 156 -> 129, 512 x 1536 -> 2 x 8960 38.8 -> 33.6.
// ---------------------------------------------------------------------------------
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void tall_load(const unsigned char* src, uint32_t off, unsigned char* dst) {
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(src), (short)0, 0x7fffffff, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)dst, 16, (int)off, 0, 0, 0);
}

template <int TM, int TN>
struct TallFrags {
    bf16x8_t a[TM], b[TN];
};

// Keeps the accumulators in their AGPRs at this point: otherwise the compiler may move them
// about inside the loop.
template <int TM, int TN>
__device__ __forceinline__ void pin_acc(f32x4_t (&acc)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) asm volatile("" : "+a"(acc[i][j]));
}

template <int TM, int EPI>
__global__ __launch_bounds__(256, 1) void gemm_tall_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
                                                           const bf16_t* __restrict__ bias, void* __restrict__ Cout,
                                                           int M, int N, int K, int ldc, int mt, int nt, int vec) {
    constexpr int TN = 8, BM = 32 * TM, BN = 256;   // a wave: TM x TN tiles of 16 x 16
    constexpr int SLOT = 256 * kPRow;               // one operand slab (64 keys), 32 KB
    constexpr int LA = BM / 32, LB = BN / 32;       // 1 KB wave loads per operand slab and wave
    __shared__ __align__(1024) unsigned char smem[5 * SLOT];

    const int T = mt * nt;
    const int per = (T + 7) / 8;
    const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (t >= T) return;
    int tm, tn;
    tile_of(t, mt, nt, tm, tn);
    const int m0 = tm * BM;
    const int n0 = (EPI == GEPI_SWIGLU) ? tn * (BN / 2) : tn * BN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int wm = wave >> 1, wn = wave & 1;

    uint32_t va[LA], vb[LB];
    {
        const int rr = lane >> 3, cs = lane & 7;
#pragma unroll
        for (int i = 0; i < LA; ++i) {
            const int r = (i * 4 + wave) * 8 + rr;
            va[i] = (uint32_t)((min(m0 + r, M - 1) * K + ((cs ^ pipe_swz(r)) << 3)) * 2);
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int r = (i * 4 + wave) * 8 + rr;
            int row;
            if (EPI == GEPI_SWIGLU) {   // 16-row blocks of up (even) and gate (odd) weights
                const int blk = r / 16;
                row = min(n0 + (blk / 2) * 16 + r % 16, N - 1) + (blk % 2) * N;
            } else {
                row = min(n0 + r, N - 1);
            }
            vb[i] = (uint32_t)((row * K + ((cs ^ pipe_swz(r)) << 3)) * 2);
        }
    }
    const int nk = K / kPBK;
    const unsigned char* pa = reinterpret_cast<const unsigned char*>(A);
    const unsigned char* pb = reinterpret_cast<const unsigned char*>(B);
    // operand slab q: A of slab q / 2 (even) or B (odd), in slot q % 5; slabs past the end
    // repeat the last one (never read, so that every step issues the same loads)
    auto slot = [&](int q) { return smem + (q % 5) * SLOT + wave * 1024; };
    auto src_a = [&](int s) { return pa + min(s, nk - 1) * kPRow; };
    auto src_b = [&](int s) { return pb + min(s, nk - 1) * kPRow; };

    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)smem);
    const int r16 = lane & 15;
    uint32_t ra[2], rb[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t c = (uint32_t)(((h * 4 + (lane >> 4)) ^ pipe_swz(r16)) << 4);
        ra[h] = lds0 + (uint32_t)((wm * (BM / 2) + r16) * kPRow) + c;
        rb[h] = lds0 + (uint32_t)((wn * (BN / 2) + r16) * kPRow) + c;
    }
    typedef TallFrags<TM, TN> Frags;
    auto tie = [&](Frags& f) {
#pragma unroll
        for (int i = 0; i < TM; ++i) asm volatile("" : "+v"(f.a[i]));
#pragma unroll
        for (int j = 0; j < TN; ++j) asm volatile("" : "+v"(f.b[j]));
    };
    auto read_one = [&](auto ic, Frags& f, uint32_t a, uint32_t b) {
        constexpr int I = decltype(ic)::value;
        if constexpr (I < TN) f.b[I] = ds_read16<I * 16 * kPRow>(b);
        else if constexpr (I < TN + TM) f.a[I - TN] = ds_read16<(I - TN) * 16 * kPRow>(a);
    };

    f32x4_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.f;
    pin_acc(acc);

#pragma unroll
    for (int i = 0; i < LA; ++i) tall_load(src_a(0), va[i], slot(0) + i * 4096);
#pragma unroll
    for (int i = 0; i < LB; ++i) tall_load(src_b(0), vb[i], slot(1) + i * 4096);
#pragma unroll
    for (int i = 0; i < LA; ++i) tall_load(src_a(1), va[i], slot(2) + i * 4096);
#pragma unroll
    for (int i = 0; i < LB; ++i) tall_load(src_b(1), vb[i], slot(3) + i * 4096);
    vm_wait<LA + LB>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Frags f0, f1;
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (read_one(std::integral_constant<int, I>{}, f0, ra[0], rb[0] + SLOT), ...);
    }(std::make_integer_sequence<int, TM + TN>{});

    // one 32-key step: MFMA I, then behind every second one of the first 2 (TM + TN) an
    // operand read of the next step, and behind the odd ones the step's DMA loads
    auto mma_step = [&](Frags& f, Frags& g, uint32_t na, uint32_t nb, auto&& dma) {
        [&]<int... I>(std::integer_sequence<int, I...>) {
            ((acc[I / TN][I % TN] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.b[I % TN], f.a[I / TN], acc[I / TN][I % TN],
                                                                            0, 0, 0),
              read_one(std::integral_constant<int, (I % 2 == 0 ? I / 2 : 99)>{}, g, na, nb),
              dma(std::integral_constant<int, I>{}), __builtin_amdgcn_sched_barrier(0)),
             ...);
        }(std::make_integer_sequence<int, TM * TN>{});
    };
    for (int s = 0; s < nk; ++s) {
        const uint32_t sa = (uint32_t)(((2 * s) % 5) * SLOT), sb = (uint32_t)(((2 * s + 1) % 5) * SLOT);
        const uint32_t xa = (uint32_t)(((2 * s + 2) % 5) * SLOT), xb = (uint32_t)(((2 * s + 3) % 5) * SLOT);
        const unsigned char* ga = src_a(s + 2);
        unsigned char* da = slot(2 * s + 4);
        lgkm_wait<0>();
        tie(f0);
        mma_step(f0, f1, ra[1] + sa, rb[1] + sb, [&](auto ic) {
            constexpr int I = decltype(ic)::value;
            if constexpr (I % 4 == 3 && I / 4 < LA) tall_load(ga, va[I / 4], da + (I / 4) * 4096);
        });
        // slab s is in registers, slab s + 1 has landed for every wave
        const unsigned char* gb = src_b(s + 2);
        unsigned char* db = slot(2 * s + 5);
        lgkm_wait<0>();
        tie(f1);
        vm_wait<LA>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        mma_step(f1, f0, ra[0] + xa, rb[0] + xb, [&](auto ic) {
            constexpr int I = decltype(ic)::value;
            if constexpr (I % 4 == 3 && I / 4 < LB) tall_load(gb, vb[I / 4], db + (I / 4) * 4096);
        });
        pin_acc(acc);
    }
    lgkm_wait<0>();
    tie(f0);
    vm_wait<0>();
    __syncthreads();   // every wave is done with the operand slots

    // Epilogue, half of the wave's row blocks at a time: the partial tile goes through the
    // wave's own 32 KB slot as fp32 (element e of tile (i, j): row 16 i + lane % 16, column
    // 16 j + (lane / 16) * 4 + e; float4 chunk c of row r at c ^ (r % 16): distinct bank
    // groups), so that the stores are whole row segments, 16 lanes to a row.
    constexpr int H = TM / 2;
    float4* const part = reinterpret_cast<float4*>(smem + wave * SLOT);
    const int seg = lane & 15;
    const int col = n0 + wn * (EPI == GEPI_SWIGLU ? 64 : 128) + seg * (EPI == GEPI_SWIGLU ? 4 : 8);
    float bv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
        bv[e] = (EPI != GEPI_SWIGLU && bias != nullptr && col + e < N) ? bf16_to_f32(bias[col + e]) : 0.f;
    auto half = [&](auto hc) {
        constexpr int i0 = decltype(hc)::value * H;
#pragma unroll
        for (int i = 0; i < H; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const f32x4_t x = acc[i0 + i][j];
                part[(i * 16 + r16) * 32 + ((j * 4 + (lane >> 4)) ^ r16)] = make_float4(x[0], x[1], x[2], x[3]);
            }
#pragma unroll 4
        for (int q = 0; q < H * 4; ++q) {
            const int r = q * 4 + (lane >> 4);
            const int row = m0 + wm * (BM / 2) + i0 * 16 + r, sw = r & 15;
            constexpr int NV = EPI == GEPI_SWIGLU ? 4 : 8;
            const int c0 = EPI == GEPI_SWIGLU ? (seg >> 2) * 8 + (seg & 3) : seg * 2;
            const float4 x = part[r * 32 + (c0 ^ sw)], y = part[r * 32 + ((c0 + (EPI == GEPI_SWIGLU ? 4 : 1)) ^ sw)];
            float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
            for (int e = 0; e < NV; ++e) {
                if constexpr (EPI == GEPI_SWIGLU) v[e] = silu_f32(round_bf16(v[4 + e])) * round_bf16(v[e]);
                else if (bias != nullptr) v[e] += bv[e];
            }
            if (row >= M) continue;
            const size_t at = (size_t)row * ldc + col;
            if constexpr (EPI == GEPI_F32) {
                float* o = reinterpret_cast<float*>(Cout) + at;
                if (vec) {
                    if (col < N) {
                        *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
                        *reinterpret_cast<float4*>(o + 4) = make_float4(v[4], v[5], v[6], v[7]);
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < NV; ++e)
                        if (col + e < N) o[e] = v[e];
                }
            } else {
                bf16_t* o = reinterpret_cast<bf16_t*>(Cout) + at;
                if (vec) {
                    if (col < N) {
                        if constexpr (NV == 8) *reinterpret_cast<uint4*>(o) = pack8(v);
                        else *reinterpret_cast<uint2*>(o) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < NV; ++e)
                        if (col + e < N) o[e] = (bf16_t)f32_to_bf16(v[e]);
                }
            }
        }
    };
    half(std::integral_constant<int, 0>{});
    half(std::integral_constant<int, 1>{});
}

// ---------------------------------------------------------------------------------
// K split over the waves of a workgroup: for launches whose tiles are too few to keep the
// CUs busy by themselves. The pipelined kernel's four waves share every slab, so one wave
// runs a single 32 x 32 MFMA tile (64 x 64 workgroup tiles) between two barriers: 512 x
// 1536 -> 2048 takes 24 slabs at 0.5 us. Here each of KW waves owns a contiguous range of
// the slabs and the whole 32 TM x 32 TN tile, with an S-deep LDS ring of its own: no
// barrier until the partial tiles are summed through LDS, in wave order.
//  * A slab's operand reads are all issued one slab ahead of their MFMAs (two register
//    sets); its LDS slot is refilled as soon as they have landed.
//  * The weight rows are the MFMA's first operand, so a lane ends with four consecutive
//    columns of one row: float4 partials, 16-byte output stores.
//  * SwiGLU: the tile's first half of weight rows is up, the second gate.
// ---------------------------------------------------------------------------------
template <int TM, int TN>
struct KsplitFrags {
    bf16x8_t a[kPBK / 16][TM], b[kPBK / 16][TN];
};

template <int TM, int TN, int KW, int S, int EPI, int WPE>
__global__ __launch_bounds__(KW * kWave, WPE) void gemm_ksplit_kernel(const bf16_t* __restrict__ A,
                                                                 const bf16_t* __restrict__ B,
                                                                 const bf16_t* __restrict__ bias,
                                                                 void* __restrict__ Cout, int M, int N, int K, int ldc,
                                                                 int mt, int nt, int vec, int kslices, int slice_slabs) {
    constexpr int BM = 32 * TM, BN = 32 * TN, KSN = kPBK / 16;
    constexpr int OC = EPI == GEPI_SWIGLU ? BN / 2 : BN;   // output columns per tile
    constexpr int STAGE = (BM + BN) * kPRow, RING = S * STAGE;
    constexpr int LA = BM / 8, LPS = (BM + BN) / 8;        // 1 KB wave loads per slab
    constexpr int CH = BN / 4;                             // float4 chunks per partial row
    static_assert(S >= 2 && S * LPS <= 63 && BM * BN * 4 <= RING, "bad K-split shape");
    __shared__ __align__(1024) unsigned char smem[KW * RING];

    // GEPI_PARTIAL: work unit t covers slice t / (mt * nt) of the slabs
    const int T = mt * nt * kslices;
    const int per = (T + 7) / 8;
    const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (t >= T) return;
    const int slice = t / (mt * nt);
    int tm, tn;
    tile_of(t % (mt * nt), mt, nt, tm, tn);
    const int m0 = tm * BM, n0 = tn * OC;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid % kWave;

    // DMA sources: 32-bit byte offsets (the host keeps both operands under 2 GB); rows past
    // the matrix repeat its last row (their outputs are not stored)
    uint32_t voff[LPS];
    {
        const int rr = lane >> 3, cs = lane & 7;
#pragma unroll
        for (int i = 0; i < LPS; ++i) {
            const int r = i * 8 + rr;
            int row;
            if (i < LA) {
                row = min(m0 + r, M - 1);
            } else {
                const int br = r - BM;
                const int gate = EPI == GEPI_SWIGLU && br >= OC;
                row = min(n0 + br - gate * OC, N - 1) + gate * N;
            }
            voff[i] = (uint32_t)((row * K + ((cs ^ pipe_swz(r)) << 3)) * 2);
        }
    }
    unsigned char* const ring = smem + wave * RING;
    const int s0 = slice * slice_slabs, nk = min(K / kPBK - s0, slice_slabs);
    const int k_begin = s0 + wave * nk / KW, n_slabs = s0 + (wave + 1) * nk / KW - k_begin;
    const unsigned char* pa = reinterpret_cast<const unsigned char*>(A) + (size_t)k_begin * kPRow;
    const unsigned char* pb = reinterpret_cast<const unsigned char*>(B) + (size_t)k_begin * kPRow;
    auto issue = [&](int slab) {
        const unsigned char* sa = pa + slab * kPRow;
        const unsigned char* sb = pb + slab * kPRow;
        unsigned char* dst = ring + (slab % S) * STAGE;
#pragma unroll
        for (int i = 0; i < LPS; ++i)
            __builtin_amdgcn_global_load_lds(static_cast<const void*>((i < LA ? sa : sb) + voff[i]),
                                             (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, 0, 0);
    };
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)ring);
    const int r32 = lane & 31;
    uint32_t roff[KSN];   // row r32, chunk of key step ks (32-row blocks differ by an immediate)
#pragma unroll
    for (int ks = 0; ks < KSN; ++ks)
        roff[ks] = lds0 + (uint32_t)(r32 * kPRow + (((ks * 2 + (lane >> 5)) ^ pipe_swz(r32)) << 4));
    typedef KsplitFrags<TM, TN> Frags;
    auto read = [&](Frags& f, int slab) {
        const uint32_t so = (uint32_t)((slab % S) * STAGE);
#pragma unroll
        for (int ks = 0; ks < KSN; ++ks) {
            f.a[ks][0] = ds_read16<0>(roff[ks] + so);
            if constexpr (TM == 2) f.a[ks][TM - 1] = ds_read16<32 * kPRow>(roff[ks] + so);
            f.b[ks][0] = ds_read16<BM * kPRow>(roff[ks] + so);
            if constexpr (TN == 2) f.b[ks][TN - 1] = ds_read16<(BM + 32) * kPRow>(roff[ks] + so);
        }
    };

    f32x16_t acc[TN][TM];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[j][i][e] = 0.f;

    // slab i: its reads (issued before) have landed in `f`; refill its slot, issue the
    // reads of slab i + 1 into `g`, and run its MFMAs
    auto step = [&](int i, Frags& f, Frags& g) {
        lgkm_wait<0>();
#pragma unroll
        for (int ks = 0; ks < KSN; ++ks) {
#pragma unroll
            for (int x = 0; x < TM; ++x) asm volatile("" : "+v"(f.a[ks][x]));
#pragma unroll
            for (int x = 0; x < TN; ++x) asm volatile("" : "+v"(f.b[ks][x]));
        }
        if (i + S < n_slabs) issue(i + S);
        if (i + 1 < n_slabs) {
            vm_wait_slabs<LPS>(min(S - 1, n_slabs - 2 - i));
            asm volatile("" ::: "memory");
            read(g, i + 1);
        }
#pragma unroll
        for (int ks = 0; ks < KSN; ++ks)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int x = 0; x < TM; ++x)
                    acc[j][x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[ks][j], f.a[ks][x], acc[j][x], 0, 0, 0);
    };
    if (n_slabs > 0) {
        for (int p = 0; p < min(S, n_slabs); ++p) issue(p);
        vm_wait_slabs<LPS>(min(S, n_slabs) - 1);
        asm volatile("" ::: "memory");
        Frags f, g;
        read(f, 0);
        for (int i = 0; i < n_slabs; i += 2) {
            step(i, f, g);
            if (i + 1 < n_slabs) step(i + 1, g, f);
        }
    }

    // partial tile: float4 chunk c of row m at c ^ swz(m) (distinct bank groups for 16
    // lanes on 16 rows, and for 16 consecutive chunks)
    auto swz = [](int m) { return CH >= 16 ? (m & 15) : ((m >> 1) & 7); };
    float4* part = reinterpret_cast<float4*>(ring);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int x = 0; x < TM; ++x)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int m = x * 32 + r32, c = j * 8 + g * 2 + (lane >> 5);
                part[m * CH + (c ^ swz(m))] =
                    make_float4(acc[j][x][g * 4], acc[j][x][g * 4 + 1], acc[j][x][g * 4 + 2], acc[j][x][g * 4 + 3]);
            }
    __syncthreads();
    auto total = [&](int m, int c) {
        float4 v = reinterpret_cast<const float4*>(smem)[m * CH + (c ^ swz(m))];
#pragma unroll
        for (int w = 1; w < KW; ++w) {
            const float4 u = reinterpret_cast<const float4*>(smem + w * RING)[m * CH + (c ^ swz(m))];
            v.x += u.x;
            v.y += u.y;
            v.z += u.z;
            v.w += u.w;
        }
        return v;
    };
    constexpr int OCH = OC / 4;
    for (int idx = tid; idx < BM * OCH; idx += KW * kWave) {
        const int m = idx / OCH, c = idx % OCH, row = m0 + m, col = n0 + c * 4;
        if (row >= M || col >= N) continue;
        const float4 t0 = total(m, c);
        float v[4] = {t0.x, t0.y, t0.z, t0.w};
        if constexpr (EPI == GEPI_SWIGLU) {
            const float4 t1 = total(m, c + OCH);
            const float g[4] = {t1.x, t1.y, t1.z, t1.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = silu_f32(round_bf16(g[e])) * round_bf16(v[e]);
        } else if (bias != nullptr) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += col + e < N ? bf16_to_f32(bias[col + e]) : 0.f;
        }
        const size_t at = (size_t)(EPI == GEPI_PARTIAL ? slice * M + row : row) * ldc + col;
        if (EPI == GEPI_F32 || EPI == GEPI_PARTIAL) {
            float* o = reinterpret_cast<float*>(Cout) + at;
            if (vec) {
                *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (col + e < N) o[e] = v[e];
            }
        } else {
            bf16_t* o = reinterpret_cast<bf16_t*>(Cout) + at;
            if (vec) {
                uint2 w;
                w.x = pack_bf16x2(v[0], v[1]);
                w.y = pack_bf16x2(v[2], v[3]);
                *reinterpret_cast<uint2*>(o) = w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (col + e < N) o[e] = (bf16_t)f32_to_bf16(v[e]);
            }
        }
    }
}

// Split-K reduction: out[r, c] = sum over slices s = 0, 1, ... (in that order) of
// part[s, r, c], + bias[c], as bf16 or fp32. Four columns per thread (N % 4 == 0).
constexpr int kMaxSlices = 8;
template <bool F32OUT>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(const float* __restrict__ part, int ksplit, int M,
                                                                 int N, const bf16_t* __restrict__ bias,
                                                                 void* __restrict__ Cout) {
    const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x;   // float4 index
    const size_t plane = (size_t)M * N;
    if (q * 4 >= plane) return;
    // every plane's load in flight at once (kMaxSlices of them; past the plan's slices the
    // last plane again, not added)
    float4 v[kMaxSlices];
#pragma unroll
    for (int sl = 0; sl < kMaxSlices; ++sl)
        v[sl] = *reinterpret_cast<const float4*>(part + (size_t)min(sl, ksplit - 1) * plane + q * 4);
    float4 acc = v[0];
#pragma unroll
    for (int sl = 1; sl < kMaxSlices; ++sl)
        if (sl < ksplit) {
            acc.x += v[sl].x;
            acc.y += v[sl].y;
            acc.z += v[sl].z;
            acc.w += v[sl].w;
        }
    const int col = (int)((q * 4) % (size_t)N);
    if (bias != nullptr) {
        acc.x += bf16_to_f32(bias[col + 0]);
        acc.y += bf16_to_f32(bias[col + 1]);
        acc.z += bf16_to_f32(bias[col + 2]);
        acc.w += bf16_to_f32(bias[col + 3]);
    }
    if (F32OUT) {
        reinterpret_cast<float4*>(Cout)[q] = acc;
    } else {
        uint2 pk;
        pk.x = pack_bf16x2(acc.x, acc.y);
        pk.y = pack_bf16x2(acc.z, acc.w);
        reinterpret_cast<uint2*>(Cout)[q] = pk;
    }
}

template <int BM, int BN, int S, int EPI>
static void gemm_pipe_launch(int M, int N, int K, const bf16_t* A, const bf16_t* B, const bf16_t* bias, void* C,
                             int ldc, hipStream_t stream) {
    const int ocols = (EPI == GEPI_SWIGLU) ? BN / 2 : BN;
    const int mt = (M + BM - 1) / BM, nt = (N + ocols - 1) / ocols;
    const int grid = 8 * ((mt * nt + 7) / 8);
    hipLaunchKernelGGL((gemm_pipe_kernel<BM, BN, S, EPI>), dim3(grid), dim3(kGemmThreads), 0, stream, A, B, bias, C,
                       M, N, K, ldc, mt, nt, 1, K / kPBK);
}

template <int TM, int EPI>
static void gemm_tall_launch(int M, int N, int K, const bf16_t* A, const bf16_t* B, const bf16_t* bias, void* C, int ldc,
                             hipStream_t stream) {
    const int ocols = (EPI == GEPI_SWIGLU) ? 128 : 256;
    const int mt = (M + 32 * TM - 1) / (32 * TM), nt = (N + ocols - 1) / ocols;
    const int grid = 8 * ((mt * nt + 7) / 8);
    const int vec = N % 8 == 0 && ldc % 8 == 0 && (reinterpret_cast<uintptr_t>(C) & 15u) == 0;
    hipLaunchKernelGGL((gemm_tall_kernel<TM, EPI>), dim3(grid), dim3(256), 0, stream, A, B, bias, C, M, N, K, ldc, mt, nt,
                       vec);
}

template <int TM, int TN, int KW, int S, int EPI, int WPE>
static void gemm_ksplit_launch(int M, int N, int K, const bf16_t* A, const bf16_t* B, const bf16_t* bias, void* C,
                               int ldc, hipStream_t stream, int kslices = 1, int slice_slabs = 1 << 30) {
    const int oc = (EPI == GEPI_SWIGLU) ? 16 * TN : 32 * TN;
    const int mt = (M + 32 * TM - 1) / (32 * TM), nt = (N + oc - 1) / oc;
    const int grid = 8 * ((mt * nt * kslices + 7) / 8);
    const int vec = N % 4 == 0 && ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15u) == 0;
    hipLaunchKernelGGL((gemm_ksplit_kernel<TM, TN, KW, S, EPI, WPE>), dim3(grid), dim3(KW * kWave), 0, stream, A, B, bias,
                       C, M, N, K, ldc, mt, nt, vec, kslices, slice_slabs);
}

int prefill_cus();

// Which tile of the K-split kernel (four waves) an unsliced launch takes: 0 none, 1: 32 x 32
// (two workgroups per CU), 2: 64 x 32, 3: 64 x 64 (one per CU). It pays while every tile has
// a CU of its own, smallest tile first, and for up to 32 rows at any width, where the larger
// kernels' tiles are mostly padding. Up to 64 rows, or K below 8192 (beyond, the other
// kernels' slices over workgroups are the better split); a wave wants 3 slabs (K of 768; a
// 64 x 64 tile 5): the pipelined kernel's ring nearly holds shorter rows (40 x 512 -> 256 5.1
// / 5.1, 40 x 256 -> 512 4.7 / 4.3, 40 x 768 -> 1024 4.9 / 6.3).
// Measured on MI355X (us, this kernel / the pipelined one): 37 x 1536 -> 2048 4.4 / 9.9,
// 19 x 896 -> 1152 4.3 / 6.7, 24 x 1536 -> 17920 14.2 / 20.0, 256 x 1536 -> 2048 6.2 / 10.0,
// 100 x 3584 -> 4608 15.9 / 19.3, 512 x 1536 -> 2048 9.2 / 10.4, 24 x 8960 -> 1536 13.6 /
// 17.4 (sliced); not: 1344 x 2048 -> 2560 37.9 / 25.2, 256 x 3584 -> 4608 28.7 / 30.1.
// SwiGLU: 24 x 1536 -> 8960 14.6 / 16.7, 16 x 3584 -> 18944 48.1 / 67.8, 60 x 896 -> 4864
// 7.6 / 9.9; not: 60 x 1536 -> 8960 22.4 / 17.9.
static bool offsets_fit(long M, long b_rows, long K) {   // 32-bit byte offsets into both operands
    return M * K * 2 < 0x7fffffffL && b_rows * K * 2 < 0x7fffffffL;
}
static int ksplit_tile(int M, int N, int K, bool swiglu) {
    const int cus = prefill_cus(), nk = K / kPBK;
    if (K % kPBK != 0 || nk < 12 || !offsets_fit(M, swiglu ? 2L * N : N, K)) return 0;
    if (M <= 32) return 1;
    const long mt32 = (M + 31) / 32, mt64 = (M + 63) / 64, nt32 = ((long)N + 31) / 32, nt64 = ((long)N + 63) / 64;
    if (swiglu) return M <= 64 && mt64 * nt32 <= cus ? 3 : 0;
    if (M > 64 && nk >= 128) return 0;
    if (mt32 * nt32 <= cus) return 1;
    if (mt64 * nt32 <= cus) return 2;
    return mt64 * nt64 <= cus && nk >= 20 ? 3 : 0;
}

// Split-K plan for a plain (non-SwiGLU) projection with K % 64 == 0 and K >= 4096 whose
// tiles leave the chip's workgroup slots empty; ksplit 0 = no split over workgroups. Each
// slice covers at least 16 slabs (1024 keys). Measured on MI355X (us):
//  * up to 32 rows, and up to 64 with at most 64 MB of weights: the K-split kernel's 32 x 32
//    (64 x 32) tiles, as many slices as leave the fewest slabs to the busiest CU, at two
//    (one) workgroups per CU: 24 x 8960 -> 1536 17.4 -> 8.9, 19 x 4864 -> 896 17.6 -> 7.3,
//    60 x 11008 -> 2048 22.3 -> 16.6, 24 x 18944 -> 3584 35.2 -> 31.2 (128 x 128 tiles
//    before); 64 x 18944 -> 3584 stays (36.7 against 40.4);
//  * more rows, half the CUs in 64 x 64 tiles at most and at most 64 MB of weights: the
//    K-split kernel's 64 x 64 tiles, one workgroup per CU: 300 x 8960 -> 1536 24.0 -> 19.9,
//    128 x 8960 -> 1536 20.1 -> 13.4, 300 x 4864 -> 896 20.7 -> 12.9; 128 x 18944 -> 3584
//    stays (39.5 against 49.1);
//  * K < 8192 and a 64 x 64 tile (or fewer rows: a 32 x 32 tile) for every CU: unsliced
//    (ksplit_tile): 700 x 4864 -> 896 24.2 -> 18.6;
//  * tiles for at most a third of the CUs: as many slices as fill every CU once (at most
//    8), one workgroup per CU over a 4-deep ring: 512 x 8960 -> 1536 33.6 -> 28.3 (5
//    slices, against 8 slices over 2-deep rings, two workgroups per CU), 512 x 11008 ->
//    2048 47.7 -> 39.1 (4 against 6), 768 x 8960 -> 1536 40.9 -> 39.7 (3 against 6);
//  * up to 128 tiles: about 384 workgroups over 2-deep rings, two per CU (two slices over
//    4-deep rings: 1024 x 8960 -> 1536 46.1 -> 50.9, 512 x 18944 -> 3584 101.2 -> 102.9).
struct SplitK {
    int ksplit = 0, kt_per = 0;
    int tile = 0;       // tile of the K-split kernel (ksplit_tile), or 0: 128 x 128
    bool deep = false;  // 128 x 128: 4-deep ring, one workgroup per CU (else 2-deep, two per CU)
};
static SplitK splitk_plan(int M, int N, int K) {
    SplitK p;
    if (K % kPBK != 0 || N % 4 != 0) return p;
    const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128);
    const int nk = K / kPBK;
    if (tiles > 128 || nk < 64) return p;
    const int cus = prefill_cus();
    const bool small_w = (long)N * K * 2 <= (64L << 20);
    const long mt32 = (M + 31) / 32, mt64 = (M + 63) / 64, nt32 = (N + 31) / 32, nt64 = (N + 63) / 64;
    const int most = std::min(8, nk / 16);
    int ks = 0;
    if (M <= 32 || (M <= 64 && small_w)) {
        p.tile = M <= 32 ? 1 : 2;
        const long t = M <= 32 ? mt32 * nt32 : mt64 * nt32, slots = (M <= 32 ? 2L : 1L) * cus;
        ks = 1;
        for (int n = 2; n <= most && t * n <= slots; ++n) {   // fewest (workgroups on a CU) / n
            const long a = (t * n + cus - 1) / cus * ks, b = (t * ks + cus - 1) / cus * n;
            if (a <= b) ks = n;
        }
    } else if (nk < 128 && mt32 * nt32 <= cus) {
        return p;
    } else if (2 * mt64 * nt64 <= cus && small_w) {
        p.tile = 3;
        ks = (int)std::min<long>(most, cus / (mt64 * nt64));
    } else if (nk < 128 && mt64 * nt64 <= cus) {
        return p;
    } else {
        const int fill = (int)std::min<long>(most, cus / tiles);
        if (fill >= 3) {
            ks = fill;
            p.deep = true;
        } else {
            ks = (int)std::min<long>(8, (384 + tiles - 1) / tiles);
            ks = std::min(ks, nk / 16);
        }
    }
    if (ks < 2 || (p.tile != 0 && !offsets_fit(M, N, K))) return SplitK{};
    p.kt_per = (nk + ks - 1) / ks;
    p.ksplit = (nk + p.kt_per - 1) / p.kt_per;
    return p;
}
static size_t splitk_bytes(int M, int N, int K) {
    const SplitK p = splitk_plan(M, N, K);
    return p.ksplit == 0 ? 0 : (size_t)p.ksplit * M * N * sizeof(float);
}

// C = A . B^T (+ bias) through ksplit fp32 partial planes in `part`, then the ordered
// reduction.
static void gemm_splitk_launch(int M, int N, int K, const bf16_t* A, const bf16_t* B, const bf16_t* bias, void* C,
                               bool f32out, float* part, const SplitK& p, hipStream_t stream) {
    const int mt = (M + 127) / 128, nt = (N + 127) / 128;
    const int grid = 8 * ((mt * nt * p.ksplit + 7) / 8);
    if (p.tile == 1)
        gemm_ksplit_launch<1, 1, 4, 2, GEPI_PARTIAL, 2>(M, N, K, A, B, nullptr, part, N, stream, p.ksplit, p.kt_per);
    else if (p.tile == 2)
        gemm_ksplit_launch<2, 1, 4, 2, GEPI_PARTIAL, 1>(M, N, K, A, B, nullptr, part, N, stream, p.ksplit, p.kt_per);
    else if (p.tile == 3)
        gemm_ksplit_launch<2, 2, 4, 2, GEPI_PARTIAL, 1>(M, N, K, A, B, nullptr, part, N, stream, p.ksplit, p.kt_per);
    else if (p.deep)
        hipLaunchKernelGGL((gemm_pipe_kernel<128, 128, 4, GEPI_PARTIAL>), dim3(grid), dim3(kGemmThreads), 0, stream, A,
                           B, nullptr, part, M, N, K, N, mt, nt, p.ksplit, p.kt_per);
    else
        hipLaunchKernelGGL((gemm_pipe_kernel<128, 128, 2, GEPI_PARTIAL>), dim3(grid), dim3(kGemmThreads), 0, stream, A,
                           B, nullptr, part, M, N, K, N, mt, nt, p.ksplit, p.kt_per);
    const size_t quads = (size_t)M * N / 4;
    const dim3 rgrid((unsigned)((quads + 255) / 256));
    if (f32out) hipLaunchKernelGGL((gemm_splitk_reduce_kernel<true>), rgrid, dim3(256), 0, stream, part, p.ksplit, M, N, bias, C);
    else hipLaunchKernelGGL((gemm_splitk_reduce_kernel<false>), rgrid, dim3(256), 0, stream, part, p.ksplit, M, N, bias, C);
}

template <int EPI>
static int gemm_dispatch(int M, int N, int K, const bf16_t* A, const bf16_t* B, const bf16_t* bias, void* C, int ldc,
                         hipStream_t stream) {
    // Output columns per tile: BN (SwiGLU: BN / 2).
    auto tiles = [&](int bm, int bn) {
        const int ocols = (EPI == GEPI_SWIGLU) ? bn / 2 : bn;
        return (long)((M + bm - 1) / bm) * ((N + ocols - 1) / ocols);
    };
    const dim3 block(kGemmThreads);
    const int tile_knob = kernel_knob(EFM_KNOB_GEMM_TILE);
    const long b_rows = (EPI == GEPI_SWIGLU) ? 2L * N : (long)N;
    const bool wide_ok = K % kPBK == 0 && offsets_fit(M, b_rows, K);
    if (tile_knob == 0) {
        switch (ksplit_tile(M, N, K, EPI == GEPI_SWIGLU)) {
            case 1:
                gemm_ksplit_launch<1, 1, 4, 2, EPI, 2>(M, N, K, A, B, bias, C, ldc, stream);
                return check_launch("gemm_bf16");
            case 2:
                if constexpr (EPI != GEPI_SWIGLU) {
                    gemm_ksplit_launch<2, 1, 4, 2, EPI, 1>(M, N, K, A, B, bias, C, ldc, stream);
                    return check_launch("gemm_bf16");
                }
                break;
            case 3:
                gemm_ksplit_launch<2, 2, 4, 2, EPI, 1>(M, N, K, A, B, bias, C, ldc, stream);
                return check_launch("gemm_bf16");
            default: break;
        }
    }
    if (wide_ok && tile_knob != 1) {
        // Rounds of resident workgroups times the cost of one round: 100 for 192 x 256 tiles
        // (one per CU), 127 for 256 x 256, 106 for 512 tiles of 128 x 128 (two per CU; 96
        // below K 1536, where the larger tiles' first loads and epilogue weigh more), 75 for
        // a last round of one per CU. Measured on MI355X (us, 192 / 256 / 128 x 128): 4096 x
        // 3584 -> 4608 129 / 162 / 161, 4096 x 3584 -> 3584 123 / 91 / 125, 4096 x 3584 -> 2 x
        // 18944 909 / 855 / 1286, 1344 x 2048 -> 2 x 11008 122 / 146 / 147, 4096 x 1536 -> 2048
        // 32.7 / 42.8 / 33.9, 1344 x 2048 -> 2560 35.3 / 48.0 / 25.2, 700 x 896 -> 2 x 4864 21.6
        // / 26.2 / 20.4. The choice is the fastest or within 3 % of it at all 27 shapes swept
        // (1.5B, 3B, 7B and 0.5B projections at 300 to 16384 rows).
        const long cus = 256, t128 = tiles(128, 128);
        const long two = K < 1536 ? 96 : 106, rem = t128 % (2 * cus);
        const long c128 = t128 / (2 * cus) * two + (rem == 0 ? 0 : rem <= cus ? 75 : two);
        const long c192 = (tiles(192, 256) + cus - 1) / cus * 100, c256 = (tiles(256, 256) + cus - 1) / cus * 127;
        if (tile_knob == 3 || (tile_knob == 0 && c192 < std::min(c256, c128))) {
            gemm_tall_launch<6, EPI>(M, N, K, A, B, bias, C, ldc, stream);
            return check_launch("gemm_bf16");
        }
        if (tile_knob == 2 || c256 < c128) {
            gemm_tall_launch<8, EPI>(M, N, K, A, B, bias, C, ldc, stream);
            return check_launch("gemm_bf16");
        }
    }
    if (K % kPBK == 0) {
        // Tile choice from sweeps of the prefill shapes on MI355X: 128 x 128 double-
        // buffered (two workgroups per CU) once there are >= 1.5 tiles per CU (>= 1 for
        // SwiGLU); K >= 4096 with 129 to one-per-CU 128 x 128 tiles: those tiles over a
        // 4-deep ring, one workgroup per CU (1344 x 11008 -> 2048 129.2 -> 106.6 us,
        // 1024 x 18944 -> 3584 237.6 -> 182.8; at 132 tiles, 1344 x 8960 -> 1536, 80.2 ->
        // 86.1); else 128 x 64 over a 3-deep ring (two per CU; 1024 x 1536 -> 2048 20.2 ->
        // 18.3 against the 2-deep ring, no shape slower); else 64 x 64 (64 x 128 for
        // SwiGLU) with shallow pipelines. Every tile shape sums each output over K in the
        // same order: results are bit-identical whichever is chosen.
        if constexpr (EPI != GEPI_SWIGLU) {
            const long t = tiles(128, 128);
            if (K / kPBK >= 64 && t > 128 && t < 384 && t <= prefill_cus()) {
                gemm_pipe_launch<128, 128, 4, EPI>(M, N, K, A, B, bias, C, ldc, stream);
                return check_launch("gemm_bf16");
            }
        }
        if (tiles(128, 128) >= ((EPI == GEPI_SWIGLU) ? 256 : 384)) {
            gemm_pipe_launch<128, 128, 2, EPI>(M, N, K, A, B, bias, C, ldc, stream);
        } else if constexpr (EPI == GEPI_SWIGLU) {
            gemm_pipe_launch<64, 128, 3, EPI>(M, N, K, A, B, bias, C, ldc, stream);
        } else {
            if (tiles(128, 64) >= 256) gemm_pipe_launch<128, 64, 3, EPI>(M, N, K, A, B, bias, C, ldc, stream);
            else gemm_pipe_launch<64, 64, 4, EPI>(M, N, K, A, B, bias, C, ldc, stream);
        }
        return check_launch("gemm_bf16");
    }
    if (tiles(128, 128) >= 256) {
        const int oc = (EPI == GEPI_SWIGLU) ? 64 : 128;
        dim3 grid((M + 127) / 128, (N + oc - 1) / oc);
        hipLaunchKernelGGL((gemm_bf16_kernel<128, 128, EPI>), grid, block, 0, stream, A, B, bias, C, M, N, K, ldc);
    } else {
        if constexpr (EPI == GEPI_SWIGLU) {
            dim3 grid((M + 63) / 64, (N + 63) / 64);
            hipLaunchKernelGGL((gemm_bf16_kernel<64, 128, EPI>), grid, block, 0, stream, A, B, bias, C, M, N, K, ldc);
        } else {
            dim3 grid((M + 63) / 64, (N + 63) / 64);
            hipLaunchKernelGGL((gemm_bf16_kernel<64, 64, EPI>), grid, block, 0, stream, A, B, bias, C, M, N, K, ldc);
        }
    }
    return check_launch("gemm_bf16");
}

static int gemm_check(int64_t M, int64_t N, int64_t K, const void* A, const void* B, const void* C) {
    if (A == nullptr || B == nullptr || C == nullptr) return set_error(EFM_ERR_INVALID_ARGUMENT, "gemm: null pointer");
    if (K <= 0 || K % kBK != 0)
        return set_error(EFM_ERR_UNSUPPORTED, "gemm: in_features must be a positive multiple of %d (got %lld)", kBK,
                         (long long)K);
    if (M > 0x7fffffff / 2 || N > 0x7fffffff / 2 || K > 0x7fffffff / 2)
        return set_error(EFM_ERR_UNSUPPORTED, "gemm: shape too large");
    if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B)) & 15u)
        return set_error(EFM_ERR_INVALID_ARGUMENT, "gemm: operands must be 16-byte aligned");
    return EFM_OK;
}

int gemm_bf16(int64_t M, int64_t N, int64_t K, const void* A, const void* B, const void* bias, void* C,
              int32_t out_dtype, hipStream_t stream) {
    int rc = gemm_check(M, N, K, A, B, C);
    if (rc) return rc;
    if (M == 0 || N == 0) return EFM_OK;
    const bf16_t* a = static_cast<const bf16_t*>(A);
    const bf16_t* b = static_cast<const bf16_t*>(B);
    const bf16_t* bi = static_cast<const bf16_t*>(bias);
    if (out_dtype == EFM_DTYPE_BF16) return gemm_dispatch<GEPI_BF16>((int)M, (int)N, (int)K, a, b, bi, C, (int)N, stream);
    if (out_dtype == EFM_DTYPE_F32) return gemm_dispatch<GEPI_F32>((int)M, (int)N, (int)K, a, b, bi, C, (int)N, stream);
    return set_error(EFM_ERR_UNSUPPORTED, "linear: output dtype %d not supported", out_dtype);
}

size_t gemm_bf16_workspace_bytes(int64_t M, int64_t N, int64_t K) {
    if (M <= 1 || M > 0x7fffffff / 2 || N > 0x7fffffff / 2 || K > 0x7fffffff / 2) return 0;
    return splitk_bytes((int)M, (int)N, (int)K);
}

int gemm_bf16_ws(int64_t M, int64_t N, int64_t K, const void* A, const void* B, const void* bias, void* C,
                 int32_t out_dtype, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    int rc = gemm_check(M, N, K, A, B, C);
    if (rc) return rc;
    if (M == 0 || N == 0) return EFM_OK;
    if (out_dtype != EFM_DTYPE_BF16 && out_dtype != EFM_DTYPE_F32)
        return set_error(EFM_ERR_UNSUPPORTED, "linear: output dtype %d not supported", out_dtype);
    const SplitK p = splitk_plan((int)M, (int)N, (int)K);
    const size_t need = (p.ksplit == 0) ? 0 : (size_t)p.ksplit * M * N * sizeof(float);
    if (p.ksplit == 0 || workspace == nullptr || workspace_bytes < need ||
        (reinterpret_cast<uintptr_t>(workspace) & 15u) != 0)
        return gemm_bf16(M, N, K, A, B, bias, C, out_dtype, stream);
    gemm_splitk_launch((int)M, (int)N, (int)K, static_cast<const bf16_t*>(A), static_cast<const bf16_t*>(B),
                       static_cast<const bf16_t*>(bias), C, out_dtype == EFM_DTYPE_F32, static_cast<float*>(workspace),
                       p, stream);
    return check_launch("gemm_bf16 split-K");
}

int gemm_swiglu(int64_t M, int64_t inter, int64_t K, const void* A, const void* W, void* out, hipStream_t stream) {
    int rc = gemm_check(M, inter, K, A, W, out);
    if (rc) return rc;
    if (M == 0) return EFM_OK;
    return gemm_dispatch<GEPI_SWIGLU>((int)M, (int)inter, (int)K, static_cast<const bf16_t*>(A),
                                      static_cast<const bf16_t*>(W), nullptr, out, (int)inter, stream);
}

// Gate/up + SwiGLU with a workspace: the SwiGLU is the MFMA kernel's epilogue, so no
// shape uses the workspace.
size_t gemm_swiglu_workspace_bytes(int64_t, int64_t, int64_t) { return 0; }

int gemm_swiglu_ws(int64_t M, int64_t inter, int64_t K, const void* A, const void* W, void* out, void*, size_t,
                   hipStream_t stream) {
    return gemm_swiglu(M, inter, K, A, W, out, stream);
}

}  // namespace efm

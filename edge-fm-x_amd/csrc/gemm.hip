// Prefill projections on the gfx950 matrix cores: C[M, N] = A[M, K] . B[N, K]^T in
// bf16 with fp32 accumulation (v_mfma_f32_16x16x32_bf16 in the slab kernel, 32x32x16). A
// holds activations (one row per token) and B the weights in their [out, in] layout, so both
// operands are K-contiguous and feed the MFMA lanes with 16-byte loads.
//
//  * K % 64 == 0 (every Qwen2.5 projection), kernels fed by global_load_lds DMA into
//    XOR-swizzled LDS rings, operand reads software-pipelined against the MFMAs and a
//    grouped tile order per XCD:
//      - the slab kernel (gemm_tall_kernel): 256 x 256 to 64 x 64 tiles on four waves, one
//        or two workgroups per CU, plus its split-K form; a cost model (rounds of resident
//        workgroups) picks the tile;
//      - few rows, or few tiles and long K: the K-split kernel, whose four waves take a
//        quarter of K each over 32 x 32 to 64 x 64 tiles.
//  * Other K: a register-staged kernel with a padded LDS row pitch (40 bf16).
//  * Epilogues: bf16 (+bias, the cuBLASLt BIAS epilogue), fp32, and SwiGLU, where the
//    B tile holds blocks of up and of gate weights so that a lane meets u and g of the same
//    output element: out = bf16(silu(bf16(g)) * bf16(u)).
//  * Every kernel sums each output's keys in the same order (the 16 x 16 x 32 MFMA as two of
//    the 32 x 32 x 16 one), so results are bit-identical across kernels and tile shapes
//    (K-split and split-K aside, which add the sums of contiguous ranges of K in order).
#include "common.hpp"

#include <algorithm>
#include <iterator>
#include <type_traits>
#include <utility>

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

constexpr int vm_count(int loads) { return loads < 63 ? loads : 63; }   // the counter holds 63

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
// Slab kernel: a 32 TM x 32 TN tile on four waves, each owning a 16 TM x 16 TN block of 16 x
// 16 MFMA tiles (256 x 256: 128 x 128 blocks, 256 accumulator registers, one wave per SIMD),
// over 64-key slabs that buffer loads bring into LDS: a wave's 1 KB load is 8 rows x 128
// bytes, and lane l fetches chunk (l % 8) ^ pipe_swz(row), so that the operand reads (16 rows
// of one chunk) spread over the banks.
//  * What bounds the large tiles is the card's power: on zero operands the same launches run at 1.6-1.7
//    PF/s, on N(0, 1) ones at 1.3-1.4, and removing the DMA or the operand reads changes the
//    rate through what they consume. So the layout moves as little as it can: a 128 x 128
//    block reads two thirds of the LDS bytes per MFMA of a 128 x 64 one, rows of 64 keys
//    are whole 128-byte lines, buffer loads carry 32-bit offsets, and the 16 x 16 x 32 MFMA
//    sustains 1.97 PF/s on random operands where the 32 x 32 x 16 one sustains 1.65 (2 waves
//    a SIMD; the two give the same bits).
//  * 64-key operand slabs in a ring of D + 1 slabs of A and one of D slabs of B. Step 0 of
//    slab s runs with its second half's operand reads and the loads of A(s + D); then one
//    barrier (slab s is in registers everywhere, slab s + 1 has landed), and step 1 runs with
//    the first reads of slab s + 1 and the loads of B(s + D) into the slab that B(s) has left.
//  * The weight rows are the MFMA's first operand: a lane ends with four consecutive columns
//    of one row. SwiGLU interleaves 16-row blocks of up and gate weights.
//  * Small tiles are bound by the latency of their slabs: D of 3 or 4 where LDS allows.
//  Measured (us, before: an 8-wave kernel over 32-key stages for the large tiles, a shared
//  ring with a barrier before every slab's reads for the small ones): 4096 x 3584 -> 2 x 18944
//  SwiGLU 1103 -> 850 (1.31 PF/s), 4096 x 18944 -> 3584 515 -> 405, 4096 x 3584 -> 4608 156 ->
//  120, 1344 x 11008 -> 2048 107 -> 89, 1000 x 3584 -> 4608 66 -> 35, 1344 x 2048 -> 2560 25.7
//  -> 19.0, 512 x 1536 -> 2048 10.0 -> 8.0, 700 x 896 -> 1152 7.3 -> 5.8.
// ---------------------------------------------------------------------------------
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// N consecutive columns of an output row, `left` of them inside the matrix. Whole segments go
// as 16-byte (bf16 of four: 8-byte) stores whatever their alignment, which the hardware takes:
// rows of a ragged N start anywhere (3052 x 64 -> 36014: 191 us with a store per column).
template <int N, typename T>
__device__ __forceinline__ void store_cols(T* o, const float* v, int left) {
    if (left >= N) {
        if constexpr (sizeof(T) == 4) {
            __builtin_memcpy(o, v, N * 4);
        } else {
            uint32_t w[N / 2];
#pragma unroll
            for (int e = 0; e < N; e += 2) w[e / 2] = pack_bf16x2(v[e], v[e + 1]);
            __builtin_memcpy(o, w, N * 2);
        }
    } else {
#pragma unroll
        for (int e = 0; e < N; ++e)
            if (e < left) {
                if constexpr (sizeof(T) == 4) o[e] = v[e];
                else o[e] = (bf16_t)f32_to_bf16(v[e]);
            }
    }
}

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

// LDS of the slab kernel: D + 1 slabs of A and D of B.
constexpr int tall_lds(int tm, int tn, int d) { return 32 * kPRow * ((d + 1) * tm + d * tn); }

template <int TM, int TN, int D, int EPI>
__global__ __launch_bounds__(256, tall_lds(TM, TN, D) <= 80 * 1024 ? 2 : 1) void gemm_tall_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ B,
                                                           const bf16_t* __restrict__ bias, void* __restrict__ Cout,
                                                           int M, int N, int K, int ldc, int mt, int nt,
                                                           int kslices, int slice_slabs) {
    constexpr int BM = 32 * TM, BN = 32 * TN;       // a wave: TM x TN tiles of 16 x 16
    constexpr int ASZ = BM * kPRow, BSZ = BN * kPRow;   // an operand slab (64 keys)
    constexpr int B0 = (D + 1) * ASZ;                   // the B ring, behind D + 1 slabs of A
    constexpr int LA = BM / 32, LB = BN / 32;       // 1 KB wave loads per operand slab and wave
    constexpr int NM = TM * TN, NR = TM + TN, NL = LA > LB ? LA : LB;   // MFMAs, reads, loads of a step
    constexpr int RS = NM >= 2 * NR ? 2 : 1;        // MFMAs per operand read
    constexpr int DS = NM / NL;                     // and per DMA load
    static_assert(NM >= NR && DS >= 2, "a step's memory instructions go out behind its MFMAs");
    __shared__ __align__(1024) unsigned char smem[B0 + D * BSZ];

    // GEPI_PARTIAL: work unit t covers slice t / (mt * nt) of the slabs
    const int T = mt * nt * kslices;
    const int per = (T + 7) / 8;
    const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (t >= T) return;
    const int slice = t / (mt * nt);
    int tm, tn;
    tile_of(t % (mt * nt), mt, nt, tm, tn);
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
            va[i] = (uint32_t)(min(r, M - 1 - m0) * K + ((cs ^ pipe_swz(r)) << 3)) * 2;
        }
#pragma unroll
        for (int i = 0; i < LB; ++i) {
            const int r = (i * 4 + wave) * 8 + rr;
            // SwiGLU: 16-row blocks of up (even) and gate (odd) weights, a wave's all of one kind
            const int row = EPI == GEPI_SWIGLU ? r / 32 * 16 + r % 16 : r;
            vb[i] = (uint32_t)(min(row, N - 1 - n0) * K + ((cs ^ pipe_swz(r)) << 3)) * 2;
        }
    }
    const int s0 = slice * slice_slabs, nk = min(K / kPBK - s0, slice_slabs);
    // 64-bit bases at the tile's first rows, 32-bit byte offsets within the tile
    const int b0 = n0 + (EPI == GEPI_SWIGLU && (wave & 2) ? N : 0);
    const unsigned char* pa = reinterpret_cast<const unsigned char*>(A + (size_t)m0 * K) + (size_t)s0 * kPRow;
    const unsigned char* pb = reinterpret_cast<const unsigned char*>(B + (size_t)b0 * K) + (size_t)s0 * kPRow;
    // slabs past the end repeat the last one (never read, so that every step issues the same
    // loads)
    unsigned char* const base = smem + wave * 1024;
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
    for (int d = 0; d < D; ++d) {
#pragma unroll
        for (int i = 0; i < LA; ++i) tall_load(src_a(d), va[i], base + d * ASZ + i * 4096);
#pragma unroll
        for (int i = 0; i < LB; ++i) tall_load(src_b(d), vb[i], base + B0 + d * BSZ + i * 4096);
    }
    vm_wait<vm_count((D - 1) * (LA + LB))>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Frags f0, f1;
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (read_one(std::integral_constant<int, I>{}, f0, ra[0], rb[0] + B0), ...);
    }(std::make_integer_sequence<int, TM + TN>{});

    // one 32-key step: MFMA I, then an operand read of the next step behind every RS-th and a
    // DMA load behind every DS-th one
    auto mma_step = [&](Frags& f, Frags& g, uint32_t na, uint32_t nb, auto&& dma) {
        [&]<int... I>(std::integer_sequence<int, I...>) {
            ((acc[I / TN][I % TN] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.b[I % TN], f.a[I / TN], acc[I / TN][I % TN],
                                                                            0, 0, 0),
              read_one(std::integral_constant<int, (I % RS == 0 ? I / RS : 99)>{}, g, na, nb),
              dma(std::integral_constant<int, I>{}), __builtin_amdgcn_sched_barrier(0)),
             ...);
        }(std::make_integer_sequence<int, TM * TN>{});
    };
    uint32_t sa = 0, sb = B0;   // offsets of A(s) and B(s); A(s + D) goes one slab behind A(s)
    for (int s = 0; s < nk; ++s) {
        const uint32_t xa = sa == (uint32_t)(D * ASZ) ? 0u : sa + ASZ;
        const uint32_t xb = sb == (uint32_t)(B0 + (D - 1) * BSZ) ? (uint32_t)B0 : sb + BSZ;
        const unsigned char* ga = src_a(s + D);
        unsigned char* da = base + (sa == 0 ? (uint32_t)(D * ASZ) : sa - ASZ);
        lgkm_wait<0>();
        tie(f0);
        mma_step(f0, f1, ra[1] + sa, rb[1] + sb, [&](auto ic) {
            constexpr int I = decltype(ic)::value;
            if constexpr (I % DS == DS - 1 && I / DS < LA) tall_load(ga, va[I / DS], da + (I / DS) * 4096);
        });
        // slab s is in registers, slab s + 1 has landed for every wave
        const unsigned char* gb = src_b(s + D);
        unsigned char* db = base + sb;
        lgkm_wait<0>();
        tie(f1);
        vm_wait<vm_count((D - 1) * LA + (D - 2) * LB)>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        mma_step(f1, f0, ra[0] + xa, rb[0] + xb, [&](auto ic) {
            constexpr int I = decltype(ic)::value;
            if constexpr (I % DS == DS - 1 && I / DS < LB) tall_load(gb, vb[I / DS], db + (I / DS) * 4096);
        });
        pin_acc(acc);
        sa = xa;
        sb = xb;
    }
    lgkm_wait<0>();
    tie(f0);
    vm_wait<0>();
    __syncthreads();   // every wave is done with the operand slots

    // Epilogue, half of the wave's row blocks at a time: the partial tile goes through the
    // wave's own quarter of the ring as fp32 (element e of tile (i, j): row 16 i + lane % 16, column 16 j +
    // (lane / 16) * 4 + e; float4 chunk c of row r at c ^ (r % 16), over fewer chunks modulo
    // theirs), so that the stores are whole row segments, LPR lanes to a row.
    constexpr int SLOT = (B0 + D * BSZ) / 4 / 1024 * 1024;
    constexpr int H = TM / 2, CPR = TN * 4, LPR = TN * 2, RPP = kWave / LPR;
    constexpr int NV = EPI == GEPI_SWIGLU ? 4 : 8;   // columns a lane stores
    static_assert(H * 16 * CPR * 16 <= SLOT, "half a wave's tile fits a slot");
    float4* const part = reinterpret_cast<float4*>(smem + wave * SLOT);
    const int seg = lane % LPR;
    const int col = n0 + wn * (LPR * NV) + seg * NV;
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
                part[(i * 16 + r16) * CPR + ((j * 4 + (lane >> 4)) ^ (r16 % CPR))] = make_float4(x[0], x[1], x[2], x[3]);
            }
#pragma unroll 4
        for (int q = 0; q < H * 16 / RPP; ++q) {
            const int r = q * RPP + lane / LPR;
            const int row = m0 + wm * (BM / 2) + i0 * 16 + r, sw = (r & 15) % CPR;
            const int c0 = EPI == GEPI_SWIGLU ? (seg >> 2) * 8 + (seg & 3) : seg * 2;
            const float4 x = part[r * CPR + (c0 ^ sw)], y = part[r * CPR + ((c0 + (EPI == GEPI_SWIGLU ? 4 : 1)) ^ sw)];
            float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
            for (int e = 0; e < NV; ++e) {
                if constexpr (EPI == GEPI_SWIGLU) v[e] = silu_f32(round_bf16(v[4 + e])) * round_bf16(v[e]);
                else if (bias != nullptr) v[e] += bv[e];
            }
            if (row >= M) continue;
            const size_t at = (size_t)(EPI == GEPI_PARTIAL ? (size_t)slice * M + row : (size_t)row) * ldc + col;
            if constexpr (EPI == GEPI_F32 || EPI == GEPI_PARTIAL) store_cols<8>(reinterpret_cast<float*>(Cout) + at, v, N - col);
            else store_cols<NV>(reinterpret_cast<bf16_t*>(Cout) + at, v, N - col);
        }
    };
    half(std::integral_constant<int, 0>{});
    half(std::integral_constant<int, 1>{});
}

// ---------------------------------------------------------------------------------
// K split over the waves of a workgroup: for launches whose tiles are too few to keep the
// CUs busy by themselves. The slab kernel's four waves share every slab and meet at a barrier
// for each. Here each of four waves owns a contiguous range of the slabs and the whole 32 TM
// x 32 TN tile, with a ring of two slabs in LDS of its own: no barrier until the partial tiles
// are summed through LDS, in wave order.
//  * A slab's operand reads are all issued one slab ahead of their MFMAs (two register
//    sets); its LDS slot is refilled as soon as they have landed.
//  * The weight rows are the MFMA's first operand, so a lane ends with four consecutive
//    columns of one row: float4 partials, 16-byte output stores.
//  * SwiGLU: the tile's first half of weight rows is up, the second gate.
// ---------------------------------------------------------------------------------
constexpr int kKsplitWaves = 4, kKsplitRing = 2;

template <int TM, int TN>
struct KsplitFrags {
    bf16x8_t a[kPBK / 16][TM], b[kPBK / 16][TN];
};

template <int TM, int TN, int EPI, int WPE>
__global__ __launch_bounds__(kKsplitWaves * kWave, WPE) void gemm_ksplit_kernel(const bf16_t* __restrict__ A,
                                                                 const bf16_t* __restrict__ B,
                                                                 const bf16_t* __restrict__ bias,
                                                                 void* __restrict__ Cout, int M, int N, int K, int ldc,
                                                                 int mt, int nt, int kslices, int slice_slabs) {
    constexpr int KW = kKsplitWaves, S = kKsplitRing;
    constexpr int BM = 32 * TM, BN = 32 * TN, KSN = kPBK / 16;
    constexpr int OC = EPI == GEPI_SWIGLU ? BN / 2 : BN;   // output columns per tile
    constexpr int STAGE = (BM + BN) * kPRow, RING = S * STAGE;
    constexpr int LA = BM / 8, LPS = (BM + BN) / 8;        // 1 KB wave loads per slab
    constexpr int CH = BN / 4;                             // float4 chunks per partial row
    static_assert(S == 2 && BM * BN * 4 <= RING, "bad K-split shape");
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

    // DMA sources: 64-bit bases at the tile's first rows, 32-bit byte offsets within the
    // tile; rows past the matrix repeat its last row (their outputs are not stored)
    uint32_t voff[LPS];
    {
        const int rr = lane >> 3, cs = lane & 7;
#pragma unroll
        for (int i = 0; i < LPS; ++i) {
            const int r = i * 8 + rr;
            const int row = i < LA ? min(r, M - 1 - m0) : min((r - BM) % OC, N - 1 - n0);
            voff[i] = (uint32_t)(row * K + ((cs ^ pipe_swz(r)) << 3)) * 2;
        }
    }
    unsigned char* const ring = smem + wave * RING;
    const int s0 = slice * slice_slabs, nk = min(K / kPBK - s0, slice_slabs);
    const int k_begin = s0 + wave * nk / KW, n_slabs = s0 + (wave + 1) * nk / KW - k_begin;
    const unsigned char* pa = reinterpret_cast<const unsigned char*>(A + (size_t)m0 * K) + (size_t)k_begin * kPRow;
    const unsigned char* pb = reinterpret_cast<const unsigned char*>(B + (size_t)n0 * K) + (size_t)k_begin * kPRow;
    const size_t gate = (size_t)N * K * 2;   // SwiGLU: from the up to the gate weights
    auto issue = [&](int slab) {
        const unsigned char* sa = pa + slab * kPRow;
        const unsigned char* sb = pb + slab * kPRow;
        unsigned char* dst = ring + (slab % S) * STAGE;
#pragma unroll
        for (int i = 0; i < LPS; ++i)
            __builtin_amdgcn_global_load_lds(static_cast<const void*>((i < LA ? sa : i < LA + OC / 8 ? sb : sb + gate) + voff[i]),
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
            if (i + 2 < n_slabs) vm_wait<LPS>();   // slab i + 2 may be in flight
            else vm_wait<0>();
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
        if (n_slabs > 1) vm_wait<LPS>();
        else vm_wait<0>();
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
        const size_t at = (size_t)(EPI == GEPI_PARTIAL ? (size_t)slice * M + row : (size_t)row) * ldc + col;
        if constexpr (EPI == GEPI_F32 || EPI == GEPI_PARTIAL) store_cols<4>(reinterpret_cast<float*>(Cout) + at, v, N - col);
        else store_cols<4>(reinterpret_cast<bf16_t*>(Cout) + at, v, N - col);
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

template <int TM, int TN, int D, int EPI>
static void gemm_tall_launch(int M, int N, int K, const bf16_t* A, const bf16_t* B, const bf16_t* bias, void* C, int ldc,
                             hipStream_t stream, int kslices = 1, int slice_slabs = 1 << 30) {
    const int ocols = (EPI == GEPI_SWIGLU) ? 16 * TN : 32 * TN;
    const int mt = (M + 32 * TM - 1) / (32 * TM), nt = (N + ocols - 1) / ocols;
    const int grid = 8 * ((mt * nt * kslices + 7) / 8);
    hipLaunchKernelGGL((gemm_tall_kernel<TM, TN, D, EPI>), dim3(grid), dim3(256), 0, stream, A, B, bias, C, M, N, K, ldc, mt, nt,
                       kslices, slice_slabs);
}

template <int TM, int TN, int EPI, int WPE>
static void gemm_ksplit_launch(int M, int N, int K, const bf16_t* A, const bf16_t* B, const bf16_t* bias, void* C,
                               int ldc, hipStream_t stream, int kslices = 1, int slice_slabs = 1 << 30) {
    const int oc = (EPI == GEPI_SWIGLU) ? 16 * TN : 32 * TN;
    const int mt = (M + 32 * TM - 1) / (32 * TM), nt = (N + oc - 1) / oc;
    const int grid = 8 * ((mt * nt * kslices + 7) / 8);
    hipLaunchKernelGGL((gemm_ksplit_kernel<TM, TN, EPI, WPE>), dim3(grid), dim3(kKsplitWaves * kWave), 0, stream, A, B,
                       bias, C, M, N, K, ldc, mt, nt, kslices, slice_slabs);
}

int prefill_cus();

// Which tile of the K-split kernel (four waves) an unsliced launch takes: 0 none, 1: 32 x 32
// (two workgroups per CU), 2: 64 x 32, 3: 64 x 64 (one per CU). It pays while every tile has
// a CU of its own, smallest tile first, and for up to 32 rows at any width, where the slab
// kernel's tiles are mostly padding. Up to 64 rows, or K below 8192 (beyond, slices over
// workgroups are the better split); a wave wants 3 slabs (K of 768: 40 x 512 -> 256 5.1 us
// against 5.1, 40 x 256 -> 512 4.7 / 4.3, 40 x 768 -> 1024 4.9 / 6.3), of a 64 x 64 tile 12.
// Measured on MI355X (us, this kernel / the slab kernel's best tile): 200 x 3584 -> 3584 14.2
// / 17.5, 100 x 3584 -> 4608 17.2 / 20, 256 x 1536 -> 2048 6.2 / 7.9; not: 512 x 1536 -> 2048
// 9.8 / 8.0, 256 x 2048 -> 2560 10.2 / 8.7. Against the kernels before either: 37 x 1536 ->
// 2048 4.4 / 9.9, 19 x 896 -> 1152 4.3 / 6.7, 24 x 1536 -> 17920 14.2 / 20.0, 24 x 8960 -> 1536
// 13.6 / 17.4 (sliced). SwiGLU only up to 32 rows: 24 x 1536 -> 8960 14.6 / 16.7, 16 x 3584 ->
// 18944 48.1 / 67.8; 60 x 896 -> 4864 7.6 / 5.8; and not where its second round of two tiles per
// CU is nearly full, which the slab kernel's 64 x 64 tiles cover in one: 5 x 896 -> 2 x 15872
// 13.7 / 12.6, up to 15 % over 70 shapes with K of 1280 to 3584, save K of 2048 and 4096, where
// this kernel stays up to 15 % ahead.
constexpr int kMaxSlabK = 1 << 21;   // 32-bit byte offsets into the 256 rows of a tile
static int ksplit_tile(int M, int N, int K, bool swiglu) {
    const int cus = prefill_cus(), nk = K / kPBK;
    if (K % kPBK != 0 || nk < 12 || K > kMaxSlabK) return 0;
    if (M <= 32) {
        const long t = swiglu ? ((long)N + 15) / 16 : 0;
        return t > 3 * cus && t <= 4 * cus && nk % 32 != 0 ? 0 : 1;
    }
    const long mt32 = (M + 31) / 32, mt64 = (M + 63) / 64, nt32 = ((long)N + 31) / 32, nt64 = ((long)N + 63) / 64;
    if (swiglu) return 0;
    if (M > 64 && nk >= 128) return 0;
    if (mt32 * nt32 <= cus) return 1;
    if (mt64 * nt32 <= cus) return 2;
    return mt64 * nt64 <= cus && nk >= 48 ? 3 : 0;
}

// Split-K plan for a plain (non-SwiGLU) projection with K % 64 == 0 and K >= 4096 whose
// tiles leave the chip's workgroup slots empty; ksplit 0 = no split over workgroups. Each
// slice covers at least 16 slabs (1024 keys). Measured on MI355X (us):
//  * up to 32 rows, and up to 64 with at most 64 MB of weights: the K-split kernel's 32 x 32
//    (64 x 32) tiles, as many slices as leave the fewest slabs to the busiest CU, at two
//    (one) workgroups per CU: 24 x 8960 -> 1536 17.4 -> 8.9, 19 x 4864 -> 896 17.6 -> 7.3,
//    60 x 11008 -> 2048 22.3 -> 16.6, 24 x 18944 -> 3584 35.2 -> 31.2 (128 x 128 tiles
//    before); 64 x 18944 -> 3584 stays (36.7 against 40.4);
//  * more rows, a third of the CUs in 64 x 64 tiles at most and at most 64 MB of weights: the
//    K-split kernel's 64 x 64 tiles, one workgroup per CU: 128 x 8960 -> 1536 20.1 -> 13.4,
//    300 x 4864 -> 896 20.7 -> 12.9. 128 x 18944 -> 3584 stays (39.5 against 49.1), and so do
//    launches with room for two slices only (118 shapes 11 % slower than 128 x 128 tiles at
//    the geometric mean, 59 with three slices 3 % faster: 188 x 11008 -> 2048 29.7 against
//    24.5, 104 x 8960 -> 1536, five slices, 15.2 against 19.2);
//  * K < 8192 and a 64 x 64 tile (or fewer rows: a 32 x 32 tile) for every CU: unsliced
//    (ksplit_tile): 700 x 4864 -> 896 24.2 -> 18.6;
//  * else 128 x 128 tiles of the slab kernel, slices chosen the same way over two workgroups
//    per CU (D 4 rings where one per CU is enough): 512 x 8960 -> 1536 29.0 -> 26.3 (5
//    slices), 300 x 18944 -> 3584 71.6 -> 57.5 (6), 1024 x 8960 -> 1536 45.6 -> 41.0 (5),
//    128 x 18944 -> 3584 35.1 -> 32.7 (8).
struct SplitK {
    int ksplit = 0, kt_per = 0;
    int tile = 0;   // tile of the K-split kernel (ksplit_tile), or 0: 128 x 128 of the slab kernel
};
static SplitK splitk_plan(int M, int N, int K) {
    SplitK p;
    if (K % kPBK != 0 || N % 4 != 0 || K > kMaxSlabK) return p;
    const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128);
    const int nk = K / kPBK;
    if (tiles > 128 || nk < 64) return p;
    const int cus = prefill_cus();
    const bool small_w = (long)N * K * 2 <= (64L << 20);
    const long mt32 = (M + 31) / 32, mt64 = (M + 63) / 64, nt32 = (N + 31) / 32, nt64 = (N + 63) / 64;
    const int most = std::min(8, nk / 16);
    // slices that leave the fewest slabs to the busiest CU, over at most `slots` workgroups
    auto fill_slices = [&](long t, long slots) {
        int ks = 1;
        for (int n = 2; n <= most && t * n <= slots; ++n)
            if ((t * n + cus - 1) / cus * ks <= (t * ks + cus - 1) / cus * n) ks = n;
        return ks;
    };
    int ks = 0;
    if (M <= 32 || (M <= 64 && small_w)) {
        p.tile = M <= 32 ? 1 : 2;
        const long t = M <= 32 ? mt32 * nt32 : mt64 * nt32, slots = (M <= 32 ? 2L : 1L) * cus;
        ks = fill_slices(t, slots);
    } else if (nk < 128 && mt32 * nt32 <= cus) {
        return p;
    } else if (3 * mt64 * nt64 <= cus && small_w) {
        p.tile = 3;
        ks = (int)std::min<long>(most, cus / (mt64 * nt64));
    } else if (nk < 128 && mt64 * nt64 <= cus) {
        return p;
    } else {
        ks = fill_slices(tiles, 2L * cus);
    }
    if (ks < 2) return SplitK{};
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
    if (p.tile == 1)
        gemm_ksplit_launch<1, 1, GEPI_PARTIAL, 2>(M, N, K, A, B, nullptr, part, N, stream, p.ksplit, p.kt_per);
    else if (p.tile == 2)
        gemm_ksplit_launch<2, 1, GEPI_PARTIAL, 1>(M, N, K, A, B, nullptr, part, N, stream, p.ksplit, p.kt_per);
    else if (p.tile == 3)
        gemm_ksplit_launch<2, 2, GEPI_PARTIAL, 1>(M, N, K, A, B, nullptr, part, N, stream, p.ksplit, p.kt_per);
    else if (mt * nt * p.ksplit <= prefill_cus())
        gemm_tall_launch<4, 4, 4, GEPI_PARTIAL>(M, N, K, A, B, nullptr, part, N, stream, p.ksplit, p.kt_per);
    else
        gemm_tall_launch<4, 4, 2, GEPI_PARTIAL>(M, N, K, A, B, nullptr, part, N, stream, p.ksplit, p.kt_per);
    const size_t quads = (size_t)M * N / 4;
    const dim3 rgrid((unsigned)((quads + 255) / 256));
    if (f32out) hipLaunchKernelGGL((gemm_splitk_reduce_kernel<true>), rgrid, dim3(256), 0, stream, part, p.ksplit, M, N, bias, C);
    else hipLaunchKernelGGL((gemm_splitk_reduce_kernel<false>), rgrid, dim3(256), 0, stream, part, p.ksplit, M, N, bias, C);
}

// Tiles of the slab kernel and what a launch of them takes, fitted to sweeps on MI355X over
// weights that rotate through the memory-side cache (us, 256 CUs). A launch is rounds of occ
// resident workgroups per CU. A round of c tiles per CU takes s us a 64-key slab: s0 at one tile on
// few CUs rising to s1 at one on each (the same work draws more power, and the clock drops),
// and from s1b just above one per CU to s2 at occ per CU; plus o us before the first and
// after the last slab, which the other workgroup of a CU hides where two share it and their
// slabs take as long. SwiGLU: the silu of a short launch is as long as its slabs; in longer
// ones the tiles that share a CU take 15 % more than the fit (1230 x 896 -> 2 x 4864 33.5 us on
// 128 x 128 tiles, 29.6 on 256 x 256). Of 680 shapes with K of 64 to 1024 the tile picked is
// 0.5 % slower than the best one at the geometric mean, of 420 of the models' dimensions 0.4 %.
// (With o hidden always 1.6 %, and up to 1.8 times: 1045 x 64 -> 2 x 4864 16.8 us on 64 x 64
// tiles, 10.6 on 192 x 128; 2871 x 64 -> 2 x 10208 52 on 256 x 256, 41 on 128 x 128.) The deep
// rings (D 3 and 4) carry launches of at most a tile per CU over the latency of the
// memory-side cache (300 x 3584 -> 4608: 128 x 64 tiles 36.9 us over 2 slabs, 20.1 over 4);
// where two workgroups share the LDS, the second one does.
struct TallTile {
    int tm, tn, occ;
    double o, s0, s1, s1b, s2;
};
constexpr TallTile kTallTiles[] = {   // EFM_KNOB_GEMM_TILE 10, 11, ...
    {8, 8, 1, 8.0, 1.05, 1.42, 0, 0},         // 256 x 256, D 2
    {6, 8, 1, 7.4, 0.72, 1.06, 0, 0},         // 192 x 256, D 2
    {6, 4, 1, 4.7, 0.47, 0.56, 0, 0},         // 192 x 128, D 3
    {4, 4, 1, 4.2, 0.36, 0.46, 0, 0},         // 128 x 128, D 4
    {4, 4, 2, 4.5, 0.47, 0.50, 0.68, 0.92},   // 128 x 128, D 2
    {4, 2, 1, 3.6, 0.235, 0.28, 0, 0},        // 128 x 64, D 4
    {4, 2, 2, 3.6, 0.38, 0.38, 0.45, 0.57},   // 128 x 64, D 2
    {2, 4, 2, 3.6, 0.235, 0.29, 0.75, 0.90},  // 64 x 128, D 3
    {2, 2, 2, 2.7, 0.21, 0.225, 0.38, 0.46},  // 64 x 64, D 4
};
static double tall_cost(const TallTile& t, long tiles, int slabs, bool swiglu, int cus) {
    const double sw = swiglu && slabs > 8 && t.occ == 2 ? 1.15 : 1;
    auto slab = [&](double c) {
        return sw * (c <= 1 ? t.s0 + (t.s1 - t.s0) * c : t.s1b + (t.s2 - t.s1b) * (c - 1) / (t.occ - 1));
    };
    const long rounds = (tiles + cus * t.occ - 1) / (cus * t.occ), last = tiles - (rounds - 1) * cus * t.occ;
    const double o = t.o + (swiglu && slabs <= 8 ? t.tm * t.tn / 32 : 0);
    const double whole = slabs * slab(t.occ), end = o + slabs * slab((double)last / cus);
    return (rounds - 1) * (t.occ == 1 ? o + whole : std::max(whole, o + whole / 2)) + end;
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
    const bool slab_ok = K % kPBK == 0 && K <= kMaxSlabK;
    if (tile_knob == 0) {
        switch (ksplit_tile(M, N, K, EPI == GEPI_SWIGLU)) {
            case 1:
                gemm_ksplit_launch<1, 1, EPI, 2>(M, N, K, A, B, bias, C, ldc, stream);
                return check_launch("gemm_bf16");
            case 2:
                if constexpr (EPI != GEPI_SWIGLU) {
                    gemm_ksplit_launch<2, 1, EPI, 1>(M, N, K, A, B, bias, C, ldc, stream);
                    return check_launch("gemm_bf16");
                }
                break;
            case 3:
                if constexpr (EPI != GEPI_SWIGLU) {
                    gemm_ksplit_launch<2, 2, EPI, 1>(M, N, K, A, B, bias, C, ldc, stream);
                    return check_launch("gemm_bf16");
                }
                break;
            default: break;
        }
    }
    if (slab_ok) {
        // the cheapest tile (EFM_KNOB_GEMM_TILE 1: of the tiles up to 128 x 128), or the knob's
        int pick = tile_knob >= 10 ? tile_knob - 10 : tile_knob == 3 ? 1 : 0;
        if (tile_knob < 2) {
            const int cus = prefill_cus();
            double best = 0;
            for (int i = tile_knob == 1 ? 3 : 0; i < (int)std::size(kTallTiles); ++i) {
                const double c = tall_cost(kTallTiles[i], tiles(32 * kTallTiles[i].tm, 32 * kTallTiles[i].tn), K / kPBK,
                                          EPI == GEPI_SWIGLU, cus);
                if (best == 0 || c < best) best = c, pick = i;
            }
        }
        switch (pick) {
            case 0: gemm_tall_launch<8, 8, 2, EPI>(M, N, K, A, B, bias, C, ldc, stream); break;
            case 1: gemm_tall_launch<6, 8, 2, EPI>(M, N, K, A, B, bias, C, ldc, stream); break;
            case 2: gemm_tall_launch<6, 4, 3, EPI>(M, N, K, A, B, bias, C, ldc, stream); break;
            case 3: gemm_tall_launch<4, 4, 4, EPI>(M, N, K, A, B, bias, C, ldc, stream); break;
            case 4: gemm_tall_launch<4, 4, 2, EPI>(M, N, K, A, B, bias, C, ldc, stream); break;
            case 5: gemm_tall_launch<4, 2, 4, EPI>(M, N, K, A, B, bias, C, ldc, stream); break;
            case 6: gemm_tall_launch<4, 2, 2, EPI>(M, N, K, A, B, bias, C, ldc, stream); break;
            case 7: gemm_tall_launch<2, 4, 3, EPI>(M, N, K, A, B, bias, C, ldc, stream); break;
            case 8: gemm_tall_launch<2, 2, 4, EPI>(M, N, K, A, B, bias, C, ldc, stream); break;
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

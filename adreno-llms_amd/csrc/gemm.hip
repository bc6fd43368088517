// Prefill GEMM for gfx950: out[M,N] = x[M,K] * W[N,K]^T on the matrix cores, with the weight
// dequantisation fused into the tile load.  fp16 activations, fp16 or per-row int8 weights,
// fp32 accumulation (v_mfma_f32_32x32x16_f16), fp16 output.
//
// Semantics follow the reference's M > 1 path: row i of out is the GEMV of row i of x
// (LF/src/model.cpp:243-250); for int8 the per-row scale multiplies the fp32 sum once, in the
// epilogue, as the int8 GEMV does (LF/kernels/gemv_m1_int8.cl:69-77).  int8 weights convert
// exactly to fp16, so every product is exact in fp32; only the order of the fp32 additions
// differs from the GEMV kernels (results agree to fp32 rounding, not bit for bit).
//
// Both operands are K-contiguous, so a block stages a BM x 64 tile of x and a BN x 64 tile of W
// through LDS (rows padded to 72 halves: 16-byte reads of 8 consecutive rows then fall in
// 8 different bank groups; two LDS stages) while the loads of the next three K-tiles are
// already in flight in registers.  Four wavefronts per block, each owning a WM x WN sub-tile as (WM/32) x (WN/32)
// accumulators of 32 x 32.
#include "common.h"
#include "device_math.h"
#include "plan_keep.h"
#include <hip/hip_fp16.h>
#include <algorithm>
#include <type_traits>
#include <utility>

namespace mi {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kKT = 64;            // K-tile, elements
constexpr int kLd = kKT + 8;       // LDS row stride, halves
constexpr int kThreads = 256;

__device__ __forceinline__ uint16_t to_half_bits(float f) {
    asm volatile("" : "+v"(f));    // round the fp32 value first, then convert (two roundings, as the GEMV path)
    return __half_as_ushort(__float2half_rn(f));
}

// Four int8 in one dword -> four fp16 (two dwords), exact: byte ^ 0x80 is q + 128, the byte
// permute builds the halves 1024 + (q + 128), and subtracting 1152 leaves q.
__device__ __forceinline__ void i8x4_to_h4(uint32_t v, uint32_t& lo, uint32_t& hi) {
    const uint32_t u = v ^ 0x80808080u;
    const uint32_t a = __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u);
    const uint32_t b = __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u);
    const __half2 k = __builtin_bit_cast(__half2, 0x64806480u);               // 1152, 1152
    lo = __builtin_bit_cast(uint32_t, __hsub2(__builtin_bit_cast(__half2, a), k));
    hi = __builtin_bit_cast(uint32_t, __hsub2(__builtin_bit_cast(__half2, b), k));
}

// Byte B of v holds two Q4 values, low nibble first.  Returns them as a pair of fp16 times the
// pair s2: the nibbles are placed into the mantissas of 1024 (unit 1) and of 64 (unit 1/16, which
// is where a high nibble sits), 1032 and 72 are subtracted (exact), and the product with the
// scale is rounded to fp16 once.
template <int B>
__device__ __forceinline__ uint32_t q4x2_to_h2(uint32_t v, __half2 s2) {
    const uint32_t t = __builtin_amdgcn_perm(0u, v, 0x0C000C00u | (B << 16) | B);
    const uint32_t h = (t & 0x00F0000Fu) | 0x54006400u;
    const __half2 k = __builtin_bit_cast(__half2, 0xD480E408u);               // -1032, -72
    return __builtin_bit_cast(uint32_t, __hmul2(__hadd2(__builtin_bit_cast(__half2, h), k), s2));
}

// Further matrices of one launch that multiply the same x (q | k | v, gate | up): tile `first` and up along N
// belong to the next one.  A block (in the streaming kernel a wavefront) finds its matrix from its tile and does
// from there on what it does in a launch of that matrix alone, so the results are those of separate launches bit
// for bit.  What it is for: a launch of a small matrix takes 4 to 9 us whatever its size (one block's serial K, the
// chip mostly idle), and k and v of a layer are 128 to 320 rows.
// Measured: the seven int8 projections of a layer with 896 / 4864 channels, given together, at 16 rows 34.6 -> 26.6 us (q | k | v
// and gate | up in one streaming launch each), at 2048 rows 121.7 -> 106.7 us; a launch of one matrix as before.
struct MoreMats {
    int n = 0, tiles = 0;                                    // further matrices; tiles along N of all of them (n > 0)
    struct { const uint8_t* W; const uint16_t* scale; uint16_t* out; int N, first; } m[kMaxSegments - 1] = {};
};
__device__ __forceinline__ void pick_matrix(const MoreMats& mm, int& tile, const uint8_t* __restrict__& W,
                                            const uint16_t* __restrict__& scale, uint16_t* __restrict__& out, int& N) {
    int first = 0;
    #pragma unroll
    for (int q = 0; q < kMaxSegments - 1; ++q)
        if (q < mm.n && tile >= mm.m[q].first) {
            W = mm.m[q].W; scale = mm.m[q].scale; out = mm.m[q].out; N = mm.m[q].N; first = mm.m[q].first;
        }
    tile -= first;
}

// Blocks go to the 8 XCDs round-robin, each with an L2 of its own.  With the tiles in their order an XCD keeps to its share
// of the columns of tiles where their number is even; where it is odd it comes through all of them, and XCD x takes the
// x-th eighth of a list instead that runs through bands of 512 columns of outputs, down M inside a band.  us, int8, tiles in
// order / in bands: 15 columns of 64, 2048 x 960 x 960 16.2 / 12.2, 25, 700 x 1600 x 960 13.4 / 11.2, 45, 320 x 2880 x 576 8.4 / 7.3;
// even: 40, 700 x 2560 x 960 10.5 / 13.1, 76, 300 x 4864 x 896 11.1 / 12.0.  The list costs a few divisions ahead of the first load,
// which pay from about 75 tiles on: 9 tiles, 60 x 576 x 576 5.5 / 5.7, 45, 192 x 960 x 960 9.8 / 10.0, 72, 512 x 576 x 576 6.5 / 7.0;
// 75, 320 x 960 x 960 10.4 / 10.0, 99, 700 x 576 x 576 7.7 / 6.3.
inline bool tiles_in_bands(long tiles_n, long tiles_m) { return tiles_n % 2 != 0 && tiles_n * tiles_m >= 75; }

template <int BM, int BN, int WM, int WN, int KIND, bool BANDS>
__global__ __launch_bounds__(kThreads) void gemm_kernel(const uint16_t* __restrict__ X,
                                                        const uint8_t* __restrict__ W,
                                                        const uint16_t* __restrict__ scale,
                                                        uint16_t* __restrict__ out, int M, int N, int K,
                                                        MoreMats more) {
    static_assert((BM / WM) * (BN / WN) == 4, "four wavefronts per block");
    constexpr int TM = WM / 32, TN = WN / 32;
    constexpr int A_CHUNKS = BM * (kKT / 8) / kThreads;                      // 16-byte chunks of x per thread
    constexpr int B_BYTES = KIND == WK_I8 ? 1 : 2;
    constexpr int B_CPR = kKT * B_BYTES / 16;                                // 16-byte chunks per W row and K-tile
    constexpr int B_CHUNKS = BN * B_CPR / kThreads;
    static_assert(A_CHUNKS >= 1 && B_CHUNKS >= 1, "tile too small for 256 threads");

    // Two LDS stages (x tile then W tile in each) and kStages register stages: the global
    // loads of K-tile i + kStages are issued while tile i is multiplied, which is what hides
    // the HBM / L2 latency (one tile ahead is far too short for it).
    extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
    constexpr int kStageHalves = (BM + BN) * kLd;

    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const int wm = wave / (BN / WN), wn = wave % (BN / WN);
    // Block -> tile: see tiles_in_bands
    int tile_m, tile_n;
    if constexpr (!BANDS) {                                                  // (a grid of tiles: no divisions)
        tile_m = blockIdx.y;
        tile_n = blockIdx.x;
    } else {
        constexpr int kBand = 512 / BN;
        const int tiles_n = more.n ? more.tiles : (N + BN - 1) / BN;
        const int tiles_m = (M + BM - 1) / BM, total = tiles_m * tiles_n;
        const int per_xcd = (total + 7) / 8, l = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
        if (l >= total) return;
        const int band = l / (kBand * tiles_m);
        const int width = tiles_n - band * kBand < kBand ? tiles_n - band * kBand : kBand;
        const int in_band = l - band * kBand * tiles_m;
        // (the divisions were done on the vector units: scalars again, for what is computed from them)
        tile_m = __builtin_amdgcn_readfirstlane(in_band / width);
        tile_n = __builtin_amdgcn_readfirstlane(band * kBand + in_band % width);
    }
    pick_matrix(more, tile_n, W, scale, out, N);
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int gk = lane / 32, li = lane % 32;

    floatx16 acc[TM][TN];
    #pragma unroll
    for (int t = 0; t < TM; ++t)
        #pragma unroll
        for (int u = 0; u < TN; ++u)
            #pragma unroll
            for (int r = 0; r < 16; ++r) acc[t][u][r] = 0.0f;

    struct Regs { u32x4 a[A_CHUNKS]; u32x4 b[B_CHUNKS]; };
    auto load_tile = [&](Regs& R, int k0) {
        #pragma unroll
        for (int i = 0; i < A_CHUNKS; ++i) {
            const int c = tid + i * kThreads, row = c / (kKT / 8), kc = c % (kKT / 8);
            const int m = m0 + row < M ? m0 + row : M - 1;          // rows past M are never stored
            R.a[i] = *reinterpret_cast<const u32x4*>(X + static_cast<size_t>(m) * K + k0 + kc * 8);
        }
        #pragma unroll
        for (int i = 0; i < B_CHUNKS; ++i) {
            const int c = tid + i * kThreads, row = c / B_CPR, kc = c % B_CPR;
            const int n = n0 + row < N ? n0 + row : N - 1;
            R.b[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(
                W + (static_cast<size_t>(n) * K + k0) * B_BYTES + kc * 16));
        }
    };
    auto store_tile = [&](const Regs& R, uint16_t* As, uint16_t* Bs) {
        #pragma unroll
        for (int i = 0; i < A_CHUNKS; ++i) {
            const int c = tid + i * kThreads, row = c / (kKT / 8), kc = c % (kKT / 8);
            *reinterpret_cast<u32x4*>(&As[row * kLd + kc * 8]) = R.a[i];
        }
        #pragma unroll
        for (int i = 0; i < B_CHUNKS; ++i) {
            const int c = tid + i * kThreads, row = c / B_CPR, kc = c % B_CPR;
            if constexpr (KIND == WK_I8) {
                uint32_t h[8];
                i8x4_to_h4(R.b[i].x, h[0], h[1]);
                i8x4_to_h4(R.b[i].y, h[2], h[3]);
                i8x4_to_h4(R.b[i].z, h[4], h[5]);
                i8x4_to_h4(R.b[i].w, h[6], h[7]);
                *reinterpret_cast<u32x4*>(&Bs[row * kLd + kc * 16]) = u32x4{h[0], h[1], h[2], h[3]};
                *reinterpret_cast<u32x4*>(&Bs[row * kLd + kc * 16 + 8]) = u32x4{h[4], h[5], h[6], h[7]};
            } else {
                *reinterpret_cast<u32x4*>(&Bs[row * kLd + kc * 8]) = R.b[i];
            }
        }
    };
    auto multiply = [&](const uint16_t* As, const uint16_t* Bs) {
        #pragma unroll
        for (int kk = 0; kk < kKT / 16; ++kk) {
            // lane group gk supplies k = 32 gk + 8 kk .. +7 of the tile, for both operands
            const int kcol = 32 * gk + 8 * kk;
            half8 a[TM], b[TN];
            #pragma unroll
            for (int t = 0; t < TM; ++t)
                a[t] = *reinterpret_cast<const half8*>(&As[(wm * WM + t * 32 + li) * kLd + kcol]);
            #pragma unroll
            for (int u = 0; u < TN; ++u)
                b[u] = *reinterpret_cast<const half8*>(&Bs[(wn * WN + u * 32 + li) * kLd + kcol]);
            #pragma unroll
            for (int t = 0; t < TM; ++t)
                #pragma unroll
                for (int u = 0; u < TN; ++u)
                    acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t], b[u], acc[t][u], 0, 0, 0);
        }
    };

    const int nk = K / kKT;
    Regs R0, R1, R2;
    load_tile(R0, 0);
    load_tile(R1, (1 < nk ? 1 : nk - 1) * kKT);
    load_tile(R2, (2 < nk ? 2 : nk - 1) * kKT);
    // One step: tile i goes registers -> LDS stage i % 2; one barrier publishes it (and, being
    // the second barrier since stage i % 2 was last read, also guards the overwrite); the
    // freed registers take tile i + 3; the matrix cores run on tile i.
#define MI_GEMM_STEP(R)                                                        \
    {                                                                          \
        uint16_t* As = lds + (i & 1) * kStageHalves;                           \
        uint16_t* Bs = As + BM * kLd;                                          \
        store_tile(R, As, Bs);                                                 \
        __syncthreads();                                                       \
        load_tile(R, (i + 3 < nk ? i + 3 : nk - 1) * kKT);                     \
        multiply(As, Bs);                                                      \
        if (++i >= nk) break;                                                  \
    }
    for (int i = 0;;) {
        MI_GEMM_STEP(R0)
        MI_GEMM_STEP(R1)
        MI_GEMM_STEP(R2)
    }
#undef MI_GEMM_STEP

    // D[i][j]: j = lane % 32 (a W row, i.e. an output column), i = 8 (r / 4) + 4 (lane / 32) + r % 4.
    #pragma unroll
    for (int u = 0; u < TN; ++u) {
        const int n = n0 + wn * WN + u * 32 + li;
        if (n >= N) continue;
        float s = 1.0f;
        if constexpr (KIND == WK_I8) s = __half2float(__ushort_as_half(scale[n]));
        #pragma unroll
        for (int t = 0; t < TM; ++t) {
            #pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm * WM + t * 32 + 8 * (r / 4) + 4 * gk + r % 4;
                if (m < M) {
                    const float v = KIND == WK_I8 ? acc[t][u][r] * s : acc[t][u][r];
                    out[static_cast<size_t>(m) * N + n] = to_half_bits(v);
                }
            }
        }
    }
}

// ---- wide tiles fed by direct global -> LDS loads (int8, Q4 and fp16 weights) ----------
//
// What bounds the kernel above is the rate at which a CU can fill LDS (about 150 bytes/ns,
// against 530 bytes/ns for reads and one 32x32x16 MFMA per 15.6 ns per SIMD) and the fragment
// reads that are not overlapped with the MFMAs of the same wavefront.  This kernel therefore
//  * keeps quantised W as it is stored (int8, or Q4 nibbles with their block scales) in LDS
//    (a half or a quarter of the fill bytes) and converts a fragment to fp16 in registers after
//    reading it; the four wavefronts of a block own disjoint rows of W (64 each, so the block
//    covers 256 rows of W) and share the 32*TM rows of x, so no fragment of W is converted twice;
//  * fills LDS with global_load_lds_dwordx4 (no registers, no ds_write), three to eight stages of
//    K = 64; 16-byte chunks are XOR-swizzled inside a row so that fragment reads are conflict-free
//    without padding (a wavefront's load always fills 1 KB of consecutive LDS);
//  * reads the fragments of the next 32 values of K before issuing the MFMAs of the current
//    ones, with one barrier per stage placed in the middle of a stage, where the data of the
//    next stage is known to have landed;
//  * orders K inside a group of 32 so that a lane's 16 consecutive weights feed two MFMAs: lanes
//    0-31 supply k = 0..7 then 8..15, lanes 32-63 supply 16..23 then 24..31, for W and x alike.
// W is the MFMA "A" operand and x the "B" operand, so a lane ends up with four consecutive
// output columns of one output row and stores them as 8 bytes.
namespace wide {

constexpr int kBN = 256;                    // rows of W per block
// LDS stages (K = 64 each) for 32 * tm rows of x.  A stage is requested stages - 2 stage times
// before it is needed, which is what covers the load latency.  Tall tiles (tm >= 3) take as many
// stages as 160 KB hold.  Low tiles of quantised weights take half of the LDS (3 or 4 stages), so
// that two blocks share a CU: they belong to shapes with many small tiles, where one block's
// prologue and epilogue then overlap the other's main loop (lm_head at M = 16: 37 -> 29 us).
constexpr int stages_for(int kind, int tm) {
    return kind == WK_Q4 ? (tm >= 5 ? 5 : tm == 4 ? 6 : tm == 3 ? 7 : 4)
         : kind == WK_F16 ? (tm >= 3 ? 3 : 4)
                          : (tm >= 4 ? 4 : tm == 3 ? 5 : tm == 2 ? 3 : 4);
}
// blocks of such a tile that fit one CU
constexpr int blocks_per_cu(int kind, int tm) { return kind != WK_F16 && tm <= 2 ? 2 : 1; }
// bytes of W per stage: int8 rows of 64 bytes; fp16 rows of 128 bytes; Q4 rows of 32 bytes of
// packed nibbles followed by the 256 rows' two block scales (fp16) each
constexpr int w_stage_bytes(int kind) {
    return kind == WK_Q4 ? kBN * 32 + kBN * 4 : kind == WK_F16 ? kBN * 128 : kBN * 64;
}
typedef __attribute__((address_space(3))) uint8_t lds_u8;
typedef __attribute__((address_space(1))) const uint8_t glb_u8;

__device__ __forceinline__ void lds_fill16(const uint8_t* g, uint8_t* l) {
    __builtin_amdgcn_global_load_lds((glb_u8*)g, (lds_u8*)l, 16, 0, 0);   // address-space casts
}
__device__ __forceinline__ void lds_fill4(const uint8_t* g, uint8_t* l) {
    __builtin_amdgcn_global_load_lds((glb_u8*)g, (lds_u8*)l, 4, 0, 0);
}
#define MI_LDS_READ8(dst, addr, imm) \
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "i"(imm))
#define MI_LDS_READ4(dst, addr, imm) \
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "i"(imm))
#define MI_LDS_READ16(dst, addr, imm) \
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "i"(imm))
#define MI_WAIT_LGKM(n) asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(n) : "memory")
#define MI_WAIT_VM(n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(n) : "memory")
#define MI_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

template <int... I, typename F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): indices are compile-time
// constants inside f (immediate operands, register array subscripts)
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

typedef float float2v __attribute__((ext_vector_type(2)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
// two fp32 values, already rounded to fp32, to a pair of fp16 (round to nearest even): one
// v_cvt_pk_f16_f32
__device__ __forceinline__ uint32_t pack_half2(float a, float b) {
    float2v v = {a, b};
    asm volatile("" : "+v"(v));    // keep the fp32 rounding of the products: no fused multiply-convert
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, half2v));
}

template <int TM>
struct Frags {
    u32x4 w[2];          // int8: 16 weights of two 32-row fragments of W, as read from LDS
    uint2 w4[2];         // Q4: the same, 8 bytes
    uint32_t ws[2];      // Q4: the two block scales of the stage, of the lane's row in either fragment
    uint32_t wf[2][2][4];  // the same as fp16: [fragment][MFMA of the pair][4 dwords = 8 halves]
    uint32_t wg[2][2][4];  // Q4 in two terms: the second term
    u32x4 wh[2][2];        // fp16 weights: read from LDS as they are used
    u32x4 x[2][TM];      // [MFMA of the pair][32-row fragment of x], 8 halves each
};

template <int TM, int KIND, int TERMS>
__global__ __launch_bounds__(256) void gemm_wide(const uint16_t* __restrict__ X,
                                                   const uint8_t* __restrict__ W,
                                                   const uint16_t* __restrict__ scale,
                                                   uint16_t* __restrict__ out, int M, int N, int K,
                                                   float* __restrict__ partial, int splits, MoreMats more,
                                                   int glu) {
    constexpr int BM = 32 * TM;
    constexpr int kXStage = BM * 128;                    // bytes of x (fp16) per stage
    constexpr bool Q4 = KIND == WK_Q4, F16 = KIND == WK_F16;
    constexpr int kWRow = Q4 ? 32 : F16 ? 128 : 64;      // bytes of one row of W per stage
    constexpr int kWLoads = Q4 ? 3 : F16 ? 8 : 4;        // Q4: two loads of nibbles, one of scales
    constexpr int kWReads = Q4 || F16 ? 4 : 2;           // Q4: two fragments, two scale pairs; fp16: two fragments for two MFMAs
    constexpr int kConv = F16 ? 0 : 8;                   // conversions per set of fragments
    constexpr int kScaleAt = kXStage + kBN * 32;         // Q4: the scales of a stage, 4 bytes per row of W
    constexpr int kStage = kXStage + w_stage_bytes(KIND);
    constexpr int kLoads = TM + kWLoads;                 // global -> LDS loads per wavefront and stage
    constexpr int kStages = stages_for(KIND, TM);
    constexpr int kReads = kWReads + 2 * TM;             // LDS reads per set of fragments
    constexpr int kMfmas = 4 * TM * TERMS;               // MFMAs per half stage (K = 32)
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];

    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, li = lane & 31;
    // Block -> tile.  Blocks go to the 8 XCDs round-robin and every XCD has its own L2, so XCD x
    // takes the x-th contiguous eighth of the tile list, and the list runs through bands of 4
    // tiles along N, down M inside a band: the tiles that are in flight on one XCD at the same
    // time then share rows of x and of W and fetch them into that L2 once.
    // With splits > 1 the list holds every tile once per slice of K (slice-major); a block then
    // sums its slice only and leaves fp32 partial sums for reduce_partials.
    int tile_m, tile_n, split;
    {
        const int tiles_m = (M + BM - 1) / BM, tiles_n = more.n ? more.tiles : (N + kBN - 1) / kBN;
        const int tiles = tiles_m * tiles_n;
        const int total = tiles * splits;
        const int per_xcd = (total + 7) / 8;
        int l = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
        if (blockIdx.x >= 8 * per_xcd || l >= total) return;          // whole block, before any barrier
        split = l / tiles;
        l -= split * tiles;
        constexpr int kBand = 4;
        const int band = l / (kBand * tiles_m);
        const int width = tiles_n - band * kBand < kBand ? tiles_n - band * kBand : kBand;
        const int in_band = l - band * kBand * tiles_m;
        tile_m = in_band / width;
        tile_n = band * kBand + in_band % width;
        pick_matrix(more, tile_n, W, scale, out, N);
    }
    const int m0 = tile_m * BM, n0 = tile_n * kBN;
    const uint32_t lbase = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_u8*)lds));

    // per-row scales of this lane's output columns, requested before anything else so that they
    // are in registers long before the epilogue: sc[u][rq] = 4 fp16 scales of columns nq .. nq + 3
    // (Q4 has no per-row scale: the block scales travel with the weights)
    const bool cols4 = (N % 4) == 0 && reinterpret_cast<uintptr_t>(scale) % 8 == 0;
    uint2 sc[2][4];
    #pragma unroll
    for (int u = 0; u < 2; ++u) {
        #pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
            const int nq = n0 + 64 * w + 32 * u + 8 * rq + 4 * g;
            if constexpr (Q4 || F16) {
                sc[u][rq] = uint2{0u, 0u};
            } else if (cols4 && nq + 3 < N) {
                sc[u][rq] = *reinterpret_cast<const uint2*>(scale + nq);
            } else {
                uint32_t h[4];
                #pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = scale[nq + e < N ? nq + e : N - 1];
                sc[u][rq] = uint2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
            }
        }
    }

    // --- fill side: lane i of load j writes LDS bytes [1024 j + 16 i, +16) of its region --------
    // x: load j covers rows 8j..8j+7 (128 bytes each, 8 chunks); slot p of row r holds chunk p ^ ((r >> 1) & 7)
    // W: load j covers rows 16j..16j+15 (64 bytes each, 4 chunks); slot p of row r holds chunk p ^ ((r >> 2) & 3)
    // W, Q4: load j covers rows 32j..32j+31 (32 bytes each, 2 chunks); slot p of row r holds chunk
    //        p ^ ((r >> 3) & 1); a third load of 4 bytes per lane brings the two block scales of
    //        the wavefront's own 64 rows
    // W, fp16: as x, load j covers rows 8j..8j+7, eight loads for the wavefront's own 64 rows
    uint32_t xsrc[TM], wsrc[F16 ? 8 : 4];
    #pragma unroll
    for (int jj = 0; jj < TM; ++jj) {
        const int r = 8 * (w + 4 * jj) + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        const int m = m0 + r < M ? m0 + r : M - 1;
        xsrc[jj] = static_cast<uint32_t>(m) * K * 2u + c * 16u;
    }
    if constexpr (Q4) {
        #pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int r = 32 * (2 * w + jj) + (lane >> 1);
            const int c = (lane & 1) ^ ((r >> 3) & 1);
            const int n = n0 + r < N ? n0 + r : N - 1;
            wsrc[jj] = static_cast<uint32_t>(n) * (K / 2) + c * 16u;
        }
        const int r = 64 * w + lane;
        const int n = n0 + r < N ? n0 + r : N - 1;
        wsrc[2] = static_cast<uint32_t>(n) * (K / 32) * 2u;
        wsrc[3] = 0u;
    } else if constexpr (F16) {
        #pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
            const int r = 8 * (8 * w + jj) + (lane >> 3);
            const int c = (lane & 7) ^ ((r >> 1) & 7);
            const int n = n0 + r < N ? n0 + r : N - 1;
            wsrc[jj] = static_cast<uint32_t>(n) * K * 2u + c * 16u;
        }
    } else {
        #pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            const int r = 16 * (4 * w + jj) + (lane >> 2);
            const int c = (lane & 3) ^ ((r >> 2) & 3);
            const int n = n0 + r < N ? n0 + r : N - 1;
            wsrc[jj] = static_cast<uint32_t>(n) * K + c * 16u;
        }
    }
    const uint8_t* Sb = reinterpret_cast<const uint8_t*>(scale);  // Q4: advanced like W below
    const uint8_t* Xb = reinterpret_cast<const uint8_t*>(X);     // both advanced to the block's first K-stage below
    // load j (0 .. kLoads - 1) of this wavefront for K-stage stage_k into LDS slot `slot`
    auto fill_one = [&](int stage_k, int slot, auto jc) {
        constexpr int j = decltype(jc)::value;
        uint8_t* xs = lds + slot * kStage;
        if constexpr (j < TM)
            lds_fill16(Xb + static_cast<size_t>(stage_k) * 128 + xsrc[j], xs + 1024 * (w + 4 * j));
        else if constexpr (F16)
            lds_fill16(W + static_cast<size_t>(stage_k) * 128 + wsrc[j - TM], xs + kXStage + 1024 * (8 * w + (j - TM)));
        else if constexpr (!Q4)
            lds_fill16(W + static_cast<size_t>(stage_k) * 64 + wsrc[j - TM], xs + kXStage + 1024 * (4 * w + (j - TM)));
        else if constexpr (j - TM < 2)
            lds_fill16(W + static_cast<size_t>(stage_k) * 32 + wsrc[j - TM], xs + kXStage + 1024 * (2 * w + (j - TM)));
        else
            lds_fill4(Sb + static_cast<size_t>(stage_k) * 4 + wsrc[2], xs + kScaleAt + 256 * w);
    };
    auto fill_stage = [&](int stage_k, int slot) {
        static_for<kLoads>([&](auto jc) { fill_one(stage_k, slot, jc); });
    };

    // --- read side -------------------------------------------------------------------------------
    // pair S (0, 1) of a stage, MFMA e (0, 1) of the pair: x chunk 4S + 2g + e, W chunk 2S + g
    const uint32_t xrow = lbase + li * 128u, xq = (2u * g) ^ ((li >> 1) & 7u);
    // Q4: bytes 16 S + 8 g .. + 7 of the row: chunk S, its lower or upper half
    // fp16: as x (the swizzle of rows li and li + 32 is the same)
    const uint32_t wrow = lbase + kXStage + (64u * w + li) * kWRow, wq = Q4 ? (li >> 3) & 1u : g ^ ((li >> 2) & 3u);
    const uint32_t soff = lbase + kScaleAt + (64u * w + li) * 4u;
    uint32_t xoff[2][2], woff[2], whoff[2][2];
    #pragma unroll
    for (int S = 0; S < 2; ++S) {
        #pragma unroll
        for (int e = 0; e < 2; ++e) {
            xoff[S][e] = xrow + (((4u * S + e) ^ xq) << 4);
            whoff[S][e] = wrow + (((4u * S + e) ^ xq) << 4);
        }
        woff[S] = Q4 ? wrow + ((S ^ wq) << 4) + 8u * g : wrow + (((2u * S) ^ wq) << 4);
    }
    // LDS read j (0 .. kReads - 1) of a set: the two W fragments first, then x for the first and
    // the second MFMA of the pair
    auto read_one = [&](Frags<TM>& F, uint32_t slot_bytes, auto Sc, auto jc) {
        constexpr int S = decltype(Sc)::value, j = decltype(jc)::value;
        if constexpr (F16 && j < kWReads) {
            const uint32_t a = whoff[S][j % 2] + slot_bytes;
            MI_LDS_READ16(F.wh[j / 2][j % 2], a, (j / 2) * 32 * kWRow);
        } else if constexpr (j < 2) {
            const uint32_t a = woff[S] + slot_bytes;
            if constexpr (Q4) {
                MI_LDS_READ8(F.w4[j], a, j * 32 * kWRow);
            } else {
                MI_LDS_READ16(F.w[j], a, j * 32 * kWRow);
            }
        } else if constexpr (j < kWReads) {
            const uint32_t a = soff + slot_bytes;
            MI_LDS_READ4(F.ws[j - 2], a, (j - 2) * 32 * 4);
        } else {
            constexpr int e = (j - kWReads) / TM, t = (j - kWReads) % TM;
            const uint32_t a = xoff[S][e] + slot_bytes;
            MI_LDS_READ16(F.x[e][t], a, t * 4096);
        }
    };
    // conversion j (0 .. 7) of a set: dword j % 4 of W fragment j / 4 becomes four halves
    // Q4 (S = pair of the stage, which selects the block scale): bytes 2 (d % 2), 2 (d % 2) + 1 of
    // dword d / 2 of fragment j / 4 become four halves, scaled
    auto convert_one = [&](Frags<TM>& F, auto Sc, auto jc) {
        constexpr int j = decltype(jc)::value, u = j / 4, d = j % 4;
        if constexpr (Q4) {
            constexpr int S = decltype(Sc)::value;
            const uint32_t sb = __builtin_amdgcn_perm(0u, F.ws[u], S ? 0x03020302u : 0x01000100u);
            const uint32_t v = d / 2 ? F.w4[u].y : F.w4[u].x;
            if constexpr (TERMS == 2) {
                // scale = hi + lo with 7 and 4 significant bits: q * hi and q * lo are exact in
                // fp16 and add up to q * scale in the fp32 accumulator
                const uint32_t hi = sb & 0xFFF0FFF0u;
                const __half2 s2 = __builtin_bit_cast(__half2, hi);
                const __half2 r2 = __hsub2(__builtin_bit_cast(__half2, sb), s2);
                F.wf[u][d / 2][2 * (d % 2)] = q4x2_to_h2<2 * (d % 2)>(v, s2);
                F.wf[u][d / 2][2 * (d % 2) + 1] = q4x2_to_h2<2 * (d % 2) + 1>(v, s2);
                F.wg[u][d / 2][2 * (d % 2)] = q4x2_to_h2<2 * (d % 2)>(v, r2);
                F.wg[u][d / 2][2 * (d % 2) + 1] = q4x2_to_h2<2 * (d % 2) + 1>(v, r2);
            } else {
                const __half2 s2 = __builtin_bit_cast(__half2, sb);
                F.wf[u][d / 2][2 * (d % 2)] = q4x2_to_h2<2 * (d % 2)>(v, s2);
                F.wf[u][d / 2][2 * (d % 2) + 1] = q4x2_to_h2<2 * (d % 2) + 1>(v, s2);
            }
        } else {
            i8x4_to_h4(F.w[u][d], F.wf[u][d / 2][2 * (d % 2)], F.wf[u][d / 2][2 * (d % 2) + 1]);
        }
    };

    floatx16 acc[2][TM];
    #pragma unroll
    for (int u = 0; u < 2; ++u)
        #pragma unroll
        for (int t = 0; t < TM; ++t)
            #pragma unroll
            for (int r = 0; r < 16; ++r) acc[u][t][r] = 0.0f;

    // MFMA n (0 .. kMfmas - 1) of a half stage; consecutive n use different accumulators
    auto mfma_one = [&](const Frags<TM>& F, auto nc) {
        constexpr int n = decltype(nc)::value, c = n / (2 * TM), e = c % 2, u = (n / TM) % 2, t = n % TM;
        const u32x4 wv = F16 ? F.wh[u][e]
                       : c / 2 ? u32x4{F.wg[u][e][0], F.wg[u][e][1], F.wg[u][e][2], F.wg[u][e][3]}
                               : u32x4{F.wf[u][e][0], F.wf[u][e][1], F.wf[u][e][2], F.wf[u][e][3]};
        acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, wv),
                                                          __builtin_bit_cast(half8, F.x[e][t]), acc[u][t], 0, 0, 0);
    };

    // One half stage.  An MFMA keeps the matrix pipe busy for 32 cycles but issues in 4, and a
    // wavefront issues in order: whatever else has to happen (LDS fills for a later stage, the
    // LDS reads of the next fragments, their int8 -> fp16 conversion) is dealt out between the
    // MFMAs, so that it runs in their shadow instead of draining the pipe.
    //   C  = fragments being multiplied; Nx = fragments being prepared (LDS slot at next_bytes,
    //   pair NS of that stage); FILL: also issue this wavefront's fills of stage fill_k.
    auto half_stage = [&](Frags<TM>& C, Frags<TM>& Nx, uint32_t next_bytes, auto NSc, auto fillc,
                          int fill_k, int fill_slot) {
        constexpr bool FILL = decltype(fillc)::value;
        constexpr int nF = FILL ? kLoads : 0;
        constexpr int A = nF + kReads + (kConv ? 1 + kConv : 0);   // fills, reads, wait for W, conversions
        static_for<kMfmas>([&](auto nc) {
            constexpr int n = decltype(nc)::value;
            mfma_one(C, nc);
            MI_SCHED_FENCE();
            constexpr int a0 = n * A / kMfmas, a1 = (n + 1) * A / kMfmas;
            static_for<a1 - a0>([&](auto kc) {
                constexpr int a = a0 + decltype(kc)::value;
                if constexpr (a < nF) {
                    fill_one(fill_k, fill_slot, std::integral_constant<int, a>{});
                } else if constexpr (a < nF + kReads) {
                    read_one(Nx, next_bytes, NSc, std::integral_constant<int, a - nF>{});
                } else if constexpr (a == nF + kReads) {
                    // LDS returns in order: the two W reads are back.  The registers are operands
                    // of the wait so that the conversions that read them cannot be moved above it.
                    if constexpr (F16)
                        ;
                    else if constexpr (Q4)
                        asm volatile("s_waitcnt lgkmcnt(%4)"
                                     : "+v"(Nx.w4[0]), "+v"(Nx.w4[1]), "+v"(Nx.ws[0]), "+v"(Nx.ws[1])
                                     : "n"(kReads - kWReads) : "memory");
                    else
                        asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(Nx.w[0]), "+v"(Nx.w[1]) : "n"(kReads - kWReads) : "memory");
                    MI_SCHED_FENCE();
                } else {
                    convert_one(Nx, NSc, std::integral_constant<int, a - nF - kReads - 1>{});
                }
            });
            MI_SCHED_FENCE();
        });
        // The reads into Nx complete before this straight-line block ends: the compiler takes the
        // asm outputs for ready values, so they must be, wherever it may place a register copy.
        MI_WAIT_LGKM(0);
        MI_SCHED_FENCE();
    };

    // waits until at most `stages` of this wavefront's stage fills are still in flight
    auto wait_fills = [&](int stages) {
        bool done = false;
        #pragma unroll
        for (int d = kStages - 2; d >= 1; --d) {
            if (!done && stages >= d) {
                MI_WAIT_VM(d * kLoads);
                done = true;
            }
        }
        if (!done) MI_WAIT_VM(0);
    };

    // this block's K-stages: [k_first, k_first + nk) of the K / 64 stages
    const int k_first = static_cast<int>(static_cast<long>(K / 64) * split / splits);
    const int nk = static_cast<int>(static_cast<long>(K / 64) * (split + 1) / splits) - k_first;
    Xb += static_cast<size_t>(k_first) * 128;
    W += static_cast<size_t>(k_first) * kWRow;
    Sb += static_cast<size_t>(k_first) * 4;
    Frags<TM> FA, FB;
    #pragma unroll
    for (int st = 0; st < kStages - 1; ++st)
        if (st < nk) fill_stage(st, st);
    wait_fills((nk < kStages - 1 ? nk : kStages - 1) - 1);          // stage 0 has landed
    __builtin_amdgcn_s_barrier();
    MI_SCHED_FENCE();
    static_for<kReads>([&](auto jc) { read_one(FA, 0u, std::integral_constant<int, 0>{}, jc); });
    if constexpr (Q4)
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(FA.w4[0]), "+v"(FA.w4[1]), "+v"(FA.ws[0]), "+v"(FA.ws[1]) : : "memory");
    else if constexpr (F16)
        MI_WAIT_LGKM(0);
    else
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(FA.w[0]), "+v"(FA.w[1]) : : "memory");
    MI_SCHED_FENCE();
    static_for<kConv>([&](auto jc) { convert_one(FA, std::integral_constant<int, 0>{}, jc); });

    // Stage i lives in slot i % kStages.  In the middle of stage i every wavefront waits for its
    // own fills of stage i + 1 and meets the others at the barrier; behind it stage i + 1 is
    // complete and stage i - 1 is no longer read, so its slot takes stage i + kStages - 1.
    auto stage = [&](int i, int slot, auto fillc) {
        const int next = slot + 1 == kStages ? 0 : slot + 1;
        const int prev = slot == 0 ? kStages - 1 : slot - 1;
        half_stage(FA, FB, static_cast<uint32_t>(slot) * kStage, std::integral_constant<int, 1>{},
                   std::false_type{}, 0, 0);
        MI_SCHED_FENCE();
        const int last = i + kStages - 2 < nk - 1 ? i + kStages - 2 : nk - 1;   // newest stage requested so far
        wait_fills(last - (i + 1));
        __builtin_amdgcn_s_barrier();
        MI_SCHED_FENCE();
        // (after the last stage the fragments read here are not used)
        half_stage(FB, FA, static_cast<uint32_t>(next) * kStage, std::integral_constant<int, 0>{},
                   fillc, i + kStages - 1, prev);
        MI_SCHED_FENCE();
    };
    int slot = 0, i = 0;
    for (; i + kStages - 1 < nk; ++i) {
        stage(i, slot, std::true_type{});
        slot = slot + 1 == kStages ? 0 : slot + 1;
    }
    for (; i < nk; ++i) {
        stage(i, slot, std::false_type{});
        slot = slot + 1 == kStages ? 0 : slot + 1;
    }

    // --- epilogue ----------------------------------------------------------------------------------
    // D[i][j]: i = 8 (r / 4) + 4 (lane / 32) + r % 4 is a row of W (an output column), j = lane % 32
    // a row of x (an output row): a lane holds 4 consecutive output columns per r / 4.  The
    // scaled fp16 values go through LDS (rows of 64 columns, padded to 144 bytes) so that the
    // stores to out are 16 bytes per lane and 128 consecutive bytes per 8 lanes.
    if (partial) {
        // slice of K: the raw fp32 sums, 16 bytes per lane, into partial[split][M][N]
        float* pout = partial + static_cast<size_t>(split) * M * N;
        const bool vec4 = (N % 4) == 0;
        #pragma unroll
        for (int u = 0; u < 2; ++u) {
            #pragma unroll
            for (int rq = 0; rq < 4; ++rq) {
                const int nq = n0 + 64 * w + 32 * u + 8 * rq + 4 * g;
                #pragma unroll
                for (int t = 0; t < TM; ++t) {
                    const int m = m0 + 32 * t + li;
                    if (m >= M) continue;
                    float* dst = pout + static_cast<size_t>(m) * N + nq;
                    if (vec4 && nq + 3 < N) {
                        *reinterpret_cast<float4*>(dst) = float4{acc[u][t][4 * rq], acc[u][t][4 * rq + 1],
                                                                 acc[u][t][4 * rq + 2], acc[u][t][4 * rq + 3]};
                    } else {
                        #pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (nq + e < N) dst[e] = acc[u][t][4 * rq + e];
                    }
                }
            }
        }
        return;
    }
    MI_WAIT_LGKM(0);
    __builtin_amdgcn_s_barrier();                        // nobody reads operands from LDS any more
    MI_SCHED_FENCE();
    if (glu) {
        // rows 16 and up of a fragment of W belong to the up matrix, the 16 below to the same columns of the
        // gate matrix (see launch_gemm_glu): a lane holds both of 4 columns in sums 8 apart, and half as many
        // columns go out, 64 consecutive bytes per 4 lanes
        constexpr int kGRow = 80;
        const int glu_n = N / 2;
        uint8_t* gbase = lds + w * (BM * kGRow);
        #pragma unroll
        for (int u = 0; u < 2; ++u) {
            #pragma unroll
            for (int rq = 0; rq < 2; ++rq) {
                float s4[8] = {1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f};
                if constexpr (!Q4 && !F16) {
                    const uint2 sg = sc[u][rq], su = sc[u][rq + 2];
                    const uint32_t s2[4] = {sg.x, sg.y, su.x, su.y};
                    #pragma unroll
                    for (int e = 0; e < 8; ++e) s4[e] = h_f(static_cast<uint16_t>(e % 2 ? s2[e / 2] >> 16 : s2[e / 2] & 0xFFFFu));
                }
                #pragma unroll
                for (int t = 0; t < TM; ++t) {
                    const floatx16& a = acc[u][t];
                    const uint32_t g0 = pack_half2(a[4 * rq] * s4[0], a[4 * rq + 1] * s4[1]);
                    const uint32_t g1 = pack_half2(a[4 * rq + 2] * s4[2], a[4 * rq + 3] * s4[3]);
                    const uint32_t u0 = pack_half2(a[4 * rq + 8] * s4[4], a[4 * rq + 9] * s4[5]);
                    const uint32_t u1 = pack_half2(a[4 * rq + 10] * s4[6], a[4 * rq + 11] * s4[7]);
                    *reinterpret_cast<uint2*>(gbase + (32 * t + li) * kGRow + (16 * u + 8 * rq + 4 * g) * 2) =
                        uint2{swiglu_h2(g0, u0), swiglu_h2(g1, u1)};
                }
            }
        }
        const int gcol = n0 / 2 + 32 * w + 8 * (lane & 3);
        #pragma unroll
        for (int j = 0; j < BM / 16; ++j) {
            const int row = 16 * j + (lane >> 2);
            const u32x4 v = *reinterpret_cast<const u32x4*>(gbase + row * kGRow + (lane & 3) * 16);
            if (m0 + row < M && gcol < glu_n)                // (the width is a multiple of 16, out is aligned)
                __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(out + static_cast<size_t>(m0 + row) * glu_n + gcol));
        }
        return;
    }
    constexpr int kERow = 144;
    uint8_t* ebase = lds + w * (BM * kERow);
    #pragma unroll
    for (int u = 0; u < 2; ++u) {
        #pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
            float s4[4] = {1.0f, 1.0f, 1.0f, 1.0f};
            if constexpr (!Q4 && !F16) {
                s4[0] = __half2float(__ushort_as_half(static_cast<uint16_t>(sc[u][rq].x & 0xFFFFu)));
                s4[1] = __half2float(__ushort_as_half(static_cast<uint16_t>(sc[u][rq].x >> 16)));
                s4[2] = __half2float(__ushort_as_half(static_cast<uint16_t>(sc[u][rq].y & 0xFFFFu)));
                s4[3] = __half2float(__ushort_as_half(static_cast<uint16_t>(sc[u][rq].y >> 16)));
            }
            #pragma unroll
            for (int t = 0; t < TM; ++t) {
                const uint32_t lo = pack_half2(acc[u][t][4 * rq] * s4[0], acc[u][t][4 * rq + 1] * s4[1]);
                const uint32_t hi = pack_half2(acc[u][t][4 * rq + 2] * s4[2], acc[u][t][4 * rq + 3] * s4[3]);
                *reinterpret_cast<uint2*>(ebase + (32 * t + li) * kERow + (32 * u + 8 * rq + 4 * g) * 2) = uint2{lo, hi};
            }
        }
    }
    // each wavefront reads back only what it wrote itself
    const int ncol = n0 + 64 * w + 8 * (lane & 7);       // first of this lane's 8 output columns
    const bool cols8 = (N % 8) == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    #pragma unroll
    for (int j = 0; j < BM / 8; ++j) {
        const int row = 8 * j + (lane >> 3);
        const u32x4 v = *reinterpret_cast<const u32x4*>(ebase + row * kERow + (lane & 7) * 16);
        const int m = m0 + row;
        if (m >= M) continue;
        uint16_t* dst = out + static_cast<size_t>(m) * N + ncol;
        if (cols8 && ncol + 7 < N) {
            // streaming store: all blocks of a round write their tiles at about the same time, 20 MB at
            // M = 2048, N = 4864, and nothing reads them back soon (measured: 25.8 -> 24.2 us there)
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(dst));
        } else {
            #pragma unroll
            for (int e = 0; e < 8; ++e)
                if (ncol + e < N) dst[e] = static_cast<uint16_t>(v[e / 2] >> (16 * (e % 2)));
        }
    }
}

// out[m][n] = fp16((sum over slices of partial[slice][m][n]) * scale[n]) (no factor when scale is
// null); slices are added in index order, so the result does not depend on how the blocks were
// scheduled.
__global__ __launch_bounds__(256) void reduce_partials(const float* __restrict__ partial, int splits,
                                                       const uint16_t* __restrict__ scale,
                                                       uint16_t* __restrict__ out, long MN, int N) {
    const long i4 = (static_cast<long>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (i4 >= MN) return;
    const bool vec = (N % 4) == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0;
    if (vec) {
        // eight, four, two slices are requested at a time and then added in index order: a few trips
        // to memory instead of one per slice (16 slices of 64 x 896: 5.4 -> 3.5 us)
        float4 a = *reinterpret_cast<const float4*>(partial + i4);
        int z = 1;
        auto add_batch = [&](auto nc) {
            constexpr int n = decltype(nc)::value;
            float4 b[n];
            #pragma unroll
            for (int u = 0; u < n; ++u) b[u] = *reinterpret_cast<const float4*>(partial + (z + u) * MN + i4);
            #pragma unroll
            for (int u = 0; u < n; ++u) { a.x += b[u].x; a.y += b[u].y; a.z += b[u].z; a.w += b[u].w; }
            z += n;
        };
        while (splits - z >= 8) add_batch(std::integral_constant<int, 8>{});
        if (splits - z >= 4) add_batch(std::integral_constant<int, 4>{});
        if (splits - z >= 2) add_batch(std::integral_constant<int, 2>{});
        if (splits - z >= 1) add_batch(std::integral_constant<int, 1>{});
        const int n = static_cast<int>(i4 % N);
        float s0 = 1.0f, s1 = 1.0f, s2 = 1.0f, s3 = 1.0f;
        if (scale) {
            s0 = __half2float(__ushort_as_half(scale[n])), s1 = __half2float(__ushort_as_half(scale[n + 1]));
            s2 = __half2float(__ushort_as_half(scale[n + 2])), s3 = __half2float(__ushort_as_half(scale[n + 3]));
        }
        __builtin_nontemporal_store(u32x2{pack_half2(a.x * s0, a.y * s1), pack_half2(a.z * s2, a.w * s3)},
                                    reinterpret_cast<u32x2*>(out + i4));
    } else {
        for (int e = 0; e < 4 && i4 + e < MN; ++e) {
            float a = partial[i4 + e];
            for (int z = 1; z < splits; ++z) a += partial[z * MN + i4 + e];
            out[i4 + e] = to_half_bits(scale ? a * __half2float(__ushort_as_half(scale[(i4 + e) % N])) : a);
        }
    }
}

// The same for interleaved gate and up columns (see launch_gemm_glu): out[m][c] = swiglu of the two, four columns per
// thread; the sums are added and rounded as above.  N: columns of both.
__global__ __launch_bounds__(256) void reduce_partials_glu(const float* __restrict__ partial, int splits,
                                                           const uint16_t* __restrict__ scale, uint16_t* __restrict__ out,
                                                           long MN, int N) {
    const long o4 = (static_cast<long>(blockIdx.x) * 256 + threadIdx.x) * 4;       // element of out
    if (o4 >= MN / 2) return;
    const long m = o4 / (N / 2);
    const int c = static_cast<int>(o4 - m * (N / 2)), n = 32 * (c / 16) + c % 16;
    const float* p = partial + m * N + n;
    float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 16);
    int z = 1;
    auto add_batch = [&](auto nc) {
        constexpr int k = decltype(nc)::value;
        float4 x[k], y[k];
        #pragma unroll
        for (int u = 0; u < k; ++u) {
            x[u] = *reinterpret_cast<const float4*>(p + (z + u) * MN);
            y[u] = *reinterpret_cast<const float4*>(p + (z + u) * MN + 16);
        }
        #pragma unroll
        for (int u = 0; u < k; ++u) {
            a.x += x[u].x; a.y += x[u].y; a.z += x[u].z; a.w += x[u].w;
            b.x += y[u].x; b.y += y[u].y; b.z += y[u].z; b.w += y[u].w;
        }
        z += k;
    };
    while (splits - z >= 4) add_batch(std::integral_constant<int, 4>{});
    if (splits - z >= 2) add_batch(std::integral_constant<int, 2>{});
    if (splits - z >= 1) add_batch(std::integral_constant<int, 1>{});
    float s[8] = {1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f, 1.0f};
    if (scale) {
        #pragma unroll
        for (int e = 0; e < 4; ++e) { s[e] = h_f(scale[n + e]); s[4 + e] = h_f(scale[n + 16 + e]); }
    }
    *reinterpret_cast<uint2*>(out + o4) =
        uint2{swiglu_h2(pack_half2(a.x * s[0], a.y * s[1]), pack_half2(b.x * s[4], b.y * s[5])),
              swiglu_h2(pack_half2(a.z * s[2], a.w * s[3]), pack_half2(b.z * s[6], b.w * s[7]))};
}

// the kernel writes splits x M x N fp32 partial sums and gives every slice at least two K-stages
inline bool slices_fit(int splits, int M, int N, int K, size_t partial_bytes) {
    return K / 64 >= 2 * splits && static_cast<double>(splits) * M * N * 4 <= static_cast<double>(partial_bytes);
}

template <int TM, int KIND, int TERMS>
bool launch(hipStream_t s, int M, int N, int K, const void* x, const void* W, const void* scale, void* out,
            float* partial, size_t partial_bytes, int splits, const MoreMats& more, bool glu) {
    if (splits < 1 || (splits > 1 && (more.n || !partial || !slices_fit(splits, M, N, K, partial_bytes)))) {
        MI_ERROR_FMT("gemm: %d slices of K do not fit (M=%d N=%d K=%d, %zu bytes of workspace)", splits, M, N, K,
                     partial_bytes);
        return false;
    }
    constexpr size_t lds_bytes = static_cast<size_t>(stages_for(KIND, TM)) * (32 * TM * 128 + w_stage_bytes(KIND));
    auto* kern = gemm_wide<TM, KIND, TERMS>;
    if (lds_bytes > 65536 &&
        !MI_ONCE_OK(MI_HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes))))
        return false;
    const long total = static_cast<long>(more.n ? more.tiles : (N + kBN - 1) / kBN) * ((M + 32 * TM - 1) / (32 * TM)) * splits;
    const dim3 grid(static_cast<unsigned>(8 * ((total + 7) / 8)), 1, 1);      // see the block -> tile map in the kernel
    hipLaunchKernelGGL(kern, grid, dim3(256), lds_bytes, s, static_cast<const uint16_t*>(x),
                       static_cast<const uint8_t*>(W), static_cast<const uint16_t*>(scale),
                       static_cast<uint16_t*>(out), M, N, K, splits > 1 ? partial : nullptr, splits, more, static_cast<int>(glu));
    if (!MI_HIP_OK(hipGetLastError())) return false;
    if (splits > 1 && !out) return true;                 // the sums stay where they are (launch_gemm_slices)
    if (splits > 1 && glu) {
        const long MN = static_cast<long>(M) * N;
        hipLaunchKernelGGL(reduce_partials_glu, dim3(static_cast<unsigned>((MN / 8 + 255) / 256)), dim3(256), 0, s, partial, splits,
                           KIND == WK_I8 ? static_cast<const uint16_t*>(scale) : nullptr, static_cast<uint16_t*>(out), MN, N);
        if (!MI_HIP_OK(hipGetLastError())) return false;
    } else if (splits > 1) {
        const long MN = static_cast<long>(M) * N;
        hipLaunchKernelGGL(reduce_partials, dim3(static_cast<unsigned>((MN / 4 + 256) / 256)), dim3(256), 0, s,
                           partial, splits, KIND == WK_I8 ? static_cast<const uint16_t*>(scale) : nullptr,
                           static_cast<uint16_t*>(out), MN, N);
        if (!MI_HIP_OK(hipGetLastError())) return false;
    }
    return true;
}

// Estimated time (us) of the wide kernel with 32 * tm rows of x per block and K cut into
// `splits` slices.  Fitted to measurements on MI355X: a block takes about 2.6 + 0.5 tm us of
// prologue and epilogue plus, per K-stage of 64, 0.27 + 0.10 tm us for int8 weights, 0.56 + 0.10 tm
// for Q4 weights rounded to fp16 once and 0.49 + 0.22 tm for Q4 weights in two terms; a fully
// occupied chip runs the same cycles about 1.56 times slower (clock under load, shared L2 and
// fabric) than a nearly empty one.  Slices cost a second launch and the partial sums' trip
// through memory.
inline double estimate_us(int kind, int terms, int tm, int splits, int M, int N, int K, int cus) {
    const long blocks = static_cast<long>((M + 32 * tm - 1) / (32 * tm)) * ((N + kBN - 1) / kBN) * splits;
    const int stages = (K / 64 + splits - 1) / splits;
    const double stage_us = kind == WK_Q4 ? (terms == 2 ? 0.49 + 0.22 * tm : 0.56 + 0.10 * tm)
                          : kind == WK_F16 ? 0.35 + 0.10 * tm : 0.27 + 0.10 * tm;
    // two blocks on one CU take about 1.4 times as long each as one alone (the dispatcher puts a
    // second block on a CU only when every CU has one)
    const int per_cu = blocks > cus ? blocks_per_cu(kind, tm) : 1;
    const double block_us = (2.6 + 0.5 * tm + stages * stage_us) * (per_cu == 2 ? 1.4 : 1.0);
    const long slots = static_cast<long>(cus) * per_cu;
    const long full = (blocks - 1) / slots, rem = blocks - full * slots;     // the last round, full or not, is `rem`
    // (64-row tiles of int8 / fp16 weights, unsliced, on more than half of the CUs and at most one per CU,
    //  run nearly as on an empty chip: 512 x 4864 x 896 in 11.2 us where the general factor says 13.6 and the
    //  64 x 64 tiles, estimated at 13.5, take 13.2; 2048 x 1152 x 896 13.2 against 15.9, 512 x 4608 x 1024 12.1
    //  against 14.5, 4096 x 576 x 1536 18.9 against 33.5.  With fewer blocks the long serial K of such
    //  shapes decides and the general factor holds: 2048 x 896 x 4864 unsliced 47 against 37 us in two slices.
    //  32-row tiles likewise at a K of 1280 to 3072, where the 64 x 64 tiles slow down as soon as a CU holds
    //  two of them: 1536 x 576 x 1536 19.2 -> 14.6 us, 1024 x 2048 x 2048 23.2 -> 18.4, 192 x 8192 x 2048 21.6 ->
    //  17.3, fp16 1536 x 1024 x 2560 29.6 -> 22.7, and from K = 1024 on (2048 x 1024 x 1024: 12.2 against 14.5 us);
    //  at a shorter K the 64 x 64 tiles stay ahead (1536 x 1152 x 896 10.2 against 11.2), at a longer one
    //  slices do (1536 x 896 x 4864 32.6 against 37.7).
    //  Q4 weights in two terms behave the same there (1024 x 2048 x 2048 in 32-row tiles 29.1 us against 34.0
    //  in two slices, 256 x 8192 x 2048 29.2 against 35.0, 2048 x 576 x 1536 21.7 against 24.2), and their tall
    //  tiles, one block per CU and twice the matrix work per byte, lose less to a full chip than the general
    //  factors say: 2048 x 4864 x 896 in 160-row tiles 34.8 us (a block alone: 27.4), 4096 x 8192 x 2048 in
    //  128-row tiles 231 us for four rounds of 48.4, against 258 us for the 64-row tiles the factors preferred.)
    //  fp16 weights do so at any number of blocks and from 9 stages on: 300 x 4864 x 896 9.7 us, 416 x 5120 x 960 11.5, 917 x 3072 x
    //  576 8.5, where the general factor put the 64 x 64 tiles ahead, which take 11.8, 12.5 and 9.3.
    const bool bands = stages <= 16 && tiles_in_bands((N + 63) / 64, (M + 63) / 64);      // (the 64 x 64 tiles are the faster then)
    const bool f16_roomy = kind == WK_F16 && splits == 1 && blocks <= cus && tm <= 2 && stages <= 48 && !bands;
    // (int8, 32-row tiles of 14 or 15 stages: 304 x 4864 x 896 9.4 us, 192 x 9728 x 896 9.6, 320 x 5120 x 960 9.9, the 64 x 64 tiles
    //  9.6, 9.6 and 10.0, which leave the SwiGLU to a launch of its own.  Not where those go in bands: int8 2048 x 960 x 960 11.4
    //  against 10.4, fp16 1184 x 1600 x 960 12.5 against 10.4, 1408 x 960 x 576 7.7 against 7.2; at a longer K the wide tiles keep up:
    //  1856 x 576 x 1536 13.6 against 14.4)
    const bool i8_short = kind == WK_I8 && splits == 1 && tm == 1 && blocks > cus / 2 && blocks <= cus && (stages == 14 || stages == 15) && !bands;
    const bool roomy = splits == 1 && blocks > cus / 2 && blocks <= cus &&
                       (tm == 2 || (tm == 1 && stages >= 16 && stages <= 48));
    const bool q4_tall = kind == WK_Q4 && terms == 2 && tm >= 3 && splits == 1;
    const double crowd = f16_roomy ? (blocks * 5 > slots * 4 ? 0.2 : 0.05) : i8_short ? 0.4 : roomy ? 0.2 : q4_tall ? 0.3 : 0.56;
    const double round = q4_tall ? 1.25 : 1.56;
    double t = full * round * block_us + (rem ? (1.0 + crowd * rem / slots) * block_us : 0.0);
    // every row of tiles streams W again: not faster than that many bytes at about 6.8 TB/s, or,
    // for a W that stays in the memory-side cache (40 MB taken as the limit: fp16 8192 x 2048, 33.5 MB, still
    // runs eight rows of tiles in 25.9 us, and the choices at 50 MB and more are right as they are), 2.2 times that for
    // the reads after the first
    const double w_once = static_cast<double>(N) * K * (kind == WK_F16 ? 2.0 : kind == WK_I8 ? 1.0 : 0.5625);
    const int tiles_m = (M + 32 * tm - 1) / (32 * tm);
    const double w_bytes = w_once <= 40.0e6 ? w_once * (1.0 + (tiles_m - 1) / 2.2) : w_once * tiles_m;
    if (t < 2.5 + w_bytes / 6.8e6) t = 2.5 + w_bytes / 6.8e6;
    if (splits > 1) t += 2.5 + 2.0 * splits * M * static_cast<double>(N) * 4 / 4.0e6;   // ~4 TB/s there and back
    return t;
}

// Rows of x per block (in units of 32) and slices of K with the smallest estimated time; slices
// only as far as their fp32 partial sums fit the workspace.
inline void pick_shape(int kind, int terms, int M, int N, int K, int cus, size_t workspace_bytes, int* tm_out,
                       int* splits_out, double* best_us) {
    static const int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24};
    double best_t = 1e30;
    for (int tm = 1; tm <= 5; ++tm) {
        if (32 * (tm - 1) >= M) break;                   // no tile taller than x needs (16 x 49 152 x 576: 7.8 against 8.7 us)
        for (int sp : kSplits) {
            if (sp > 1 && (K / 64 < 2 * sp || static_cast<double>(sp) * M * N * 4 > static_cast<double>(workspace_bytes)))
                continue;
            const double t = estimate_us(kind, terms, tm, sp, M, N, K, cus);
            if (t < best_t) { best_t = t; *tm_out = tm; *splits_out = sp; }
        }
    }
    if (best_us) *best_us = best_t;
}

// The same among two slices and more: false where none fits.
inline bool pick_sliced(int kind, int terms, int M, int N, int K, int cus, size_t workspace_bytes, int* tm_out, int* splits_out,
                        double* best_us) {
    *best_us = 1e30;
    for (int tm = 1; tm <= 5 && 32 * (tm - 1) < M; ++tm)
        for (int sp : {2, 3, 4, 6, 8, 12, 16, 24}) {
            if (!slices_fit(sp, M, N, K, workspace_bytes)) continue;
            const double t = estimate_us(kind, terms, tm, sp, M, N, K, cus);
            if (t < *best_us) { *best_us = t; *tm_out = tm; *splits_out = sp; }
        }
    return *best_us < 1e30;
}

template <int KIND, int TERMS>
bool launch_any(int tm, hipStream_t s, int M, int N, int K, const void* x, const void* W,
                const void* scale, void* out, float* partial, size_t partial_bytes, int splits, const MoreMats& more,
                bool glu) {
    switch (tm) {
        case 1: return launch<1, KIND, TERMS>(s, M, N, K, x, W, scale, out, partial, partial_bytes, splits, more, glu);
        case 2: return launch<2, KIND, TERMS>(s, M, N, K, x, W, scale, out, partial, partial_bytes, splits, more, glu);
        case 3: return launch<3, KIND, TERMS>(s, M, N, K, x, W, scale, out, partial, partial_bytes, splits, more, glu);
        case 4: return launch<4, KIND, TERMS>(s, M, N, K, x, W, scale, out, partial, partial_bytes, splits, more, glu);
        default: return launch<5, KIND, TERMS>(s, M, N, K, x, W, scale, out, partial, partial_bytes, splits, more, glu);
    }
}

}  // namespace wide

// ---- 256 x 256 blocks, 128 x 128 per wavefront (int8 weights) --------------------------------------
//
// The wide kernel above gives a wavefront 64 rows of W against up to 160 rows of x: per MFMA it reads
// (2 + 2 TM) / (4 TM) fragments from LDS, and at 160 rows that traffic (133 KB per stage of K = 64) takes
// the LDS four fifths as long as the MFMAs take the matrix cores, overlapped by less than half.  Here the
// four wavefronts sit two along x by two along W and each owns 128 x 128 of the block's 256 x 256 outputs:
// sixteen 32 x 32 accumulators (all 256 AGPRs), four fragments of W and four of x per 16 MFMAs, 37 % less
// LDS read traffic and 19 % less fill traffic per MFMA.  Same LDS layout, swizzles, K permutation, fills
// and barrier scheme as the wide kernel; three stages of 48 KB.  It needs whole rounds of 256-row tiles to
// pay: a few hundred tiles at least, and a long K (each block's prologue and epilogue stand alone on its CU).
namespace quad {

constexpr int kBM = 256, kBN = 256, kStages = 3;
constexpr int kXStage = kBM * 128, kWStage = kBN * 64, kStage = kXStage + kWStage;
constexpr int kXLoads = 8, kWLoads = 4, kLoads = kXLoads + kWLoads;   // 1 KB loads per wavefront and stage
constexpr int kReads = 12, kConv = 16, kMfmas = 32;                   // per half stage (K = 32)
constexpr int kERow = 272;                                            // epilogue: 128 columns of fp16 + 16 bytes

struct Frags {
    u32x4 w[4];                // 16 int8 weights of four 32-row fragments of W
    uint32_t wf[4][2][4];      // the same as fp16: [fragment][MFMA of the pair][4 dwords = 8 halves]
    u32x4 x[2][4];             // [MFMA of the pair][32-row fragment of x]
};

using wide::lds_fill16;
using wide::static_for;
using wide::pack_half2;

__global__ __launch_bounds__(256) void gemm_quad(const uint16_t* __restrict__ X, const uint8_t* __restrict__ W,
                                                 const uint16_t* __restrict__ scale, uint16_t* __restrict__ out,
                                                 int M, int N, int K) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = w >> 1, wc = w & 1;                  // this wavefront's 128 rows of x, 128 rows of W
    const int g = lane >> 5, li = lane & 31;
    // block -> tile: as in the wide kernel (an XCD takes a contiguous eighth of the list, bands of 4 tiles along N)
    int tile_m, tile_n;
    {
        const int tiles_m = (M + kBM - 1) / kBM, tiles_n = (N + kBN - 1) / kBN, total = tiles_m * tiles_n;
        const int per_xcd = (total + 7) / 8;
        const int l = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
        if (blockIdx.x >= 8 * per_xcd || l >= total) return;          // whole block, before any barrier
        constexpr int kBand = 4;
        const int band = l / (kBand * tiles_m);
        const int width = tiles_n - band * kBand < kBand ? tiles_n - band * kBand : kBand;
        const int in_band = l - band * kBand * tiles_m;
        tile_m = in_band / width;
        tile_n = band * kBand + in_band % width;
    }
    const int m0 = tile_m * kBM, n0 = tile_n * kBN;
    const uint32_t lbase = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((wide::lds_u8*)lds));

    // fill side: x load j covers rows 8 (w + 4 j) .. + 7 of the tile (128 bytes each, chunk p of row r in slot
    // p ^ ((r >> 1) & 7)); W load j rows 16 (4 w + j) .. + 15 (64 bytes each, slot p ^ ((r >> 2) & 3))
    uint32_t xsrc[kXLoads], wsrc[kWLoads];
    #pragma unroll
    for (int j = 0; j < kXLoads; ++j) {
        const int r = 8 * (w + 4 * j) + (lane >> 3);
        const int c = (lane & 7) ^ ((r >> 1) & 7);
        const int m = m0 + r < M ? m0 + r : M - 1;
        xsrc[j] = static_cast<uint32_t>(m) * K * 2u + c * 16u;
    }
    #pragma unroll
    for (int j = 0; j < kWLoads; ++j) {
        const int r = 16 * (4 * w + j) + (lane >> 2);
        const int c = (lane & 3) ^ ((r >> 2) & 3);
        const int n = n0 + r < N ? n0 + r : N - 1;
        wsrc[j] = static_cast<uint32_t>(n) * K + c * 16u;
    }
    const uint8_t* Xb = reinterpret_cast<const uint8_t*>(X);
    auto fill_one = [&](int stage_k, int slot, auto jc) {
        constexpr int j = decltype(jc)::value;
        uint8_t* xs = lds + slot * kStage;
        if constexpr (j < kXLoads)
            lds_fill16(Xb + static_cast<size_t>(stage_k) * 128 + xsrc[j], xs + 1024 * (w + 4 * j));
        else
            lds_fill16(W + static_cast<size_t>(stage_k) * 64 + wsrc[j - kXLoads], xs + kXStage + 1024 * (4 * w + (j - kXLoads)));
    };
    auto fill_stage = [&](int stage_k, int slot) {
        static_for<kLoads>([&](auto jc) { fill_one(stage_k, slot, jc); });
    };

    // read side: pair S of a stage, MFMA e of the pair: x chunk 4 S + 2 g + e, W chunk 2 S + g
    const uint32_t xrow = lbase + (128u * wr + li) * 128u, xq = (2u * g) ^ ((li >> 1) & 7u);
    const uint32_t wrow = lbase + kXStage + (128u * wc + li) * 64u, wq = g ^ ((li >> 2) & 3u);
    uint32_t xoff[2][2], woff[2];
    #pragma unroll
    for (int S = 0; S < 2; ++S) {
        #pragma unroll
        for (int e = 0; e < 2; ++e) xoff[S][e] = xrow + (((4u * S + e) ^ xq) << 4);
        woff[S] = wrow + (((2u * S) ^ wq) << 4);
    }
    // read j of a set: the four W fragments first, then x for the first and the second MFMA of the pair
    auto read_one = [&](Frags& F, uint32_t slot_bytes, auto Sc, auto jc) {
        constexpr int S = decltype(Sc)::value, j = decltype(jc)::value;
        if constexpr (j < 4) {
            const uint32_t a = woff[S] + slot_bytes;
            MI_LDS_READ16(F.w[j], a, j * 32 * 64);
        } else {
            constexpr int e = (j - 4) / 4, t = (j - 4) % 4;
            const uint32_t a = xoff[S][e] + slot_bytes;
            MI_LDS_READ16(F.x[e][t], a, t * 4096);
        }
    };
    auto convert_one = [&](Frags& F, auto jc) {
        constexpr int j = decltype(jc)::value, u = j / 4, d = j % 4;
        i8x4_to_h4(F.w[u][d], F.wf[u][d / 2][2 * (d % 2)], F.wf[u][d / 2][2 * (d % 2) + 1]);
    };

    floatx16 acc[4][4];
    #pragma unroll
    for (int u = 0; u < 4; ++u)
        #pragma unroll
        for (int t = 0; t < 4; ++t)
            #pragma unroll
            for (int r = 0; r < 16; ++r) acc[u][t][r] = 0.0f;

    auto mfma_one = [&](const Frags& F, auto nc) {
        constexpr int n = decltype(nc)::value, e = n / 16, u = (n / 4) % 4, t = n % 4;
        const u32x4 wv = u32x4{F.wf[u][e][0], F.wf[u][e][1], F.wf[u][e][2], F.wf[u][e][3]};
        acc[u][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, wv),
                                                          __builtin_bit_cast(half8, F.x[e][t]), acc[u][t], 0, 0, 0);
    };

    // one half stage: the fills of a later stage, the reads and conversions of the next fragments, dealt out
    // between the MFMAs of the current ones
    auto half_stage = [&](Frags& C, Frags& Nx, uint32_t next_bytes, auto NSc, auto fillc, int fill_k, int fill_slot) {
        constexpr bool FILL = decltype(fillc)::value;
        constexpr int nF = FILL ? kLoads : 0;
        constexpr int A = nF + kReads + 1 + kConv;
        static_for<kMfmas>([&](auto nc) {
            constexpr int n = decltype(nc)::value;
            mfma_one(C, nc);
            MI_SCHED_FENCE();
            constexpr int a0 = n * A / kMfmas, a1 = (n + 1) * A / kMfmas;
            static_for<a1 - a0>([&](auto kc) {
                constexpr int a = a0 + decltype(kc)::value;
                if constexpr (a < nF) {
                    fill_one(fill_k, fill_slot, std::integral_constant<int, a>{});
                } else if constexpr (a < nF + kReads) {
                    read_one(Nx, next_bytes, NSc, std::integral_constant<int, a - nF>{});
                } else if constexpr (a == nF + kReads) {
                    // LDS returns in order: with the eight x reads outstanding, the four W reads are back
                    asm volatile("s_waitcnt lgkmcnt(8)" : "+v"(Nx.w[0]), "+v"(Nx.w[1]), "+v"(Nx.w[2]), "+v"(Nx.w[3]) : : "memory");
                    MI_SCHED_FENCE();
                } else {
                    convert_one(Nx, std::integral_constant<int, a - nF - kReads - 1>{});
                }
            });
            MI_SCHED_FENCE();
        });
        MI_WAIT_LGKM(0);
        MI_SCHED_FENCE();
    };
    // at most `stages` (0 or 1) of this wavefront's stage fills still in flight
    auto wait_fills = [&](int stages) {
        if (stages >= 1) MI_WAIT_VM(kLoads); else MI_WAIT_VM(0);
    };

    const int nk = K / 64;
    Frags FA, FB;
    #pragma unroll
    for (int st = 0; st < kStages - 1; ++st)
        if (st < nk) fill_stage(st, st);
    wait_fills((nk < kStages - 1 ? nk : kStages - 1) - 1);          // stage 0 has landed
    __builtin_amdgcn_s_barrier();
    MI_SCHED_FENCE();
    static_for<kReads>([&](auto jc) { read_one(FA, 0u, std::integral_constant<int, 0>{}, jc); });
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(FA.w[0]), "+v"(FA.w[1]), "+v"(FA.w[2]), "+v"(FA.w[3]) : : "memory");
    MI_SCHED_FENCE();
    static_for<kConv>([&](auto jc) { convert_one(FA, jc); });

    auto stage = [&](int i, int slot, auto fillc) {
        const int next = slot + 1 == kStages ? 0 : slot + 1;
        const int prev = slot == 0 ? kStages - 1 : slot - 1;
        half_stage(FA, FB, static_cast<uint32_t>(slot) * kStage, std::integral_constant<int, 1>{}, std::false_type{}, 0, 0);
        MI_SCHED_FENCE();
        const int last = i + kStages - 2 < nk - 1 ? i + kStages - 2 : nk - 1;   // newest stage requested so far
        wait_fills(last - (i + 1));
        __builtin_amdgcn_s_barrier();
        MI_SCHED_FENCE();
        half_stage(FB, FA, static_cast<uint32_t>(next) * kStage, std::integral_constant<int, 0>{}, fillc, i + kStages - 1, prev);
        MI_SCHED_FENCE();
    };
    int slot = 0, i = 0;
    for (; i + kStages - 1 < nk; ++i) {
        stage(i, slot, std::true_type{});
        slot = slot + 1 == kStages ? 0 : slot + 1;
    }
    for (; i < nk; ++i) {
        stage(i, slot, std::false_type{});
        slot = slot + 1 == kStages ? 0 : slot + 1;
    }

    // epilogue: D[i][j], i = 8 (r / 4) + 4 g + r % 4 a row of W (an output column), j = li a row of x.  The scaled
    // fp16 values go through LDS (this wavefront's own 128 x 128 patch, rows padded to 272 bytes) so that the
    // stores are 16 bytes per lane, 256 consecutive bytes per 16 lanes.
    MI_WAIT_LGKM(0);
    __builtin_amdgcn_s_barrier();                        // nobody reads operands from LDS any more
    MI_SCHED_FENCE();
    uint8_t* ebase = lds + w * (128 * kERow);
    const bool cols4 = (N % 4) == 0 && reinterpret_cast<uintptr_t>(scale) % 8 == 0;
    #pragma unroll
    for (int u = 0; u < 4; ++u) {
        #pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
            const int nq = n0 + 128 * wc + 32 * u + 8 * rq + 4 * g;
            uint32_t h[4];
            if (cols4 && nq + 3 < N) {
                const uint2 v = *reinterpret_cast<const uint2*>(scale + nq);
                h[0] = v.x & 0xFFFFu; h[1] = v.x >> 16; h[2] = v.y & 0xFFFFu; h[3] = v.y >> 16;
            } else {
                #pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = scale[nq + e < N ? nq + e : N - 1];
            }
            float s4[4];
            #pragma unroll
            for (int e = 0; e < 4; ++e) s4[e] = __half2float(__ushort_as_half(static_cast<uint16_t>(h[e])));
            #pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t lo = pack_half2(acc[u][t][4 * rq] * s4[0], acc[u][t][4 * rq + 1] * s4[1]);
                const uint32_t hi = pack_half2(acc[u][t][4 * rq + 2] * s4[2], acc[u][t][4 * rq + 3] * s4[3]);
                *reinterpret_cast<uint2*>(ebase + (32 * t + li) * kERow + (32 * u + 8 * rq + 4 * g) * 2) = uint2{lo, hi};
            }
        }
    }
    // each wavefront reads back only what it wrote itself
    const int ncol = n0 + 128 * wc + 8 * (lane & 15);    // first of this lane's 8 output columns
    const bool cols8 = (N % 8) == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
    #pragma unroll 4
    for (int j = 0; j < 32; ++j) {
        const int row = 4 * j + (lane >> 4);
        const u32x4 v = *reinterpret_cast<const u32x4*>(ebase + row * kERow + (lane & 15) * 16);
        const int m = m0 + 128 * wr + row;
        if (m >= M) continue;
        uint16_t* dst = out + static_cast<size_t>(m) * N + ncol;
        if (cols8 && ncol + 7 < N) {
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(dst));
        } else {
            #pragma unroll
            for (int e = 0; e < 8; ++e)
                if (ncol + e < N) dst[e] = static_cast<uint16_t>(v[e / 2] >> (16 * (e % 2)));
        }
    }
}

bool launch(hipStream_t s, int M, int N, int K, const void* x, const void* W, const void* scale, void* out) {
    constexpr size_t lds_bytes = static_cast<size_t>(kStages) * kStage;
    static_assert(4 * 128 * kERow <= kStages * kStage, "the epilogue's patches fit the operand stages");
    if (!MI_ONCE_OK(MI_HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_quad),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes))))
        return false;
    const long total = static_cast<long>((N + kBN - 1) / kBN) * ((M + kBM - 1) / kBM);
    hipLaunchKernelGGL(gemm_quad, dim3(static_cast<unsigned>(8 * ((total + 7) / 8))), dim3(256), lds_bytes, s,
                       static_cast<const uint16_t*>(x), static_cast<const uint8_t*>(W),
                       static_cast<const uint16_t*>(scale), static_cast<uint16_t*>(out), M, N, K);
    return MI_HIP_OK(hipGetLastError());
}

}  // namespace quad

// ---- a few rows of x, and tiles of as many: the weights stream past them, as in the GEMV --------
//
// With up to 64 rows of x the contraction is bound by the weights' bytes, like the GEMV, not by the matrix cores, and the
// tiles above leave most of the chip idle (19 tiles at N = 4864).  Here a wavefront takes strips of 16 rows of W through
// v_mfma_f32_16x16x32_f16 against 16 MT rows of x, 64 values of K (a unit) at a time:
//   A = W strip: lane l supplies row l % 16, 8 values of K starting at 16 (l / 16) + 8 s of the unit's 64 (s = 0, 1: the two
//       MFMAs of a unit);
//   B = x^T: lane l supplies row l % 16 of the x tile at the same values of K;
//   D[i][j] (lane l: i = 4 (l / 16) + r, j = l % 16) = out[row j of the x tile][row i of the strip]:
//       four consecutive output columns per lane.
// How both get there, and how K is shared out: skinny_tile.
namespace skinny {

typedef float floatx4 __attribute__((ext_vector_type(4)));
constexpr int kMaxM = 64;
constexpr int kWaves = 8;                // wavefronts per block

// The sums of a 16 x 16 tile's kb slices of K, each in one wavefront of a block of its own, meet in memory: the
// wavefront that arrives last takes all of them in slice order (a lane the sums of the lanes of its number) and goes
// on with their total; the others return false.  Sums and counter travel as agent-scope accesses, which pass the
// XCDs' own L2s: a store that has been acknowledged (vmcnt) is where every other CU's such load looks for it.  No
// block waits for another.  The counter starts at 0 (add_workspace) and is left at 0; launches on a stream are ordered.
// What it replaces is a second launch over 1 KB per tile and slice, which in a prompt or a batch waits for this one and
// holds up the next: a prompt of 37 fp16 tokens 1618 -> 1576 us in 32 layers (960 x 2560 each); at 64 rows equal.
__device__ __forceinline__ bool meet_slices(floatx4& acc, float* __restrict__ sums, uint32_t* __restrict__ counter, const int by,
                                            const int kb, const int lane) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    auto* at = reinterpret_cast<uint64_t*>(sums) + lane;                 // [kb][2][64] pairs
    #pragma unroll
    for (int h = 0; h < 2; ++h)
        __hip_atomic_store(at + (by * 2 + h) * 64, __builtin_bit_cast(uint64_t, f32x2{acc[2 * h], acc[2 * h + 1]}),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint32_t before = 0;
    if (lane == 0) before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    before = __builtin_amdgcn_readfirstlane(before);
    if (before + 1 != static_cast<uint32_t>(kb)) return false;
    asm volatile("" ::: "memory");
    if (lane == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    constexpr int kMost = 8;                                             // slices over blocks (pick_shape), asked for together
    f32x2 v[kMost][2];
    #pragma unroll
    for (int y = 0; y < kMost; ++y)
        #pragma unroll
        for (int h = 0; h < 2; ++h)
            v[y][h] = __builtin_bit_cast(f32x2, __hip_atomic_load(at + ((y < kb ? y : 0) * 2 + h) * 64, __ATOMIC_RELAXED,
                                                                  __HIP_MEMORY_SCOPE_AGENT));
    #pragma unroll
    for (int y = 0; y < kMost; ++y)
        if (y < kb) {
            #pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = y == 0 ? v[y][r / 2][r % 2] : acc[r] + v[y][r / 2][r % 2];
        }
    return true;
}

// Up to 64 rows of x, or tiles of as many.  A wavefront owns a tile of 16 S columns of the output (S strips of 16 rows of W) and a slice of K, and
// works for itself: it asks for its slice of x and of W, 64 values of K at a time, by direct global -> LDS loads into a ring of
// its own, waits for its own loads only, and multiplies.  ks wavefronts of a block share a tile; their sums meet in LDS, in
// slice order, behind the one barrier of the kernel.
//
// What bounds such a launch is the way to memory, and how much of it is asked for at once: a few us of latency and one pass
// over the weights.  So
//  * everything a block needs is on its way before anything is used, up to 160 KB of LDS per CU and without registers;
//  * a load instruction covers whole pieces of rows, 64 or 128 bytes of each (8 lanes to a row of x).  As fragments straight
//    from memory neighbouring lanes are in different rows, and a load of 64 lanes is 64 lookups in the L1, for x as often
//    as a block has strips: that bounded the launch;
//  * the 16-byte pieces of a row are XOR-swizzled so that fragment reads are free of bank conflicts without padding.
// us per launch, weights from HBM, with fragments (x copied to LDS first where it fitted) -> this: fp16, 37 rows of 960 x 2560 9.7 ->
// 8.1, 1600 x 960 6.1 -> 5.3, 960 x 960 6.0 -> 4.5, 5120 x 960 with the SwiGLU 7.6 -> 6.6, 64 rows of 576 x 1536 9.8 -> 5.9; int8, 16 rows of
// 896 x 896 4.2 -> 3.7, 9728 x 896 with the SwiGLU 7.0 -> 6.7; Q4, 24 rows of 896 x 4864 9.8 -> 7.4; the floor of a launch is 1.6.
// An int8 weight becomes fp16 in the registers (exactly).  Q4: q * scale as two exact fp16 terms (scale = hi + lo with 7 and
// 4 significant bits, as in the wide kernel), or rounded to fp16 once with TERMS = 1.
// GLU: see launch_gemm_glu; the tile's strips are the gate's and the up matrix's in turn (S = 2, 4).
// MEET: kb slices of K over blocks, which meet as told at meet_slices (an instance of its own, S = 1).
// Without MEET and with `partial` the sums go there, [slice over blocks][M][N], for a launch that adds them (N a multiple of 4).
template <int KIND, int MT, int S>
struct Unit {                                            // what 64 values of K take in a wavefront's ring
    static constexpr int kX = MT * 2048;                 // rows of 128 bytes
    static constexpr int kW = KIND == WK_F16 ? S * 2048 : KIND == WK_I8 ? S * 1024 : S * 512;
    static constexpr int kBytes = kX + kW + (KIND == WK_Q4 ? S * 64 : 0);              // Q4: two block scales per row
    static constexpr int kSums = MT * S * 1024;          // the tile's fp32 sums, which take the place of the ring
    static constexpr int kLoads = 2 * MT + (KIND == WK_F16 ? 2 * S : KIND == WK_I8 ? S : 2);
};
constexpr int kMaxRing = 8;                              // units in a ring

template <int LOADS>
__device__ __forceinline__ void wait_for_all_but(int units) {           // the loads of the last `units` units may be under way
    #define MI_CASE(u) case u: MI_WAIT_VM((u) * LOADS < 63 ? (u) * LOADS : 63); break;
    switch (units) {
        MI_CASE(0) MI_CASE(1) MI_CASE(2) MI_CASE(3) MI_CASE(4) MI_CASE(5) MI_CASE(6)
        default: MI_WAIT_VM(7 * LOADS < 63 ? 7 * LOADS : 63);
    }
    #undef MI_CASE
}

// A unit's fragments from LDS (the wait stands in the block that reads: the registers are in flight until then).
#define MI_X1 "ds_read_b128 %[p0], %[a]\n\tds_read_b128 %[q0], %[b]\n\t"
#define MI_X2 MI_X1 "ds_read_b128 %[p1], %[a] offset:2048\n\tds_read_b128 %[q1], %[b] offset:2048\n\t"
#define MI_X3 MI_X2 "ds_read_b128 %[p2], %[a] offset:4096\n\tds_read_b128 %[q2], %[b] offset:4096\n\t"
#define MI_X4 MI_X3 "ds_read_b128 %[p3], %[a] offset:6144\n\tds_read_b128 %[q3], %[b] offset:6144\n\t"
#define MI_OX1 [p0] "=&v"(x[0][0]), [q0] "=&v"(x[0][1])
#define MI_OX2 MI_OX1, [p1] "=&v"(x[1][0]), [q1] "=&v"(x[1][1])
#define MI_OX3 MI_OX2, [p2] "=&v"(x[2][0]), [q2] "=&v"(x[2][1])
#define MI_OX4 MI_OX3, [p3] "=&v"(x[3][0]), [q3] "=&v"(x[3][1])
#define MI_F1 "ds_read_b128 %[w0], %[a] offset:%[o0]\n\tds_read_b128 %[v0], %[b] offset:%[o0]\n\t"
#define MI_F2 MI_F1 "ds_read_b128 %[w1], %[a] offset:%[o1]\n\tds_read_b128 %[v1], %[b] offset:%[o1]\n\t"
#define MI_F4 MI_F2 "ds_read_b128 %[w2], %[a] offset:%[o2]\n\tds_read_b128 %[v2], %[b] offset:%[o2]\n\t" \
              "ds_read_b128 %[w3], %[a] offset:%[o3]\n\tds_read_b128 %[v3], %[b] offset:%[o3]\n\t"
#define MI_OF1 [w0] "=&v"(w[0][0]), [v0] "=&v"(w[0][1])
#define MI_OF2 MI_OF1, [w1] "=&v"(w[1][0]), [v1] "=&v"(w[1][1])
#define MI_OF4 MI_OF2, [w2] "=&v"(w[2][0]), [v2] "=&v"(w[2][1]), [w3] "=&v"(w[3][0]), [v3] "=&v"(w[3][1])
#define MI_I1 "ds_read_b128 %[w0], %[d]\n\t"
#define MI_I2 MI_I1 "ds_read_b128 %[w1], %[d] offset:1024\n\t"
#define MI_I4 MI_I2 "ds_read_b128 %[w2], %[d] offset:2048\n\tds_read_b128 %[w3], %[d] offset:3072\n\t"
#define MI_OI1 [w0] "=&v"(w[0][0])
#define MI_OI2 MI_OI1, [w1] "=&v"(w[1][0])
#define MI_OI4 MI_OI2, [w2] "=&v"(w[2][0]), [w3] "=&v"(w[3][0])
#define MI_Q1 "ds_read_b64 %[w0], %[d]\n\tds_read_b32 %[v0], %[e]\n\t"
#define MI_Q2 MI_Q1 "ds_read_b64 %[w1], %[d] offset:512\n\tds_read_b32 %[v1], %[e] offset:64\n\t"
#define MI_OQ1 [w0] "=&v"(w4[0]), [v0] "=&v"(ws[0])
#define MI_OQ2 MI_OQ1, [w1] "=&v"(w4[1]), [v1] "=&v"(ws[1])
#define MI_READ_MT(MTN, WS, OWS, ...)                                                                      \
    if constexpr (MT == MTN)                                                                               \
        asm volatile(MI_X##MTN WS "s_waitcnt lgkmcnt(0)" : MI_OX##MTN, OWS : [a] "v"(a), [b] "v"(b), __VA_ARGS__ : "memory");
#define MI_READ_S(SN, L, ...)                                                                              \
    if constexpr (S == SN) {                                                                               \
        MI_READ_MT(1, MI_##L##SN, MI_O##L##SN, __VA_ARGS__)                                                \
        MI_READ_MT(2, MI_##L##SN, MI_O##L##SN, __VA_ARGS__)                                                \
        MI_READ_MT(3, MI_##L##SN, MI_O##L##SN, __VA_ARGS__)                                                \
        MI_READ_MT(4, MI_##L##SN, MI_O##L##SN, __VA_ARGS__)                                                \
    }
template <int KIND, int MT, int S>
struct UnitFrags {
    u32x4 x[MT][2];
    u32x4 w[S][2];                                       // int8: only the first, 16 weights
    u32x2 w4[S];                                         // Q4: 16 weights and the row's two block scales
    uint32_t ws[S];
    // a, b: the lane's pieces 2c and 2c + 1 of its row of the first x tile; d: of the first strip; e: its scales
    __device__ __forceinline__ void read(uint32_t a, uint32_t b, uint32_t d, uint32_t e) {
        if constexpr (KIND == WK_F16) {
            MI_READ_S(1, F, [o0] "i"(MT * 2048))
            MI_READ_S(2, F, [o0] "i"(MT * 2048), [o1] "i"(MT * 2048 + 2048))
            MI_READ_S(4, F, [o0] "i"(MT * 2048), [o1] "i"(MT * 2048 + 2048), [o2] "i"(MT * 2048 + 4096), [o3] "i"(MT * 2048 + 6144))
        } else if constexpr (KIND == WK_I8) {
            MI_READ_S(1, I, [d] "v"(d))
            MI_READ_S(2, I, [d] "v"(d))
            MI_READ_S(4, I, [d] "v"(d))
        } else {
            MI_READ_S(1, Q, [d] "v"(d), [e] "v"(e))
            MI_READ_S(2, Q, [d] "v"(d), [e] "v"(e))
        }
    }
};

template <int KIND, int MT, int S, int TERMS, bool GLU, bool MEET>
__device__ __forceinline__ void skinny_tile(const uint16_t* __restrict__ X, const uint8_t* __restrict__ W,
                                            const uint16_t* __restrict__ scale, uint16_t* __restrict__ out, const int M, int N,
                                            const int K, const int ks, const int ring_units, float* __restrict__ partial,
                                            uint32_t* __restrict__ counters, const MoreMats& more, const int bx, const int waves,
                                            const int by, const int kb, const int bz) {
    static_assert(!GLU || S % 2 == 0, "strips of either matrix");
    constexpr bool F16 = KIND == WK_F16, Q4 = KIND == WK_Q4;
    typedef Unit<KIND, MT, S> U;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, c = lane >> 4;
    const int slice = wave & (ks - 1);
    int tile = bx * (waves / ks) + wave / ks;
    if constexpr (!GLU) pick_matrix(more, tile, W, scale, out, N);
    const int n0 = 16 * S * tile, m0 = 16 * MT * bz;
    const bool live = n0 < N;                            // (a block's last tiles may lie past the matrix: they take part in the barrier only)
    const int nb = live ? n0 : 0;

    // K is cut over kb blocks and, inside a block, over ks wavefronts
    const int its = K / 64, b0 = its * by / kb, b1 = its * (by + 1) / kb;
    const int it0 = b0 + (b1 - b0) * slice / ks, n = live ? b0 + (b1 - b0) * (slice + 1) / ks - it0 : 0;

    uint32_t sc[S][4];
    if constexpr (KIND == WK_I8) {                       // asked for first: used last
        #pragma unroll
        for (int s = 0; s < S; ++s)
            #pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int nq = nb + 16 * s + 4 * c + r;
                sc[s][r] = scale[nq < N ? nq : N - 1];
            }
    }

    // --- fill side: lane l of a load writes LDS bytes [16 l, +16) of its KB ---
    // x, fp16 W: a load covers 8 rows of 128 bytes; slot p of row r holds piece p ^ ((r >> 1) & 7)
    // int8: 16 rows of 64 bytes, piece p ^ ((r >> 2) & 3); Q4: 16 rows of 32 bytes (S of them), piece p ^ ((r >> 3) & 1)
    const size_t wrowb = Q4 ? static_cast<size_t>(K) / 2 : F16 ? static_cast<size_t>(K) * 2 : static_cast<size_t>(K);
    const uint8_t* const Xb = reinterpret_cast<const uint8_t*>(X) + static_cast<size_t>(m0) * K * 2 + static_cast<size_t>(it0) * 128;
    const uint8_t* const Wb = W + static_cast<size_t>(nb) * wrowb + static_cast<size_t>(it0) * (Q4 ? 32 : F16 ? 128 : 64);
    const int wlast = N - 1 - nb, xlast = M - 1 - m0;    // rows past N and M are read as the last row
    constexpr int kWL = F16 ? 2 * S : Q4 ? 1 : S;
    uint32_t xoff[2 * MT], woff[kWL];
    #pragma unroll
    for (int j = 0; j < 2 * MT; ++j) {
        const int r = 8 * j + (lane >> 3), m = r < xlast ? r : xlast;
        xoff[j] = static_cast<uint32_t>(m) * static_cast<uint32_t>(K) * 2u + 16u * ((lane & 7) ^ ((r >> 1) & 7));
    }
    #pragma unroll
    for (int j = 0; j < kWL; ++j) {
        int r, piece;
        if constexpr (F16) { r = 8 * j + (lane >> 3); piece = (lane & 7) ^ ((r >> 1) & 7); }
        else if constexpr (Q4) { r = lane >> 1; piece = (lane & 1) ^ ((r >> 3) & 1); }
        else { r = 16 * j + (lane >> 2); piece = (lane & 3) ^ ((r >> 2) & 3); }
        woff[j] = static_cast<uint32_t>(r < wlast ? r : wlast) * static_cast<uint32_t>(wrowb) + 16u * piece;
    }
    [[maybe_unused]] const uint8_t* Sb = nullptr;
    [[maybe_unused]] uint32_t soff = 0;
    if constexpr (Q4) {
        Sb = reinterpret_cast<const uint8_t*>(scale) + static_cast<size_t>(nb) * (K / 16) + static_cast<size_t>(it0) * 4;
        const int r = lane & (16 * S - 1);
        soff = static_cast<uint32_t>(r < wlast ? r : wlast) * static_cast<uint32_t>(K / 16);
    }
    const int stride = ring_units * U::kBytes > U::kSums ? ring_units * U::kBytes : U::kSums;
    uint8_t* const ring = lds + wave * stride;
    auto fill = [&](int u, int slot) {                   // unit u of the slice
        uint8_t* l = ring + slot * U::kBytes;
        #pragma unroll
        for (int j = 0; j < 2 * MT; ++j) wide::lds_fill16(Xb + static_cast<size_t>(u) * 128 + xoff[j], l + 1024 * j);
        const uint8_t* w = Wb + static_cast<size_t>(u) * (Q4 ? 32 : F16 ? 128 : 64);
        if constexpr (Q4) {
            if (lane < 32 * S) wide::lds_fill16(w + woff[0], l + U::kX);
            if (lane < 16 * S) wide::lds_fill4(Sb + static_cast<size_t>(u) * 4 + soff, l + U::kX + U::kW);
        } else {
            #pragma unroll
            for (int j = 0; j < kWL; ++j) wide::lds_fill16(w + woff[j], l + U::kX + 1024 * j);
        }
    };
    const int lead = n < ring_units ? n : ring_units;
    for (int u = 0; u < lead; ++u) fill(u, u);

    // --- read side ---
    const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((wide::lds_u8*)ring));
    const uint32_t xa = base + i * 128 + 16 * ((2 * c) ^ (i >> 1));
    const uint32_t wa = base + U::kX + (Q4 ? i * 32 + 16 * ((c >> 1) ^ (i >> 3)) + 8 * (c & 1) : i * 64 + 16 * (c ^ (i >> 2)));
    const uint32_t sa = base + U::kX + U::kW + i * 4;
    floatx4 acc[MT][S];
    #pragma unroll
    for (int t = 0; t < MT; ++t)
        #pragma unroll
        for (int s = 0; s < S; ++s) acc[t][s] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    int slot = 0;
    for (int u = 0; u < n; ++u) {
        const int issued = u + ring_units < n ? u + ring_units : n;
        wait_for_all_but<U::kLoads>(issued - u - 1);
        UnitFrags<KIND, MT, S> F;
        const uint32_t at = slot * U::kBytes;
        F.read(xa + at, (xa + at) ^ 16u, wa + at, sa + at);
        if (u + ring_units < n) fill(u + ring_units, slot);
        slot = slot + 1 == ring_units ? 0 : slot + 1;
        #pragma unroll
        for (int s = 0; s < S; ++s) {
            half8 a[TERMS][2];
            if constexpr (F16) {
                a[0][0] = __builtin_bit_cast(half8, F.w[s][0]);
                a[0][1] = __builtin_bit_cast(half8, F.w[s][1]);
            } else if constexpr (Q4) {
                const uint32_t both = __builtin_amdgcn_perm(0u, F.ws[s], c >> 1 ? 0x03020302u : 0x01000100u);
                __half2 st[TERMS];
                if constexpr (TERMS == 2) {
                    st[0] = __builtin_bit_cast(__half2, both & 0xFFF0FFF0u);
                    st[1] = __hsub2(__builtin_bit_cast(__half2, both), st[0]);
                } else {
                    st[0] = __builtin_bit_cast(__half2, both);
                }
                #pragma unroll
                for (int e = 0; e < 2; ++e)
                    #pragma unroll
                    for (int z = 0; z < TERMS; ++z)
                        a[z][e] = __builtin_bit_cast(half8, u32x4{q4x2_to_h2<0>(F.w4[s][e], st[z]), q4x2_to_h2<1>(F.w4[s][e], st[z]),
                                                                  q4x2_to_h2<2>(F.w4[s][e], st[z]), q4x2_to_h2<3>(F.w4[s][e], st[z])});
            } else {
                uint32_t h[8];
                #pragma unroll
                for (int d = 0; d < 4; ++d) i8x4_to_h4(F.w[s][0][d], h[2 * d], h[2 * d + 1]);
                a[0][0] = __builtin_bit_cast(half8, u32x4{h[0], h[1], h[2], h[3]});
                a[0][1] = __builtin_bit_cast(half8, u32x4{h[4], h[5], h[6], h[7]});
            }
            #pragma unroll
            for (int z = 0; z < TERMS; ++z)
                #pragma unroll
                for (int e = 0; e < 2; ++e)
                    #pragma unroll
                    for (int t = 0; t < MT; ++t)
                        acc[t][s] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[z][e], __builtin_bit_cast(half8, F.x[t][e]), acc[t][s], 0, 0, 0);
        }
    }

    // The slices' sums meet in LDS, each where its wavefront's ring was; sum t S + s of the tile (GLU: both sums of rows t) is
    // then finished by the tile's wavefront of that number mod ks, which adds them in slice order.
    auto sums_of = [&](int w) { return reinterpret_cast<floatx4*>(lds + w * stride); };
    if (ks > 1) {                                        // (the same for every wavefront of the block)
        #pragma unroll
        for (int t = 0; t < MT; ++t)
            #pragma unroll
            for (int s = 0; s < S; ++s) sums_of(wave)[(t * S + s) * 64 + lane] = acc[t][s];
        __syncthreads();
    }
    if (!live) return;
    const bool cols4 = (N % 4) == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0;
    #pragma unroll
    for (int t = 0; t < MT; ++t) {
        [[maybe_unused]] uint2 h[S];
        #pragma unroll
        for (int s = 0; s < S; ++s) {
            if (((GLU ? t : t * S + s) & (ks - 1)) != slice) continue;
            const int strip = tile * S + s;
            if (16 * strip >= N) continue;
            floatx4 v = acc[t][s];
            if (ks > 1) {
                v = sums_of(wave - slice)[(t * S + s) * 64 + lane];
                for (int z = 1; z < ks; ++z) {
                    const floatx4 o = sums_of(wave - slice + z)[(t * S + s) * 64 + lane];
                    #pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] += o[r];
                }
            }
            const int nq = 16 * strip + 4 * c, m = m0 + 16 * t + i;      // first of this lane's 4 output columns, its row
            if constexpr (MEET) {
                const int met = (bz * ((N + 15) / 16) + strip) * MT + t;
                if (kb > 1 && !meet_slices(v, partial + static_cast<size_t>(met) * kb * 256, counters + met, by, kb, lane))
                    continue;
            } else if constexpr (!GLU) {
                if (partial) {                           // (N is a multiple of 4 then)
                    if (m < M && nq < N) *reinterpret_cast<floatx4*>(partial + (static_cast<size_t>(by) * M + m) * N + nq) = v;
                    continue;
                }
            }
            if constexpr (KIND == WK_I8) {
                #pragma unroll
                for (int r = 0; r < 4; ++r) v[r] *= h_f(static_cast<uint16_t>(sc[s][r]));
            }
            const uint32_t lo = wide::pack_half2(v[0], v[1]), hi = wide::pack_half2(v[2], v[3]);
            if constexpr (GLU) {
                h[s] = uint2{lo, hi};
                continue;
            }
            if (m >= M || nq >= N) continue;
            uint16_t* dst = out + static_cast<size_t>(m) * N + nq;
            if (cols4 && nq + 3 < N) {
                *reinterpret_cast<uint2*>(dst) = uint2{lo, hi};
            } else {
                #pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (nq + r < N) dst[r] = static_cast<uint16_t>((r / 2 ? hi : lo) >> (16 * (r % 2)));
            }
        }
        if constexpr (GLU) {
            if ((t & (ks - 1)) == slice && m0 + 16 * t + i < M) {
                #pragma unroll
                for (int s = 0; s < S; s += 2)
                    if (n0 + 16 * s < N)
                        *reinterpret_cast<uint2*>(out + static_cast<size_t>(m0 + 16 * t + i) * (N / 2) + (n0 + 16 * s) / 2 + 4 * c) =
                            uint2{swiglu_h2(h[s].x, h[s + 1].x), swiglu_h2(h[s].y, h[s + 1].y)};
            }
        }
    }
}

template <int KIND, int MT, int S, int TERMS, bool GLU, bool MEET>
__global__ __launch_bounds__(64 * kWaves) void gemm_skinny(const uint16_t* __restrict__ X, const uint8_t* __restrict__ W,
                                                           const uint16_t* __restrict__ scale, uint16_t* __restrict__ out,
                                                           int M, int N, int K, int ks, int ring_units, float* __restrict__ partial,
                                                           uint32_t* __restrict__ counters, MoreMats more) {
    skinny_tile<KIND, MT, S, TERMS, GLU, MEET>(X, W, scale, out, M, N, K, ks, ring_units, partial, counters, more, blockIdx.x,
                                               blockDim.x >> 6, blockIdx.y, gridDim.y, blockIdx.z);
}

constexpr size_t kLdsLimit = 160 * 1024;
inline size_t unit_bytes(int kind, int mt, int S) {      // Unit::kBytes
    return static_cast<size_t>(mt) * 2048 + (kind == WK_F16 ? S * 2048 : kind == WK_I8 ? S * 1024 : S * 576);
}

// bytes of partial sums that kb slices of K over blocks leave in the workspace (meet_slices)
inline size_t partial_bytes(int mt, int N, int kb) { return static_cast<size_t>((N + 15) / 16) * kb * mt * 1024; }

// ks: wavefronts that share a tile, the fewest of 4 and 8 that give the chip four wavefronts per CU (4 at least: with two, 9728 x 896 at
// 16 rows 7.2 us, with four 6.7); 8 only where a ring holds two units then (fp16 at more than 48 rows: 3072 x 576 5.2 us in 4
// slices, 6.0 in 8) and, one strip to a wavefront, from a K of 768 on: below, a wavefront has one unit or two, and more of them only
// meet later (int8, 16 rows of 1536 x 576 3.8 in 4 slices, 4.0 in 8; of 960 x 576 3.5 / 3.8; 1600 x 960 as fast either way).  kb: slices over
// blocks where one block per tile still leaves most CUs idle and the trip of the sums through memory, 2.5 us, is less than
// what it saves, from more than 4 units per wavefront on (896 x 4864 at 16 rows: 8.7 us in 8 slices, 7.1 in 8 x 4; 2048 x 2048 at 8 Q4 rows
// 5.6 in 8, 6.6 in 8 x 2, int8 5.5 / 6.5).  S: two strips per wavefront where one per wavefront is more blocks than CUs: x is
// fetched half as often (4864 x 896 at 48 int8 rows 6.7 -> 6.1 us), up to 16 rows only from five blocks per CU on (Q4 32 000 x 320 8.0 with one, 6.0
// with two); fewer blocks than CUs with two lose (1152 x 896 at 16 rows 3.7 against 4.1).
struct Shape { int ks, kb, S; };
// before: the slices that estimate_us was fitted with
inline Shape pick_shape(int kind, int M, int N, int K, int cus, size_t workspace_bytes, bool before = false) {
    const int mt = (M + 15) / 16;
    const long strips = (N + 15) / 16;
    const int its = K / 64;
    Shape sh{1, 1, strips > cus && (mt > 1 || strips > 5L * cus) ? 2 : 1};
    const long tiles = (strips + sh.S - 1) / sh.S;
    const int most = 2 * kWaves * unit_bytes(kind, mt, 2) <= kLdsLimit ? kWaves : kWaves / 2;
    while (sh.ks < most && (sh.ks < 4 || tiles * sh.ks < (sh.S == 2 ? 5L : 4L) * cus) && its >= 2 * sh.ks) sh.ks *= 2;
    if (sh.S == 1 && sh.ks == 8 && its < 12 && !before) sh.ks = 4;
    if (sh.ks == most) {
        while (sh.kb < 8 && strips * sh.kb * 2 <= cus && its >= 4 * sh.ks * sh.kb + !before && strips * mt <= kSliceCounters &&
               partial_bytes(mt, N, 2 * sh.kb) <= workspace_bytes)
            sh.kb *= 2;
    }
    return sh;
}
// The slices of a launch whose sums another launch adds: as many over blocks as give every CU one, 4 in a block (us at kb = 1 /
// these / twice as many: fp16, 37 rows of 960 x 2560 8.8 / 4.9 / 5.0, 960 x 960 4.6 / 3.6 / 3.8, int8, 16 rows of 896 x 4864 8.9 / 4.6 / 4.5).
// kb = 1: none, the launch would save nothing.
inline Shape pick_apart(int kind, int M, int N, int K, int cus, size_t workspace_bytes) {
    const long strips = (N + 15) / 16;
    const int its = K / 64;
    Shape sh{4, 1, 1};
    while (sh.kb < 8 && strips * (sh.kb + 1) <= cus && its >= sh.ks * (sh.kb + 1) &&
           static_cast<size_t>(sh.kb + 1) * M * N * 4 <= workspace_bytes)
        ++sh.kb;
    return sh;
}

// Where the streaming kernel is the library's own choice, against the tiles above (us, weights from HBM).
//  - Up to 64 rows: 2560 x 1024 at 24 / 40 / 64 rows 4.4 / 4.7 / 5.2 (fp16 5.0 / 5.6 / 6.2) against 8.7 to 9.6 for the 64 x 64 tiles, 896 x
//    4864 at 64 fp16 rows 9.1 against 14 (the wide kernel in slices), 8192 x 2048 12.6 against 16.2.
//  - Fewer of many rows of W, where the tiles fetch x once per 64 of them: fp16 up to 32 beyond 8192 (9728 x 896 at 32 / 48 / 64 rows 8.5 / 9.6 /
//    10.5 against 8.8 / 9.3 / 9.7); int8 up to 48 beyond 12 288 (64 rows of 14 592 x 896 9.7 / 9.4, 19 456 x 896 12.4 / 11.9), 32 beyond 24 576
//    (48 of 32 000 x 320 7.6 / 6.9).  int8 of a K up to 512 beyond 48 rows goes in tiles of 32 rows, 16 columns each: 64 rows of 1024 x 512 3.6
//    against 4.0 here.
//  - Not beyond 36 MB of weights, nor, above 13.5 MB, 80 rows of W per CU: the wide kernel's higher streaming rate wins there (int8
//    49 152 x 576 at 16 rows 11.2 against 7.3).
inline bool preferred(int kind, int M, int N, int K, int cus) {
    const double w_bytes = static_cast<double>(N) * K * (kind == WK_F16 ? 2.0 : kind == WK_Q4 ? 0.5625 : 1.0);
    const long strips = (N + 15) / 16;
    const int rows = kind == WK_F16 ? (strips > 2L * cus ? 32 : 64)
                   : kind == WK_I8 ? (strips > 6L * cus ? 32 : strips > 3L * cus || K <= 512 ? 48 : 64) : 64;
    return M <= rows && (w_bytes <= 13.5e6 ? strips <= (M > 48 ? 10L : 16L) * cus : w_bytes <= 36.0e6 && strips <= 5L * cus);
}

// ---- more rows of x than a tile holds: tiles of 16 mt rows by 16 S columns ----
//
// us per launch, weights from HBM, the 64 x 64 tiles or the wide kernel -> these: int8 100 / 300 / 600 rows of 1152 x 896 8.6 / 9.3 / 9.4 ->
// 4.7 / 5.6 / 7.2, 100 rows of 9728 x 896 with the SwiGLU 10.8 -> 9.8, Q4 300 rows of 896 x 896 12.0 -> 5.7, of 9728 x 896 with the SwiGLU
// 17.8 -> 15.8, 100 fp16 rows of 896 x 4864 14.2 -> 8.2.  From about 600 rows on by many columns the wide kernel's larger tiles
// win: a block here pulls 1 byte into LDS for 25 to 60 multiplications, there for 140.
//
// A launch takes 3.5 us and more the larger the tile, and for every round of blocks on the CUs the tile's end and what a block pulls
// into LDS: int8 and fp16 fitted to 4600 launches of 65 to 2048 rows, every tile at each of 310 calls (8 % rms; the tile it picks is 1 %
// behind the best one in the mean), Q4 to 1300 (10 %).  Blocks beyond one per CU come in rounds, a last round that is not full
// at about 0.6 of its price (the blocks in it have the L2s to themselves).  Tiles of 64 columns leave a CU with one block and wait
// for more before they begin, which a short K does not pay back (512 rows of 1536 x 576 fp16 7.5 us, with 32 columns 6.5); with Q4 never the best.
struct RowShape { int mt = 0, S = 1, ks = 4, kb = 1; double us = 1e30; };
inline double rows_us(int kind, int mt, int S, int kb, int M, int N, int K, int cus) {
    const long blocks = static_cast<long>((M + 16 * mt - 1) / (16 * mt)) * ((N + 16 * S - 1) / (16 * S)) * kb;
    const double unit = static_cast<double>(unit_bytes(kind, mt, S)), its = K / 64.0 / kb, mean = static_cast<double>(blocks) / cus;
    const long full = (blocks + cus - 1) / cus;
    auto rounds = [&](double f) { return full == 1 ? 1.0 : f * full + (1.0 - f) * mean; };
    if (kind == WK_Q4) return 4.1 + rounds(0.7) * its * unit / 57.0e3 * (S == 1 ? 0.72 : 1.0);
    if (kind == WK_F16)
        return 3.43 + 0.047 * mt * S + (S == 4 ? 0.25 : 0.0) +
               rounds(0.58) * (0.043 * mt * S + its * unit / 80.4e3 * (S == 4 ? 1.16 : S == 1 ? 0.92 : 1.0));
    return 3.51 + 0.047 * mt * S + (S == 4 ? 0.6 : 0.0) +
           rounds(0.64) * (0.022 * mt * S + its * unit / 74.6e3 * (S == 4 ? 1.26 : S == 1 ? 0.85 : 1.0));
}
// Slices of K inside a block, by what a launch by itself, one among several matrices and one with the SwiGLU have in
// common, since they decide the order of the sums.
inline int rows_ks(int M, int N, int K) {
    int ks = N > 8192 ? 2 : N > 1536 || M > 400 ? 4 : 8;
    while (ks > 1 && K / 64 < ks) ks /= 2;
    return ks;
}
// (a grid counts 65 535 tiles of rows)
inline bool rows_fit(int kind, int mt, int S, int ks, int M) {
    if ((static_cast<long>(M) + 16 * mt - 1) / (16 * mt) > 65535) return false;
    const size_t unit = unit_bytes(kind, mt, S), sums = static_cast<size_t>(mt) * S * 1024;
    return (ks < 4 ? 4 : ks) * (unit > sums ? unit : sums) <= kLdsLimit;
}
inline RowShape pick_rows(int kind, int M, int N, int K, int cus, bool glu) {
    RowShape best;
    for (int mt = 2; mt <= 4; ++mt)
        for (int S = 1; S <= 4; S *= 2) {
            const int ks = rows_ks(M, N, K);
            if ((S == 4 && (mt == 2 || kind == WK_Q4)) || (glu && S == 1) || !rows_fit(kind, mt, S, ks, M)) continue;
            const double us = rows_us(kind, mt, S, 1, M, N, K, cus);
            if (us < best.us) best = RowShape{mt, S, ks, 1, us};
        }
    return best;
}
// Where they are the choice over the kernels above, by the estimates of all (us, weights from HBM, tiles of rows / the other).
//  - Up to 64 rows of W per CU with Q4, 48 otherwise: beyond, the others stream better (80 int8 rows of 19 456 x 896 14.9 / 12.1, 100
//    Q4 rows 18.2 / 16.1, 56 fp16 rows of 14 592 x 896 13.6 / 10.3).
//  - Up to 8192 outputs per CU, about five rounds of tiles, from where 140 multiplications per byte pulled into LDS beat 25 to 60 (int8 512
//    rows of 4096 x 512 7.7 / 6.7); 9600 with Q4, which the wide kernel multiplies twice (3072 rows of 1536 x 576 20.4 / 16.2, 2600 of
//    1152 x 896 18.9 / 16.6), and at a long K up to 2e7 products per CU (600 rows of 2048 x 8192 67 / 51; 2560 x 2560 at 600 / 800 rows
//    25 / 27 and 37 / 32).  Many columns, the gate and up matrices of a prompt, whose SwiGLU rides in the launch: 300 x 9728 x 896 Q4 17.6 / 16.1
//    without it, but the prompt of 300 tokens 1477 / 1545.  Fewer rows for them: 600 x 3072 x 576 int8 9.0 / 8.2, 600 x 5120 x 960 17.5 / 14.1.
//    fp16 to 1280 rows (2048 x 896 x 896 11.6 / 10.1), int8 to 3072 (4096 x 333 x 1920 24.1 / 20.9).
//  - The estimates' own errors: the wide kernel's is 5 to 10 % too low without slices of K and 20 to 50 % too high with them (1200 x 896 x
//    4864 in three 25.6 us, estimated at 32.6; fp16 130 x 2048 x 8192 20.1, at 24.4), for a few rows of fp16 0.5 us too low on top (300 x
//    5120 x 960 12.5 against 10.7 here); the 64 x 64 tiles' is for weights in the caches, from HBM up to 1.5 us too low, the less the
//    shorter K (200 rows of 4096 x 256 6.0 / 4.4 as they were chosen with 1.5 for any K); this one's 8 % too low for int8 beyond 8192 rows of W,
//    in two slices of K.
// Of 2016 calls (30 shapes of W, 40 to 4096 rows, every kind) 20 are 3 to 16 % slower than with the kernels above alone, by 0.2 to 1.5 us: int8 1200 x
// 1536 x 576 8.8 / 7.6, fp16 300 x 3072 x 576 7.1 / 6.5, int8 600 x 1536 x 576 6.9 / 6.5.  Their layers, calls together, and prompts are
// the faster for them (a layer of 600 int8 rows 17.9 / 23.0 us, of 1200 29.4 / 32.8, 30 layers of 300 fp16 rows 1230 / 1360).
inline bool rows_preferred(int kind, const RowShape& r, double wide_us, int wide_slices, double tiled_us, int M, int N, int K, int cus) {
    const double outs = static_cast<double>(M) * N, us = r.us * (kind == WK_I8 && N > 8192 ? 1.08 : 1.0);
    if (N > (kind == WK_Q4 ? 64L : 48L) * cus || outs > (kind != WK_Q4 ? 8192.0 : N > 2560 ? 16000.0 : 9600.0) * cus || (kind == WK_Q4 && outs * K > 2.0e7 * cus)) return false;
    if ((N > 2560 && M > (kind == WK_Q4 ? 512 : 304)) || M > (kind == WK_F16 ? 1280 : kind == WK_I8 ? 3072 : 1 << 30)) return false;
    if (wide_slices > 1) wide_us *= kind == WK_F16 ? 0.82 : M <= 1024 ? 0.85 : 0.7;
    else if (kind != WK_Q4) wide_us = kind == WK_I8 ? 1.05 * wide_us : 1.1 * wide_us + (M <= 304 ? 0.5 : 0.0);
    return us < wide_us && (kind == WK_Q4 || us < tiled_us + (K < 640 ? (K - 128) / 345.0 : 1.5));
}
// The same cut into slices over blocks for a launch that adds them (mt = 0: not worth it).
inline RowShape pick_rows_apart(int kind, int M, int N, int K, int cus, size_t workspace_bytes) {
    RowShape best;
    const int its = K / 64;
    if (its < 14 || static_cast<long>((M + 47) / 48) * ((N + 31) / 32) > cus * 9L / 5) return best;
    for (int mt = 2; mt <= 4; ++mt)
        for (int S = 1; S <= 4; S *= 2) {
            if ((S == 4 && (mt == 2 || kind == WK_Q4)) || !rows_fit(kind, mt, S, 4, M)) continue;
            for (int kb = 2; kb <= 6 && its >= 4 * kb && static_cast<size_t>(kb) * M * N * 4 <= workspace_bytes; ++kb) {
                const double us = rows_us(kind, mt, S, kb, M, N, K, cus) + kb * 4.0e-6 * M * N / 4.0;
                if (us < best.us) best = RowShape{mt, S, 4, kb, us};
            }
        }
    return best;
}

// Estimated time (us): what decides between this kernel and rows of GEMV below 16 rows.  Fitted to the kernel that took fragments
// from memory, with its slices, and 0.3 to 1 us too high: 8 to 15 rows of a small matrix stay rows of GEMV, whose results are the
// reference's order bit for bit, though 16 rows of a 0.5B layer take 7.4 us here and 8 rows 12 there.
inline double estimate_us(int kind, int M, int N, int K, int cus, size_t workspace_bytes) {
    const Shape sh = pick_shape(kind, M, N, K, cus, workspace_bytes, true);
    const double w_bytes = static_cast<double>(N) * K * (kind == WK_F16 ? 2.0 : kind == WK_Q4 ? 0.5625 : 1.0);
    // (Q4 weights: the two-term feed costs 0.6 us more, 1.1 with K over blocks)
    const double q4_us = kind == WK_Q4 ? (sh.kb > 1 ? 1.1 : 0.6) : 0.0;
    // (x from the caches: 0.07 us per row where several strips of a block read it, 0.03 where the block's
    //  eight wavefronts share one strip, 0.06 with K over blocks as well)
    const double xg_us = sh.kb > 1 ? 5.4 + 0.06 * M : sh.ks == kWaves ? 3.6 + 0.03 * M : 3.6 + 0.07 * M;
    // (more than 13.5 MB: 19 456 x 896 at 8 int8 rows 8.6)
    return q4_us + (sh.ks < kWaves ? 3.75 + 0.035 * M : xg_us) + w_bytes / 8.0e6 + (w_bytes > 13.5e6 ? 2.4 : 0.0);
}

// ---- calls that share no x, in one launch ----
//
// Calls of a batch that cannot observe one another's results (the batch's host code checks that) and that the streaming
// kernel serves, each as its own plan has it (the same slices of K in the same order: the same bits as a launch of its
// own), a block per call and group of strips.  A launch of a few hundred rows of W takes 4 to 5 us whatever its size:
// the seven int8 projections of a 0.5B layer at 16 rows, four launches and one for the slices' sums, 26.6 -> 14.0 us (7.5 since
// the kernel loads by rows).
constexpr int kMaxManyGemm = 32;
struct SkinnyCalls {
    int n = 0, M = 0, ring = 1;
    uint16_t first[kMaxManyGemm] = {};                   // a call's first block
    struct Call {
        const uint16_t* X;
        const uint8_t* W;
        const uint16_t* scale;
        uint16_t* out;
        float* partial;
        uint32_t* counters;
        int N, K;
        uint16_t blocks;                                 // blocks along N; for every slice over blocks and tile of rows as many
        uint8_t ks, kb;                                  // slices inside a block and over blocks
    } c[kMaxManyGemm] = {};
};
static_assert(sizeof(SkinnyCalls) <= 4096, "kernel arguments");

// S = 1: up to 64 rows of x, slices over blocks may meet; S = 2: tiles of rows.
template <int KIND, int MT, int S, int TERMS>
__global__ __launch_bounds__(64 * kWaves) void gemm_skinny_many(const SkinnyCalls) {
    // (the argument is read where it lies: indexed by a run-time number it would be copied to scratch first)
    const auto* L = (const __attribute__((address_space(4))) SkinnyCalls*)__builtin_amdgcn_kernarg_segment_ptr();
    const int lane = threadIdx.x & 63, n = L->n, b = blockIdx.x;
    const int mine = L->first[lane < kMaxManyGemm ? lane : 0];
    const int q = __popcll(__ballot(lane < n && b >= mine)) - 1;
    const int blocks = L->c[q].blocks, at = b - L->first[q], kb = L->c[q].kb;
    const int piece = S == 2 || kb > 1 ? at / blocks : 0;                // slice over blocks, or tile of rows
    const MoreMats none{};
    skinny_tile<KIND, MT, S, TERMS, false, S == 1>(L->c[q].X, L->c[q].W, L->c[q].scale, L->c[q].out, L->M, L->c[q].N, L->c[q].K, L->c[q].ks,
                                                   L->ring, L->c[q].partial, L->c[q].counters, none, at - piece * blocks, kWaves,
                                                   S == 1 ? piece : 0, kb, S == 1 ? 0 : piece);
}

// Units of K in a wavefront's ring: its whole slice where `per_cu` such blocks fit the LDS of a CU.
inline int ring_units(size_t unit, int waves, long per_cu, int K, int ks, int kb) {
    const int its = (K / 64 + kb - 1) / kb, most = (its + ks - 1) / ks;
    int ring = static_cast<int>(kLdsLimit / static_cast<size_t>(per_cu < 1 ? 1 : per_cu > 4 ? 4 : per_cu) / (waves * unit));
    if (ring > kMaxRing) ring = kMaxRing;
    if (ring > most) ring = most;
    return ring < 1 ? 1 : ring;
}

template <int KIND, int MT, int S, int TERMS, bool GLU, bool MEET>
bool launch_one(hipStream_t s, int M, int N, int K, const void* x, const void* W, const void* scale, void* out, Shape sh,
                float* partial, uint32_t* counters, const MoreMats& more) {
    const int ks = sh.ks, waves = ks < 4 ? 4 : ks;
    const long tiles = more.n ? more.tiles : (N + 16 * S - 1) / (16 * S), per_block = waves / ks;
    const long blocks = (tiles + per_block - 1) / per_block;
    const int cus = device_info().cus;
    constexpr size_t unit = Unit<KIND, MT, S>::kBytes;
    const long tiles_m = (M + 16 * MT - 1) / (16 * MT);
    const int ring = ring_units(unit, waves, (blocks * sh.kb * tiles_m + cus - 1) / cus, K, ks, sh.kb);
    const size_t lds = waves * (ring * unit > Unit<KIND, MT, S>::kSums ? ring * unit : Unit<KIND, MT, S>::kSums);
    auto* kern = gemm_skinny<KIND, MT, S, TERMS, GLU, MEET>;
    if (lds > 65536 &&
        !MI_ONCE_OK(MI_HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kLdsLimit)))))
        return false;
    hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(sh.kb), static_cast<unsigned>(tiles_m)), dim3(64 * waves), lds, s,
                       static_cast<const uint16_t*>(x), static_cast<const uint8_t*>(W), static_cast<const uint16_t*>(scale),
                       static_cast<uint16_t*>(out), M, N, K, ks, ring, partial, counters, more);
    return MI_HIP_OK(hipGetLastError());
}

// glu, or sums for another launch (`apart`), or neither
template <int KIND, int MT, int TERMS>
bool launch_mt(hipStream_t s, int M, int N, int K, const void* x, const void* W, const void* scale, void* out, Shape sh,
               float* partial, const MoreMats& more, bool glu, bool apart) {
    if (glu) return launch_one<KIND, MT, 2, TERMS, true, false>(s, M, N, K, x, W, scale, out, sh, nullptr, nullptr, more);
    if (sh.kb > 1 && !apart)
        return launch_one<KIND, MT, 1, TERMS, false, true>(s, M, N, K, x, W, scale, out, sh, partial, slice_counters(partial), more);
    float* sums = apart ? partial : nullptr;
    return sh.S == 2 ? launch_one<KIND, MT, 2, TERMS, false, false>(s, M, N, K, x, W, scale, out, sh, sums, nullptr, more)
                     : launch_one<KIND, MT, 1, TERMS, false, false>(s, M, N, K, x, W, scale, out, sh, sums, nullptr, more);
}

template <int KIND, int TERMS>
bool launch(hipStream_t s, int M, int N, int K, const void* x, const void* W, const void* scale, void* out, Shape sh,
            void* workspace, size_t workspace_bytes, const MoreMats& more, bool glu, bool apart = false) {
    if (M < 1 || M > kMaxM || !(sh.ks == 1 || sh.ks == 2 || sh.ks == 4 || sh.ks == 8) || sh.kb < 1 || (sh.kb > 1 && more.n) ||
        (glu && sh.kb > 1) || (apart && (!workspace || static_cast<size_t>(sh.kb) * M * N * 4 > workspace_bytes)) ||
        (sh.kb > 1 && !apart && (!workspace || partial_bytes((M + 15) / 16, N, sh.kb) > workspace_bytes ||
                       (N + 15) / 16 * ((M + 15) / 16) > kSliceCounters))) {
        MI_ERROR_FMT("gemm: the streaming kernel takes up to %d rows of x, 1, 2, 4 or 8 slices of K per block "
                     "and a workspace for slices over blocks (M=%d K=%d, %d slices, %d slices over blocks, %zu bytes)",
                     kMaxM, M, K, sh.ks, sh.kb, workspace_bytes);
        return false;
    }
    auto* partial = static_cast<float*>(workspace);
    switch ((M + 15) / 16) {
        case 1: return launch_mt<KIND, 1, TERMS>(s, M, N, K, x, W, scale, out, sh, partial, more, glu, apart);
        case 2: return launch_mt<KIND, 2, TERMS>(s, M, N, K, x, W, scale, out, sh, partial, more, glu, apart);
        case 3: return launch_mt<KIND, 3, TERMS>(s, M, N, K, x, W, scale, out, sh, partial, more, glu, apart);
        default: return launch_mt<KIND, 4, TERMS>(s, M, N, K, x, W, scale, out, sh, partial, more, glu, apart);
    }
}

template <int KIND, int MT, int TERMS>
bool launch_rows_mt(hipStream_t s, int M, int N, int K, const void* x, const void* W, const void* scale, void* out, int S, Shape sh,
                    float* sums, const MoreMats& more, bool glu) {
    if constexpr (MT > 2 && KIND != WK_Q4) {
        if (S == 4)
            return glu ? launch_one<KIND, MT, 4, TERMS, true, false>(s, M, N, K, x, W, scale, out, sh, nullptr, nullptr, more)
                       : launch_one<KIND, MT, 4, TERMS, false, false>(s, M, N, K, x, W, scale, out, sh, sums, nullptr, more);
    }
    if (glu) return launch_one<KIND, MT, 2, TERMS, true, false>(s, M, N, K, x, W, scale, out, sh, nullptr, nullptr, more);
    return S == 2 ? launch_one<KIND, MT, 2, TERMS, false, false>(s, M, N, K, x, W, scale, out, sh, sums, nullptr, more)
                  : launch_one<KIND, MT, 1, TERMS, false, false>(s, M, N, K, x, W, scale, out, sh, sums, nullptr, more);
}
// sums: null, or where the sums of kb slices go (for a launch that adds them)
template <int KIND, int TERMS>
bool launch_rows(hipStream_t s, int M, int N, int K, const void* x, const void* W, const void* scale, void* out, const RowShape& r,
                 float* sums, const MoreMats& more, bool glu) {
    const Shape sh{r.ks, r.kb, r.S};
    switch (r.mt) {
        case 2: return launch_rows_mt<KIND, 2, TERMS>(s, M, N, K, x, W, scale, out, r.S, sh, sums, more, glu);
        case 3: return launch_rows_mt<KIND, 3, TERMS>(s, M, N, K, x, W, scale, out, r.S, sh, sums, more, glu);
        default: return launch_rows_mt<KIND, 4, TERMS>(s, M, N, K, x, W, scale, out, r.S, sh, sums, more, glu);
    }
}

// The calls of L as one launch with `lds` bytes per block.
template <int KIND, int MT, int S, int TERMS>
bool launch_calls(hipStream_t s, const SkinnyCalls& L, unsigned blocks, size_t lds) {
    auto* kern = gemm_skinny_many<KIND, MT, S, TERMS>;
    if (lds > 65536 &&
        !MI_ONCE_OK(MI_HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kLdsLimit)))))
        return false;
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * kWaves), lds, s, L);
    return MI_HIP_OK(hipGetLastError());
}
template <int KIND, int TERMS>
bool launch_calls_mt(hipStream_t s, const SkinnyCalls& L, int mt, unsigned blocks, size_t lds) {
    if (L.M > kMaxM) return mt == 3 ? launch_calls<KIND, 3, 2, TERMS>(s, L, blocks, lds) : launch_calls<KIND, 4, 2, TERMS>(s, L, blocks, lds);
    switch (mt) {
        case 1: return launch_calls<KIND, 1, 1, TERMS>(s, L, blocks, lds);
        case 2: return launch_calls<KIND, 2, 1, TERMS>(s, L, blocks, lds);
        case 3: return launch_calls<KIND, 3, 1, TERMS>(s, L, blocks, lds);
        default: return launch_calls<KIND, 4, 1, TERMS>(s, L, blocks, lds);
    }
}

// n calls of one M and weight kind in as few launches as hold them.  Calls whose slices meet in memory go first, so that
// their last blocks' trips run under the others' work.  More than 64 rows: in the fewest tiles of at most 64 (fp16: 48) rows, 32
// columns wide, the longest K first, and as much LDS as lets two blocks share a CU, one's loads under the other's products (one
// block per CU: 130 int8 rows of 0.5B 21.1 against 15.5, 200 Q4 rows of 360M 25.9 against 21.0; fp16 in tiles of 64: 400 rows of 0.5B 35.9
// against 33.4).  us per layer, launches of their own -> together: 80 fp16 rows of 135M 17.4 -> 8.0, 130 int8 rows of 0.5B 27.9 -> 15.5,
// 700 int8 rows of 360M 49.8 -> 38.9, 2048 int8 rows of 0.5B (q, k, v and o) 105.0 -> 99.1.
inline int many_mt(int kind, int M) {
    const int tiles_m = (M + kMaxM - 1) / kMaxM, mt = ((M + tiles_m - 1) / tiles_m + 15) / 16;
    return tiles_m > 1 && (mt < 3 || kind == WK_F16) ? 3 : mt;
}
bool launch_many(hipStream_t s, const GemvCall* calls, int n, int terms, void* workspace, size_t workspace_bytes) {
    const WeightKind kind = calls[0].kind;
    const int M = calls[0].M, mt = many_mt(kind, M), S = M > kMaxM ? 2 : 1, rows_m = (M + 16 * mt - 1) / (16 * mt);
    const size_t unit = std::max(unit_bytes(kind, mt, S), static_cast<size_t>(mt) * S * 1024);
    SkinnyCalls L;
    long blocks = 0;
    size_t sums = 0;
    int counters = 0;
    auto flush = [&]() {
        if (L.n == 0) return true;
        L.M = M;
        const int cus = device_info().cus;
        for (int j = 0; j < L.n; ++j) {
            const int ring = ring_units(unit, kWaves, S == 2 ? 2 : (blocks + cus - 1) / cus, L.c[j].K, L.c[j].ks, L.c[j].kb);
            if (ring > L.ring) L.ring = ring;
        }
        const auto nb = static_cast<unsigned>(blocks);
        const size_t lds = kWaves * L.ring * unit;
        const bool ok = kind == WK_Q4 ? (terms == 1 ? launch_calls_mt<WK_Q4, 1>(s, L, mt, nb, lds) : launch_calls_mt<WK_Q4, 2>(s, L, mt, nb, lds))
                      : kind == WK_F16 ? launch_calls_mt<WK_F16, 1>(s, L, mt, nb, lds) : launch_calls_mt<WK_I8, 1>(s, L, mt, nb, lds);
        L = SkinnyCalls{};
        blocks = 0;
        sums = 0;
        counters = 0;
        return ok;
    };
    int longest = 0;
    for (int i = 0; i < n; ++i) longest = calls[i].K > longest ? calls[i].K : longest;
    for (int pass = 0; pass < 2; ++pass) {               // slices over blocks, or the longest K; the others
        for (int i = 0; i < n; ++i) {
            const GemvCall& c = calls[i];
            const Shape sh = M > kMaxM ? Shape{rows_ks(M, c.N, c.K), 1, S} : pick_shape(kind, M, c.N, c.K, device_info().cus, workspace_bytes);
            if (pass != (sh.kb > 1 || (M > kMaxM && c.K == longest) ? 0 : 1)) continue;
            const int strips = (c.N + 15) / 16, per_block = kWaves / sh.ks;
            const long along_n = ((c.N + 16 * S - 1) / (16 * S) + per_block - 1) / per_block, nb = along_n * sh.kb * (S == 2 ? rows_m : 1);
            if (nb > 65535) {
                MI_ERROR_FMT("gemm: a call beyond a launch of several (M=%d N=%d K=%d)", M, c.N, c.K);
                return false;
            }
            const size_t bytes = sh.kb > 1 ? partial_bytes(mt, c.N, sh.kb) : 0;
            if (L.n == kMaxManyGemm || blocks + nb > 65535 || sums + bytes > workspace_bytes ||
                counters + (bytes ? strips * mt : 0) > kSliceCounters) {
                if (!flush()) return false;
            }
            SkinnyCalls::Call& d = L.c[L.n];
            d.X = static_cast<const uint16_t*>(c.x);
            d.W = static_cast<const uint8_t*>(c.W);
            d.scale = static_cast<const uint16_t*>(c.scale);
            d.out = static_cast<uint16_t*>(c.y);
            d.N = c.N; d.K = c.K;
            d.blocks = static_cast<uint16_t>(along_n);
            d.ks = static_cast<uint8_t>(sh.ks);
            d.kb = static_cast<uint8_t>(sh.kb);
            if (bytes) {
                d.partial = reinterpret_cast<float*>(static_cast<char*>(workspace) + sums);
                d.counters = slice_counters(workspace) + counters;
                sums += bytes;
                counters += strips * mt;
            }
            L.first[L.n++] = static_cast<uint16_t>(blocks);
            blocks += nb;
        }
    }
    return flush();
}

}  // namespace skinny

template <int BM, int BN, int WM, int WN, int KIND, bool BANDS>
bool launch_tile_as(hipStream_t s, int M, int N, int K, const void* x, const void* W, const void* scale, void* out, const dim3& grid,
                    const MoreMats& more) {
    constexpr size_t lds_bytes = 2u * (BM + BN) * kLd * sizeof(uint16_t);
    auto* kern = gemm_kernel<BM, BN, WM, WN, KIND, BANDS>;
    // more than 64 KB of LDS per block has to be asked for once per kernel
    if (lds_bytes > 65536 &&
        !MI_ONCE_OK(MI_HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes))))
        return false;
    hipLaunchKernelGGL(kern, grid, dim3(kThreads), lds_bytes, s, static_cast<const uint16_t*>(x), static_cast<const uint8_t*>(W),
                       static_cast<const uint16_t*>(scale), static_cast<uint16_t*>(out), M, N, K, more);
    return MI_HIP_OK(hipGetLastError());
}

template <int BM, int BN, int WM, int WN>
bool launch_tile(hipStream_t s, WeightKind kind, int M, int N, int K, const void* x, const void* W,
                 const void* scale, void* out, const MoreMats& more) {
    const int tiles_n = more.n ? more.tiles : (N + BN - 1) / BN, tiles_m = (M + BM - 1) / BM;
    const long total = static_cast<long>(tiles_n) * tiles_m;
    if (tiles_in_bands(tiles_n, tiles_m)) {
        const dim3 list(static_cast<unsigned>(8 * ((total + 7) / 8)));
        return kind == WK_I8 ? launch_tile_as<BM, BN, WM, WN, WK_I8, true>(s, M, N, K, x, W, scale, out, list, more)
                             : launch_tile_as<BM, BN, WM, WN, WK_F16, true>(s, M, N, K, x, W, scale, out, list, more);
    }
    const dim3 grid(tiles_n, tiles_m);
    return kind == WK_I8 ? launch_tile_as<BM, BN, WM, WN, WK_I8, false>(s, M, N, K, x, W, scale, out, grid, more)
                         : launch_tile_as<BM, BN, WM, WN, WK_F16, false>(s, M, N, K, x, W, scale, out, grid, more);
}

inline long tiles(int M, int N, int bm, int bn) {
    return static_cast<long>((M + bm - 1) / bm) * ((N + bn - 1) / bn);
}

}  // namespace

bool gemm_supported(WeightKind kind, int M, int N, int K, const void* x, const void* W, const void* scale) {
    if (!(kind == WK_I8 || kind == WK_F16 || kind == WK_Q4) || M < 2 || N < 1 || K < kKT || K % kKT != 0) return false;
    if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(W) % 16) return false;
    if (kind != WK_F16 && !scale) return false;
    return kind != WK_Q4 || reinterpret_cast<uintptr_t>(scale) % 4 == 0;
}

namespace {

bool wide_reaches(WeightKind kind, int M, int N, int K) {     // 32-bit byte offsets
    return static_cast<double>(M) * K * 2 < 4294967296.0 &&
           static_cast<double>(N) * K * (kind == WK_F16 ? 2 : 1) < 4294967296.0;
}

// The 64 x 64 tiles are bound either by one tile's serial K loop (about 0.4 us per K-tile, up to
// 1.3 times that as the chip fills) or by throughput (1.2 to 1.55 ns per tile and K-tile);
// fitted to measurements.
double tiled_estimate_us(int M, int N, int K) {
    const int nk = K / kKT;
    const long t64 = tiles(M, N, 64, 64);
    const double serial = (0.9 + nk * 0.4) * (1.0 + 0.3 * (t64 < 128 ? t64 / 128.0 : 1.0));
    // (the CUs that hold a second tile set the time: 192 x 8192 x 2048, 384 tiles, takes the 22 us of 512
    //  tiles; whole rounds of CUs at such a K, halfway there at a short one: 16 x 19 456 x 896, 304 tiles,
    //  10.6 us, 1024 x 1152 x 896, 288 tiles, 9.5 us)
    const int cus = device_info().cus;
    const long rounds = (t64 + cus - 1) / cus * cus;
    const long counted = t64 <= cus ? t64 : nk >= 20 ? rounds : (t64 + rounds) / 2;
    const double bulk = 3.3 + counted * nk * (nk > 32 ? 0.00155 : 0.0012);
    return serial > bulk ? serial : bulk;
}

}  // namespace

double gemm_estimate_us(WeightKind kind, int M, int N, int K, size_t workspace_bytes) {
    const int terms = kind == WK_Q4 ? 2 : 1;
    double wide_us = 1e30;
    int tm = 1, splits = 1;
    if (wide_reaches(kind, M, N, K))
        wide::pick_shape(kind, terms, M, N, K, device_info().cus, workspace_bytes, &tm, &splits, &wide_us);
    if (M <= skinny::kMaxM && skinny::preferred(kind, M, N, K, device_info().cus))
        return skinny::estimate_us(kind, M, N, K, device_info().cus, workspace_bytes);
    if (kind == WK_Q4) return wide_us;
    const double tiled_us = tiled_estimate_us(M, N, K);
    return wide_us < tiled_us ? wide_us : tiled_us;
}

static GemmPlan make_plan(int mode, WeightKind kind, int M, int N, int K, size_t workspace_bytes);

GemmPlan plan_gemm(hipStream_t s, WeightKind kind, int M, int N, int K, size_t workspace_bytes) {
    const int set = gemm_mode(s), mode = set == 4 && kind != WK_Q4 ? 0 : set;   // mode 4 only concerns Q4 weights
    return kept_plan<GemmPlan>(PlanKey{mode, device_info().cus, kind, M, N, K, workspace_bytes},
                               [&] { return make_plan(mode, kind, M, N, K, workspace_bytes); });
}

static GemmPlan make_plan(int mode, WeightKind kind, int M, int N, int K, size_t workspace_bytes) {
    GemmPlan p;
    // 100 s + 10 + t: the wide kernel pinned to 32 t rows of x per block and s slices of K
    int pin_splits = 0;
    if (mode >= 111) { pin_splits = mode / 100; mode %= 100; }
    const int cus = device_info().cus;
    const bool wide_fits = wide_reaches(kind, M, N, K);
    int tm = 1, splits = 1;
    if (kind == WK_Q4) {
        // Q4 weights have the streaming kernel (a few rows of x; mode 5 asks for it by name) and the
        // wide kernel; modes 3 and 11..15 pin the latter to one slice of K.
        // Mode 4 feeds every weight as the single fp16 number nearest to q * scale (half the
        // MFMAs, an error of up to 2^-12 sum |w x|); all other modes feed q * scale exactly, as
        // two fp16 terms.
        if (mode == 2) return p;
        p.terms = mode == 4 ? 1 : 2;
        if (M <= skinny::kMaxM && (mode == 5 || ((mode == 0 || mode == 4) && skinny::preferred(WK_Q4, M, N, K, cus)))) {
            const skinny::Shape sh = skinny::pick_shape(WK_Q4, M, N, K, cus, workspace_bytes);
            p.kernel = 4; p.tile_rows = 16 * ((M + 15) / 16); p.k_slices = sh.ks * sh.kb;
            return p;
        }
        if (!wide_fits || mode == 5) return p;
        const bool may_slice = mode == 0 || mode == 4;
        double wide_us = 0.0;
        wide::pick_shape(WK_Q4, p.terms, M, N, K, cus, may_slice ? workspace_bytes : 0, &tm, &splits, &wide_us);
        if (may_slice || mode == 6) {
            const skinny::RowShape r = skinny::pick_rows(kind, M, N, K, cus, false);
            if (mode == 6 && !r.mt) return p;            // more rows than the grid counts
            if (mode == 6 || skinny::rows_preferred(kind, r, wide_us, splits, 0.0, M, N, K, cus)) {
                p.kernel = 6; p.tile_rows = 16 * r.mt; p.ks = r.ks; p.strips = r.S;
                return p;
            }
        }
        if (mode >= 11 && mode <= 15) tm = mode - 10;
        if (pin_splits) splits = pin_splits;
        p.kernel = 1; p.tile_rows = 32 * tm; p.k_slices = splits;
        return p;
    }
    // The 256 x 256 blocks (int8 weights): by name (mode 30), or by themselves where they pay, which takes
    // several full rounds of such tiles and a long K.  Measured against the 160-row wide tiles: 8192 x 8192 x
    // 8192 884 against 968 us, 8192 x 8192 x 2048 247 against 264 us; but 4096 x 4864 x 4864 (304 tiles, 1.2
    // rounds) 229 against 177 us and 4096 x 9728 x 896 (K of 14 stages) 89 against 78 us.
    if (kind == WK_I8 && wide_fits && (mode == 30 || mode == 0)) {
        const long t256 = static_cast<long>((M + 255) / 256) * ((N + 255) / 256);
        const long rounds = (t256 + cus - 1) / cus;
        if (mode == 30 || (K >= 2048 && rounds >= 4 && t256 * 10 >= rounds * cus * 9)) {
            p.kernel = 5; p.tile_rows = 256;
            return p;
        }
    }
    if (mode == 30) return p;
    // int8 and fp16, a few rows of x: the streaming kernel (mode 5 asks for it by name, up to 64 rows)
    if (M <= skinny::kMaxM && (mode == 5 || (mode == 0 && skinny::preferred(kind, M, N, K, cus)))) {
        const skinny::Shape sh = skinny::pick_shape(kind, M, N, K, cus, workspace_bytes);
        p.kernel = 4; p.tile_rows = 16 * ((M + 15) / 16); p.k_slices = sh.ks * sh.kb;
        return p;
    }
    if (mode == 5) return p;
    // the same in tiles of rows, where its estimated time beats that of the other two
    const skinny::RowShape r = mode == 0 || mode == 6 ? skinny::pick_rows(kind, M, N, K, cus, false) : skinny::RowShape{};
    auto rows = [&]() {
        p.kernel = 6; p.tile_rows = 16 * r.mt; p.ks = r.ks; p.strips = r.S;
        return p;
    };
    if (mode == 6) return r.mt ? rows() : p;               // (none: more rows than the grid counts)
    // the wide kernel where its estimated time beats that of the 64 x 64 tiles
    if (wide_fits && (mode == 0 || mode == 3 || (mode >= 11 && mode <= 15))) {
        double wide_us = 0.0;
        // modes 3 and 11..15 pin the plain kernel; slices of K are the library's own choice (mode 0)
        wide::pick_shape(kind, 1, M, N, K, cus, mode == 0 ? workspace_bytes : 0, &tm, &splits, &wide_us);
        if (mode >= 11) tm = mode - 10;
        if (pin_splits) splits = pin_splits;
        const double tiled_us = tiled_estimate_us(M, N, K);
        // (64 x 64 tiles in bands keep up from fewer outputs on: 2048 x 960 x 960 int8 12.2 us there, 12.3 in tiles of rows, 1200 x 1600 x 960 fp16
        // 12.6 / 13.0; but 1500 x 960 x 960 int8 11.9 / 10.5, 1200 rows 11.7 / 8.9, fp16 12.4 / 9.5.  Where 960 columns keep them, fewer columns
        // by such a K do too, which may go out with them: the layer of 360M at 2048 int8 rows 91.8 us, with k and v apart from q 95.3.)
        const bool banded = K <= 1024 && tiles_in_bands((N + 63) / 64, (M + 63) / 64) &&
                            (static_cast<double>(M) * N > 7000.0 * cus || (K >= 768 && M > 7 * cus));
        if (mode == 0 && !banded && skinny::rows_preferred(kind, r, wide_us, splits, tiled_us, M, N, K, cus)) return rows();
        if (mode != 0 || wide_us < tiled_us) {
            p.kernel = 1; p.tile_rows = 32 * tm; p.k_slices = splits;
            return p;
        }
    } else if (mode == 3 || mode >= 11) {
        return p;
    }
    // 128 x 128 tiles once they fill every CU twice over (two blocks are resident per CU);
    // below that the 64 x 64 tile spreads the work over more CUs and wins (measured).
    const bool big = mode != 2 && M > 64 && tiles(M, N, 128, 128) >= 2L * cus;
    p.kernel = big ? 3 : 2; p.tile_rows = big ? 128 : 64;
    return p;
}

namespace {

bool launch_planned(hipStream_t s, const GemmPlan& p, WeightKind kind, int M, int N, int K, const void* x, const void* W,
                    const void* scale, void* out, void* workspace, size_t ws_bytes, const MoreMats& more, bool glu = false) {
    auto* partial = static_cast<float*>(workspace);
    switch (p.kernel) {
        case 1: {
            const int tm = p.tile_rows / 32, ks = p.k_slices;
            if (kind == WK_Q4)
                return p.terms == 1 ? wide::launch_any<WK_Q4, 1>(tm, s, M, N, K, x, W, scale, out, partial, ws_bytes, ks, more, glu)
                                    : wide::launch_any<WK_Q4, 2>(tm, s, M, N, K, x, W, scale, out, partial, ws_bytes, ks, more, glu);
            if (kind == WK_F16) return wide::launch_any<WK_F16, 1>(tm, s, M, N, K, x, W, scale, out, partial, ws_bytes, ks, more, glu);
            return wide::launch_any<WK_I8, 1>(tm, s, M, N, K, x, W, scale, out, partial, ws_bytes, ks, more, glu);
        }
        case 4:
        {
            const skinny::Shape sh = skinny::pick_shape(kind, M, N, K, device_info().cus, ws_bytes);
            if (kind == WK_Q4)
                return p.terms == 1 ? skinny::launch<WK_Q4, 1>(s, M, N, K, x, W, scale, out, sh, workspace, ws_bytes, more, glu)
                                    : skinny::launch<WK_Q4, 2>(s, M, N, K, x, W, scale, out, sh, workspace, ws_bytes, more, glu);
            return kind == WK_F16 ? skinny::launch<WK_F16, 1>(s, M, N, K, x, W, scale, out, sh, workspace, ws_bytes, more, glu)
                                  : skinny::launch<WK_I8, 1>(s, M, N, K, x, W, scale, out, sh, workspace, ws_bytes, more, glu);
        }
        case 5: return quad::launch(s, M, N, K, x, W, scale, out);
        case 6: {
            const skinny::RowShape r{p.tile_rows / 16, p.strips, p.ks, 1, 0.0};
            if (kind == WK_Q4)
                return p.terms == 1 ? skinny::launch_rows<WK_Q4, 1>(s, M, N, K, x, W, scale, out, r, nullptr, more, glu)
                                    : skinny::launch_rows<WK_Q4, 2>(s, M, N, K, x, W, scale, out, r, nullptr, more, glu);
            return kind == WK_F16 ? skinny::launch_rows<WK_F16, 1>(s, M, N, K, x, W, scale, out, r, nullptr, more, glu)
                                  : skinny::launch_rows<WK_I8, 1>(s, M, N, K, x, W, scale, out, r, nullptr, more, glu);
        }
        case 2: return launch_tile<64, 64, 32, 32>(s, kind, M, N, K, x, W, scale, out, more);
        case 3: return launch_tile<128, 128, 64, 64>(s, kind, M, N, K, x, W, scale, out, more);
        default:
            MI_ERROR_FMT("gemm: mode %d has no kernel for kind=%d M=%d N=%d K=%d (Q4 weights have no tile kernel; the "
                         "streaming kernel takes up to 64 rows of x; the wide kernel's 32-bit offsets reach 4 GiB of x and "
                         "of W)", gemm_mode(s), static_cast<int>(kind), M, N, K);
            return false;
    }
}

}  // namespace

bool launch_gemm(hipStream_t s, WeightKind kind, int M, int N, int K, const void* x, const void* W,
                 const void* scale, void* out, void* workspace, size_t workspace_bytes) {
    if (!gemm_supported(kind, M, N, K, x, W, scale)) {
        MI_ERROR_FMT("gemm: unsupported kind=%d M=%d N=%d K=%d, or x / W not 16-byte aligned, or int8 / Q4 "
                     "without a (4-byte aligned) scale", static_cast<int>(kind), M, N, K);
        return false;
    }
    const size_t ws_bytes = workspace ? workspace_bytes : 0;
    return launch_planned(s, plan_gemm(s, kind, M, N, K, ws_bytes), kind, M, N, K, x, W, scale, out, workspace, ws_bytes,
                          MoreMats{});
}

// The SwiGLU of a stacked gate | up projection in the projection's own launch (or in the launch that adds its slices of
// K).  W holds 16 rows of the gate matrix, the same 16 of the up matrix, the next 16 of the gate matrix, and so on: a
// lane of the wide kernel then holds gate and up of a column in one accumulator, and a wavefront of the streaming kernel
// has them in neighbouring strips.  Both are rounded to fp16 as launch_gemm stores them, and the operations are swiglu_h's: the
// result is that of the two launches bit for bit.  What it saves is the trip of 2 x inter columns through memory:
// 2048 rows of 4864 + 4864 columns, 40 MB written and read again.
// Measured: a 2048-token int8 prompt 4253 -> 4147 us, 300 Q4 tokens behind 900 2206 -> 2172, 37 fp16 tokens 1661 -> 1609;
// less than the 13.5, 4.4 and 2.6 us per layer that the launch took, for the arithmetic (about 60 instructions per
// column) now stands in the epilogue.
int launch_gemm_glu(hipStream_t s, WeightKind kind, int M, int N, int K, const void* x, const void* W, const void* scale,
                    void* out, void* workspace, size_t workspace_bytes) {
    if (N % 32 || reinterpret_cast<uintptr_t>(out) % 16 || !gemm_supported(kind, M, N, K, x, W, scale)) return 0;
    const size_t ws_bytes = workspace ? workspace_bytes : 0;
    GemmPlan p = plan_gemm(s, kind, M, N, K, ws_bytes);
    if (p.kernel == 6) {                                 // (the slices of K as planned: they are the order of the sums)
        const skinny::RowShape r = skinny::pick_rows(kind, M, N, K, device_info().cus, true);
        p.tile_rows = 16 * r.mt; p.strips = r.S;
    }
    if (!(p.kernel == 1 || p.kernel == 6 ||
          (p.kernel == 4 && skinny::pick_shape(kind, M, N, K, device_info().cus, ws_bytes).kb == 1)))
        return 0;
    return launch_planned(s, p, kind, M, N, K, x, W, scale, out, workspace, ws_bytes, MoreMats{}, true) ? 1 : -1;
}

namespace {

// kernel 4 (shape few), 6 (shape rows) or 1 (wide: `plan`) in slices; 0: none
struct SlicePlan { int kernel = 0, terms = 1; skinny::Shape few{}; skinny::RowShape rows{}; GemmPlan plan{}; };

SlicePlan make_slice_plan(int mode, GemmPlan p, WeightKind kind, int M, int N, int K, size_t workspace_bytes) {
    SlicePlan sp;
    sp.terms = kind == WK_Q4 ? p.terms : 1;
    const int cus = device_info().cus;
    const bool own = mode == 0 || mode == 4;
    // (a few rows: the streaming kernel's own slices, whatever the plan for a launch by itself.  Prompts of 10 / 24 / 37 / 64
    //  tokens, int8 0.5B, int8 360M, fp16 360M, int8 0.5B, with its new loads in all: 973 / 1354 / 1514 / 1338 -> 927 / 1186 / 1208 / 1104 us)
    if (M <= skinny::kMaxM && own) {
        sp.few = skinny::pick_apart(kind, M, N, K, cus, workspace_bytes);
        if (sp.few.kb > 1) { sp.kernel = 4; return sp; }
    }
    if (own && p.kernel >= 1 && p.kernel != 5) {
        // (of this very plan: gemm_estimate_us counts two terms for Q4 weights in every mode)
        const double uncut = p.kernel == 1   ? wide::estimate_us(kind, sp.terms, p.tile_rows / 32, p.k_slices, M, N, K, cus)
                             : p.kernel == 6 ? skinny::rows_us(kind, p.tile_rows / 16, p.strips, 1, M, N, K, cus)
                             : p.kernel == 4 ? 1e30 : tiled_estimate_us(M, N, K);
        int tm = 1, splits = 1;
        double cut = 1e30;
        if (wide_reaches(kind, M, N, K)) wide::pick_sliced(kind, sp.terms, M, N, K, cus, workspace_bytes, &tm, &splits, &cut);
        // Tiles of rows: against the wide kernel's slices and the plan, which also leaves the next launch a pass over its fp16 result,
        // 1 us per 400 rows: 400 tokens of 0.5B int8 / fp16, whose q | k | v is estimated 1.1 / 1.25 us longer in slices, 1628 / 1726 us with them, 1577 /
        // 1676 without; 500 Q4 tokens of 360M, o 0.9 longer, 2138 / 2184.
        sp.rows = skinny::pick_rows_apart(kind, M, N, K, cus, workspace_bytes);
        if (sp.rows.mt && sp.rows.us < cut - 2.5 && sp.rows.us < uncut + M / 400.0) { sp.kernel = 6; return sp; }
        if (p.kernel != 4 && !(p.kernel == 1 && p.k_slices > 1) && cut - 2.5 < uncut) {
            p.kernel = 1;
            p.tile_rows = 32 * tm;
            p.k_slices = splits;
        }
    }
    if (p.kernel == 1 && p.k_slices > 1) { sp.kernel = 1; sp.plan = p; }
    return sp;
}

template <int KIND, int TERMS>
bool launch_streaming_slices(hipStream_t s, const SlicePlan& sp, int M, int N, int K, const void* x, const void* W, const void* scale,
                             void* workspace, size_t workspace_bytes) {
    if (sp.kernel == 6) return skinny::launch_rows<KIND, TERMS>(s, M, N, K, x, W, scale, nullptr, sp.rows, static_cast<float*>(workspace), MoreMats{}, false);
    return skinny::launch<KIND, TERMS>(s, M, N, K, x, W, scale, nullptr, sp.few, workspace, workspace_bytes, MoreMats{}, false, true);
}

}  // namespace

// A GEMM with K cut into slices, up to their sums: fp32 [slices][M][N] at the start of the workspace, for a launch that
// adds them in index order and goes on with the result (decode.hip).  As launch_gemm would cut it, or, where that has no
// slices, as many as pay without the launch that would add them: that launch is counted as 2.5 us in the estimate.
// Returns the number of slices; 0: none (nothing was launched); -1: an error.  Prompts of 80 / 300 / 600
// tokens without and with these launches: int8 0.5B 1472 / 1802 / 2247 -> 1360 / 1706 / 2116 us, Q4 360M 2112 / 2585 / 3069 ->
// 1875 / 2329 / 2838.
int launch_gemm_slices(hipStream_t s, WeightKind kind, int M, int N, int K, const void* x, const void* W, const void* scale,
                       void* workspace, size_t workspace_bytes) {
    if (!workspace || !gemm_supported(kind, M, N, K, x, W, scale)) return 0;
    const GemmPlan p = plan_gemm(s, kind, M, N, K, workspace_bytes);
    const int mode = gemm_mode(s);
    const SlicePlan sp = kept_plan<SlicePlan>(PlanKey{mode, device_info().cus, kind, M, N, K, workspace_bytes},
                                              [&] { return make_slice_plan(mode, p, kind, M, N, K, workspace_bytes); });
    if (sp.kernel == 0) return 0;
    if (sp.kernel == 1)
        return launch_planned(s, sp.plan, kind, M, N, K, x, W, scale, nullptr, workspace, workspace_bytes, MoreMats{}) ? sp.plan.k_slices : -1;
    const bool ok = kind == WK_Q4 ? (sp.terms == 1 ? launch_streaming_slices<WK_Q4, 1>(s, sp, M, N, K, x, W, scale, workspace, workspace_bytes)
                                                   : launch_streaming_slices<WK_Q4, 2>(s, sp, M, N, K, x, W, scale, workspace, workspace_bytes))
                  : kind == WK_F16 ? launch_streaming_slices<WK_F16, 1>(s, sp, M, N, K, x, W, scale, workspace, workspace_bytes)
                                   : launch_streaming_slices<WK_I8, 1>(s, sp, M, N, K, x, W, scale, workspace, workspace_bytes);
    return !ok ? -1 : sp.kernel == 6 ? sp.rows.kb : sp.few.kb;
}

// One launch serves the leading matrices whose own plans sum K in the same order, so that each result is what
// launch_gemm gives: the same kernel and number of slices, none of them over blocks (their partial sums meet in one
// workspace).  The wide kernel's tile height does not enter a sum: where the library chooses it, it is chosen for
// all matrices side by side.
int launch_gemm_group(hipStream_t s, WeightKind kind, int n, const GemmMat* mat, int M, int K, const void* x, void* workspace,
                      size_t workspace_bytes) {
    const size_t ws_bytes = workspace ? workspace_bytes : 0;
    const int cus = device_info().cus;
    GemmPlan p = plan_gemm(s, kind, M, mat[0].N, K, ws_bytes);
    skinny::Shape sh{};
    if (p.kernel == 4) sh = skinny::pick_shape(kind, M, mat[0].N, K, cus, ws_bytes);
    if (p.kernel == 6) {
        long all = 0;
        for (int j = 0; j < n; ++j) all += mat[j].N;
        const skinny::RowShape r = skinny::pick_rows(kind, M, all < (1 << 30) ? static_cast<int>(all) : mat[0].N, K, cus, false);
        if (r.mt && skinny::rows_fit(kind, r.mt, r.S, p.ks, M)) { p.tile_rows = 16 * r.mt; p.strips = r.S; }
    }
    if (!(p.kernel == 2 || p.kernel == 3 || p.kernel == 6 || (p.kernel == 1 && p.k_slices == 1) || (p.kernel == 4 && sh.kb == 1))) return 0;
    const int width = p.kernel == 1 ? wide::kBN : p.kernel == 2 ? 64 : p.kernel == 3 ? 128 : p.kernel == 6 ? 16 * p.strips : 16 * sh.S;
    auto tiles_of = [&](int N) { return N / width + (N % width != 0); };
    MoreMats more;
    more.tiles = tiles_of(mat[0].N);
    int g = 1;
    for (; g < n && g < kMaxSegments; ++g) {
        const GemmMat& c = mat[g];
        if (!gemm_supported(kind, M, c.N, K, x, c.W, c.scale)) break;
        const GemmPlan q = plan_gemm(s, kind, M, c.N, K, ws_bytes);
        if (q.kernel != p.kernel || q.terms != p.terms || q.k_slices != p.k_slices || q.ks != p.ks) break;
        if (p.kernel == 4) {
            const skinny::Shape t = skinny::pick_shape(kind, M, c.N, K, cus, ws_bytes);
            if (t.ks != sh.ks || t.S != sh.S || t.kb != 1) break;
        }
        if (static_cast<long>(more.tiles) + tiles_of(c.N) > 65535) break;
        more.m[g - 1].W = static_cast<const uint8_t*>(c.W);
        more.m[g - 1].scale = static_cast<const uint16_t*>(c.scale);
        more.m[g - 1].out = static_cast<uint16_t*>(c.out);
        more.m[g - 1].N = c.N;
        more.m[g - 1].first = more.tiles;
        more.tiles += tiles_of(c.N);
        more.n = g;
    }
    if (g == 1) return 0;
    if (p.kernel == 1 && (gemm_mode(s) == 0 || gemm_mode(s) == 4)) {
        int tm = 1, splits = 1;
        wide::pick_shape(kind, p.terms, M, more.tiles * wide::kBN, K, cus, 0, &tm, &splits, nullptr);
        p.tile_rows = 32 * tm;
    }
    return launch_planned(s, p, kind, M, mat[0].N, K, x, mat[0].W, mat[0].scale, mat[0].out, workspace, ws_bytes, more) ? g : -1;
}

GemmRoute gemm_route(hipStream_t s, const GemvCall& c, size_t workspace_bytes) {
    if (!gemm_supported(c.kind, c.M, c.N, c.K, c.x, c.W, c.scale)) return GemmRoute::kRefused;
    const GemmPlan p = plan_gemm(s, c.kind, c.M, c.N, c.K, workspace_bytes);
    if (p.kernel < 1 || (p.kernel == 1 && p.k_slices > 1 && !wide::slices_fit(p.k_slices, c.M, c.N, c.K, workspace_bytes)))
        return GemmRoute::kRefused;
    // Tiles of rows: as many as a launch of several counts, in its slices.  They take its tile there, 32 columns wide: a call that fills the
    // chip more than twice over with them goes alone where its own tile saves the time of a launch, 3.4 us (the down projection of 0.5B
    // in int8: with q and o the layer of 2304 rows takes 131 us, alone 120; of 600 rows 44.5, alone 46).
    const int cus = device_info().cus, mt = skinny::many_mt(c.kind, c.M);
    const long blocks = static_cast<long>((c.N + 31) / 32) * ((c.M + 16 * mt - 1) / (16 * mt));
    const bool rows = p.kernel == 6 && c.M > skinny::kMaxM && p.ks == skinny::rows_ks(c.M, c.N, c.K) && blocks <= 65535 &&
                      (blocks <= 2L * cus || skinny::rows_us(c.kind, mt, 2, 1, c.M, c.N, c.K, cus) <
                                                 skinny::rows_us(c.kind, p.tile_rows / 16, p.strips, 1, c.M, c.N, c.K, cus) + 3.4);
    return (p.kernel == 4 || rows) && (c.N + 15) / 16 <= 8191 ? GemmRoute::kShares : GemmRoute::kAlone;
}

bool launch_gemm_many(hipStream_t s, const GemvCall* calls, int n, void* workspace, size_t workspace_bytes) {
    const size_t ws_bytes = workspace ? workspace_bytes : 0;
    for (int i = 0; i < n; ++i) {
        if (calls[i].M != calls[0].M || calls[i].kind != calls[0].kind || gemm_route(s, calls[i], ws_bytes) != GemmRoute::kShares) {
            MI_ERROR_FMT("gemm: a call that does not fit a launch of several (M=%d N=%d K=%d)", calls[i].M, calls[i].N, calls[i].K);
            return false;
        }
    }
    const GemmPlan p = plan_gemm(s, calls[0].kind, calls[0].M, calls[0].N, calls[0].K, ws_bytes);
    return skinny::launch_many(s, calls, n, p.terms, workspace, ws_bytes);
}

}  // namespace mi

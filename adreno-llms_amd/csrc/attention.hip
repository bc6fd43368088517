// Causal attention of a prompt on the matrix cores: rows pos0 .. pos0 + M - 1 of a sequence against
// cache rows 0 .. their own position, softmax(q k / sqrt(D)) v per query head, key/value heads shared by
// n_heads / n_kv_heads query heads (QW/kernels/attention.cl gqa_attn_scores, gqa_softmax, gqa_attn_out).
//
// The kernels of decode.hip that keep the reference's order of operations are bound by that order: one
// chain of additions over the keys per output element and per denominator, on the vector units.  Where
// a layer's projections run on the matrix cores, the sums run in another order anyway, and this
// kernel takes their place: fp16 products, fp32 sums, scores kept in fp32 (the reference order rounds them
// to fp16), exponentials rounded to fp16 once, before they are summed and before they meet the values (the
// reference order sums them in fp32 and rounds exponential and probability).  The denominator takes the rounded
// ones too because an error of one then moves the output by that key's distance from it only.  Error of an fp16
// output against fp64 in a numpy model of the roundings (37 to 2048 keys, scores of standard deviation 0.3 to 4,
// values of mean 0 to 3), 2-norm: reference order 1.9e-4 to 1.5e-3, this order 1.9e-4 to 3.2e-4, with unrounded
// terms in the denominator up to 2 % more.  Logits after 8 layers, 37 to 2048 rows, against an fp64 model: 1.2e-3 to
// 3.2e-3 either way (mean of 14 prompts 2.1e-3).
#include "common.h"
#include "device_math.h"

namespace mi {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kKeys = 64;                        // keys per tile
constexpr int kRows = 16;                        // queries per wavefront (of one head)
constexpr float kNone = -3.402823466e+38f;       // the score of a key that the query does not see
constexpr float kStart = -1.0e30f;               // the running maximum of a query that has seen no key
constexpr float kSlack = 8.0f;                   // see the main loop

// The greater of a lane's value and those of the lanes 16, 32 and 48 away.
__device__ __forceinline__ float max_of_groups(float a) {
    unsigned u = __float_as_uint(a);
    auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    u = __float_as_uint(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
    r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{a, b}, half2v));
}

constexpr size_t tile_bytes(int D) { return static_cast<size_t>(kKeys) * (2 * D + 16) + static_cast<size_t>(D) * (2 * kKeys + 8); }
constexpr size_t merge_bytes(int D) { return static_cast<size_t>(D / 4 + 2) * 64 * 4; }     // a wavefront's sums, see the end of the kernel
constexpr size_t flash_lds(int D, int KS) { return 2 * KS * tile_bytes(D); }

// A wavefront owns 16 queries of one head ("a set"), KS wavefronts of the block share them, wavefront k of
// the KS taking key tiles k, k + KS, ...; the block's WAVES / KS sets belong to one key/value head and share
// its tiles, KS of them at a time, in LDS.
//
// Scores are computed transposed (A = keys, B = queries), so that lane (query i = lane % 16, group g =
// lane / 16) ends up with keys 4 g .. 4 g + 3 of every 16 keys for its query: maximum and sum are taken
// inside the lane and across the four groups (two register swaps), and two such quadruples are, as they
// stand, the B operand of the product with the values (k = 8 values per lane; which keys they are does
// not matter as long as the A operand brings the same ones), so probabilities never go through LDS.  The
// values are transposed on their way into LDS, 4 keys x 4 elements per thread in registers.
// LDS pitches: key rows 2 D + 16 bytes (16-byte reads of 16 consecutive rows), value rows (one element,
// 64 keys) 136 bytes (8-byte reads of 16 consecutive rows): the addresses of either spread over all banks (the counters
// below show conflicts all the same; the value rows' writes, four rows apart, meet two to a bank).
//
// What bounds it: a wavefront alone on its SIMD takes 0.8 us per tile; the reads from LDS (16 KB per wavefront and
// tile), the exponentials and the waits between the phases overlap only across wavefronts.  Counters at 2048 rows,
// 14 heads over 2: matrix cores busy 17 % of the SIMD-cycles, LDS 52 % of the CU-cycles (38 % of that bank conflicts).
// us per launch, launches back to back: 433 in the reference's order (attention_group_kernel), 22.7 here (0.33
// PFLOP/s, causal half counted; a large matrix product reaches 1.5); 300 rows at position 900: 96 -> 11.4.
// Requesting tiles two ahead, forming the next tile's scores under the current tile's exponentials, and two sets
// per wavefront were no faster.
template <int D, int WAVES, int KS>
__global__ __launch_bounds__(64 * WAVES) void flash_rows_kernel(const uint16_t* __restrict__ QR, const uint16_t* __restrict__ kc,
                                                         const uint16_t* __restrict__ vc, uint16_t* __restrict__ out, int M,
                                                         int pos0, int n_heads, int n_kv_heads, float scale_log2, int mirror) {
    constexpr int kThreads = 64 * WAVES, kSets = WAVES / KS;                            // sets of queries per block
    constexpr int kKPitch = 2 * D + 16, kVPitch = 2 * kKeys + 8;
    constexpr int kKTile = kKeys * kKPitch, kVTile = D * kVPitch;
    constexpr int kKPieces = KS * kKeys * (D / 8) / kThreads;  // 16-byte pieces of KS key tiles per thread
    constexpr int kVBlocks = KS * (kKeys / 4) * (D / 4) / kThreads;   // 4 x 4 blocks of KS value tiles per thread
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    uint8_t* const kbuf = lds;                                 // [2][KS][kKTile]
    uint8_t* const vbuf = lds + 2 * KS * kKTile;               // [2][KS][kVTile]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int slice = wave % KS;
    const int nrep = n_heads / n_kv_heads, kvd = n_kv_heads * D, qd = n_heads * D;
    const int sets = (M + kRows - 1) / kRows * nrep;           // of a key/value head
    const int per_head = (sets + kSets - 1) / kSets;
    // Longest rows first.  (mirror > 0: the blocks from number `mirror` on, the second of their CU, are taken from
    // the short end: they share it with the longest ones.)
    int rank = blockIdx.x;
    if (mirror && rank >= mirror) rank = per_head * n_kv_heads - 1 - (rank - mirror);
    const int kvh = rank % n_kv_heads, b = per_head - 1 - rank / n_kv_heads;
    const int last_set = (b + 1) * kSets < sets ? (b + 1) * kSets - 1 : sets - 1;
    const int q_end = last_set / nrep * kRows + kRows;         // one past the block's last query
    const int keys = pos0 + (q_end < M ? q_end : M);           // keys the block reads
    const int tiles = (keys + kKeys - 1) / kKeys, steps = (tiles + KS - 1) / KS;
    // (a set past the last and rows past M: computed as the last ones, not stored)
    const int set = b * kSets + wave / KS < sets ? b * kSets + wave / KS : sets - 1;
    const int q0 = set / nrep * kRows, head = kvh * nrep + set % nrep;
    const bool live = b * kSets + wave / KS < sets && q0 + i < M;
    const int row = q0 + i < M ? q0 + i : M - 1, my_pos = pos0 + row;
    half8 q[D / 32];
    #pragma unroll
    for (int j = 0; j < D / 32; ++j)
        q[j] = *reinterpret_cast<const half8*>(QR + static_cast<size_t>(row) * qd + head * D + 8 * g + 32 * j);

    // Tiles travel memory -> registers -> LDS.  A request's address is a scalar base per tile plus a thread's
    // constant offset.  Keys past the block's last are read as the last one, never what lies there, and masked; past
    // the last tile that one is read again.
    struct Regs { u32x4 k[kKPieces]; u32x2 v[kVBlocks][4]; };
    const uint32_t row_bytes = static_cast<uint32_t>(kvd) * 2;
    const uint8_t* kbase = reinterpret_cast<const uint8_t*>(kc + kvh * D);
    const uint8_t* vbase = reinterpret_cast<const uint8_t*>(vc + kvh * D);
    const int row_last = keys - 1 - (steps - 1) * KS * kKeys;  // the last key's row in the last step's tiles
    uint32_t koff[2][kKPieces], voff[2][kVBlocks][4];          // of any step, of the last
    #pragma unroll
    for (int p = 0; p < kKPieces; ++p) {
        const int r = (tid + kThreads * p) / (D / 8), c = 16 * ((tid + kThreads * p) % (D / 8));
        koff[0][p] = r * row_bytes + c;
        koff[1][p] = (r < row_last ? r : row_last) * row_bytes + c;
    }
    #pragma unroll
    for (int p = 0; p < kVBlocks; ++p)
        #pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int r = 4 * ((tid + kThreads * p) / (D / 4)) + e, c = 8 * ((tid + kThreads * p) % (D / 4));
            voff[0][p][e] = r * row_bytes + c;
            voff[1][p][e] = (r < row_last ? r : row_last) * row_bytes + c;
        }
    auto fetch = [&](Regs& R, int step) {
        const int t = step < steps ? step : steps - 1;
        const bool last = t == steps - 1;
        const size_t at = static_cast<size_t>(t) * KS * kKeys * row_bytes;
        const uint8_t *kb = kbase + at, *vb = vbase + at;
        #pragma unroll
        for (int p = 0; p < kKPieces; ++p) R.k[p] = *reinterpret_cast<const u32x4*>(kb + (last ? koff[1][p] : koff[0][p]));
        #pragma unroll
        for (int p = 0; p < kVBlocks; ++p)
            #pragma unroll
            for (int e = 0; e < 4; ++e) R.v[p][e] = *reinterpret_cast<const u32x2*>(vb + (last ? voff[1][p][e] : voff[0][p][e]));
    };
    auto stash = [&](const Regs& R, int buf) {
        #pragma unroll
        for (int p = 0; p < kKPieces; ++p) {
            const int idx = tid + kThreads * p;
            *reinterpret_cast<u32x4*>(kbuf + buf * KS * kKTile + idx / (D / 8) * kKPitch + 16 * (idx % (D / 8))) = R.k[p];
        }
        #pragma unroll
        for (int p = 0; p < kVBlocks; ++p) {
            const int idx = tid + kThreads * p, k4 = idx / (D / 4);          // 4 keys
            uint8_t* dst = vbuf + (buf * KS + k4 / (kKeys / 4)) * kVTile + 4 * (idx % (D / 4)) * kVPitch + 8 * (k4 % (kKeys / 4));
            const u32x2 (&v)[4] = R.v[p];
            #pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t sel = e & 1 ? 0x07060302u : 0x05040100u;
                *reinterpret_cast<u32x2*>(dst + e * kVPitch) =
                    u32x2{__builtin_amdgcn_perm(v[1][e / 2], v[0][e / 2], sel), __builtin_amdgcn_perm(v[3][e / 2], v[2][e / 2], sel)};
            }
        }
    };

    floatx4 acc[D / 16];
    #pragma unroll
    for (int d = 0; d < D / 16; ++d) acc[d] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    // running maximum of the query's scores, times scale_log2; sum of the probabilities (as they meet the values, rounded
    // to fp16: a row of ones beside the values' rows, the same number in every register)
    float base = kStart;
    floatx4 l = {0.0f, 0.0f, 0.0f, 0.0f};
    half8 ones;
    #pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = static_cast<_Float16>(1.0f);
    auto multiply = [&](int buf, int k0) {
        const uint8_t* ktile = kbuf + (buf * KS + slice) * kKTile + i * kKPitch + 16 * g;
        const uint8_t* vtile = vbuf + (buf * KS + slice) * kVTile + i * kVPitch + 8 * g;
        floatx4 s[4];
        #pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            s[kt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            #pragma unroll
            for (int j = 0; j < D / 32; ++j)
                s[kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const half8*>(ktile + 16 * kt * kKPitch + 64 * j), q[j], s[kt], 0, 0, 0);
        }
        const bool masked = k0 + kKeys - 1 > pos0 + q0;        // (keys up to the set's first query need no mask)
        if (masked) {
            #pragma unroll
            for (int kt = 0; kt < 4; ++kt)
                #pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (k0 + 16 * kt + 4 * g + r > my_pos) s[kt][r] = kNone;
        }
        // A score may exceed the running maximum by 2^kSlack before the sums are rescaled: exponentials up to
        // that are as good in fp16 as those up to 1, and the test needs the lane's own keys only.
        float top = kNone;
        #pragma unroll
        for (int kt = 0; kt < 4; ++kt) top = fmaxf(top, fmaxf(fmaxf(s[kt][0], s[kt][1]), fmaxf(s[kt][2], s[kt][3])));
        top *= scale_log2;
        if (__any(top > base + kSlack)) {
            top = fmaxf(base, max_of_groups(top));
            const float alpha = __builtin_amdgcn_exp2f(base - top);
            l *= alpha;
            #pragma unroll
            for (int d = 0; d < D / 16; ++d) acc[d] *= alpha;
            base = top;
        }
        // (a query without a key so far: every score is kNone, and its exponentials must be 0)
        const float sub = base == kStart ? 0.0f : base;
        uint32_t p[4][2];
        #pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            float e[4];
            #pragma unroll
            for (int r = 0; r < 4; ++r) e[r] = __builtin_amdgcn_exp2f(fmaf(s[kt][r], scale_log2, -sub));
            p[kt][0] = pack2(e[0], e[1]);
            p[kt][1] = pack2(e[2], e[3]);
        }
        half8 pb[2];
        #pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
            pb[kp] = __builtin_bit_cast(half8, u32x4{p[2 * kp][0], p[2 * kp][1], p[2 * kp + 1][0], p[2 * kp + 1][1]});
            l = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, pb[kp], l, 0, 0, 0);
        }
        // `from` + the tile's product for elements 16 d ..; `keep` takes the 4 values of the lane's keys 16 n + 4 g ..
        auto product = [&](int d, floatx4 from, auto keep) {
            #pragma unroll
            for (int kp = 0; kp < 2; ++kp) {
                const u32x2 lo = keep(*reinterpret_cast<const u32x2*>(vtile + 16 * d * kVPitch + 64 * kp), 2 * kp);
                const u32x2 hi = keep(*reinterpret_cast<const u32x2*>(vtile + 16 * d * kVPitch + 64 * kp + 32), 2 * kp + 1);
                from = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, u32x4{lo.x, lo.y, hi.x, hi.y}), pb[kp], from, 0, 0, 0);
            }
            return from;
        };
        auto all = [](u32x2 v, int) { return v; };
        if (!masked) {
            #pragma unroll
            for (int d = 0; d < D / 16; ++d) acc[d] = product(d, acc[d], all);
            return;
        }
        // A masked key has probability 0, but 0 x inf and 0 x NaN are NaN: where a NaN comes up, the tile is multiplied
        // once more per query of the set, with the values that query does not see as zeros, and the query's column kept.
        floatx4 sums[D / 16];
        bool nan = false;
        #pragma unroll
        for (int d = 0; d < D / 16; ++d) {
            sums[d] = product(d, acc[d], all);
            #pragma unroll
            for (int r = 0; r < 4; ++r) nan |= sums[d][r] != sums[d][r];
        }
        if (!__any(nan)) {
            #pragma unroll
            for (int d = 0; d < D / 16; ++d) acc[d] = sums[d];
        } else {
            #pragma unroll 1
            for (int j = 0; j < kRows; ++j) {
                asm volatile("" ::: "memory");     // (read again per query: kept, the values take the registers of the CU's second block)
                const int seen = pos0 + q0 + j + 1 - k0 - 4 * g;           // of the keys 4 g .. of the tile, this many
                auto own = [&](u32x2 v, int n) {
                    #pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int left = seen - 16 * n - 2 * h;
                        v[h] = left >= 2 ? v[h] : left == 1 ? v[h] & 0xffffu : 0u;
                    }
                    return v;
                };
                #pragma unroll
                for (int d = 0; d < D / 16; ++d) {
                    const floatx4 mine = product(d, acc[d], own);
                    if (i == j) acc[d] = mine;
                }
            }
        }
    };
    const int w_last = pos0 + (q0 + kRows < M ? q0 + kRows : M) - 1;       // the set's last query
    Regs R;
    fetch(R, 0);
    for (int t = 0; t < steps; ++t) {
        // registers -> LDS, the next tiles requested, one barrier (a buffer is written again two barriers after it
        // was last read), the wavefront's tile multiplied unless its queries end before it
        stash(R, t & 1);
        fetch(R, t + 1);
        __syncthreads();
        const int k0 = (t * KS + slice) * kKeys;
        if (k0 <= w_last) multiply(t & 1, k0);
    }
    float sum = l[0];
    if constexpr (KS > 1) {
        // the KS wavefronts' sums meet in LDS: slices 1 .. KS - 1 leave theirs, slice 0 merges them in order
        __syncthreads();
        float* mine = reinterpret_cast<float*>(lds) + wave * static_cast<int>(merge_bytes(D) / 4) + lane;
        if (slice > 0) {
            mine[0] = base;
            mine[64] = sum;
            #pragma unroll
            for (int d = 0; d < D / 16; ++d)
                #pragma unroll
                for (int r = 0; r < 4; ++r) mine[(2 + 4 * d + r) * 64] = acc[d][r];
        }
        __syncthreads();
        if (slice > 0) return;
        #pragma unroll
        for (int z = 1; z < KS; ++z) {
            const float* other = mine + z * static_cast<int>(merge_bytes(D) / 4);
            const float bz = other[0], lz = other[64];
            const float top = fmaxf(base, bz);                 // (slice 0 always has key 0: top is of a score)
            const float a = __builtin_amdgcn_exp2f(base - top), c = __builtin_amdgcn_exp2f(bz - top);
            sum = sum * a + lz * c;
            #pragma unroll
            for (int d = 0; d < D / 16; ++d)
                #pragma unroll
                for (int r = 0; r < 4; ++r) acc[d][r] = acc[d][r] * a + other[(2 + 4 * d + r) * 64] * c;
            base = top;
        }
    }
    if (!live) return;
    const float inv = __fdiv_rn(1.0f, sum + 1e-20f);           // (the reference's: 0 where every score is -inf)
    uint16_t* dst = out + static_cast<size_t>(row) * qd + head * D + 4 * g;
    #pragma unroll
    for (int d = 0; d < D / 16; ++d)
        *reinterpret_cast<u32x2*>(dst + 16 * d) = u32x2{pack2(acc[d][0] * inv, acc[d][1] * inv), pack2(acc[d][2] * inv, acc[d][3] * inv)};
}

// Blocks of a launch of WAVES wavefronts per block, KS per set.
inline int flash_blocks(int M, int n_heads, int n_kv_heads, int WAVES, int KS) {
    const int sets = (M + kRows - 1) / kRows * (n_heads / n_kv_heads), per_block = WAVES / KS;
    return (sets + per_block - 1) / per_block * n_kv_heads;
}

template <int D, int WAVES, int KS>
bool launch_flash(hipStream_t s, const uint16_t* QR, const uint16_t* kc, const uint16_t* vc, uint16_t* out, int M, int pos0,
                  int n_heads, int n_kv_heads, float scale) {
    constexpr size_t lds = flash_lds(D, KS);
    static_assert(lds <= 160 * 1024 && (KS == 1 || WAVES * merge_bytes(D) <= lds), "tiles and merge buffer fit");
    auto* kern = flash_rows_kernel<D, WAVES, KS>;
    if (lds > 65536 &&
        !MI_ONCE_OK(MI_HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                  static_cast<int>(lds)))))
        return false;
    // More blocks than CUs and at most two per CU, all resident at once: a CU's second block is one of the shortest where
    // its first is one of the longest.  us with / without, 2048 rows: 14 heads over 2 22.7 / 24.6, 15 over 5 23.0 / 24.9,
    // 9 over 3 21.1 / 21.6, width 128, 16 over 4 49.5 / 54.0.  Where LDS holds one block, the second round has to go on
    // with the long ones (width 128 in two slices at 1000 rows 29.0 / 24.4).
    const int total = flash_blocks(M, n_heads, n_kv_heads, WAVES, KS), cus = device_info().cus;
    const bool mirror = 2 * lds <= 160 * 1024 && total > cus && total <= 2 * cus;
    hipLaunchKernelGGL(kern, dim3(total), dim3(64 * WAVES), lds, s, QR, kc, vc, out, M, pos0, n_heads, n_kv_heads,
                       scale * 1.44269504088896341f, mirror ? cus : 0);
    return MI_HIP_OK(hipGetLastError());
}

}  // namespace

bool attention_prompt_supported(int head_dim) { return head_dim == 64 || head_dim == 128; }

bool launch_attention_prompt(hipStream_t s, const uint16_t* QR, const uint16_t* kc, const uint16_t* vc, uint16_t* out, int M,
                             int pos0, int n_heads, int n_kv_heads, int head_dim, float scale) {
#define MI_FLASH(D, WAVES, KS) return launch_flash<D, WAVES, KS>(s, QR, kc, vc, out, M, pos0, n_heads, n_kv_heads, scale)
    // A set's chain of tiles bounds the launch (0.8 us per tile while a wavefront has its SIMD to itself), so the
    // keys of a set go over several wavefronts, and as many of those share a CU as there are blocks for.  us, launches
    // back to back, eight wavefronts / 2 per set, 4 / 2, 8 / 4, head width 64, at 14 heads over 2 (15 over 5 within 0.3
    // of it) and 9 over 3:
    //   2048 rows 22.2 / 28.9 / 37.4, 21.1 / 21.9 / 25.8; 1000 rows 12.2 / 12.2 / 14.7, 11.9 / 11.7 / 10.3 (8 / 4 by
    //   the rule): enough blocks of 8 / 2 for the chip;
    //   300 rows at 900 14.2 / 13.4 / 11.4, 14.1 / 13.4 / 11.3; 40 at 1500 16.9 / 16.4 / 13.8, 16.7 / 16.3 / 13.8: few
    //   blocks, long chains (in between, 600 rows, 8.9 / 8.6 / 10.0 and 8.8 / 8.2 / 8.4, the line is not at its best);
    //   100 rows 4.7 / 4.0 / 5.5, 40 at 300 6.8 / 6.1 / 6.9: a tile or a few per wavefront either way.
    const int cus = device_info().cus;
    if (head_dim == 64) {
        if (flash_blocks(M, n_heads, n_kv_heads, 8, 2) * 4 >= cus * 3) MI_FLASH(64, 8, 2);
        if (pos0 + M <= 512) MI_FLASH(64, 4, 2);
        MI_FLASH(64, 8, 4);
    }
    // (head width 128, 16 heads over 4, four wavefronts, 1 / 2 per set: 2048 rows 49.5 / 77.2, 1000 rows 25.9 / 24.4,
    //  300 at 900 29.9 / 23.0)
    if (flash_blocks(M, n_heads, n_kv_heads, 4, 1) >= cus) MI_FLASH(128, 4, 1);
    MI_FLASH(128, 4, 2);
#undef MI_FLASH
}

}  // namespace mi

// A Qwen2-shaped greedy decode step that stays on the device: the small kernels that sit between
// the projections (QW/kernels/{embedding,rmsnorm,bias_add,rope,attention,mlp,utils}.cl), the
// projections themselves as GEMV launches that also carry the RMSNorm ahead of them or the
// residual add behind them, and the argmax.  Graph of a step:
// QW/src/model.cpp:243-376, QW/src/layers/attention.cpp:336-674, QW/src/layers/mlp.cpp:97-237.
//
// Position and token live in device memory (the reference's counter buffer, QW/src/model.cpp:
// 490-500): every kernel reads them there and the last kernel of a step advances them, so a step
// is the same sequence of launches with the same arguments at every position: one captured
// graph replays for the whole generation, and no token returns to the host between steps.
//
// These kernels are the harness around the matmul path, not the path: they are written for
// exactness against the CPU restatement (same operations in the same order, so that the token
// lists can be compared for identity), and are launch-bound at batch 1 whatever they do.
#include "common.h"
#include <type_traits>
#include "device_math.h"
#include "step_record.h"
#include "../../include/mi_decode.h"
#include "../../include/mi_linear.h"

#include <cmath>
#include <vector>

namespace mi {
namespace {

struct State {
    int pos;
    int token;
    int next;       // written by the argmax, moved into token by advance_kernel
};

__device__ __forceinline__ float rcp_rn(float x) { return __fdiv_rn(1.0f, x); }

// h[c] = embed[token][c]   (QW/kernels/embedding.cl).  The first launch of a step also copies the
// rotary table's row of the current position to rope_now (cosines, then sines: 2 D values), so
// that the attention launches of the step find it without waiting for the position first.
__global__ void embed_kernel(const uint16_t* __restrict__ embed, const State* __restrict__ st,
                             uint16_t* __restrict__ h, int hidden, int vocab, const uint16_t* __restrict__ cosT,
                             const uint16_t* __restrict__ sinT, uint16_t* __restrict__ rope_now, int D, int max_pos) {
    int t = st->token;
    t = t < 0 ? 0 : (t >= vocab ? vocab - 1 : t);
    int pos = st->pos;
    pos = pos < 0 ? 0 : (pos >= max_pos ? max_pos - 1 : pos);
    for (int c = threadIdx.x; c < D; c += blockDim.x) {
        rope_now[c] = cosT[static_cast<size_t>(pos) * D + c];
        rope_now[D + c] = sinT[static_cast<size_t>(pos) * D + c];
    }
    for (int c = threadIdx.x; c < hidden; c += blockDim.x) h[c] = embed[static_cast<size_t>(t) * hidden + c];
}

// out[c] = fp16((x[c] * inv) * w[c]), inv = 1 / sqrt(mean(x^2) + eps); the sum of squares runs
// over 64 work-items in float4 strides and a 32..1 tree (QW/kernels/rmsnorm.cl).  One wavefront.
// Used where the norm cannot ride in the projection's own launch (see mi_decoder_step).
__global__ __launch_bounds__(64) void rmsnorm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                     uint16_t* __restrict__ out, int cols, float eps) {
    // Work-item lid owns the float4 groups lid, lid + 64, ...: it squares and normalises the
    // same elements, so x and w are read once, all loads are in flight together, and the
    // kernel costs one memory round trip.  Up to kGroups groups per work-item live in registers
    // (cols <= 256 kGroups); the tail that is not a whole group, and longer rows, go through memory.
    constexpr int kGroups = 8;
    const int lid = threadIdx.x, c4n = cols >> 2;
    x += static_cast<size_t>(blockIdx.x) * cols;       // block b takes row b (a prompt's rows; one row in a decode step)
    out += static_cast<size_t>(blockIdx.x) * cols;
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    u16x4 xv[kGroups], wv[kGroups];
    float acc = 0.0f;
    #pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        const int c4 = lid + 64 * g;
        if (c4 < c4n) {
            xv[g] = *reinterpret_cast<const u16x4*>(x + 4 * c4);
            wv[g] = *reinterpret_cast<const u16x4*>(w + 4 * c4);
        }
    }
    #pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        if (lid + 64 * g < c4n) {
            const float v0 = h_f(xv[g][0]), v1 = h_f(xv[g][1]), v2 = h_f(xv[g][2]), v3 = h_f(xv[g][3]);
            float d = v0 * v0;
            d = fmaf(v1, v1, d);
            d = fmaf(v2, v2, d);
            d = fmaf(v3, v3, d);
            acc = acc + d;
        }
    }
    for (int c4 = lid + 64 * kGroups; c4 < c4n; c4 += 64) {           // rows longer than the registers hold
        float v[4];
        #pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = h_f(x[4 * c4 + e]);
        float d = v[0] * v[0];
        d = fmaf(v[1], v[1], d);
        d = fmaf(v[2], v[2], d);
        d = fmaf(v[3], v[3], d);
        acc = acc + d;
    }
    for (int c = c4n * 4 + lid; c < cols; c += 64) {                    // cols not a multiple of 4
        const float v = h_f(x[c]);
        acc = fmaf(v, v, acc);
    }
    const float total = wave_tree_sum(acc);
    // sqrtf is the correctly rounded one (-fhip-fp32-correctly-rounded-divide-sqrt); the
    // __fsqrt_rn intrinsic is not, despite its name: it is off by an ulp for one input in six
    const float inv = rcp_rn(sqrtf(__fdiv_rn(total, static_cast<float>(cols)) + eps));
    #pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        const int c4 = lid + 64 * g;
        if (c4 < c4n) {
            u16x4 o;
            #pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = f_h((h_f(xv[g][e]) * inv) * h_f(wv[g][e]));
            *reinterpret_cast<u16x4*>(out + 4 * c4) = o;
        }
    }
    for (int c4 = lid + 64 * kGroups; c4 < c4n; c4 += 64)
        for (int e = 0; e < 4; ++e) out[4 * c4 + e] = f_h((h_f(x[4 * c4 + e]) * inv) * h_f(w[4 * c4 + e]));
    for (int c = c4n * 4 + lid; c < cols; c += 64) out[c] = f_h((h_f(x[c]) * inv) * h_f(w[c]));
}

// One block per query head: q/k/v bias (QW/kernels/bias_add.cl), rotary embedding of q and k at the
// current position (QW/kernels/rope.cl), k and v into the caches (rows as QW/src/layers/
// attention.cpp:560-600), then single-query grouped-query attention (QW/kernels/attention.cl:
// gqa_attn_scores, gqa_softmax, gqa_attn_out); each value rounded to fp16 where the separate
// kernels would store it.  Sums run in the order the CPU restatement uses: the score over D in
// float4 groups, the softmax denominator over the keys in index order, the output over the keys
// in index order.
// Every head of a group prepares the group's k and v of the current position for itself (in
// LDS; the values are the same in all of them) and reads only older rows from the caches; the
// group's first head writes the new row.  raw = the projections' outputs; q_out, k_out, v_out
// receive them after bias and rotary embedding.
// Dynamic LDS: 6 bytes per position (fp32 exponentials, fp16 scores) + 6 D bytes.
__global__ __launch_bounds__(256) void rope_attention_kernel(const uint16_t* __restrict__ q_raw, const uint16_t* __restrict__ k_raw,
                                      const uint16_t* __restrict__ v_raw, const uint16_t* __restrict__ bq,
                                      const uint16_t* __restrict__ bk, const uint16_t* __restrict__ bv,
                                      const uint16_t* __restrict__ cosT, const uint16_t* __restrict__ sinT,
                                      uint16_t* __restrict__ kc, uint16_t* __restrict__ vc,
                                      uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_out,
                                      uint16_t* __restrict__ v_out, uint16_t* __restrict__ out,
                                      const State* __restrict__ st, int n_heads, int n_kv_heads, int D, int max_pos,
                                      float scale) {
    extern __shared__ __attribute__((aligned(16))) uint16_t qv[];          // q, then k and v of the current position:
    uint16_t* kcur = qv + D;                                               // 3 D halves (a multiple of 8 bytes)
    uint16_t* vcur = kcur + D;
    float* ex = reinterpret_cast<float*>(vcur + D);                        // [max_pos] exponentials
    uint16_t* sc = reinterpret_cast<uint16_t*>(ex + max_pos);              // [max_pos] scores
    __shared__ float red[64];
    __shared__ float inv_s;
    int pos = st->pos;
    pos = pos < 0 ? 0 : (pos >= max_pos ? max_pos - 1 : pos);
    const int nrep = n_heads / n_kv_heads;
    const int seq_k = pos + 1, qh = blockIdx.x, kvd = n_kv_heads * D, kvh = qh / nrep, hd2 = D / 2;
    const bool writer = qh % nrep == 0;
    const int tid = threadIdx.x, nt = blockDim.x;
    const uint16_t* cr = cosT + static_cast<size_t>(pos) * D;
    const uint16_t* sr = sinT + static_cast<size_t>(pos) * D;
    for (int i = tid; i < hd2; i += nt) {
        const float c = h_f(cr[i]), sn = h_f(sr[i]);
        {
            const uint16_t* buf = q_raw + qh * D;
            const uint16_t* bias = bq + qh * D;
            const float x1 = h_f(f_h(h_f(buf[i]) + h_f(bias[i])));
            const float x2 = h_f(f_h(h_f(buf[i + hd2]) + h_f(bias[i + hd2])));
            const uint16_t r1 = f_h(fmaf(x1, c, -(x2 * sn))), r2 = f_h(fmaf(x2, c, x1 * sn));
            qv[i] = r1;
            qv[i + hd2] = r2;
            q_out[qh * D + i] = r1;
            q_out[qh * D + i + hd2] = r2;
        }
        {
            const uint16_t* buf = k_raw + kvh * D;
            const uint16_t* bias = bk + kvh * D;
            const float x1 = h_f(f_h(h_f(buf[i]) + h_f(bias[i])));
            const float x2 = h_f(f_h(h_f(buf[i + hd2]) + h_f(bias[i + hd2])));
            const uint16_t r1 = f_h(fmaf(x1, c, -(x2 * sn))), r2 = f_h(fmaf(x2, c, x1 * sn));
            kcur[i] = r1;
            kcur[i + hd2] = r2;
            if (writer) {
                uint16_t* dst = kc + static_cast<size_t>(pos) * kvd + kvh * D;
                dst[i] = r1;
                dst[i + hd2] = r2;
                k_out[kvh * D + i] = r1;
                k_out[kvh * D + i + hd2] = r2;
            }
        }
    }
    for (int e = tid; e < D; e += nt) {
        const uint16_t r = f_h(h_f(v_raw[kvh * D + e]) + h_f(bv[kvh * D + e]));
        vcur[e] = r;
        if (writer) {
            vc[static_cast<size_t>(pos) * kvd + kvh * D + e] = r;
            v_out[kvh * D + e] = r;
        }
    }
    __syncthreads();
    for (int tk = tid; tk < seq_k; tk += nt) {
        // a key row is read in 8-byte pieces (rows start at multiples of 8 bytes: D % 4 == 0)
        typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
        const u16x4* kv = reinterpret_cast<const u16x4*>(tk == pos ? kcur : kc + static_cast<size_t>(tk) * kvd + kvh * D);
        const u16x4* qq = reinterpret_cast<const u16x4*>(qv);
        float acc = 0.0f;
        for (int d4 = 0; d4 < D / 4; ++d4) {
            const u16x4 a = qq[d4], b = kv[d4];
            float t = h_f(a[0]) * h_f(b[0]);
            t = fmaf(h_f(a[1]), h_f(b[1]), t);
            t = fmaf(h_f(a[2]), h_f(b[2]), t);
            t = fmaf(h_f(a[3]), h_f(b[3]), t);
            acc = acc + t;
        }
        sc[tk] = f_h(acc * scale);
    }
    __syncthreads();
    // maximum (any order gives the same value)
    float m = -3.402823466e+38f;
    for (int c = tid; c < seq_k; c += nt) m = fmaxf(m, h_f(sc[c]));
    if (tid < 64) red[tid] = -3.402823466e+38f;
    __syncthreads();
    for (int s = 32; s > 0; s >>= 1) m = fmaxf(m, __shfl_down(m, s, 64));
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    float maxv = red[0];
    for (int i = 1; i < (nt + 63) / 64; ++i) maxv = fmaxf(maxv, red[i]);
    for (int c = tid; c < seq_k; c += nt) {
        const float e = exp_poly(h_f(sc[c]) - maxv);
        ex[c] = e;
        sc[c] = f_h(e);
    }
    __syncthreads();
    if (tid == 0) {
        float sum = 0.0f;
        for (int c = 0; c < seq_k; ++c) sum = sum + ex[c];
        inv_s = rcp_rn(sum + 1e-20f);
    }
    __syncthreads();
    const float inv = inv_s;
    for (int c = tid; c < seq_k; c += nt) sc[c] = f_h(h_f(sc[c]) * inv);
    __syncthreads();
    for (int e = tid; e < D; e += nt) {
        // keys 0 .. pos - 1 from the cache, eight loads in flight at a time, then the current one
        const uint16_t* col = vc + kvh * D + e;
        float acc = 0.0f;
        int tk = 0;
        for (; tk + 8 <= pos; tk += 8) {
            uint16_t v[8];
            #pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = col[static_cast<size_t>(tk + u) * kvd];
            #pragma unroll
            for (int u = 0; u < 8; ++u) acc = fmaf(h_f(sc[tk + u]), h_f(v[u]), acc);
        }
        for (; tk < pos; ++tk) acc = fmaf(h_f(sc[tk]), h_f(col[static_cast<size_t>(tk) * kvd]), acc);
        acc = fmaf(h_f(sc[pos]), h_f(vcur[e]), acc);
        out[qh * D + e] = f_h(acc);
    }
}

// The same launch for head widths known at compile time (64 and 128): one block of 512 threads per query
// head, the arithmetic and its order those of rope_attention_kernel.
//
// What bounds it at a long context are the two serial chains that order leaves: the sum of the exponentials (to 900 positions;
// beyond, ordered_sum) and, per output element, the sum over the keys.  A dependent addition takes 8 shader cycles (3.55 ns)
// whatever else the CU does, so the launch cannot be faster than 7.1 (3.6) ns per position.  Everything else is kept off
// the chains' path:
//  * scores, exponentials and probabilities are spread over all eight wavefronts (a key per thread, from a
//    tile of key rows in LDS; the next tile is requested while one is worked on);
//  * the sum's terms and the probabilities are read from LDS sixteen bytes at a time, a batch ahead;
//  * the values reach the chain transposed, eight keys of one element per 16-byte read, and are multiplied as
//    fp16 straight out of the pair they lie in (v_fma_mix_f32): one instruction per key.  Wavefronts 4 to 7 fill
//    the ring of value tiles (4 keys x 4 elements per thread, turned in registers) while wavefront 0 (and 1 at
//    head width 128) runs down the chain.
// us per launch, 256 threads with everything but the scores in the first wavefront -> this: 14 heads at position 1900
// 47.6 -> 25.3 (the two chains are 13.5 of it), 9 heads at 210 8.75 -> 7.24, 14 heads at 40 4.64 -> 4.63.
//
// At a short context (up to kShort keys, all of them in the first tiles) the launch is a chain of memory
// round trips and barriers instead, so everything that does not depend on an earlier result is requested at once
// (the first kShort rows of both caches before the position is known; rows that turn out not to be needed
// arrive unused), and wavefront 0 does the softmax and, at head width 64, the rest alone, without barriers.
//
// The current position's key and value take their places in the tiles as rows like the others.  Sums run in
// whole batches of kBatch positions: exponentials and probabilities past the last key are zeros, and so are
// value rows, which leaves a sum as it is: x + 0 = x and fma(0, 0, x) = x for every x but -0, and a sum that
// starts at +0 never becomes -0.
constexpr int kAttnThreads = 512;
constexpr int kShort = 128;
constexpr int kBatch = 32;
__host__ __device__ inline int padded_positions(int max_pos) { return (max_pos + kBatch - 1) / kBatch * kBatch; }
constexpr int kMaxPositions = 8192;                      // longest context a decoder is created for
// Bytes of LDS for tiles: a tile of key rows (padded by 16 bytes against bank conflicts), later two value tiles; at a
// short context kShort rows of either.
constexpr int kTileData = 65536;
constexpr size_t tile_area(int D) { return static_cast<size_t>(kTileData) / (2 * D) * (2 * D + 16); }

// A value of the lane `SH` below inside a row of 16, of the last lane of the row below, of lane 31 (DPP moves); a lane
// without one keeps its own.
template <int CTRL, int ROWS> __device__ __forceinline__ uint32_t from_below(uint32_t a) {
    return __builtin_amdgcn_update_dpp(static_cast<int>(a), static_cast<int>(a), CTRL, ROWS, 0xf, false);
}
// f(step): for every step of a scan over the 64 lanes, from_below's controls and the lowest lane its value covers last
template <typename F> __device__ __forceinline__ void scan_steps(F&& f, int lane) {
    f(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{}, (lane & 15) >= 1 ? lane - 1 : -1);      // row_shr:1
    f(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{}, (lane & 15) >= 2 ? lane - 2 : -1);
    f(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{}, (lane & 15) >= 4 ? lane - 4 : -1);
    f(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{}, (lane & 15) >= 8 ? lane - 8 : -1);
    f(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{}, lane & 16 ? (lane & 48) - 1 : -1);      // row_bcast:15
    f(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{}, lane & 32 ? 31 : -1);                   // row_bcast:31
}

// The sum of ex[0 .. n) in index order, as one chain of fp32 additions from 0 gives it bit for bit, by a wavefront whose
// lanes each hold a run of the terms; n a multiple of 4 and at most 256 * QUADS, terms not negative, the result in every lane.
//
// A running sum S >= 0 that stays in its binade, S = m u with u the unit in its last place, grows by a multiple of u
// with every term: fp32(S + e) - S depends on e and, where e / u ends in exactly a half, on whether m is even.  So a
// lane adds its terms to two stand-ins for the sum in front of them, an even and an odd one of the same binade (a plain sum
// of everything ahead tells which that is); what either gained is what the true sum gains, in units of u the
// difference of the bit patterns.  Gains of neighbouring lanes in one binade are put together by a scan: "from an even
// sum k0 units, from an odd one k1".  Runs in which the sum passes into the next binade, seven or so of 64, are added
// term by term, and so is everything whose binade turns out another when the true sum gets there: nothing rests on the plain sum.
// 8 steps of the decoder, int8 0.5B at position 1030 / 1900 6028 / 7690 -> 5850 / 6990 us, Q4 360M at 2400 11 560 -> 10 470, fp16 0.5B at
// 3800 12 070 -> 10 490.  (With its lanes' terms read from LDS where they are used and its scans through LDS: no gain at 1900.)
template <int QUADS>
__device__ __forceinline__ float ordered_sum(const float* ex, const int n) {
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const f32x4* e4 = reinterpret_cast<const f32x4*>(ex);
    const int lane = threadIdx.x & 63;
    // quadruples of terms per lane (an odd number: 16-byte reads that far apart fall on all banks); of all; this lane's
    const int run = ((n + 255) / 256) | 1, quads = n / 4;
    const int q0 = lane * run, mine = q0 + run <= quads ? run : q0 < quads ? quads - q0 : 0;
    f32x4 e[QUADS];
    #pragma unroll
    for (int j = 0; j < QUADS; ++j) {
        e[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (j < mine) e[j] = e4[q0 + j];
    }
    f32x4 a = e[0];
    #pragma unroll
    for (int j = 1; j < QUADS; ++j) a += e[j];
    float upto = (a[0] + a[1]) + (a[2] + a[3]);                // a plain sum of the terms up to the run's end, then of those ahead of it
    scan_steps([&](auto ctrl, auto rows, int last) {
        const float o = __uint_as_float(from_below<decltype(ctrl)::value, decltype(rows)::value>(__float_as_uint(upto)));
        upto += last >= 0 ? o : 0.0f;
    }, lane);
    const float before = __shfl_up(upto, 1, 64);
    // (it is off by less than 2^-10 of itself: n is at most 2^13)
    const float lo = before * (1.0f - 0x1p-10f), hi = upto * (1.0f + 0x1p-10f);
    const uint32_t binade = __float_as_uint(lo) >> 23;
    bool steady = lane > 0 && mine > 0 && lo > 1e-30f && hi < 1e30f && binade == __float_as_uint(hi) >> 23;
    const uint32_t even = __float_as_uint(before) & ~1u;
    float s0 = __uint_as_float(even), s1 = __uint_as_float(even | 1u);
    #pragma unroll
    for (int j = 0; j < QUADS; ++j)
        #pragma unroll
        for (int r = 0; r < 4; ++r) {
            s0 = s0 + e[j][r];
            s1 = s1 + e[j][r];
        }
    uint32_t k0 = __float_as_uint(s0) - even, k1 = __float_as_uint(s1) - (even | 1u);
    steady = steady && __float_as_uint(s0) >> 23 == binade && __float_as_uint(s1) >> 23 == binade;
    // runs of neighbouring steady lanes of one binade, in one piece each: a head is a lane that does not go on with the one below
    const uint32_t below = __shfl_up(steady ? binade : 0u, 1, 64);
    const uint64_t heads = __ballot(lane == 0 || !steady || below != binade);
    const int from = 63 - __clzll(heads & (~0ull >> (63 - lane)));
    scan_steps([&](auto ctrl, auto rows, int last) {
        const uint32_t p0 = from_below<decltype(ctrl)::value, decltype(rows)::value>(k0), p1 = from_below<decltype(ctrl)::value, decltype(rows)::value>(k1);
        const uint32_t n0 = p0 + (p0 & 1u ? k1 : k0), n1 = p1 + (p1 & 1u ? k0 : k1);
        if (last >= from) { k0 = n0; k1 = n1; }
    }, lane);
    // from head to head with the true sum (lanes that hold terms are the lowest ones)
    const uint64_t steadies = __ballot(steady);
    const int lanes = (quads + run - 1) / run;
    uint64_t left = heads & (~0ull >> (64 - lanes));
    float sum = 0.0f;
    while (left) {
        const int first = __ffsll(static_cast<unsigned long long>(left)) - 1;
        left &= left - 1;
        const int next = left ? __ffsll(static_cast<unsigned long long>(left)) - 1 : lanes;
        if (steadies >> first & 1) {
            const uint32_t b = __builtin_amdgcn_readlane(binade, first), g0 = __builtin_amdgcn_readlane(k0, next - 1),
                           g1 = __builtin_amdgcn_readlane(k1, next - 1);
            const uint32_t at = __builtin_amdgcn_readfirstlane(__float_as_uint(sum)), to = at + (at & 1u ? g1 : g0);
            if (at >> 23 == b && to >> 23 == b) {
                sum = __uint_as_float(to);
                continue;
            }
        }
        for (int l = first; l < next; ++l) {                   // every lane goes on with its own terms, lane l's is the sum
            float t = sum;
            #pragma unroll
            for (int j = 0; j < QUADS; ++j)
                #pragma unroll
                for (int r = 0; r < 4; ++r) t = t + e[j][r];
            sum = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(t), l));
        }
    }
    return sum;
}
// Positions (in whole batches) from which on the sum is spread over the lanes (even at about 800), and the most of them: a lane holds its
// terms in registers, 9 quadruples up to 2304 positions, 17 up to 4096 (idle ones add zeros).  Longer contexts keep the one
// chain: 33 quadruples in a lane were not tried.  (8 steps of int8 0.5B at position 2100 with 17 / 9: 7487 / 7344 us.)
constexpr int kSpreadFrom = 928, kSpreadQuads = 17, kSpreadMost = 256 * (kSpreadQuads - 1);

template <int D>
// (Arguments in the order of need: the first 14 dwords arrive in registers with the wavefront, and the
//  first thing the kernel does is ask for the cache tiles and the position.)
__global__ __launch_bounds__(kAttnThreads) void rope_attention_tiled(uint16_t* __restrict__ kc, uint16_t* __restrict__ vc,
                                      const State* __restrict__ st, int n_heads, int n_kv_heads, int max_pos,
                                      float scale, const uint16_t* __restrict__ q_raw, const uint16_t* __restrict__ k_raw,
                                      const uint16_t* __restrict__ v_raw, const uint16_t* __restrict__ bq,
                                      const uint16_t* __restrict__ bk, const uint16_t* __restrict__ bv,
                                      const uint16_t* __restrict__ rope_now,
                                      uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_out,
                                      uint16_t* __restrict__ v_out, uint16_t* __restrict__ out) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int kRowH = D + 8;                           // halves between key rows in LDS
    constexpr int kPieces = D / 8;                         // 16-byte pieces per row
    constexpr int kPassRows = kAttnThreads / kPieces;      // key rows that 512 threads request at once
    constexpr int kKeyRows = kTileData / (2 * D);          // key rows per tile (512 / 256)
    constexpr int kPasses = kKeyRows / kPassRows;
    constexpr int kShortPasses = kShort / kPassRows;
    constexpr int kValueRows = kKeyRows / 2;               // value rows per tile of the ring
    constexpr int kDG = D / 4;                             // groups of 4 elements
    constexpr int kShortBlocks = kShort / 4 * kDG / kAttnThreads;         // 4 x 4 blocks per thread, short context
    constexpr int kRingThreads = 256;                                      // wavefronts 4 .. 7 fill the ring
    constexpr int kRingBlocks = kValueRows / 4 * kDG / kRingThreads;
    constexpr int kChainWaves = D / 64;
    extern __shared__ __attribute__((aligned(16))) uint16_t qv[];
    uint16_t* vcur = qv + D;
    const int mp = padded_positions(max_pos);
    float* ex = reinterpret_cast<float*>(vcur + D);                        // [mp] exponentials, then probabilities; 16-byte aligned
    uint16_t* sc = reinterpret_cast<uint16_t*>(ex + mp);                   // [mp] scores
    float* red = reinterpret_cast<float*>(sc + mp);                        // [8] maxima of the wavefronts
    uint16_t* ktile = reinterpret_cast<uint16_t*>(red + 8);                // 16-byte aligned
    uint8_t* vring = reinterpret_cast<uint8_t*>(ktile);                    // [2][kValueRows / 8][D][8 keys], where the keys were
    uint8_t* vshort = reinterpret_cast<uint8_t*>(ktile + kShort * kRowH);
    const int nrep = n_heads / n_kv_heads;
    const int qh = blockIdx.x, kvd = n_kv_heads * D, kvh = qh / nrep, hd2 = D / 2;
    const bool writer = qh % nrep == 0;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // piece p of this thread in a key tile: row tid / kPieces + p kPassRows, 16-byte piece tid % kPieces
    const int krow = tid / kPieces, kpiece = tid % kPieces;
    auto request_keys = [&](int row0, int p) {
        const int at = row0 + krow + p * kPassRows, tk = at < max_pos ? at : max_pos - 1;
        return *reinterpret_cast<const u32x4*>(kc + static_cast<size_t>(tk) * kvd + kvh * D + 8 * kpiece);
    };
    // 4 keys x 4 elements of the values
    struct VBlock { u32x2 r[4]; };
    auto request_values = [&](int key0, int dg) {
        VBlock b;
        #pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int tk = key0 + e < max_pos ? key0 + e : max_pos - 1;
            b.r[e] = *reinterpret_cast<const u32x2*>(vc + static_cast<size_t>(tk) * kvd + kvh * D + 4 * dg);
        }
        return b;
    };
    u32x4 kreg[kPasses];
    VBlock vreg[kRingBlocks];
    int pos = st->pos;
    kreg[0] = request_keys(0, 0);
    asm volatile("" ::: "memory");
    // What the current position needs (projections, biases, the rotary row: a few bytes per thread, behind pointers that
    // have to be fetched) is asked for next, ahead of the other rows.  Wavefront 0 prepares q, 1 k, 2 and 3 v; every
    // thread loads from a valid address whether it has an element or not, so the number of loads in flight is the same.
    const int role = wave < 3 ? wave : 2;
    const int i = role < 2 ? (lane < hd2 ? lane : hd2 - 1) : (tid >= 128 && tid - 128 < D ? tid - 128 : D - 1);
    const int i2 = role < 2 ? i + hd2 : i;
    const uint16_t* buf = role == 0 ? q_raw + qh * D : role == 1 ? k_raw + kvh * D : v_raw + kvh * D;
    const uint16_t* bias = role == 0 ? bq + qh * D : role == 1 ? bk + kvh * D : bv + kvh * D;
    const uint16_t raw1 = buf[i], raw2 = buf[i2], bias1 = bias[i], bias2 = bias[i2];
    const uint16_t cos_i = rope_now[role < 2 ? i : 0], sin_i = rope_now[D + (role < 2 ? i : 0)];   // embed_kernel's row
    asm volatile("" ::: "memory");                             // these first
    #pragma unroll
    for (int p = 1; p < kShortPasses; ++p) kreg[p] = request_keys(0, p);
    #pragma unroll
    for (int p = 0; p < kShortBlocks; ++p) vreg[p] = request_values(4 * ((tid + kAttnThreads * p) / kDG), (tid + kAttnThreads * p) % kDG);
    __builtin_amdgcn_sched_barrier(0);                         // and nothing that waits for one of them in between

    pos = pos < 0 ? 0 : (pos >= max_pos ? max_pos - 1 : pos);
    const int seq_k = pos + 1, padded = (seq_k + kBatch - 1) / kBatch * kBatch;
    const bool is_short = seq_k <= kShort;
    if (!is_short) {
        #pragma unroll
        for (int p = kShortPasses; p < kPasses; ++p) kreg[p] = request_keys(0, p);
    }
    // (computed by every thread, stored by those that have an element: a load that is only used under a
    //  condition would be moved there, behind the tiles)
    const float c = h_f(cos_i), sn = h_f(sin_i);
    const float x1 = h_f(f_h(h_f(raw1) + h_f(bias1)));
    const float x2 = h_f(f_h(h_f(raw2) + h_f(bias2)));
    const uint16_t r1 = f_h(fmaf(x1, c, -(x2 * sn))), r2 = f_h(fmaf(x2, c, x1 * sn));
    const bool has_pair = wave < 2 && lane < hd2, has_v = tid >= 128 && tid - 128 < D;
    const uint16_t rv = f_h(x1);                               // fp16(v + bias), rounded once
    if (has_pair && wave == 0) {
        qv[i] = r1;
        qv[i + hd2] = r2;
    } else if (has_v) {
        vcur[tid - 128] = rv;
    }
    // A tile's key rows from registers to LDS; the current position's row comes from its wavefront (k above).
    auto keep_keys = [&](int row0, int p) {
        const int row = krow + p * kPassRows;
        if (row0 + row != pos) *reinterpret_cast<u32x4*>(ktile + row * kRowH + 8 * kpiece) = kreg[p];
    };
    auto keep_current_key = [&](int row0) {
        if (wave == 1 && lane < hd2 && pos >= row0 && pos < row0 + kKeyRows) {
            ktile[(pos - row0) * kRowH + i] = r1;
            ktile[(pos - row0) * kRowH + i + hd2] = r2;
        }
    };
    // Four keys of four elements, transposed, into a value tile [8 keys each][cell][8 keys], zeros past the last key.
    // Cell c is element 4 (c % kDG) + c / kDG: the threads of a wavefront then write next to each other (element
    // order had eight of them on the same banks: 3.4 us per launch at position 1900). vcur must be in LDS (the block that holds the
    // current position takes its row from there).
    auto keep_values = [&](uint8_t* tile, const VBlock& b, int key0, int kg, int dg) {
        u32x2 v[4];
        #pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = key0 + e < pos ? b.r[e] : u32x2{0u, 0u};
        if (key0 <= pos && pos < key0 + 4) {
            const u32x2 own = *reinterpret_cast<const u32x2*>(vcur + 4 * dg);
            #pragma unroll
            for (int e = 0; e < 4; ++e)
                if (key0 + e == pos) v[e] = own;
        }
        uint8_t* dst = tile + ((kg / 2) * D + dg) * 16 + (kg & 1) * 8;
        #pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t sel = e & 1 ? 0x07060302u : 0x05040100u;
            *reinterpret_cast<u32x2*>(dst + e * kDG * 16) =
                u32x2{__builtin_amdgcn_perm(v[1][e / 2], v[0][e / 2], sel), __builtin_amdgcn_perm(v[3][e / 2], v[2][e / 2], sel)};
        }
    };
    // The outputs a caller may inspect and the cache rows (after the first tile is in LDS: a store in flight counts
    // like a load that has not arrived, and would make the waits above wait for later requests than they need).
    auto store_current = [&]() {
        if (has_pair) {
            if (wave == 0) {
                q_out[qh * D + i] = r1;
                q_out[qh * D + i + hd2] = r2;
            } else if (writer) {
                uint16_t* dst = kc + static_cast<size_t>(pos) * kvd + kvh * D;
                dst[i] = r1;
                dst[i + hd2] = r2;
                k_out[kvh * D + i] = r1;
                k_out[kvh * D + i + hd2] = r2;
            }
        } else if (has_v && writer) {
            const int e = tid - 128;
            vc[static_cast<size_t>(pos) * kvd + kvh * D + e] = rv;
            v_out[kvh * D + e] = rv;
        }
    };
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    struct Query { u16x4 v[D / 4]; };
    auto read_query = [&]() {
        Query q;
        #pragma unroll
        for (int d4 = 0; d4 < D / 4; ++d4) q.v[d4] = reinterpret_cast<const u16x4*>(qv)[d4];
        return q;
    };
    auto score = [&](const uint16_t* row, const Query& q) {
        const u16x4* kv = reinterpret_cast<const u16x4*>(row);
        float acc = 0.0f;
        #pragma unroll
        for (int d4 = 0; d4 < D / 4; ++d4) {
            const u16x4 a = q.v[d4], b = kv[d4];
            float t = h_f(a[0]) * h_f(b[0]);
            t = fmaf(h_f(a[1]), h_f(b[1]), t);
            t = fmaf(h_f(a[2]), h_f(b[2]), t);
            t = fmaf(h_f(a[3]), h_f(b[3]), t);
            acc = acc + t;
        }
        return f_h(acc * scale);
    };
    // sum of ex[0 .. padded) in index order, by every lane of the wavefront (the same reads, the same sum)
    auto sum_in_order = [&]() {
        const f32x4* e4 = reinterpret_cast<const f32x4*>(ex);
        f32x4 t[2][kBatch / 4];
        auto read = [&](f32x4 (&b)[kBatch / 4], int c0) {
            #pragma unroll
            for (int j = 0; j < kBatch / 4; ++j) b[j] = e4[c0 / 4 + j];
            asm volatile("" ::: "memory");                     // asked for here, not where it is used
        };
        float sum = 0.0f;
        auto add = [&](const f32x4 (&b)[kBatch / 4]) {
            #pragma unroll
            for (int j = 0; j < kBatch / 4; ++j) {
                sum = sum + b[j][0];
                sum = sum + b[j][1];
                sum = sum + b[j][2];
                sum = sum + b[j][3];
            }
        };
        // (the batch behind the last is the last again: with a request for every addition made the number in flight is a
        //  constant, and only then does the wait for one batch leave the next one in flight)
        read(t[0], 0);
        for (int c0 = 0;;) {
            read(t[1], c0 + kBatch < padded ? c0 + kBatch : c0);
            add(t[0]);
            c0 += kBatch;
            if (c0 >= padded) break;
            read(t[0], c0 + kBatch < padded ? c0 + kBatch : c0);
            add(t[1]);
            c0 += kBatch;
            if (c0 >= padded) break;
        }
        return sum;
    };
    // acc + sum over keys 0 .. n - 1 (n a multiple of kBatch) of a value tile, in index order; p: the probabilities from
    // the tile's first key on, as fp32 (an fp16 first factor makes the compiler put a wait state of 4 cycles behind each
    // v_fma_mix_f32: 5.1 instead of 3.5 ns per key); e: the cell
    auto chain = [&](float acc, const uint8_t* tile, const float* p, int e, int n) {
        u32x4 v[2][kBatch / 8];
        f32x4 q[2][kBatch / 4];
        auto read = [&](int b, int r0) {
            #pragma unroll
            for (int j = 0; j < kBatch / 8; ++j) {
                v[b][j] = *reinterpret_cast<const u32x4*>(tile + ((r0 / 8 + j) * D + e) * 16);
                q[b][2 * j] = *reinterpret_cast<const f32x4*>(p + r0 + 8 * j);
                q[b][2 * j + 1] = *reinterpret_cast<const f32x4*>(p + r0 + 8 * j + 4);
            }
            asm volatile("" ::: "memory");                     // asked for here, not where it is used
        };
        auto run = [&](int b) {
            #pragma unroll
            for (int j = 0; j < kBatch / 4; ++j) {
                const uint32_t v01 = v[b][j / 2][2 * (j % 2)], v23 = v[b][j / 2][2 * (j % 2) + 1];
                acc = fmaf(q[b][j][0], h_f(static_cast<uint16_t>(v01 & 0xffffu)), acc);
                acc = fmaf(q[b][j][1], h_f(static_cast<uint16_t>(v01 >> 16)), acc);
                acc = fmaf(q[b][j][2], h_f(static_cast<uint16_t>(v23 & 0xffffu)), acc);
                acc = fmaf(q[b][j][3], h_f(static_cast<uint16_t>(v23 >> 16)), acc);
            }
        };
        read(0, 0);
        for (int r0 = 0;;) {                                   // (requests as in sum_in_order)
            read(1, r0 + kBatch < n ? r0 + kBatch : r0);
            run(0);
            r0 += kBatch;
            if (r0 >= n) break;
            read(0, r0 + kBatch < n ? r0 + kBatch : r0);
            run(1);
            r0 += kBatch;
            if (r0 >= n) break;
        }
        return acc;
    };

    const int element = 4 * (tid % kDG) + tid / kDG;           // of the thread's cell (tid < D)
    if (is_short) {
        #pragma unroll
        for (int p = 0; p < kShortPasses; ++p)
            if (p * kPassRows < seq_k) keep_keys(0, p);
        keep_current_key(0);
        __syncthreads();                                       // (vcur is read by whoever holds the current position's block)
        #pragma unroll
        for (int p = 0; p < kShortBlocks; ++p) {
            const int kg = (tid + kAttnThreads * p) / kDG, dg = (tid + kAttnThreads * p) % kDG;
            if (4 * kg < padded) keep_values(vshort, vreg[p], 4 * kg, kg, dg);
        }
        store_current();
        if (tid < seq_k) sc[tid] = score(ktile + tid * kRowH, read_query());
        __syncthreads();
        // softmax by the first wavefront alone: its LDS accesses are ordered, so the steps need no
        // barrier between them (a short context is all barrier otherwise)
        if (wave == 0) {
            float m = -3.402823466e+38f;                       // maximum: any order gives the same value
            for (int k = tid; k < seq_k; k += 64) m = fmaxf(m, h_f(sc[k]));
            const float maxv = wave_max(m);
            for (int k = tid; k < padded; k += 64) ex[k] = k < seq_k ? exp_poly(h_f(sc[k]) - maxv) : 0.0f;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // every lane reads what the others wrote
            __builtin_amdgcn_wave_barrier();
            const float inv = rcp_rn(sum_in_order() + 1e-20f);
            for (int k = tid; k < padded; k += 64) ex[k] = h_f(f_h(h_f(f_h(ex[k])) * inv));     // probabilities, rounded to fp16
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
            __builtin_amdgcn_wave_barrier();
        }
        if constexpr (kChainWaves > 1) __syncthreads();
        if (wave < kChainWaves) out[qh * D + element] = f_h(chain(0.0f, vshort, ex, tid, padded));
        return;
    }

    // scores, tile by tile; a thread keeps the greatest of its own
    float m = -3.402823466e+38f;
    {
        #pragma unroll
        for (int p = 0; p < kPasses; ++p) keep_keys(0, p);
        keep_current_key(0);
        store_current();
        __syncthreads();                                       // q and the first tile are in LDS
        const Query query = read_query();
        for (int row0 = 0; row0 < seq_k; row0 += kKeyRows) {
            if (row0 + kKeyRows < seq_k) {
                #pragma unroll
                for (int p = 0; p < kPasses; ++p) kreg[p] = request_keys(row0 + kKeyRows, p);
            }
            if (row0 > 0) __syncthreads();                     // the tile is in LDS
            if (tid < kKeyRows && row0 + tid < seq_k) {
                const uint16_t s = score(ktile + tid * kRowH, query);
                sc[row0 + tid] = s;
                m = fmaxf(m, h_f(s));
            }
            if (row0 + kKeyRows < seq_k) {
                __syncthreads();                               // and has been used
                #pragma unroll
                for (int p = 0; p < kPasses; ++p) keep_keys(row0 + kKeyRows, p);
                keep_current_key(row0 + kKeyRows);
            }
        }
    }
    // wavefronts 4 .. 7 keep value tiles coming: tile u of the ring holds keys u kValueRows ..
    const bool feeds = wave >= 4;
    const int rt = tid - (kAttnThreads - kRingThreads);
    auto request_tile = [&](int u) {
        #pragma unroll
        for (int p = 0; p < kRingBlocks; ++p)
            vreg[p] = request_values(u * kValueRows + 4 * ((rt + kRingThreads * p) / kDG), (rt + kRingThreads * p) % kDG);
    };
    auto keep_tile = [&](int u) {
        #pragma unroll
        for (int p = 0; p < kRingBlocks; ++p) {
            const int kg = (rt + kRingThreads * p) / kDG, dg = (rt + kRingThreads * p) % kDG;
            keep_values(vring + (u & 1) * (kValueRows * D * 2), vreg[p], u * kValueRows + 4 * kg, kg, dg);
        }
    };
    const int vtiles = (seq_k + kValueRows - 1) / kValueRows;
    if (feeds) request_tile(0);
    m = wave_max(m);
    if (lane == 0) red[wave] = m;
    __syncthreads();                                           // scores and maxima are in LDS, the key tile has been used
    m = fmaxf(fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])), fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7])));
    for (int k = tid; k < padded; k += kAttnThreads) ex[k] = k < seq_k ? exp_poly(h_f(sc[k]) - m) : 0.0f;
    __syncthreads();                                           // exponentials
    if (feeds) {
        keep_tile(0);
        if (vtiles > 1) { request_tile(1); keep_tile(1); }
        if (vtiles > 2) request_tile(2);
    } else if (wave == 0) {
        const float sum = padded < kSpreadFrom || padded > kSpreadMost ? sum_in_order()
                        : padded <= 256 * 9                           ? ordered_sum<9>(ex, padded) : ordered_sum<kSpreadQuads>(ex, padded);
        const float inv = rcp_rn(sum + 1e-20f);
        if (tid == 0) red[0] = inv;
    }
    __syncthreads();                                           // the sum
    {
        const float inv = red[0];
        for (int k = tid; k < padded; k += kAttnThreads) ex[k] = h_f(f_h(h_f(f_h(ex[k])) * inv));
    }
    __syncthreads();                                           // probabilities and the first two value tiles
    float acc = 0.0f;
    for (int u = 0; u < vtiles; ++u) {
        if (wave < kChainWaves) {
            const int n = padded - u * kValueRows < kValueRows ? padded - u * kValueRows : kValueRows;
            acc = chain(acc, vring + (u & 1) * (kValueRows * D * 2), ex + u * kValueRows, tid, n);
        }
        if (u + 2 < vtiles) {
            __syncthreads();                                   // tile u has been used; tile u + 1 is behind an earlier barrier
            if (feeds) {
                keep_tile(u + 2);
                if (u + 3 < vtiles) request_tile(u + 3);
            }
        } else if (u + 1 < vtiles) {
            __syncthreads();
        }
    }
    if (wave < kChainWaves) out[qh * D + element] = f_h(acc);
}

// ---- attention with the keys of a head split over several blocks (an arithmetic mode, not the default) ----
//
// The launch above keeps the reference's order of operations, and at a long context that order is two
// chains of dependent additions as long as the context, in one wavefront per head.  Here block (head, s) takes
// run s of `splits` consecutive runs of the keys: scores as above (fp32 dot product, rounded to fp16 like
// the reference's), its own maximum m, e = exp(score - m) in fp32, their sum l and o[d] = sum e v[d]; a
// second launch merges the parts of a head: M = max m, out = sum_s exp(m_s - M) o_s / sum_s exp(m_s - M) l_s.
// The same real numbers as softmax(q k) v, summed in another order and without the fp16 roundings of the
// probabilities: within the stated tolerance of the reference-order launch, not bit-identical.
// part: [n_heads][splits][D + 2] floats: m, l, o[D].
//
// The launch is a chain of trips to memory: the position, then the block's rows of both caches.  They are asked for
// at once, 16 bytes per lane (a tile of keys and a tile of values in registers), and turned over to LDS as they are
// needed: a thread takes the score of a key from the key tile, then one element of the output over every kGroups-th
// key from the value tile.  14 heads at position 3701 in 16 splits, us per launch: rows read by a thread each and
// values 2 bytes at a time, 32 in flight, 10.2 -> this 8.7 (6.8 either way at
// position 2000, where 32 in flight is all there are).  The heads of a group that read the same run put on one XCD: no gain.
constexpr int kSplitThreads = 256;
constexpr int kMaxSplits = 32;
constexpr int split_tile(int D) { return 16384 / D; }          // keys per tile (256 / 128)
constexpr int split_groups(int D) { return kSplitThreads / D; }
// Floats of LDS for the exponentials: per group its keys one behind the other, rows of whole 16 bytes
__host__ __device__ inline int split_group_cap(int D, int chunk_cap) { return ((chunk_cap + split_groups(D) - 1) / split_groups(D) + 3) & ~3; }

template <int D>
__global__ __launch_bounds__(kSplitThreads) void attention_split_kernel(
        uint16_t* __restrict__ kc, uint16_t* __restrict__ vc, const State* __restrict__ st, int n_heads, int n_kv_heads,
        int max_pos, float scale, const uint16_t* __restrict__ q_raw, const uint16_t* __restrict__ k_raw,
        const uint16_t* __restrict__ v_raw, const uint16_t* __restrict__ bq, const uint16_t* __restrict__ bk,
        const uint16_t* __restrict__ bv, const uint16_t* __restrict__ rope_now, uint16_t* __restrict__ q_out,
        uint16_t* __restrict__ k_out, uint16_t* __restrict__ v_out, float* __restrict__ part, int chunk_cap) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    constexpr int kTile = split_tile(D), kGroups = split_groups(D);
    constexpr int kPieces = D / 8, kPassRows = kSplitThreads / kPieces, kPasses = kTile / kPassRows;
    constexpr int kRowH = D + 8;                               // halves between key rows in LDS (values: D)
    extern __shared__ __attribute__((aligned(16))) float sm[];
    const int gcap = split_group_cap(D, chunk_cap);
    float* ex = sm;                                            // [kGroups][gcap] scores, then exponentials
    float* red = ex + kGroups * gcap;                          // [8] block reductions
    float* osum = red + 8;                                     // [kSplitThreads / D][D] partial outputs
    uint16_t* qv = reinterpret_cast<uint16_t*>(osum + kSplitThreads);   // [D] q
    uint16_t* tile = qv + D;                                   // [kTile][kRowH] keys, then [kTile][D] values
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int qh = blockIdx.x, sp = blockIdx.y, splits = gridDim.y;
    const int nrep = n_heads / n_kv_heads, kvh = qh / nrep, kvd = n_kv_heads * D, hd2 = D / 2;
    int pos = st->pos;
    // what the current position needs, a few bytes per thread behind other pointers, rides along with the position:
    // threads 0 .. D/2 - 1 take a pair of q, 64 .. a pair of k, 128 .. an element of v
    const int role = tid < 64 ? 0 : tid < 128 ? 1 : 2;
    const int i = role < 2 ? ((tid & 63) < hd2 ? tid & 63 : hd2 - 1) : (tid - 128 < D ? tid - 128 : D - 1);
    const int i2 = role < 2 ? i + hd2 : i;
    const uint16_t* buf = role == 0 ? q_raw + qh * D : role == 1 ? k_raw + kvh * D : v_raw + kvh * D;
    const uint16_t* bias = role == 0 ? bq + qh * D : role == 1 ? bk + kvh * D : bv + kvh * D;
    const uint16_t raw1 = buf[i], raw2 = buf[i2], bias1 = bias[i], bias2 = bias[i2];
    const uint16_t cos_i = rope_now[role < 2 ? i : 0], sin_i = rope_now[D + (role < 2 ? i : 0)];

    pos = pos < 0 ? 0 : (pos >= max_pos ? max_pos - 1 : pos);
    const int seq_k = pos + 1;
    const int chunk = (seq_k + splits - 1) / splits;           // <= chunk_cap: the host sizes it for max_pos
    const int k0 = sp * chunk, k1 = k0 + chunk < seq_k ? k0 + chunk : seq_k, n = k1 - k0;
    float* mine = part + (static_cast<size_t>(qh) * splits + sp) * (D + 2);
    if (n <= 0) {                                              // no keys for this block at this position
        if (tid == 0) { mine[0] = -3.402823466e+38f; mine[1] = 0.0f; }
        if (tid < D) mine[2 + tid] = 0.0f;
        return;
    }
    const bool has_current = k1 == seq_k;                      // the block whose run ends with the current position
    // piece p of this thread in a tile: row tid / kPieces + p kPassRows, 16-byte piece tid % kPieces; rows past the
    // run's last key are read as that key's and not used
    const int prow = tid / kPieces, piece = tid % kPieces;
    u32x4 kreg[kPasses], vreg[kPasses];
    auto request = [&](u32x4 (&reg)[kPasses], const uint16_t* cache, int t0) {
        #pragma unroll
        for (int p = 0; p < kPasses; ++p)
            if (t0 + p * kPassRows < n) {                      // (uniform)
                const int row = t0 + prow + p * kPassRows, c = k0 + (row < n ? row : n - 1);
                reg[p] = *reinterpret_cast<const u32x4*>(cache + static_cast<size_t>(c) * kvd + kvh * D + 8 * piece);
            }
    };
    auto keep = [&](const u32x4 (&reg)[kPasses], int stride, int t0) {
        #pragma unroll
        for (int p = 0; p < kPasses; ++p)
            if (t0 + p * kPassRows < n) {
                const int row = prow + p * kPassRows;
                if (k0 + t0 + row != pos) *reinterpret_cast<u32x4*>(tile + row * stride + 8 * piece) = reg[p];
            }
    };
    request(kreg, kc, 0);
    request(vreg, vc, 0);

    const float cs = h_f(cos_i), sn = h_f(sin_i);
    const float x1 = h_f(f_h(h_f(raw1) + h_f(bias1)));
    const float x2 = h_f(f_h(h_f(raw2) + h_f(bias2)));
    const uint16_t r1 = f_h(fmaf(x1, cs, -(x2 * sn))), r2 = f_h(fmaf(x2, cs, x1 * sn));
    const uint16_t rv = f_h(x1);                               // fp16(v + bias), rounded once
    const bool is_q = tid < hd2, is_k = has_current && tid >= 64 && tid < 64 + hd2, is_v = has_current && tid >= 128 && tid < 128 + D;
    const int cur = pos - k0;                                  // the current position's row of the run
    // Scores, tile by tile, a thread per key (key c of the run is thread c % 256's); the current position's key goes
    // into its tile straight from the threads that made it.
    float m = -3.402823466e+38f;
    if (is_q) {
        qv[i] = r1;
        qv[i + hd2] = r2;
    }
    for (int t0 = 0; t0 < n; t0 += kTile) {
        if (t0 > 0) __syncthreads();                           // the last tile has been used
        keep(kreg, kRowH, t0);
        if (is_k && cur >= t0 && cur < t0 + kTile) {
            tile[(cur - t0) * kRowH + i] = r1;
            tile[(cur - t0) * kRowH + i + hd2] = r2;
        }
        __syncthreads();
        if (t0 + kTile < n) request(kreg, kc, t0 + kTile);
        const int row = tid - t0 % kSplitThreads;              // (a tile is 256 keys or half of them)
        if (row >= 0 && row < kTile && t0 + row < n) {
            float acc = 0.0f;
            #pragma unroll
            for (int j = 0; j < D / 8; ++j) {
                const u32x4 qq = reinterpret_cast<const u32x4*>(qv)[j], kk = *reinterpret_cast<const u32x4*>(tile + row * kRowH + 8 * j);
                #pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc = fmaf(h_f(static_cast<uint16_t>(qq[e] & 0xffffu)), h_f(static_cast<uint16_t>(kk[e] & 0xffffu)), acc);
                    acc = fmaf(h_f(static_cast<uint16_t>(qq[e] >> 16)), h_f(static_cast<uint16_t>(kk[e] >> 16)), acc);
                }
            }
            const float sco = h_f(f_h(acc * scale));
            const int c = t0 + row;
            ex[(c % kGroups) * gcap + c / kGroups] = sco;
            m = fmaxf(m, sco);
        }
    }
    // (the outputs a caller may inspect and the cache rows, behind the loads)
    if (is_q && sp == 0) { q_out[qh * D + i] = r1; q_out[qh * D + i + hd2] = r2; }
    if (qh % nrep == 0) {
        if (is_k) {
            uint16_t* dst = kc + static_cast<size_t>(pos) * kvd + kvh * D;
            dst[i] = r1; dst[i + hd2] = r2;
            k_out[kvh * D + i] = r1; k_out[kvh * D + i + hd2] = r2;
        } else if (is_v) {
            vc[static_cast<size_t>(pos) * kvd + kvh * D + i] = rv;
            v_out[kvh * D + i] = rv;
        }
    }
    m = wave_max(m);
    if (lane == 0) red[wave] = m;
    __syncthreads();                                           // scores and maxima are in LDS, the keys have been used
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float l = 0.0f;
    for (int c = tid; c < n; c += kSplitThreads) {
        float* at = ex + (c % kGroups) * gcap + c / kGroups;
        const float e = exp_poly(*at - m);
        *at = e;
        l += e;
    }
    for (int sft = 32; sft > 0; sft >>= 1) l += __shfl_xor(l, sft, 64);
    if (lane == 0) red[4 + wave] = l;
    // o[d]: kSplitThreads / D groups of D threads, group g takes the keys g, g + groups, ... of the run
    const int d = tid % D, grp = tid / D;
    const float* ep = ex + grp * gcap;
    float o = 0.0f;
    for (int t0 = 0; t0 < n; t0 += kTile) {
        if (t0 > 0) __syncthreads();                           // the last tile has been used
        keep(vreg, D, t0);
        if (is_v && cur >= t0 && cur < t0 + kTile) tile[(cur - t0) * D + i] = rv;
        __syncthreads();                                       // (and the exponentials and the waves' sums are in LDS)
        if (t0 + kTile < n) request(vreg, vc, t0 + kTile);
        const int rows = n - t0 < kTile ? n - t0 : kTile, count = (rows - grp + kGroups - 1) / kGroups, i0 = t0 / kGroups;
        const uint16_t* vp = tile + grp * D + d;
        int r = 0;
        for (; r + 8 <= count; r += 8) {                       // eight keys read ahead of their sums
            const f32x4 e0 = *reinterpret_cast<const f32x4*>(ep + i0 + r), e1 = *reinterpret_cast<const f32x4*>(ep + i0 + r + 4);
            uint16_t v[8];
            #pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = vp[(r + u) * kGroups * D];
            #pragma unroll
            for (int u = 0; u < 8; ++u) o = fmaf(u < 4 ? e0[u % 4] : e1[u % 4], h_f(v[u]), o);
        }
        for (; r < count; ++r) o = fmaf(ep[i0 + r], h_f(vp[r * kGroups * D]), o);
    }
    osum[grp * D + d] = o;
    __syncthreads();
    if (tid < D) {
        float t = osum[tid];
        #pragma unroll
        for (int g2 = 1; g2 < kGroups; ++g2) t += osum[g2 * D + tid];
        mine[2 + tid] = t;
    }
    if (tid == 0) {
        mine[0] = m;
        mine[1] = (red[4] + red[5]) + (red[6] + red[7]);
    }
}

// The parts of a head into its attention output (see attention_split_kernel).  Every load of the launch is
// asked for before the first is used: thread s takes the maximum and the sum of part s, thread d element d
// of every part.
template <int D>
__global__ __launch_bounds__(D) void attention_merge_kernel(const float* __restrict__ part, int splits,
                                                            uint16_t* __restrict__ out) {
    __shared__ float w[kMaxSplits];
    __shared__ float Ls;
    const int qh = blockIdx.x, d = threadIdx.x;
    const float* p = part + static_cast<size_t>(qh) * splits * (D + 2);
    float o_s[kMaxSplits];
    #pragma unroll
    for (int s = 0; s < kMaxSplits; ++s) o_s[s] = s < splits ? p[s * (D + 2) + 2 + d] : 0.0f;
    if (d < 64) {                                              // the first wavefront: splits <= 32 lanes of it
        const bool has = d < splits;
        const float ms = has ? p[d * (D + 2)] : -3.402823466e+38f;
        const float ls = has ? p[d * (D + 2) + 1] : 0.0f;
        const float M = wave_max(ms);
        const float ws = ls > 0.0f ? exp_poly(ms - M) : 0.0f;
        float L = ls * ws;
        for (int sft = 32; sft > 0; sft >>= 1) L += __shfl_xor(L, sft, 64);
        if (d < kMaxSplits) w[d] = ws;
        if (d == 0) Ls = L;
    }
    __syncthreads();
    float o = 0.0f;
    #pragma unroll
    for (int s = 0; s < kMaxSplits; ++s) o = fmaf(o_s[s], w[s], o);
    out[qh * D + d] = f_h(o * rcp_rn(Ls + 1e-20f));
}

inline size_t split_attention_lds(int D, int chunk_cap) {
    return (static_cast<size_t>(split_groups(D)) * split_group_cap(D, chunk_cap) + 8 + kSplitThreads) * 4 +
           (static_cast<size_t>(D) + static_cast<size_t>(split_tile(D)) * (D + 8)) * 2;
}

// gate[i] = fp16((g * sigmoid(g)) * up[i])   (QW/kernels/mlp.cl swiglu_inplace)
__global__ void swiglu_kernel(uint16_t* __restrict__ gate, const uint16_t* __restrict__ up, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        gate[i] = swiglu_h(gate[i], up[i]);
    }
}


// ---- a prompt of M tokens at once (Model::forward with seq_len = M, QW/src/model.cpp:243-376) ----
// Row r of every buffer belongs to position pos0 + r.  The kernels below repeat, row by row, the
// operations of the single-token kernels above in the same order, so that a prompt gives the
// same cache rows and logits as M single-token steps wherever the projections do (they do bit
// for bit when the M > 1 projections run as rows of GEMV, and within the GEMM's tolerance when
// they run on the matrix cores; the attention then runs there too, attention.hip, and the two
// attention kernels below serve the rows of GEMV and the head widths that kernel does not take).

// H[r][c] = embed[tokens[r]][c]   (QW/kernels/embedding.cl)
__global__ void embed_rows_kernel(const uint16_t* __restrict__ embed, const int* __restrict__ tokens,
                                  uint16_t* __restrict__ H, int hidden, int vocab) {
    int t = tokens[blockIdx.x];
    t = t < 0 ? 0 : (t >= vocab ? vocab - 1 : t);
    const uint16_t* src = embed + static_cast<size_t>(t) * hidden;
    uint16_t* dst = H + static_cast<size_t>(blockIdx.x) * hidden;
    for (int c = threadIdx.x; c < hidden; c += blockDim.x) dst[c] = src[c];
}

// One block per row: q/k/v bias, rotary embedding of q and k at position pos0 + row, k and v into
// the cache rows of that position (QW/kernels/bias_add.cl, rope.cl; rows as QW/src/layers/
// attention.cpp:560-600).
__global__ __launch_bounds__(256) void rope_rows_kernel(const uint16_t* __restrict__ Q, const uint16_t* __restrict__ Kp,
                                                        const uint16_t* __restrict__ V, const uint16_t* __restrict__ bq,
                                                        const uint16_t* __restrict__ bk, const uint16_t* __restrict__ bv,
                                                        const uint16_t* __restrict__ cosT, const uint16_t* __restrict__ sinT,
                                                        uint16_t* __restrict__ kc, uint16_t* __restrict__ vc,
                                                        uint16_t* __restrict__ QR, int pos0, int n_heads, int n_kv_heads, int D,
                                                        int ldq, int ldkv) {
    // ldq, ldkv: halves between rows of Q and of Kp / V (the widths of the projections, or of the
    // stacked q|k|v projection they are columns of)
    const int row = blockIdx.x, pos = pos0 + row, hd2 = D / 2, qd = n_heads * D, kvd = n_kv_heads * D;
    const uint16_t* cr = cosT + static_cast<size_t>(pos) * D;
    const uint16_t* sr = sinT + static_cast<size_t>(pos) * D;
    for (int j = threadIdx.x; j < (n_heads + n_kv_heads) * hd2; j += blockDim.x) {
        const int head = j / hd2, i = j - head * hd2;
        const bool isq = head < n_heads;
        const int hh = isq ? head : head - n_heads;
        const uint16_t* buf = isq ? Q + static_cast<size_t>(row) * ldq + hh * D : Kp + static_cast<size_t>(row) * ldkv + hh * D;
        const uint16_t* bias = (isq ? bq : bk) + hh * D;
        uint16_t* dst = isq ? QR + static_cast<size_t>(row) * qd + hh * D : kc + static_cast<size_t>(pos) * kvd + hh * D;
        const float c = h_f(cr[i]), sn = h_f(sr[i]);
        const float x1 = h_f(f_h(h_f(buf[i]) + h_f(bias[i])));
        const float x2 = h_f(f_h(h_f(buf[i + hd2]) + h_f(bias[i + hd2])));
        dst[i] = f_h(fmaf(x1, c, -(x2 * sn)));
        dst[i + hd2] = f_h(fmaf(x2, c, x1 * sn));
    }
    for (int e = threadIdx.x; e < kvd; e += blockDim.x)
        vc[static_cast<size_t>(pos) * kvd + e] = f_h(h_f(V[static_cast<size_t>(row) * ldkv + e]) + h_f(bv[e]));
}

// One block per (query head, row): the query of position pos0 + row against cache rows
// 0 .. pos0 + row (causal), QW/kernels/attention.cl gqa_attn_scores, gqa_softmax, gqa_attn_out with
// the sums in the order of rope_attention_kernel.  256 threads.  Dynamic LDS: 2 D (1 + kPromptTile)
// bytes + 6 bytes per position.
constexpr int kPromptTile = 64;
__global__ __launch_bounds__(256) void attention_rows_kernel(const uint16_t* __restrict__ QR, const uint16_t* __restrict__ kc,
                                                             const uint16_t* __restrict__ vc, uint16_t* __restrict__ out,
                                                             int pos0, int seq_cap, int n_heads, int n_kv_heads, int D,
                                                             float scale) {
    extern __shared__ __attribute__((aligned(16))) uint16_t qv[];
    uint16_t* tile = qv + D;                                       // [kPromptTile][D] values
    float* ex = reinterpret_cast<float*>(tile + kPromptTile * D);
    uint16_t* sc = reinterpret_cast<uint16_t*>(ex + seq_cap);
    __shared__ float red[64];
    __shared__ float inv_s;
    const int qh = blockIdx.x, row = blockIdx.y, pos = pos0 + row, seq_k = pos + 1;
    const int nrep = n_heads / n_kv_heads, kvh = qh / nrep, kvd = n_kv_heads * D, qd = n_heads * D;
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int i = tid; i < D; i += nt) qv[i] = QR[static_cast<size_t>(row) * qd + qh * D + i];
    __syncthreads();
    for (int tk = tid; tk < seq_k; tk += nt) {
        typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
        const u16x4* kv = reinterpret_cast<const u16x4*>(kc + static_cast<size_t>(tk) * kvd + kvh * D);
        const u16x4* qq = reinterpret_cast<const u16x4*>(qv);
        float acc = 0.0f;
        for (int d4 = 0; d4 < D / 4; ++d4) {
            const u16x4 a = qq[d4], b = kv[d4];
            float t = h_f(a[0]) * h_f(b[0]);
            t = fmaf(h_f(a[1]), h_f(b[1]), t);
            t = fmaf(h_f(a[2]), h_f(b[2]), t);
            t = fmaf(h_f(a[3]), h_f(b[3]), t);
            acc = acc + t;
        }
        sc[tk] = f_h(acc * scale);
    }
    __syncthreads();
    float m = -3.402823466e+38f;
    for (int c = tid; c < seq_k; c += nt) m = fmaxf(m, h_f(sc[c]));
    if (tid < 64) red[tid] = -3.402823466e+38f;
    __syncthreads();
    for (int s = 32; s > 0; s >>= 1) m = fmaxf(m, __shfl_down(m, s, 64));
    if ((tid & 63) == 0) red[tid >> 6] = m;
    __syncthreads();
    float maxv = red[0];
    for (int i = 1; i < (nt + 63) / 64; ++i) maxv = fmaxf(maxv, red[i]);
    for (int c = tid; c < seq_k; c += nt) {
        const float e = exp_poly(h_f(sc[c]) - maxv);
        ex[c] = e;
        sc[c] = f_h(e);
    }
    __syncthreads();
    if (tid == 0) {
        float sum = 0.0f;
        for (int c = 0; c < seq_k; ++c) sum = sum + ex[c];
        inv_s = rcp_rn(sum + 1e-20f);
    }
    __syncthreads();
    const float inv = inv_s;
    for (int c = tid; c < seq_k; c += nt) sc[c] = f_h(h_f(sc[c]) * inv);
    __syncthreads();
    // values: tiles of kPromptTile cache rows go through LDS (all threads fetch, 8 bytes each), then
    // thread e < D runs its sum over the tile's keys in index order
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    u16x4* tile4 = reinterpret_cast<u16x4*>(tile);
    const int d4n = D / 4;
    float acc = 0.0f;                                   // of output element tid (D <= 256 = threads)
    for (int t0 = 0; t0 < seq_k; t0 += kPromptTile) {
        const int rows = seq_k - t0 < kPromptTile ? seq_k - t0 : kPromptTile;
        for (int i = tid; i < rows * d4n; i += nt) {
            const int r = i / d4n, p = i - r * d4n;
            tile4[i] = *reinterpret_cast<const u16x4*>(vc + static_cast<size_t>(t0 + r) * kvd + kvh * D + 4 * p);
        }
        __syncthreads();
        if (tid < D)
            for (int r = 0; r < rows; ++r) acc = fmaf(h_f(sc[t0 + r]), h_f(tile[r * D + tid]), acc);
        __syncthreads();
    }
    if (tid < D) out[static_cast<size_t>(row) * qd + qh * D + tid] = f_h(acc);
}

// The same for head widths 64 and 128 with at most 8 query heads per key/value head: one block per
// (key/value head, row) serves all query heads of the group, so that a cache row is fetched once
// per group and position instead of once per head, and every fetch is a coalesced copy of a tile
// of kPromptTile rows into LDS (a thread of attention_rows_kernel walks a cache row of its own,
// which the memory pipeline serves one line per thread).  Per query the operations and their
// order are those of attention_rows_kernel: a score per thread from the key tile (rows padded by
// 8 bytes against bank conflicts), maximum, exponentials, the denominator summed by one thread
// in key order, the output element's sum in key order from the value tiles.  A (query, key)
// pair owns 4 bytes of LDS that hold, in turn, its fp16 score, its fp32 exponential and its fp16
// probability.  Wavefront w serves queries w and w + 4 in every phase but the last, where a thread
// owns one output element of up to 8 D / 256 queries.
// Dynamic LDS: 2 kPromptTile (D + 4) + 4 nrep seq_cap bytes; seq_cap is a multiple of 4.
template <int D>
__global__ __launch_bounds__(256) void attention_group_kernel(const uint16_t* __restrict__ QR, const uint16_t* __restrict__ kc,
                                                              const uint16_t* __restrict__ vc, uint16_t* __restrict__ out,
                                                              int pos0, int seq_cap, int n_heads, int n_kv_heads, float scale) {
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    constexpr int TK = kPromptTile, KS = D + 4, D4 = D / 4;
    extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
    uint16_t* tile = smem;                                          // [TK][KS] keys, then [TK][D] values
    uint32_t* slot = reinterpret_cast<uint32_t*>(tile + TK * KS);   // [nrep][seq_cap]
    __shared__ float inv_s[8];
    const int g = blockIdx.x, row = blockIdx.y, pos = pos0 + row, seq_k = pos + 1;
    const int nrep = n_heads / n_kv_heads, kvd = n_kv_heads * D, qd = n_heads * D;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint16_t* qsrc = QR + static_cast<size_t>(row) * qd + static_cast<size_t>(g) * nrep * D;   // the group's heads are adjacent
    const bool has0 = w < nrep, has1 = w + 4 < nrep;
    const int q0i = has0 ? w : 0, q1i = has1 ? w + 4 : q0i;
    // the wavefront's two query rows live in registers for the whole scores phase
    u16x4 qa[D4], qb[D4];
    #pragma unroll
    for (int d4 = 0; d4 < D4; ++d4) {
        qa[d4] = *reinterpret_cast<const u16x4*>(qsrc + q0i * D + 4 * d4);
        qb[d4] = *reinterpret_cast<const u16x4*>(qsrc + q1i * D + 4 * d4);
    }

    // A tile's rows travel global memory -> registers -> LDS; the next tile's are requested before
    // the current tile is worked on, so that their latency runs under the arithmetic.
    constexpr int kPieces = TK * D4 / 256;                          // 8-byte pieces of a tile per thread
    u16x4 pre[kPieces];
    auto fetch = [&](const uint16_t* cache, int t0) {
        #pragma unroll
        for (int u = 0; u < kPieces; ++u) {
            const int i = tid + 256 * u, r = i / D4, p = i - r * D4;
            const int tk = t0 + r < seq_k ? t0 + r : seq_k - 1;     // rows past the last key: a copy of it, never used
            pre[u] = *reinterpret_cast<const u16x4*>(cache + static_cast<size_t>(tk) * kvd + g * D + 4 * p);
        }
    };
    auto stash = [&](int stride) {
        #pragma unroll
        for (int u = 0; u < kPieces; ++u) {
            const int i = tid + 256 * u, r = i / D4, p = i - r * D4;
            *reinterpret_cast<u16x4*>(tile + r * stride + 4 * p) = pre[u];
        }
    };

    // scores: thread (key = lane, wavefront w) of a tile takes queries w and w + 4
    fetch(kc, 0);
    for (int t0 = 0; t0 < seq_k; t0 += TK) {
        const int rows = seq_k - t0 < TK ? seq_k - t0 : TK;
        __syncthreads();                                             // the last tile has been used
        stash(KS);
        __syncthreads();
        if (t0 + TK < seq_k) fetch(kc, t0 + TK);
        if (lane < rows) {
            const u16x4* kr = reinterpret_cast<const u16x4*>(tile + lane * KS);
            float acc0 = 0.0f, acc1 = 0.0f;
            #pragma unroll
            for (int d4 = 0; d4 < D4; ++d4) {
                const u16x4 b = kr[d4], a0 = qa[d4], a1 = qb[d4];
                float t = h_f(a0[0]) * h_f(b[0]);
                t = fmaf(h_f(a0[1]), h_f(b[1]), t);
                t = fmaf(h_f(a0[2]), h_f(b[2]), t);
                t = fmaf(h_f(a0[3]), h_f(b[3]), t);
                acc0 = acc0 + t;
                float u = h_f(a1[0]) * h_f(b[0]);
                u = fmaf(h_f(a1[1]), h_f(b[1]), u);
                u = fmaf(h_f(a1[2]), h_f(b[2]), u);
                u = fmaf(h_f(a1[3]), h_f(b[3]), u);
                acc1 = acc1 + u;
            }
            if (has0) slot[q0i * seq_cap + t0 + lane] = f_h(acc0 * scale);
            if (has1) slot[q1i * seq_cap + t0 + lane] = f_h(acc1 * scale);
        }
    }
    fetch(vc, 0);                                                    // the first tile of values arrives under the softmax
    __syncthreads();
    // maximum and exponentials, a wavefront per query.  A lane takes four of its entries at a time
    // (all reads ahead of the arithmetic and the writes: one LDS round trip per four entries).
    auto each4 = [&](uint32_t* sl, auto&& f) {
        for (int c0 = lane; c0 < seq_k; c0 += 256) {
            uint32_t v[4];
            #pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = sl[c0 + 64 * u < seq_k ? c0 + 64 * u : c0];
            #pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = f(v[u]);
            #pragma unroll
            for (int u = 0; u < 4; ++u)
                if (c0 + 64 * u < seq_k) sl[c0 + 64 * u] = v[u];
        }
    };
    #pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (j ? has1 : has0) {
            uint32_t* sl = slot + (j ? q1i : q0i) * seq_cap;
            float m = -3.402823466e+38f;
            for (int c0 = lane; c0 < seq_k; c0 += 256) {
                uint32_t v[4];
                #pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = sl[c0 + 64 * u < seq_k ? c0 + 64 * u : c0];
                #pragma unroll
                for (int u = 0; u < 4; ++u) m = fmaxf(m, h_f(static_cast<uint16_t>(v[u])));
            }
            for (int s = 32; s > 0; s >>= 1) m = fmaxf(m, __shfl_xor(m, s, 64));
            each4(sl, [m](uint32_t v) { return __float_as_uint(exp_poly(h_f(static_cast<uint16_t>(v)) - m)); });
        }
    }
    __syncthreads();
    // denominators: lanes 0 and 1 of a wavefront, one query each, keys in index order (sixteen
    // entries are read ahead of their additions; rows of slot start at multiples of 16 bytes)
    {
        const int qi = w + 4 * lane;
        if (lane < 2 && qi < nrep) {
            const uint32_t* sl = slot + qi * seq_cap;
            float sum = 0.0f;
            int c = 0;
            for (; c + 16 <= seq_k; c += 16) {
                uint4 v[4];
                #pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const uint4*>(sl + c + 4 * u);
                #pragma unroll
                for (int u = 0; u < 4; ++u) {
                    sum = sum + __uint_as_float(v[u].x);
                    sum = sum + __uint_as_float(v[u].y);
                    sum = sum + __uint_as_float(v[u].z);
                    sum = sum + __uint_as_float(v[u].w);
                }
            }
            for (; c < seq_k; ++c) sum = sum + __uint_as_float(sl[c]);
            inv_s[qi] = rcp_rn(sum + 1e-20f);
        }
    }
    __syncthreads();
    // probabilities: fp16(fp16(e) * inv), as the separate kernels store them
    #pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (j ? has1 : has0) {
            const int qi = j ? q1i : q0i;
            const float inv = inv_s[qi];
            each4(slot + qi * seq_cap, [inv](uint32_t v) -> uint32_t { return f_h(h_f(f_h(__uint_as_float(v))) * inv); });
        }
    }
    // values: thread (e = tid % D, tid / D) owns element e of queries tid / D + j (256 / D)
    constexpr int kStep = 256 / D, kJ = 8 / kStep;
    const int e = tid % D, qfirst = tid / D;
    int qc[kJ];
    float acc[kJ];
    #pragma unroll
    for (int j = 0; j < kJ; ++j) {
        const int qi = qfirst + j * kStep;
        qc[j] = (qi < nrep ? qi : nrep - 1) * seq_cap;
        acc[j] = 0.0f;
    }
    for (int t0 = 0; t0 < seq_k; t0 += TK) {
        const int rows = seq_k - t0 < TK ? seq_k - t0 : TK;
        __syncthreads();                                             // probabilities are in place; the last tile has been used
        stash(D);
        __syncthreads();
        if (t0 + TK < seq_k) fetch(vc, t0 + TK);
        int r = 0;
        for (; r + 8 <= rows; r += 8) {                              // eight keys read ahead of their sums
            uint16_t v[8];
            uint4 pr[kJ][2];
            #pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = tile[(r + u) * D + e];
            #pragma unroll
            for (int j = 0; j < kJ; ++j) {
                pr[j][0] = *reinterpret_cast<const uint4*>(slot + qc[j] + t0 + r);
                pr[j][1] = *reinterpret_cast<const uint4*>(slot + qc[j] + t0 + r + 4);
            }
            #pragma unroll
            for (int j = 0; j < kJ; ++j) {
                const uint32_t p8[8] = {pr[j][0].x, pr[j][0].y, pr[j][0].z, pr[j][0].w, pr[j][1].x, pr[j][1].y, pr[j][1].z, pr[j][1].w};
                #pragma unroll
                for (int u = 0; u < 8; ++u) acc[j] = fmaf(h_f(static_cast<uint16_t>(p8[u])), h_f(v[u]), acc[j]);
            }
        }
        for (; r < rows; ++r) {
            const float v = h_f(tile[r * D + e]);
            #pragma unroll
            for (int j = 0; j < kJ; ++j) acc[j] = fmaf(h_f(static_cast<uint16_t>(slot[qc[j] + t0 + r])), v, acc[j]);
        }
    }
    #pragma unroll
    for (int j = 0; j < kJ; ++j) {
        const int qi = qfirst + j * kStep;
        if (qi < nrep) out[static_cast<size_t>(row) * qd + (static_cast<size_t>(g) * nrep + qi) * D + e] = f_h(acc[j]);
    }
}

inline size_t group_attention_lds(int D, int nrep, int seq_cap) {
    return 2 * static_cast<size_t>(kPromptTile) * (D + 4) + 4 * static_cast<size_t>(nrep) * seq_cap;
}

// H[i] = fp16(H[i] + T[i]): the element-wise add behind a projection (QW/kernels/utils.cl element_add)
__global__ void add_rows_kernel(uint16_t* __restrict__ H, const uint16_t* __restrict__ T, long n) {
    for (long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += static_cast<long>(gridDim.x) * blockDim.x)
        H[i] = f_h(h_f(T[i]) + h_f(H[i]));
}

// add_rows_kernel and rmsnorm_kernel in one launch, a wavefront per row: H[r] = fp16(H[r] + T[r]),
// out[r] = rmsnorm(H[r]) * w, with the operations of the two kernels in their order (the row stays
// in registers between them).  For rows of at most 2048 elements, a multiple of 4.
__global__ __launch_bounds__(64) void add_rmsnorm_rows_kernel(uint16_t* __restrict__ H, const uint16_t* __restrict__ T,
                                                              const uint16_t* __restrict__ w, uint16_t* __restrict__ out,
                                                              int cols, float eps) {
    constexpr int kGroups = 8;
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    const int lid = threadIdx.x, c4n = cols >> 2;
    H += static_cast<size_t>(blockIdx.x) * cols;
    T += static_cast<size_t>(blockIdx.x) * cols;
    out += static_cast<size_t>(blockIdx.x) * cols;
    u16x4 xv[kGroups], tv[kGroups], wv[kGroups];
    #pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        const int c4 = lid + 64 * g;
        if (c4 < c4n) {
            xv[g] = *reinterpret_cast<const u16x4*>(H + 4 * c4);
            tv[g] = *reinterpret_cast<const u16x4*>(T + 4 * c4);
            wv[g] = *reinterpret_cast<const u16x4*>(w + 4 * c4);
        }
    }
    float acc = 0.0f;
    #pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        const int c4 = lid + 64 * g;
        if (c4 < c4n) {
            #pragma unroll
            for (int e = 0; e < 4; ++e) xv[g][e] = f_h(h_f(tv[g][e]) + h_f(xv[g][e]));
            *reinterpret_cast<u16x4*>(H + 4 * c4) = xv[g];
            const float v0 = h_f(xv[g][0]), v1 = h_f(xv[g][1]), v2 = h_f(xv[g][2]), v3 = h_f(xv[g][3]);
            float d = v0 * v0;
            d = fmaf(v1, v1, d);
            d = fmaf(v2, v2, d);
            d = fmaf(v3, v3, d);
            acc = acc + d;
        }
    }
    const float total = wave_tree_sum(acc);
    const float inv = rcp_rn(sqrtf(__fdiv_rn(total, static_cast<float>(cols)) + eps));
    #pragma unroll
    for (int g = 0; g < kGroups; ++g) {
        const int c4 = lid + 64 * g;
        if (c4 < c4n) {
            u16x4 o;
            #pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = f_h((h_f(xv[g][e]) * inv) * h_f(wv[g][e]));
            *reinterpret_cast<u16x4*>(out + 4 * c4) = o;
        }
    }
}

// Where the projection ahead of them was cut into slices of K, the launches that add the slices (wide::reduce_partials'
// operations: sums in index order, times the scale, rounded to fp16) also do what follows: the projection never goes
// through memory, and a launch of 2.5 to 5 us is saved.  300 Q4 tokens behind 900 2150 -> 1930 us, 2048 int8
// tokens 4075 -> 3970.
//
// The sums of four neighbouring columns at each of NP places.  A few rows come in up to 24 slices, and a launch is a chain
// of trips to memory: eight slices are asked for at a time, and a row is spread over as many threads as it has columns for
// (a wavefront per row, four slices at a time: 70 Q4 tokens 1743 us, 1403 like this, 1597 as launches of their own).
template <int NP>
__device__ __forceinline__ void sum_slices4(const float* const (&p)[NP], float4 (&a)[NP], int slices, long MN) {
    constexpr int kBatch = 8;
    #pragma unroll
    for (int q = 0; q < NP; ++q) a[q] = *reinterpret_cast<const float4*>(p[q]);
    for (int z = 1; z < slices; z += kBatch) {
        float4 b[kBatch][NP];
        #pragma unroll
        for (int u = 0; u < kBatch; ++u)
            #pragma unroll
            for (int q = 0; q < NP; ++q) b[u][q] = *reinterpret_cast<const float4*>(p[q] + (z + u < slices ? z + u : 0) * MN);
        #pragma unroll
        for (int u = 0; u < kBatch; ++u)
            if (z + u < slices) {
                #pragma unroll
                for (int q = 0; q < NP; ++q) { a[q].x += b[u][q].x; a[q].y += b[u][q].y; a[q].z += b[u][q].z; a[q].w += b[u][q].w; }
            }
    }
}

// The o or down projection's slices, then add_rmsnorm_rows_kernel: a block per row, a thread per four columns (`cols` a
// multiple of 4 up to 2048, 64 threads per 256 columns; 16-byte aligned sums, 8-byte aligned scales).  Lane l of
// wavefront g has the columns 4 l + 256 g .. that lane l of that kernel takes as its group g, and the squares are
// added in its order: over the groups, then over the lanes.
__global__ __launch_bounds__(512) void slices_add_rmsnorm_kernel(const float* __restrict__ sums, int slices, const uint16_t* __restrict__ scale,
                                                                 uint16_t* __restrict__ H, const uint16_t* __restrict__ w,
                                                                 uint16_t* __restrict__ out, int cols, float eps) {
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    __shared__ float sq[512];
    const int c4 = threadIdx.x, lane = threadIdx.x & 63, groups = blockDim.x >> 6;
    const bool has = c4 < cols >> 2;
    const long MN = static_cast<long>(gridDim.x) * cols;
    const int at = has ? 4 * c4 : 0;
    sums += static_cast<size_t>(blockIdx.x) * cols + at;
    H += static_cast<size_t>(blockIdx.x) * cols + at;
    out += static_cast<size_t>(blockIdx.x) * cols + at;
    u16x4 xv = *reinterpret_cast<const u16x4*>(H);
    const u16x4 wv = *reinterpret_cast<const u16x4*>(w + at);
    const u16x4 sv = scale ? *reinterpret_cast<const u16x4*>(scale + at) : u16x4{0x3c00, 0x3c00, 0x3c00, 0x3c00};   // 1.0
    float4 a[1];
    const float* const p[1] = {sums};
    sum_slices4(p, a, slices, MN);
    const float t[4] = {a[0].x, a[0].y, a[0].z, a[0].w};
    #pragma unroll
    for (int e = 0; e < 4; ++e) xv[e] = f_h(h_f(f_h(t[e] * h_f(sv[e]))) + h_f(xv[e]));
    const float v0 = h_f(xv[0]), v1 = h_f(xv[1]), v2 = h_f(xv[2]), v3 = h_f(xv[3]);
    float d = v0 * v0;
    d = fmaf(v1, v1, d);
    d = fmaf(v2, v2, d);
    d = fmaf(v3, v3, d);
    sq[threadIdx.x] = has ? d : 0.0f;                          // (a square is never -0: adding 0 changes nothing)
    if (has) *reinterpret_cast<u16x4*>(H) = xv;
    __syncthreads();
    float acc = 0.0f;
    for (int g = 0; g < groups; ++g) acc = acc + sq[64 * g + lane];
    const float total = wave_tree_sum(acc);
    const float inv = rcp_rn(sqrtf(__fdiv_rn(total, static_cast<float>(cols)) + eps));
    u16x4 o;
    #pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = f_h((h_f(xv[e]) * inv) * h_f(wv[e]));
    if (has) *reinterpret_cast<u16x4*>(out) = o;
}

// The stacked q | k | v projection's slices, then rope_rows_kernel: a block per row, four pairs of a head per thread
// (head widths that are multiples of 8, 16-byte aligned sums, 8-byte aligned scales and tables).
__global__ __launch_bounds__(256) void slices_rope_rows_kernel(const float* __restrict__ sums, int slices, const uint16_t* __restrict__ scale,
                                                               const uint16_t* __restrict__ bq, const uint16_t* __restrict__ bk,
                                                               const uint16_t* __restrict__ bv, const uint16_t* __restrict__ cosT,
                                                               const uint16_t* __restrict__ sinT, uint16_t* __restrict__ kc,
                                                               uint16_t* __restrict__ vc, uint16_t* __restrict__ QR, int pos0,
                                                               int n_heads, int n_kv_heads, int D) {
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    const int row = blockIdx.x, pos = pos0 + row, hd2 = D / 2, qd = n_heads * D, kvd = n_kv_heads * D, cols = qd + 2 * kvd;
    const long MN = static_cast<long>(gridDim.x) * cols;
    sums += static_cast<size_t>(row) * cols;
    auto finish4 = [&](const float4& a, int col, u16x4 bias) {      // four columns of the projection, with their bias
        const u16x4 sv = scale ? *reinterpret_cast<const u16x4*>(scale + col) : u16x4{0x3c00, 0x3c00, 0x3c00, 0x3c00};   // 1.0
        const float t[4] = {a.x, a.y, a.z, a.w};
        u16x4 v;
        #pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = f_h(h_f(f_h(t[e] * h_f(sv[e]))) + h_f(bias[e]));
        return v;
    };
    // (a bias starts anywhere: two bytes at a time)
    auto bias4 = [](const uint16_t* b) { return u16x4{b[0], b[1], b[2], b[3]}; };
    const int per_head = hd2 / 4, pairs = (n_heads + n_kv_heads) * per_head;
    for (int j = threadIdx.x; j < pairs + kvd / 4; j += blockDim.x) {
        if (j < pairs) {
            const int head = j / per_head, i = 4 * (j - head * per_head);
            const bool isq = head < n_heads;
            const int hh = isq ? head : head - n_heads;
            const uint16_t* bias = (isq ? bq : bk) + hh * D;
            uint16_t* dst = isq ? QR + static_cast<size_t>(row) * qd + hh * D : kc + static_cast<size_t>(pos) * kvd + hh * D;
            const u16x4 c = *reinterpret_cast<const u16x4*>(cosT + static_cast<size_t>(pos) * D + i);
            const u16x4 sn = *reinterpret_cast<const u16x4*>(sinT + static_cast<size_t>(pos) * D + i);
            const u16x4 b1 = bias4(bias + i), b2 = bias4(bias + i + hd2);
            const float* const p[2] = {sums + head * D + i, sums + head * D + i + hd2};
            float4 a[2];
            sum_slices4(p, a, slices, MN);
            const u16x4 v1 = finish4(a[0], head * D + i, b1), v2 = finish4(a[1], head * D + i + hd2, b2);
            u16x4 o1, o2;
            #pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x1 = h_f(v1[e]), x2 = h_f(v2[e]), ce = h_f(c[e]), se = h_f(sn[e]);
                o1[e] = f_h(fmaf(x1, ce, -(x2 * se)));
                o2[e] = f_h(fmaf(x2, ce, x1 * se));
            }
            *reinterpret_cast<u16x4*>(dst + i) = o1;
            *reinterpret_cast<u16x4*>(dst + i + hd2) = o2;
        } else {
            const int e0 = 4 * (j - pairs);
            const u16x4 b = bias4(bv + e0);
            const float* const p[1] = {sums + qd + kvd + e0};
            float4 a[1];
            sum_slices4(p, a, slices, MN);
            *reinterpret_cast<u16x4*>(vc + static_cast<size_t>(pos) * kvd + e0) = finish4(a[0], qd + kvd + e0, b);
        }
    }
}

// gate[i] = swiglu(gate[i], up[i]) over any number of elements, four per thread and step (n is a
// multiple of 4 and both arrays start at multiples of 8 bytes; swiglu_kernel's operations per element)
__global__ void swiglu_rows_kernel(uint16_t* __restrict__ gate, const uint16_t* __restrict__ up, long n) {
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    const long n4 = n >> 2;
    for (long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n4; i += static_cast<long>(gridDim.x) * blockDim.x) {
        u16x4 g4 = *reinterpret_cast<const u16x4*>(gate + 4 * i);
        const u16x4 u4 = *reinterpret_cast<const u16x4*>(up + 4 * i);
        #pragma unroll
        for (int e = 0; e < 4; ++e) {
            g4[e] = swiglu_h(g4[e], u4[e]);
        }
        *reinterpret_cast<u16x4*>(gate + 4 * i) = g4;
    }
}

// out[r][c] = swiglu of column c of a stacked gate | up projection ([M, 2 inter]), four columns per thread and step:
// `run` gate columns, the same up columns, and so on (run = inter: one matrix behind the other; run and inter are
// multiples of 4); swiglu_kernel's operations per element
__global__ void swiglu_stacked_kernel(const uint16_t* __restrict__ GU, uint16_t* __restrict__ out, int inter, int run, long n4) {
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    const int c4n = inter >> 2;
    for (long i = static_cast<long>(blockIdx.x) * blockDim.x + threadIdx.x; i < n4; i += static_cast<long>(gridDim.x) * blockDim.x) {
        const long r = i / c4n;
        const int c = static_cast<int>(i - r * c4n) * 4;
        const uint16_t* src = GU + r * 2 * inter + c + c / run * run;
        u16x4 g4 = *reinterpret_cast<const u16x4*>(src);
        const u16x4 u4 = *reinterpret_cast<const u16x4*>(src + run);
        #pragma unroll
        for (int e = 0; e < 4; ++e) g4[e] = swiglu_h(g4[e], u4[e]);
        *reinterpret_cast<u16x4*>(out + r * inter + c) = g4;
    }
}

// the state a prompt leaves behind for the launches that pick the next token: they read the
// last prompt position and advance it
__global__ void set_pos_kernel(State* st, int pos) { st->pos = pos; }

// Dynamic LDS of rope_attention_tiled<D>: q and v of the current position, exponentials and scores, eight maxima, tiles.
inline size_t tiled_attention_lds(int D, int max_pos) {
    return static_cast<size_t>(2 * D) * 2 + 6 * static_cast<size_t>(padded_positions(max_pos)) + 32 + tile_area(D);
}

__global__ void advance_kernel(State* st) {
    st->token = st->next;
    st->pos = st->pos + 1;
}

struct Decoder {
    mi_decoder_config c{};
    std::vector<const void*> in_norm, post_norm, bq, bk, bv, wq, wk, wv, wo, wgate, wup, wdown;
    const void* embed = nullptr;
    const void* final_norm = nullptr;
    const void* lm_head = nullptr;
    // device memory owned by the decoder
    uint16_t *kc = nullptr, *vc = nullptr, *cosT = nullptr, *sinT = nullptr;
    uint16_t *h = nullptr, *xn = nullptr, *q = nullptr, *k = nullptr, *v = nullptr, *attn = nullptr;
    uint16_t *qr = nullptr, *kr = nullptr, *vr = nullptr;      // q, k, v after bias and rotary embedding
    uint16_t* rope_now = nullptr;                              // cosines and sines of the current position (embed_kernel)
    uint16_t *gate = nullptr, *up = nullptr, *logits = nullptr;
    State* st = nullptr;
    std::vector<void*> owned;
    // rows of a prompt (mi_decoder_prefill): one allocation, made on the first prompt and again
    // only for a longer one
    void* prompt_mem = nullptr;
    int prompt_rows = 0;
    // q|k|v and gate|up of every layer as one matrix each (rows stacked, scales stacked), copies made
    // with the first prompt: a prompt's projections of one input are then one GEMM instead of three
    // or two.  An entry stays null where a layer's matrices are not of one kind.
    std::vector<void*> wqkv, wgu, stacked_mem;
    bool stacked_built = false;
    // attention with a head's keys split over blocks (mi_decoder_set_attention_splits): 0 = the reference-order launch
    int splits = 0;
    float* split_part = nullptr;                               // [n_heads][splits][head_dim + 2]
    StepRecordings<hipGraphExec_t> recordings;                 // a step's launches as graphs (mi_decoder_step)
    std::vector<WeightEntry> weights;                          // what the registry held for the decoder's weights ...
    uint64_t weights_epoch = 0;                                // ... at this registry_epoch()
    int weights_version = 0;                                   // raised whenever that turned out to have changed
};

template <typename T>
bool dev_alloc(Decoder* d, T** p, size_t bytes) {
    void* m = nullptr;
    if (!MI_HIP_OK(hipMalloc(&m, bytes ? bytes : 1))) return false;
    d->owned.push_back(m);
    *p = static_cast<T*>(m);
    return true;
}

uint16_t host_f16(float f) { return mi_f32_to_f16(f); }

}  // namespace
}  // namespace mi

using namespace mi;

extern "C" {

void* mi_decoder_create(const mi_decoder_config* cfg, const mi_decoder_weights* w) {
    if (!cfg || !w || !ensure_init()) return nullptr;
    const mi_decoder_config& c = *cfg;
    if (c.hidden <= 0 || c.inter <= 0 || c.n_heads <= 0 || c.n_kv_heads <= 0 || c.head_dim <= 0 || c.n_layers <= 0 ||
        c.vocab <= 0 || c.max_pos <= 0 || c.n_heads % c.n_kv_heads || c.head_dim % 4 || c.head_dim > 256 || c.max_pos > kMaxPositions) {
        MI_ERROR_FMT("mi_decoder_create: bad configuration");
        return nullptr;
    }
    auto* d = new Decoder;
    d->c = c;
    const int L = c.n_layers;
    auto take = [L](std::vector<const void*>& dst, const void* const* src) {
        dst.assign(src, src + L);
    };
    take(d->in_norm, w->in_norm); take(d->post_norm, w->post_norm);
    take(d->bq, w->bq); take(d->bk, w->bk); take(d->bv, w->bv);
    take(d->wq, w->wq); take(d->wk, w->wk); take(d->wv, w->wv); take(d->wo, w->wo);
    take(d->wgate, w->wgate); take(d->wup, w->wup); take(d->wdown, w->wdown);
    d->embed = w->embed; d->final_norm = w->final_norm; d->lm_head = w->lm_head;
    // (16 bytes: the GEMV launches that carry the norm in their prologue read it in 16-byte pieces)
    bool aligned = reinterpret_cast<uintptr_t>(w->final_norm) % 16 == 0;
    for (int l = 0; l < L; ++l)
        aligned = aligned && reinterpret_cast<uintptr_t>(w->in_norm[l]) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(w->post_norm[l]) % 16 == 0;
    if (!aligned || c.hidden % 4) {
        MI_ERROR_FMT("mi_decoder_create: norm weights must be 16-byte aligned and hidden a multiple of 4");
        delete d;
        return nullptr;
    }

    const int D = c.head_dim, kvd = c.n_kv_heads * D, qd = c.n_heads * D;
    if (D == 64 || D == 128) {
        // more than 64 KB of LDS per block has to be asked for once per kernel: the most any context length needs
        const size_t most = tiled_attention_lds(D, kMaxPositions);
        const void* kern = D == 64 ? reinterpret_cast<const void*>(rope_attention_tiled<64>)
                                   : reinterpret_cast<const void*>(rope_attention_tiled<128>);
        if (!MI_HIP_OK(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(most)))) {
            delete d;
            return nullptr;
        }
    }
    const size_t cache = static_cast<size_t>(L) * c.max_pos * kvd * 2;
    bool ok = dev_alloc(d, &d->kc, cache) && dev_alloc(d, &d->vc, cache) &&
              dev_alloc(d, &d->cosT, static_cast<size_t>(c.max_pos) * D * 2) &&
              dev_alloc(d, &d->sinT, static_cast<size_t>(c.max_pos) * D * 2) &&
              dev_alloc(d, &d->h, c.hidden * 2) && dev_alloc(d, &d->xn, c.hidden * 2) && dev_alloc(d, &d->q, qd * 2) &&
              dev_alloc(d, &d->k, kvd * 2) && dev_alloc(d, &d->v, kvd * 2) && dev_alloc(d, &d->qr, qd * 2) &&
              dev_alloc(d, &d->kr, kvd * 2) && dev_alloc(d, &d->vr, kvd * 2) && dev_alloc(d, &d->attn, qd * 2) &&
              dev_alloc(d, &d->gate, c.inter * 2) &&
              dev_alloc(d, &d->up, c.inter * 2) && dev_alloc(d, &d->logits, static_cast<size_t>(c.vocab) * 2) &&
              dev_alloc(d, &d->st, sizeof(State)) && dev_alloc(d, &d->rope_now, 2 * D * 2);
    if (ok) {
        // rotary tables, QW/src/layers/attention.cpp:133-172: cos/sin(t * theta^(-2i/D)), both halves alike
        std::vector<uint16_t> ct(static_cast<size_t>(c.max_pos) * D), stb(ct.size());
        for (int t = 0; t < c.max_pos; ++t)
            for (int i = 0; i < D / 2; ++i) {
                const float exponent = (2.0f * static_cast<float>(i)) / static_cast<float>(D);
                const float inv_freq = powf(c.rope_theta, -exponent);
                const float angle = static_cast<float>(t) * inv_freq;
                const uint16_t cv = host_f16(cosf(angle)), sv = host_f16(sinf(angle));
                ct[static_cast<size_t>(t) * D + i] = cv; ct[static_cast<size_t>(t) * D + i + D / 2] = cv;
                stb[static_cast<size_t>(t) * D + i] = sv; stb[static_cast<size_t>(t) * D + i + D / 2] = sv;
            }
        const State zero{0, 0, 0};
        ok = MI_HIP_OK(hipMemcpy(d->cosT, ct.data(), ct.size() * 2, hipMemcpyHostToDevice)) &&
             MI_HIP_OK(hipMemcpy(d->sinT, stb.data(), stb.size() * 2, hipMemcpyHostToDevice)) &&
             MI_HIP_OK(hipMemset(d->kc, 0, cache)) && MI_HIP_OK(hipMemset(d->vc, 0, cache)) &&
             MI_HIP_OK(hipMemcpy(d->st, &zero, sizeof zero, hipMemcpyHostToDevice));
    }
    if (!ok) {
        mi_decoder_destroy(d);
        return nullptr;
    }
    return d;
}

int mi_decoder_destroy(void* dec) {
    auto* d = static_cast<Decoder*>(dec);
    if (!d) return 1;
    for (void* p : d->owned) (void)hipFree(p);
    if (d->prompt_mem) (void)hipFree(d->prompt_mem);
    for (void* w : d->wqkv) if (w) mi_unregister_weight(w);
    for (void* w : d->wgu) if (w) mi_unregister_weight(w);
    for (void* p : d->stacked_mem) (void)hipFree(p);
    for (size_t i = 0; i < d->recordings.count(); ++i)
        (void)hipGraphExecDestroy(d->recordings.exec(i));      // (the frees above have waited for their last replay)
    delete d;
    return 1;
}

int mi_decoder_reset(void* dec, void* stream, int pos, int token) {
    auto* d = static_cast<Decoder*>(dec);
    if (!d || pos < 0 || pos >= d->c.max_pos || token < 0 || token >= d->c.vocab) {
        MI_ERROR_FMT("mi_decoder_reset: bad argument (pos=%d token=%d)", pos, token);
        return 0;
    }
    const State s{pos, token, token};
    auto st = static_cast<hipStream_t>(stream);
    return MI_HIP_OK(hipMemcpyAsync(d->st, &s, sizeof s, hipMemcpyHostToDevice, st)) && MI_HIP_OK(hipStreamSynchronize(st));
}

int mi_decoder_set_token(void* dec, void* stream, int token) {
    auto* d = static_cast<Decoder*>(dec);
    if (!d || token < 0 || token >= d->c.vocab) {
        MI_ERROR_FMT("mi_decoder_set_token: bad argument (token=%d)", token);
        return 0;
    }
    auto st = static_cast<hipStream_t>(stream);
    return MI_HIP_OK(hipMemcpyAsync(reinterpret_cast<char*>(d->st) + offsetof(State, token), &token, sizeof token,
                                    hipMemcpyHostToDevice, st)) && MI_HIP_OK(hipStreamSynchronize(st));
}

int mi_decoder_read(void* dec, void* stream, int* pos, int* token) {
    auto* d = static_cast<Decoder*>(dec);
    if (!d) return 0;
    State s{};
    auto st = static_cast<hipStream_t>(stream);
    if (!MI_HIP_OK(hipMemcpyAsync(&s, d->st, sizeof s, hipMemcpyDeviceToHost, st)) || !MI_HIP_OK(hipStreamSynchronize(st)))
        return 0;
    if (pos) *pos = s.pos;
    if (token) *token = s.token;
    return 1;
}

const void* mi_decoder_logits(void* dec) { return dec ? static_cast<Decoder*>(dec)->logits : nullptr; }

int mi_decoder_set_attention_splits(void* dec, int splits) {
    auto* d = static_cast<Decoder*>(dec);
    if (!d) return 0;
    if (splits <= 1) { d->splits = 0; return 1; }
    const int D = d->c.head_dim;
    if (splits > kMaxSplits || (D != 64 && D != 128)) {
        MI_ERROR_FMT("mi_decoder_set_attention_splits: %d splits at head_dim %d (2..%d, head_dim 64 or 128)", splits, D, kMaxSplits);
        return 0;
    }
    if (!d->split_part &&
        !dev_alloc(d, &d->split_part, static_cast<size_t>(d->c.n_heads) * kMaxSplits * (D + 2) * sizeof(float))) return 0;
    d->splits = splits;
    return 1;
}

const void* mi_decoder_buffer(void* dec, int which) {
    auto* d = static_cast<Decoder*>(dec);
    if (!d) return nullptr;
    switch (which) {
        case 0: return d->h;
        case 1: return d->qr;
        case 2: return d->kr;
        case 3: return d->vr;
        case 4: return d->attn;
        case 5: return d->gate;
        case 6: return d->cosT;
        case 7: return d->sinT;
        default: return nullptr;
    }
}

// The end of a step and of a prompt: final norm, lm_head, greedy token; the token moves into the
// device state and the position advances.  d->h holds the residual stream of the last position.
static int decoder_pick_next(Decoder* d, void* stream) {
    const mi_decoder_config& c = d->c;
    auto s = static_cast<hipStream_t>(stream);
    const int Hd = c.hidden;
    auto launched = [] { return MI_HIP_OK(hipGetLastError()); };
    // (the fused argmax's second launch also does what advance_kernel does)
    void* next = reinterpret_cast<char*>(d->st) + offsetof(State, next);
    bool fused = false;
    if (!linear_argmax(s, c.vocab, Hd, d->h, d->lm_head, d->logits, d->final_norm, c.rms_eps, 32, next, &d->st->token,
                       &d->st->pos, &fused))
        return 0;
    if (fused) return 1;
    {
        // Q4: the throughput GEMV has no norm in its prologue but takes the argmax in its epilogue, and
        // at the lm_head's size it is the faster one: norm as a launch of its own, then that kernel
        WeightKind kind = WK_F16;
        if (!fused_gemv_kind(d->lm_head, c.vocab, Hd, &kind)) return 0;
        if (kind == WK_Q4 || !gemv_takes_norm(kind, Hd)) {
            hipLaunchKernelGGL(rmsnorm_kernel, dim3(1), dim3(64), 0, s, d->h, static_cast<const uint16_t*>(d->final_norm), d->xn,
                               Hd, c.rms_eps);
            if (!launched()) return 0;
            if (!linear_argmax(s, c.vocab, Hd, d->xn, d->lm_head, d->logits, nullptr, 0.0f, 32, next, &d->st->token,
                               &d->st->pos, &fused))
                return 0;
            if (fused) return 1;
            if (!mi_linear(stream, 1, c.vocab, Hd, d->xn, d->lm_head, d->logits)) return 0;
            if (!mi_argmax_f16(stream, d->logits, c.vocab, 32, next)) return 0;
            hipLaunchKernelGGL(advance_kernel, dim3(1), dim3(1), 0, s, d->st);
            return launched() ? 1 : 0;
        }
    }
    {
        // the head's GEMV takes the norm in its prologue (checked above) but not the argmax in its epilogue
        const int N1[1] = {c.vocab};
        const void* const W1[1] = {d->lm_head};
        void* const y1[1] = {d->logits};
        if (!fused_gemv(s, 1, N1, Hd, d->h, W1, y1, d->final_norm, c.rms_eps, EPI_STORE)) return 0;
        if (!mi_argmax_f16(stream, d->logits, c.vocab, 32, next)) return 0;
    }
    hipLaunchKernelGGL(advance_kernel, dim3(1), dim3(1), 0, s, d->st);
    return launched() ? 1 : 0;
}

// The launches of a step, one by one.
// Projections of rmsnorm(h) * w.  The norm rides in the GEMV launch where the weights allow it
// (every wavefront repeats it while its first weights are in flight); otherwise it is a
// launch of its own into xn.
// With swiglu set (gate and up projection), y[0] receives swiglu(gate, up) and the SwiGLU
// rides in the same launch too where it can.
static bool norm_linear(Decoder* d, void* stream, const void* w, int n, const int* N, const void* const* W, void* const* y, bool swiglu) {
    auto s = static_cast<hipStream_t>(stream);
    const int Hd = d->c.hidden;
    const float eps = d->c.rms_eps;
    auto launched = [] { return MI_HIP_OK(hipGetLastError()); };
    WeightKind kind = WK_F16, k0 = WK_F16;
    bool fuse = true;
    for (int i = 0; i < n; ++i) {
        if (!fused_gemv_kind(W[i], N[i], Hd, &kind)) return false;
        if (i == 0) k0 = kind;
        fuse = fuse && kind == k0 && gemv_takes_norm(kind, Hd);
    }
    if (fuse && swiglu && gemv_takes_swiglu(k0, Hd)) return fused_gemv(s, n, N, Hd, d->h, W, y, w, eps, EPI_SWIGLU);
    if (fuse) {
        if (!fused_gemv(s, n, N, Hd, d->h, W, y, w, eps, EPI_STORE)) return false;
    } else {
        hipLaunchKernelGGL(rmsnorm_kernel, dim3(1), dim3(64), 0, s, d->h, static_cast<const uint16_t*>(w), d->xn, Hd,
                           eps);
        if (!launched()) return false;
        mi_linear_call calls[kMaxSegments];
        for (int i = 0; i < n; ++i) calls[i] = mi_linear_call{1, N[i], Hd, d->xn, W[i], y[i]};
        if (mi_linear_batch(stream, calls, n) != n) return false;
    }
    if (swiglu) {
        hipLaunchKernelGGL(swiglu_kernel, dim3((N[0] + 255) / 256), dim3(256), 0, s, static_cast<uint16_t*>(y[0]),
                           static_cast<const uint16_t*>(y[1]), N[0]);
        return launched();
    }
    return true;
}
// h = fp16(h + fp16(W x)): the projection and the element-wise add that follows it
// (QW/kernels/utils.cl element_add), one launch
static bool linear_into_h(Decoder* d, void* stream, int K, const void* x, const void* W) {
    const int Hd = d->c.hidden;
    const int N1[1] = {Hd};
    const void* const W1[1] = {W};
    void* const y1[1] = {d->h};
    return fused_gemv(static_cast<hipStream_t>(stream), 1, N1, K, x, W1, y1, nullptr, 0.0f, EPI_ADD);
}
// What a layer does behind its attention to the one row whose residual stream is in h: o, residual, norm, gate | up, SwiGLU, down, residual.
static bool finish_layer_of_one(Decoder* d, void* stream, int l, const void* attn) {
    const mi_decoder_config& c = d->c;
    if (!linear_into_h(d, stream, c.n_heads * c.head_dim, attn, d->wo[l])) return false;
    const int N2[2] = {c.inter, c.inter};
    const void* const W2[2] = {d->wgate[l], d->wup[l]};
    void* const y2[2] = {d->gate, d->up};
    return norm_linear(d, stream, d->post_norm[l], 2, N2, W2, y2, true) && linear_into_h(d, stream, c.inter, d->gate, d->wdown[l]);
}

static int enqueue_step(Decoder* d, void* stream) {
    const mi_decoder_config& c = d->c;
    auto s = static_cast<hipStream_t>(stream);
    const int Hd = c.hidden, D = c.head_dim, qd = c.n_heads * D, kvd = c.n_kv_heads * D;
    const float scale = 1.0f / sqrtf(static_cast<float>(D));
    auto launched = [] { return MI_HIP_OK(hipGetLastError()); };
    hipLaunchKernelGGL(embed_kernel, dim3(1), dim3(256), 0, s, static_cast<const uint16_t*>(d->embed), d->st, d->h, Hd, c.vocab,
                       d->cosT, d->sinT, d->rope_now, D, c.max_pos);
    if (!launched()) return 0;
    for (int l = 0; l < c.n_layers; ++l) {
        {
            const int N3[3] = {qd, kvd, kvd};
            const void* const W3[3] = {d->wq[l], d->wk[l], d->wv[l]};
            void* const y3[3] = {d->q, d->k, d->v};
            if (!norm_linear(d, stream, d->in_norm[l], 3, N3, W3, y3, false)) return 0;
        }
        uint16_t* kc = d->kc + static_cast<size_t>(l) * c.max_pos * kvd;
        uint16_t* vc = d->vc + static_cast<size_t>(l) * c.max_pos * kvd;
        const auto *bq = static_cast<const uint16_t*>(d->bq[l]), *bk = static_cast<const uint16_t*>(d->bk[l]),
                   *bv = static_cast<const uint16_t*>(d->bv[l]);
        if (d->splits > 1) {
            const int chunk_cap = ((c.max_pos + d->splits - 1) / d->splits + 3) & ~3;
            const size_t lds = split_attention_lds(D, chunk_cap);
            const dim3 grid(c.n_heads, d->splits);
            if (D == 64) {
                hipLaunchKernelGGL(attention_split_kernel<64>, grid, dim3(kSplitThreads), lds, s, kc, vc, d->st, c.n_heads,
                                   c.n_kv_heads, c.max_pos, scale, d->q, d->k, d->v, bq, bk, bv, d->rope_now, d->qr, d->kr,
                                   d->vr, d->split_part, chunk_cap);
                hipLaunchKernelGGL(attention_merge_kernel<64>, dim3(c.n_heads), dim3(64), 0, s, d->split_part, d->splits, d->attn);
            } else {
                hipLaunchKernelGGL(attention_split_kernel<128>, grid, dim3(kSplitThreads), lds, s, kc, vc, d->st, c.n_heads,
                                   c.n_kv_heads, c.max_pos, scale, d->q, d->k, d->v, bq, bk, bv, d->rope_now, d->qr, d->kr,
                                   d->vr, d->split_part, chunk_cap);
                hipLaunchKernelGGL(attention_merge_kernel<128>, dim3(c.n_heads), dim3(128), 0, s, d->split_part, d->splits, d->attn);
            }
        } else if (D == 64 || D == 128) {
            const size_t lds = tiled_attention_lds(D, c.max_pos);
            if (D == 64)
                hipLaunchKernelGGL(rope_attention_tiled<64>, dim3(c.n_heads), dim3(kAttnThreads), lds, s, kc, vc, d->st, c.n_heads,
                                   c.n_kv_heads, c.max_pos, scale, d->q, d->k, d->v, bq, bk, bv, d->rope_now, d->qr, d->kr,
                                   d->vr, d->attn);
            else
                hipLaunchKernelGGL(rope_attention_tiled<128>, dim3(c.n_heads), dim3(kAttnThreads), lds, s, kc, vc, d->st, c.n_heads,
                                   c.n_kv_heads, c.max_pos, scale, d->q, d->k, d->v, bq, bk, bv, d->rope_now, d->qr, d->kr,
                                   d->vr, d->attn);
        } else {
            // a whole number of wavefronts: the maximum's cross-lane steps read every lane of a wavefront
            const int at = ((D > 64 ? D : 64) + 63) & ~63;
            hipLaunchKernelGGL(rope_attention_kernel, dim3(c.n_heads), dim3(at), static_cast<size_t>(c.max_pos) * 6 + D * 6, s,
                               d->q, d->k, d->v, bq, bk, bv, d->cosT, d->sinT, kc, vc, d->qr, d->kr, d->vr, d->attn,
                               d->st, c.n_heads, c.n_kv_heads, D, c.max_pos, scale);
        }
        if (!launched()) return 0;
        if (!finish_layer_of_one(d, stream, l, d->attn)) return 0;
    }
    return decoder_pick_next(d, stream);
}

// A step is the same launches with the same arguments at every position, and a host that enqueues them one by one spends
// 3 to 4.5 us on each of 123 to 153 where the GPU needs less; as a recorded graph they cost one call of about 90 us and
// follow each other at 1.6 us instead of 2.5.  So the second of two steps in a row under the same circumstances is
// recorded (0.5 to 2 ms, once) and from then on replayed: a token of SmolLM2-135M in fp16, read back as it comes, 678 ->
// 582 us, of Qwen2.5-0.5B in int8 602 -> 482 us.
//
// It is recorded on a stream that nobody else knows (StandsFor), so that another thread that meanwhile waits for the step's
// stream, or asks about it, neither fails nor breaks into the recording.
//
// Circumstances: the stream and its workspace, the GEMV arithmetic, the attention's splits, and what the registry holds
// for the decoder's weights (looked up again whenever anything was registered or removed).  All else that the launches refer to
// belongs to the decoder.  Only on streams of mi_stream_create, which have a workspace to name; not while the caller
// records (the launches then go into its graph).
namespace {
struct StepApi {
    Decoder* d;
    hipStream_t s;
    int enqueue() { return enqueue_step(d, s); }
    int replay(hipGraphExec_t exec) { return MI_HIP_OK(hipGraphLaunch(exec, s)) ? 1 : 0; }
    // (mi_stream_destroy takes the workspace out of the table when the stream's work is over; a stream that has come
    //  since under the same address has another workspace, or one at the same address, and then the recording fits it)
    bool gone(const StepKey& k) { return own_stream_workspace(static_cast<hipStream_t>(const_cast<void*>(k.stream))) != k.workspace; }
    void drain() { (void)hipStreamSynchronize(s); }
    void drop(hipGraphExec_t exec) { (void)hipGraphExecDestroy(exec); }
    Recorded record(hipGraphExec_t* exec) {
        hipStream_t own = nullptr;
        if (hipStreamCreateWithFlags(&own, hipStreamNonBlocking) != hipSuccess) {
            (void)hipGetLastError();
            return Recorded::kRefused;
        }
        Recorded r = Recorded::kRefused;
        if (hipStreamBeginCapture(own, hipStreamCaptureModeThreadLocal) == hipSuccess) {
            hipGraph_t graph = nullptr;
            int launched = 0;
            {
                StandsFor same(own, s);
                launched = enqueue_step(d, own);
            }
            if (hipStreamEndCapture(own, &graph) == hipSuccess && graph) {
                if (!launched) r = Recorded::kLaunchFailed;
                else if (hipGraphInstantiate(exec, graph, nullptr, nullptr, 0) == hipSuccess) r = Recorded::kYes;
            }
            if (graph) (void)hipGraphDestroy(graph);
        }
        if (r != Recorded::kYes) (void)hipGetLastError();
        (void)hipStreamDestroy(own);
        return r;
    }
};
}  // namespace

int mi_decoder_step(void* dec, void* stream) {
    auto* d = static_cast<Decoder*>(dec);
    if (!d) return 0;
    auto s = static_cast<hipStream_t>(stream);
    void* ws = own_stream_workspace(s);
    if (!ws) return enqueue_step(d, stream);
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &status) != hipSuccess || status != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return enqueue_step(d, stream);
    }
    const uint64_t epoch = registry_epoch();
    if (d->weights.empty() || epoch != d->weights_epoch) {
        std::vector<WeightEntry> held;
        for (const auto* list : {&d->wq, &d->wk, &d->wv, &d->wo, &d->wgate, &d->wup, &d->wdown})
            for (const void* w : *list) held.push_back(weight_entry(w));
        held.push_back(weight_entry(d->lm_head));
        if (!(held == d->weights)) ++d->weights_version;
        d->weights.swap(held);
        d->weights_epoch = epoch;
    }
    StepKey now;
    now.stream = s;
    now.workspace = ws;
    now.gemv_mode = gemv_mode(s);
    now.splits = d->splits;
    now.weights = d->weights_version;
    StepApi api{d, s};
    return d->recordings.step(api, now);
}

// Rows of n matrices of one kind and K (and their scales) copied into one matrix, registered like
// its parts: one behind the other, or (run > 0; parts of one N, a multiple of run) `run` rows of each in turn.  Null
// when the parts are not of one kind or memory is short; *failed on a HIP error.
static void* stack_weights(Decoder* d, hipStream_t s, int n, const void* const* W, const int* N, int K, int run, bool* failed) {
    WeightKind kind = WK_F16, k0 = WK_F16;
    const void* scale[4] = {nullptr, nullptr, nullptr, nullptr};
    int total = 0;
    for (int i = 0; i < n; ++i) {
        if (!registered_weight(W[i], N[i], K, &kind, &scale[i])) return nullptr;
        if (i == 0) k0 = kind;
        if (kind != k0) return nullptr;
        total += N[i];
    }
    const size_t row = k0 == WK_F16 ? static_cast<size_t>(K) * 2 : k0 == WK_I8 ? static_cast<size_t>(K) : static_cast<size_t>(K) / 2;
    const size_t srow = k0 == WK_I8 ? 2 : k0 == WK_Q4 ? static_cast<size_t>(K / 32) * 2 : 0;
    void *w = nullptr, *sc = nullptr;
    if (hipMalloc(&w, row * total) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
    d->stacked_mem.push_back(w);
    if (srow) {
        if (hipMalloc(&sc, srow * total) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
        d->stacked_mem.push_back(sc);
    }
    size_t at = 0;
    for (int i = 0; i < n; ++i) {
        // pieces of `len` rows, n pieces apart in the stack
        const size_t len = run > 0 ? run : N[i], pieces = N[i] / len;
        auto append = [&](void* dst, const void* src, size_t row_bytes) {
            char* to = static_cast<char*>(dst) + at * row_bytes;
            return MI_HIP_OK(run > 0 ? hipMemcpy2DAsync(to, n * len * row_bytes, src, len * row_bytes, len * row_bytes, pieces,
                                                        hipMemcpyDeviceToDevice, s)
                                     : hipMemcpyAsync(to, src, len * row_bytes, hipMemcpyDeviceToDevice, s));
        };
        if (!append(w, W[i], row) || (srow && !append(sc, scale[i], srow))) { *failed = true; return nullptr; }
        at += len;
    }
    const int reg = k0 == WK_I8 ? mi_register_int8_weight(w, sc, total, K) : k0 == WK_Q4 ? mi_register_q4_weight(w, sc, total, K) : 1;
    return reg ? w : nullptr;
}

// Device rows for a prompt of up to M tokens (H, XN, T [M, hidden]; QKV [M, qd + 2 kvd]; QR, ATT
// [M, qd]; GU [M, 2 inter]; G2 [M, inter]; the token ids).  Grows only; growing waits for the
// stream (an earlier prompt may still be running in the old rows) and reallocates.
static bool ensure_prompt_rows(Decoder* d, hipStream_t s, int M) {
    if (M <= d->prompt_rows) return true;
    const mi_decoder_config& c = d->c;
    const size_t qd = static_cast<size_t>(c.n_heads) * c.head_dim, kvd = static_cast<size_t>(c.n_kv_heads) * c.head_dim;
    const size_t row_halves = 3 * static_cast<size_t>(c.hidden) + 3 * qd + 2 * kvd + 3 * static_cast<size_t>(c.inter);
    if (d->prompt_mem) {
        if (!MI_HIP_OK(hipStreamSynchronize(s))) return false;
        (void)hipFree(d->prompt_mem);
        d->prompt_mem = nullptr;
        d->prompt_rows = 0;
    }
    // every block starts at a multiple of 16 bytes: the row counts are padded to 8 halves per block
    const size_t bytes = (row_halves * M + 10 * 8) * 2 + static_cast<size_t>(M) * 4 + 16;
    if (!MI_HIP_OK(hipMalloc(&d->prompt_mem, bytes))) {
        d->prompt_mem = nullptr;
        return false;
    }
    d->prompt_rows = M;
    return true;
}

// Rows of the gate matrix, then of the up matrix, that take turns in their stack: 16, as launch_gemm_glu takes them,
// or, where the width is no multiple of 16, 0: one matrix behind the other.
static int glu_run(int inter) { return inter % 16 == 0 ? 16 : 0; }

// Every layer's q | k | v and gate | up matrices stacked into one registered matrix each, once.
static bool ensure_stacked(Decoder* d, hipStream_t s) {
    if (d->stacked_built) return true;
    const mi_decoder_config& c = d->c;
    const int Hd = c.hidden, qd = c.n_heads * c.head_dim, kvd = c.n_kv_heads * c.head_dim, I = c.inter;
    d->wqkv.assign(c.n_layers, nullptr);
    d->wgu.assign(c.n_layers, nullptr);
    bool failed = false;
    for (int l = 0; l < c.n_layers && !failed; ++l) {
        const void* const W3[3] = {d->wq[l], d->wk[l], d->wv[l]};
        const int N3[3] = {qd, kvd, kvd};
        d->wqkv[l] = stack_weights(d, s, 3, W3, N3, Hd, 0, &failed);
        const void* const W2[2] = {d->wgate[l], d->wup[l]};
        const int N2[2] = {I, I};
        if (!failed && I % 4 == 0) d->wgu[l] = stack_weights(d, s, 2, W2, N2, Hd, glu_run(I), &failed);
    }
    if (failed) {
        // nothing half-built stays behind: the next prompt starts over, and no registry entry
        // outlives the memory it names
        if (!MI_HIP_OK(hipStreamSynchronize(s))) return false;
        for (void* w : d->wqkv) if (w) mi_unregister_weight(w);
        for (void* w : d->wgu) if (w) mi_unregister_weight(w);
        for (void* p : d->stacked_mem) { mi_unregister_weight(p); (void)hipFree(p); }
        d->wqkv.clear(); d->wgu.clear(); d->stacked_mem.clear();
        return false;
    }
    d->stacked_built = true;
    return true;
}

int mi_decoder_reserve_prompt(void* dec, void* stream, int max_tokens) {
    auto* d = static_cast<Decoder*>(dec);
    if (!d || max_tokens < 1 || max_tokens > d->c.max_pos) {
        MI_ERROR_FMT("mi_decoder_reserve_prompt: bad argument (max_tokens=%d, max_pos=%d)", max_tokens, d ? d->c.max_pos : 0);
        return 0;
    }
    auto s = static_cast<hipStream_t>(stream);
    return ensure_prompt_rows(d, s, max_tokens) && ensure_stacked(d, s) && MI_HIP_OK(hipStreamSynchronize(s)) ? 1 : 0;
}

int mi_decoder_prefill(void* dec, void* stream, const int* tokens, int n_tokens, int pos0) {
    auto* d = static_cast<Decoder*>(dec);
    if (!d || !tokens || n_tokens < 1 || pos0 < 0 || static_cast<long>(pos0) + n_tokens > d->c.max_pos) {
        MI_ERROR_FMT("mi_decoder_prefill: bad argument (n_tokens=%d pos0=%d, max_pos=%d)", n_tokens, pos0,
                     d ? d->c.max_pos : 0);
        return 0;
    }
    const mi_decoder_config& c = d->c;
    auto s = static_cast<hipStream_t>(stream);
    const int M = n_tokens, Hd = c.hidden, D = c.head_dim, qd = c.n_heads * D, kvd = c.n_kv_heads * D, I = c.inter;
    const float scale = 1.0f / sqrtf(static_cast<float>(D));
    auto launched = [] { return MI_HIP_OK(hipGetLastError()); };

    // rows of the prompt (allocated here unless mi_decoder_reserve_prompt has made room already):
    // H, XN, T [M, hidden]; QKV [M, qd + 2 kvd] (q | k | v of a row side by side from the stacked
    // projection, or three blocks of their own); QR, ATT [M, qd]; GU [M, 2 inter] likewise; G2 [M, inter]; tokens
    if (!ensure_prompt_rows(d, s, M)) return 0;
    const int cap = d->prompt_rows;
    auto* base = static_cast<uint16_t*>(d->prompt_mem);
    size_t at = 0;
    auto carve = [&](size_t halves_per_row) {
        uint16_t* p = base + at;
        at += (halves_per_row * cap + 7) & ~static_cast<size_t>(7);
        return p;
    };
    uint16_t *H = carve(Hd), *XN = carve(Hd), *T = carve(Hd), *QKV = carve(qd + 2 * kvd), *QR = carve(qd), *ATT = carve(qd);
    uint16_t *GU = carve(2 * static_cast<size_t>(I)), *G2 = carve(I);
    int* tok = reinterpret_cast<int*>(base + at);

    if (!ensure_stacked(d, s)) return 0;
    if (!MI_HIP_OK(hipMemcpyAsync(tok, tokens, static_cast<size_t>(M) * 4, hipMemcpyHostToDevice, s))) return 0;
    hipLaunchKernelGGL(embed_rows_kernel, dim3(M), dim3(256), 0, s, static_cast<const uint16_t*>(d->embed), tok, H, Hd, c.vocab);
    if (!launched()) return 0;
    const long nH = static_cast<long>(M) * Hd, nI = static_cast<long>(M) * I;
    const unsigned gH = static_cast<unsigned>(nH / 256 + 1 < 4096 ? nH / 256 + 1 : 4096);
    const unsigned gI = static_cast<unsigned>(nI / 1024 + 1 < 8192 ? nI / 1024 + 1 : 8192);
    const size_t att_lds = static_cast<size_t>(D) * 2 * (1 + kPromptTile) + static_cast<size_t>(pos0 + M) * 6;
    if (att_lds > 65536) {
        // (the most any head width and context need, so that one call serves every later shape)
        if (!MI_ONCE_OK(MI_HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(attention_rows_kernel),
                                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                                      256 * 2 * (1 + kPromptTile) + kMaxPositions * 6))))
            return 0;
    }
    // A layer's attention runs on the matrix cores where any of its projections does.  Where all of them run as rows
    // of GEMV (mode 1; in the default mode a few rows, whose weights mi_linear keeps on the GEMV) the layer keeps
    // the reference's order, and a prompt of such layers leaves the cache rows and logits of single-token steps bit for bit.
    auto matrix_attention = [&](int l) {
        if (M < 2 || gemm_mode(s) == 1 || !attention_prompt_supported(D)) return false;
        auto gemm = [&](int N, int K, const void* x, const void* W) { return linear_takes_gemm(s, M, N, K, x, W); };
        return (d->wqkv[l] ? gemm(qd + 2 * kvd, Hd, XN, d->wqkv[l])
                           : gemm(qd, Hd, XN, d->wq[l]) || gemm(kvd, Hd, XN, d->wk[l]) || gemm(kvd, Hd, XN, d->wv[l])) ||
               gemm(Hd, qd, ATT, d->wo[l]) ||
               (d->wgu[l] ? gemm(2 * I, Hd, XN, d->wgu[l]) : gemm(I, Hd, XN, d->wgate[l]) || gemm(I, Hd, XN, d->wup[l])) ||
               gemm(Hd, I, d->wgu[l] ? G2 : GU, d->wdown[l]);
    };
    // one block per key/value head and row where the group's scores fit the LDS of a CU (160 KB, less
    // the kernel's few static bytes)
    constexpr size_t kGroupLdsMost = 160 * 1024 - 256;
    const int nrep = c.n_heads / c.n_kv_heads;
    const int grp_cap = (pos0 + M + 3) & ~3;             // rows of (query, key) entries start at multiples of 16 bytes
    const size_t grp_lds = group_attention_lds(D, nrep, grp_cap);
    const bool grouped = (D == 64 || D == 128) && nrep <= 8 && grp_lds <= kGroupLdsMost;
    if (grouped && grp_lds > 65536) {
        const void* kern = D == 64 ? reinterpret_cast<const void*>(attention_group_kernel<64>)
                                   : reinterpret_cast<const void*>(attention_group_kernel<128>);
        if (!MI_HIP_OK(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kGroupLdsMost)))) return 0;
    }
    // H += T, then XN = rmsnorm(H) * w: one launch where a row fits the fused kernel's registers
    const bool add_norm_fused = Hd % 4 == 0 && Hd <= 2048;
    auto add_then_norm = [&](const void* w) {
        if (add_norm_fused) {
            hipLaunchKernelGGL(add_rmsnorm_rows_kernel, dim3(M), dim3(64), 0, s, H, T, static_cast<const uint16_t*>(w), XN, Hd,
                               c.rms_eps);
            return launched();
        }
        hipLaunchKernelGGL(add_rows_kernel, dim3(gH), dim3(256), 0, s, H, T, nH);
        if (!launched()) return false;
        hipLaunchKernelGGL(rmsnorm_kernel, dim3(M), dim3(64), 0, s, H, static_cast<const uint16_t*>(w), XN, Hd, c.rms_eps);
        return launched();
    };
    // T = x W^T of the o or down projection, then add_then_norm; slices of K are added in the launch of the latter
    auto linear_add_norm = [&](int K, const uint16_t* x, const void* W, const void* w) {
        const float* sums = nullptr;
        const void* scales = nullptr;
        const int slices = add_norm_fused ? linear_slices(s, M, Hd, K, x, W, &sums, &scales) : 0;
        if (slices < 0) return false;
        if (!slices) return mi_linear(stream, M, Hd, K, x, W, T) && add_then_norm(w);
        hipLaunchKernelGGL(slices_add_rmsnorm_kernel, dim3(M), dim3((Hd + 255) / 256 * 64), 0, s, sums, slices,
                           static_cast<const uint16_t*>(scales), H, static_cast<const uint16_t*>(w), XN, Hd, c.rms_eps);
        return launched();
    };
    hipLaunchKernelGGL(rmsnorm_kernel, dim3(M), dim3(64), 0, s, H, static_cast<const uint16_t*>(d->in_norm[0]), XN, Hd,
                       c.rms_eps);
    if (!launched()) return 0;
    for (int l = 0; l < c.n_layers; ++l) {
        uint16_t* kc = d->kc + static_cast<size_t>(l) * c.max_pos * kvd;
        uint16_t* vc = d->vc + static_cast<size_t>(l) * c.max_pos * kvd;
        const auto *bq = static_cast<const uint16_t*>(d->bq[l]), *bk = static_cast<const uint16_t*>(d->bk[l]),
                   *bv = static_cast<const uint16_t*>(d->bv[l]);
        const float* sums = nullptr;
        const void* scales = nullptr;
        int slices = 0;
        if (d->wqkv[l] && D % 8 == 0) {
            slices = linear_slices(s, M, qd + 2 * kvd, Hd, XN, d->wqkv[l], &sums, &scales);
            if (slices < 0) return 0;
        }
        if (slices) {
            hipLaunchKernelGGL(slices_rope_rows_kernel, dim3(M), dim3(256), 0, s, sums, slices, static_cast<const uint16_t*>(scales), bq,
                               bk, bv, d->cosT, d->sinT, kc, vc, QR, pos0, c.n_heads, c.n_kv_heads, D);
        } else {
            uint16_t *Q = QKV, *Kp, *V;
            int ldq, ldkv;
            if (d->wqkv[l]) {
                if (!mi_linear(stream, M, qd + 2 * kvd, Hd, XN, d->wqkv[l], QKV)) return 0;
                Kp = QKV + qd;
                V = Kp + kvd;
                ldq = ldkv = qd + 2 * kvd;
            } else {
                Kp = QKV + static_cast<size_t>(cap) * qd;
                V = Kp + static_cast<size_t>(cap) * kvd;
                ldq = qd;
                ldkv = kvd;
                if (!mi_linear(stream, M, qd, Hd, XN, d->wq[l], Q) || !mi_linear(stream, M, kvd, Hd, XN, d->wk[l], Kp) ||
                    !mi_linear(stream, M, kvd, Hd, XN, d->wv[l], V))
                    return 0;
            }
            hipLaunchKernelGGL(rope_rows_kernel, dim3(M), dim3(256), 0, s, Q, Kp, V, bq, bk, bv, d->cosT, d->sinT, kc, vc, QR, pos0,
                               c.n_heads, c.n_kv_heads, D, ldq, ldkv);
        }
        if (!launched()) return 0;
        // Only the last position picks a token: behind its cache rows the last layer goes on with that row alone, which
        // becomes the single-token state (2048 int8 tokens of 0.5B 3791 -> 3702 us, 300 Q4 tokens behind 900 1682 -> 1658).
        const bool one = l + 1 == c.n_layers;
        const int rows = one ? 1 : M, first = M - rows;
        const uint16_t* q_rows = QR + static_cast<size_t>(first) * qd;
        if (matrix_attention(l)) {
            if (!launch_attention_prompt(s, q_rows, kc, vc, ATT, rows, pos0 + first, c.n_heads, c.n_kv_heads, D, scale)) return 0;
        } else if (grouped && D == 64)
            hipLaunchKernelGGL(attention_group_kernel<64>, dim3(c.n_kv_heads, rows), dim3(256), grp_lds, s, q_rows, kc, vc, ATT,
                               pos0 + first, grp_cap, c.n_heads, c.n_kv_heads, scale);
        else if (grouped)
            hipLaunchKernelGGL(attention_group_kernel<128>, dim3(c.n_kv_heads, rows), dim3(256), grp_lds, s, q_rows, kc, vc, ATT,
                               pos0 + first, grp_cap, c.n_heads, c.n_kv_heads, scale);
        else
            hipLaunchKernelGGL(attention_rows_kernel, dim3(c.n_heads, rows), dim3(256), att_lds, s, q_rows, kc, vc, ATT, pos0 + first,
                               pos0 + M, c.n_heads, c.n_kv_heads, D, scale);
        if (!launched()) return 0;
        if (one) {
            if (!MI_HIP_OK(hipMemcpyAsync(d->h, H + static_cast<size_t>(M - 1) * Hd, static_cast<size_t>(Hd) * 2,
                                          hipMemcpyDeviceToDevice, s)) ||
                !finish_layer_of_one(d, stream, l, ATT))
                return 0;
            break;
        }
        if (!linear_add_norm(qd, ATT, d->wo[l], d->post_norm[l])) return 0;
        const uint16_t* act;                      // swiglu(gate, up), [M, inter]
        if (d->wgu[l]) {
            const int run = glu_run(I), fused = run ? linear_glu(s, M, 2 * I, Hd, XN, d->wgu[l], G2) : 0;
            if (fused < 0 || (!fused && !mi_linear(stream, M, 2 * I, Hd, XN, d->wgu[l], GU))) return 0;
            if (!fused)
                hipLaunchKernelGGL(swiglu_stacked_kernel, dim3(gI), dim3(256), 0, s, GU, G2, I, run ? run : I, nI / 4);
            act = G2;
        } else {
            uint16_t *G = GU, *U = GU + static_cast<size_t>(cap) * I;
            if (!mi_linear(stream, M, I, Hd, XN, d->wgate[l], G) || !mi_linear(stream, M, I, Hd, XN, d->wup[l], U)) return 0;
            if (I % 4 == 0) {
                hipLaunchKernelGGL(swiglu_rows_kernel, dim3(gI), dim3(256), 0, s, G, U, nI);
            } else {
                if (nI > 2147483647L) return 0;
                hipLaunchKernelGGL(swiglu_kernel, dim3(gI), dim3(256), 0, s, G, U, static_cast<int>(nI));
            }
            act = G;
        }
        if (!launched()) return 0;
        if (!linear_add_norm(I, act, d->wdown[l], d->in_norm[l + 1])) return 0;         // the next layer's input norm rides along
    }
    hipLaunchKernelGGL(set_pos_kernel, dim3(1), dim3(1), 0, s, d->st, pos0 + M - 1);
    if (!launched()) return 0;
    return decoder_pick_next(d, stream);
}


}  // extern "C"

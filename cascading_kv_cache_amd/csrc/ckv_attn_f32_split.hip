// float32 attention of cached chunks on the bfloat16 matrix cores, head_dim 64 and 128: a float32 operand of ordinary size is the
// exact sum of three bfloat16 planes (high, middle, low), and a product is the six of its nine plane products that float32 can tell from
// zero (the three left out are below 2^-25 of it); all of them are exact and summed in float32.
//
// The low planes of values below 2^-109 would be smaller than any bfloat16 (at 2^-122 a value would keep 12 bits), and those of the largest
// and of infinite values are no numbers.  A part of a tile with a value that is not zero and below 2^-100, or past 3.38e38, is
// staged raw: its bits, eleven to a plane, as finite bfloat16 numbers.  Blocks of keys that meet a raw part, and those in which a row has
// a probability below 2^-100 of its largest (2^-126 for the score sums, which have no planes of it), are worked out by the
// float32 instruction from the operands put together, with exponentials down to the smallest subnormal number.  What that costs
// the others (32 heads x 256 rows x 516 + 256 keys x 128): half a microsecond each of the forward kernel's 26 and the score kernel's 16.
//
// 32 heads x 256 rows x 516 + 256 keys x 128, us, on the float32 instruction and now: forward 44.0 -> 26.5 (1.2 MB of operands a
// workgroup from the L2, 16 TB/s in all, and the first pass through the loop's instructions), scores 29.8 -> 16.6 (products and vector
// work one behind the other: exponentials beside the next tile's products measured the same), staging 10.1 -> 15.1 (5.5 of it stores:
// 1.5 times the bytes); a whole call with its update 97.3 -> 70.9 (4.5 of it by a launch less in the update), 512 rows x
// 2052 + 512 keys 207 + 147 + 15 -> 128 + 85 + 19.  Relative error against float64, 2-norm: output
// 4.4e-7 -> 2.3e-7, new scores 1.7e-7 -> 0.5e-7 (a row's largest logit and sum reach the scores apart, not as one logarithm).
//
// Why: the float32 instruction (32x32x2) takes 64 cycles for 2 terms of a sum and vector instructions do not run beside
// it; six of the bfloat16 one (32x32x16) take 192 for 16, and they do.  The planes are made once per key and query by the staging
// kernel, which puts them in the order in which the matrix instructions take them (a piece of 1 KiB: 16 bytes a lane), so that
// the kernels behind it load whole cache lines straight into operand registers.
//
//   staging  a wavefront per 32 rows and 16 + 16 dims that rotate together, or per 16 keys' values (transposed, keys in the order
//            in which S^T leaves them in its registers), a workgroup's four at a time.
//   forward  one workgroup = one kv head x 32 (position, head) rows; its eight wavefronts take the 32-key blocks in turn, each with
//            an online softmax of its own, and merge at the end through LDS.  S^T = K Q^T keeps a query in one lane pair, and
//            registers 8 ks .. 8 ks + 7 of S^T, split, are the B operand of step ks of O^T += V^T P^T.
//   colsum   one workgroup = one head x four blocks of 32 keys, held in registers; two streams of its wavefronts take the 32-row
//            query tiles, which come through LDS, in turn.  One block a workgroup where four make too few workgroups, four
//            streams then, each with its queries straight from memory.
//
// Zero times infinity is NaN, here also where a plane of a finite operand is zero: a block whose logits are not all finite
// is worked out by the float32 instruction too, and a wavefront whose accumulators are not finite goes over its keys once
// more, finite values through the matrix pipe and the others where their probability is above zero.
#include "ckv_attn_internal.h"

#include <type_traits>

namespace ckv {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kRows = 32;      // query rows of a forward workgroup
constexpr int kKeys = 32;      // keys of a block
constexpr int kFwdWaves = 8;
constexpr int kColSums = 4;    // partial sums of a key, one per query tile mod 4
constexpr int kPlanes = 3;
template <int kGroups>
struct Col {
    static constexpr int kStreams = kGroups == 1 ? 4 : 2, kWaves = kGroups * kStreams, kBlockKeys = kGroups * kKeys;
    static constexpr int kAcc = kColSums / kStreams;   // partial sums of a wavefront
    static constexpr bool kThroughLds = kGroups > 1;   // more than one wavefront takes a tile
};

template <int D>
struct Geo {
    static constexpr int kSteps = D / 16;   // of a contraction over the head dim
    static constexpr int kDB = D / 32;      // accumulators of 32 dims
    static constexpr int kPitch = D + 4;    // floats of a row in the merge area
    static constexpr int kPieces = kPlanes * kSteps;             // of 32 rows, or of 32 keys' values
    static constexpr int kTileVec = kPieces * CKV_WAVE, kTile = kTileVec * 16;
    static constexpr int kFwdLds = kTile + kFwdWaves * kRows * kPitch * 4 + 2 * kFwdWaves * kRows * 4;
    static_assert(kFwdLds <= 160 * 1024, "a compute unit's LDS");
    // A tile's word of F32Planes::odd_*: a field for each wavefront that stages a part of the tile, not zero where its part is raw.
    static constexpr int kParts = kSteps / 2, kField = 32 / kParts;   // queries and keys: steps c and c + kParts
    typedef std::conditional_t<kField == 8, uint8_t, uint16_t> Field;
    __device__ static bool raw_step(uint32_t word, int c) { return (word >> (c % kParts * kField) & 1u) != 0u; }
    __device__ static bool raw_values(uint32_t word, int ks) { return (word >> (16 * ks) & 1u) != 0u; }
};

template <int N>
struct Vec {
    float v[N];
};

__device__ inline f32x16 mma(uint4 a, uint4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ inline f32x16 mma32(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }

__device__ inline f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; i++) z[i] = 0.f;
    return z;
}

// matrix row of accumulator register v in lane half `half`
__device__ inline int acc_row(int v, int half) { return 8 * (v >> 2) + 4 * half + (v & 3); }

__device__ inline uint32_t pack2(float a, float b) {
    const f32x2 f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}
__device__ inline float low_of(uint32_t w) { return __uint_as_float(w << 16); }
__device__ inline float high_of(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// Two values' planes.  Rounding to bfloat16 leaves a rest of 16 bits and that one of 8, all of them exact.
__device__ inline void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = pack2(a, b);
    const float ra = a - low_of(h), rb = b - high_of(h);
    m = pack2(ra, rb);
    l = pack2(ra - low_of(m), rb - high_of(m));
}
// Does everything that it was shown fit the planes to the last bit, with room below for the lowest one?  The matrix instruction takes
// subnormal operands as they are, but the low plane of a value below 2^-109 would need smaller ones still, and the largest
// finite values round to infinity.  A NaN is NaN in the high plane.
struct Range {
    float top = 0.f;
    uint32_t low = ~0u;   // twice the bits (no sign), less one: zero comes last
    __device__ inline void show(float x) {
        top = fmaxf(top, fabsf(x));
        const uint32_t twice = (__float_as_uint(x) << 1) - 1u;
        low = twice < low ? twice : low;
    }
    __device__ inline bool fits() const { return top < 3.38e38f && low >= 2u * 0x0d800000u - 1u; }   // bits of 2^-100
};
// Eleven bits of a value that the planes do not take, as a finite bfloat16: sign, lower exponent and mantissa, the upper exponent being
// 01111.  Three of them are the 32.
__device__ inline uint32_t raw_word(uint32_t f) { return (f & 0x400u) << 5 | 0x3c00u | (f & 0x3ffu); }
__device__ inline uint32_t raw_bits(uint32_t w) { return (w >> 5 & 0x400u) | (w & 0x3ffu); }
// eight values' pieces of the three planes; `raw` (one for the wavefront): of their bits
__device__ inline void split8(const float (&x)[8], bool raw, uint4 (&out)[kPlanes]) {
    uint32_t w[kPlanes][4];
    if (__builtin_expect(!raw, 1)) {
#pragma unroll
        for (int i = 0; i < 4; i++) split2(x[2 * i], x[2 * i + 1], w[0][i], w[1][i], w[2][i]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t a = __float_as_uint(x[2 * i]), b = __float_as_uint(x[2 * i + 1]);
            w[0][i] = raw_word(a >> 21) | raw_word(b >> 21) << 16;
            w[1][i] = raw_word(a >> 10) | raw_word(b >> 10) << 16;
            w[2][i] = raw_word(a & 0x3ffu) | raw_word(b & 0x3ffu) << 16;
        }
    }
#pragma unroll
    for (int pl = 0; pl < kPlanes; pl++) out[pl] = make_uint4(w[pl][0], w[pl][1], w[pl][2], w[pl][3]);
}

__device__ inline uint32_t word_of(const uint4& x, int i) { return i == 0 ? x.x : i == 1 ? x.y : i == 2 ? x.z : x.w; }
// element e of three planes' pieces (raw: of its bits), put together
__device__ inline float whole_of(const uint4 (&x)[kPlanes], int e, bool raw) {
    const uint32_t h = word_of(x[0], e >> 1), m = word_of(x[1], e >> 1), l = word_of(x[2], e >> 1);
    const int at = 16 * (e & 1);
    const uint32_t bits = raw_bits(h >> at) << 21 | raw_bits(m >> at) << 10 | raw_bits(l >> at);
    const float sum = e & 1 ? high_of(h) + (high_of(m) + high_of(l)) : low_of(h) + (low_of(m) + low_of(l));
    const uint32_t pick = raw ? ~0u : 0u;   // no branch: there are sixteen of these behind each other
    return __uint_as_float((bits & pick) | (__float_as_uint(sum) & ~pick));
}

// the plane products of one step, the small ones in an accumulator of their own
__device__ inline void mma_planes(const uint4 (&a)[kPlanes], const uint4 (&b)[kPlanes], f32x16& large, f32x16& small) {
    small = mma(a[2], b[0], small);
    small = mma(a[0], b[2], small);
    small = mma(a[1], b[1], small);
    small = mma(a[1], b[0], small);
    small = mma(a[0], b[1], small);
    large = mma(a[0], b[0], large);
}

// Logits, their maxima and the normalisers between the kernels are to the base 2: the staged queries carry log2 e.  (So logits past 2.35e38
// overflow, of the 3.4e38 that float32 holds.)
__device__ inline float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }   // results below the smallest normal number are zero
constexpr float kFaint = -100.f;   // a probability's logit below the largest, from which on its planes would lose bits

// a word that no kernel of this launch writes, at a uniform index
__device__ inline uint32_t uniform_word(const uint32_t* words, int i) {
    typedef const __attribute__((address_space(4))) uint32_t* constant_words;
    return ((constant_words)(uintptr_t)words)[__builtin_amdgcn_readfirstlane(i)];
}

// Where key n of a (b, kv head) lies; behind the last one, the last one.
struct KeySource {
    const float *k, *v;
    int64_t sd, shift;
    const int64_t* pos;
    const uint8_t* mask;   // null: a key of the chunk
    __device__ KeySource(const ckv_attn_args& a, int64_t b, int64_t h, int n) {
        const int NS = (int)a.num_sink, Nc = NS + (int)a.S, last = Nc + (int)a.Q - 1;
        if (n > last) n = last;
        if (n < NS) {
            const int64_t at = b * a.sink_stride[0] + h * a.sink_stride[1] + n * a.sink_stride[2];
            k = (const float*)a.sink_k + at;
            v = (const float*)a.sink_v + at;
            sd = a.sink_stride[3];
            pos = a.sink_pos + b * a.sink_pos_stride[0] + h * a.sink_pos_stride[1] + n;
            shift = 0;
            mask = a.sink_mask + n;
        } else if (n < Nc) {
            const int64_t slot = n - NS, at = b * a.cache_stride[0] + h * a.cache_stride[1] + slot * a.cache_stride[2];
            k = (const float*)a.cache_k + at;
            v = (const float*)a.cache_v + at;
            sd = a.cache_stride[3];
            pos = a.pos + b * a.pos_stride[0] + h * a.pos_stride[1] + slot;
            shift = a.pos_shift;
            mask = a.mask + slot;
        } else {
            const int64_t m = n - Nc, at = b * a.kv_new_stride[0] + h * a.kv_new_stride[1] + m * a.kv_new_stride[2];
            k = (const float*)a.k_new + at;
            v = (const float*)a.v_new + at;
            sd = a.kv_new_stride[3];
            pos = a.q_pos + m;
            shift = 0;
            mask = nullptr;
        }
    }
};

struct F32Stage {
    ckv_attn_args a;
    uint4 *q, *k, *v;       // see F32Planes
    uint32_t *vis, *odd_q;
    uint2* odd_kv;
    float *w_ema, *w_new;   // the weights of the score sums, or null
    int w_items;            // wavefronts with weights; those behind them keep scores
    KeptScores kept;
    float post_q, post_k;   // what rotated queries and keys are multiplied by
    int nblk, q_tiles;
    int k_items, q_items, v_items, vis_items;   // wavefronts
    bool vec;               // rows of sinks, cache, chunk and queries are 16-byte pieces
};

template <int kN>
__device__ inline void load_row(const float* src, int64_t sd, bool vec, float (&x)[kN]) {   // kN elements, in pieces of up to 16 bytes
    constexpr int kPer = kN < 4 ? kN : 4;
    if (vec) {
#pragma unroll
        for (int i = 0; i < kN; i += kPer) {
            const Vec<kPer> t = *reinterpret_cast<const Vec<kPer>*>(__builtin_assume_aligned(src + i, kPer * 4));
#pragma unroll
            for (int j = 0; j < kPer; j++) x[i + j] = t.v[j];
        }
    } else {
#pragma unroll
        for (int i = 0; i < kN; i++) x[i] = src[i * sd];
    }
}

// Bound by its trips to memory and the sines and cosines, one of each a rotation pair and row.
template <int D>
__global__ void __launch_bounds__(256) stage_f32_kernel(F32Stage p) {
    using G_ = Geo<D>;
    constexpr int kPairSteps = G_::kSteps / 2;
    const ckv_attn_args& a = p.a;
    const int lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
    int id = (int)(blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6));
    const int NS = (int)a.num_sink, S = (int)a.S, Q = (int)a.Q, Nc = NS + S, N = Nc + Q, H = (int)a.H, KVH = (int)a.KVH;
    if (id < p.k_items + p.q_items) {
        const bool key = id < p.k_items;
        if (!key) id -= p.k_items;
        const int c = id % kPairSteps, tile = id / kPairSteps, tiles = key ? p.nblk : p.q_tiles;
        const int unit = tile / tiles, n = (tile - unit * tiles) * 32 + col, heads = key ? KVH : H;
        const int64_t b = unit / heads, h = unit - (int)b * heads;
        // what a wavefront needs is requested in one go, from in-bounds addresses whatever becomes of it: a load behind a branch is a
        // trip to memory of its own
        const float* src;
        const int64_t* at;
        int64_t sd, shift = 0;
        if (key) {
            const KeySource from(a, b, h, n);
            src = from.k;
            sd = from.sd;
            at = from.pos;
            shift = from.shift;
        } else {
            const int m = n < Q ? n : Q - 1;
            src = (const float*)a.q + b * a.q_stride[0] + h * a.q_stride[1] + m * a.q_stride[2];
            sd = a.q_stride[3];
            at = a.q_pos + m;
        }
        const bool there = n < (key ? N : Q);
        const int j0 = 16 * c + 8 * half;
        float x1[8], x2[8], freq[8];
        const int64_t stored_pos = *at;
#pragma unroll
        for (int e = 0; e < 8; e++) freq[e] = a.inv_freq ? a.inv_freq[j0 + e] : 0.f;
        load_row<8>(src + j0 * sd, sd, p.vec, x1);
        load_row<8>(src + (j0 + D / 2) * sd, sd, p.vec, x2);
        const float pos = (float)(stored_pos + shift), post = key ? p.post_k : p.post_q;
        // Sines and cosines in a loop that is not unrolled, by way of LDS: a range reduction is long, and eight of them one behind
        // the other are fetched instruction by instruction by a wavefront that runs them once.
        __shared__ float2 parked[4][8][CKV_WAVE];
        float2* mine = &parked[threadIdx.x >> 6][0][lane];
#pragma unroll
        for (int e = 0; e < 8; e++) mine[e * CKV_WAVE].x = freq[e];
#pragma unroll 2
        for (int e = 0; e < 8; e++) {
            const float f = a.inv_freq ? mine[e * CKV_WAVE].x : 1.0f / powf(a.rope_theta, (float)(2 * (j0 + e)) / (float)D);
            float sn, cs;
            sincosf(__fmul_rn(pos, f), &sn, &cs);
            mine[e * CKV_WAVE] = make_float2(cs, sn);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) {   // cascade_attention.py:31-35 in float32: each product rounded, then the sum, then the scale
            const float cs = mine[e * CKV_WAVE].x, sn = mine[e * CKV_WAVE].y;
            const float r1 = __fadd_rn(__fmul_rn(x1[e], cs), __fmul_rn(-x2[e], sn)), r2 = __fadd_rn(__fmul_rn(x2[e], cs), __fmul_rn(x1[e], sn));
            x1[e] = there ? __fmul_rn(r1, post) : 0.f;
            x2[e] = there ? __fmul_rn(r2, post) : 0.f;
        }
        uint4* dst = (key ? p.k : p.q) + (int64_t)tile * G_::kTileVec + lane;
        Range range;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            range.show(x1[e]);
            range.show(x2[e]);
        }
        const bool raw = __ballot(!range.fits()) != 0ull;
        uint4 w1[kPlanes], w2[kPlanes];
        split8(x1, raw, w1);
        split8(x2, raw, w2);
        typedef typename G_::Field Field;
        if (lane == 0) reinterpret_cast<Field*>(key ? &p.odd_kv[tile].x : &p.odd_q[tile])[c] = raw ? 1 : 0;
#pragma unroll
        for (int pl = 0; pl < kPlanes; pl++) {
            dst[(c * kPlanes + pl) * CKV_WAVE] = w1[pl];
            dst[((c + kPairSteps) * kPlanes + pl) * CKV_WAVE] = w2[pl];
        }
        return;
    }
    id -= p.k_items + p.q_items;
    if (id < p.v_items) {
        constexpr int DB = G_::kDB;
        const int ks = id & 1, tile = id >> 1, unit = tile / p.nblk, blk = tile - unit * p.nblk;
        const int64_t b = unit / KVH, h = unit - (int)b * KVH;
        // each lane finds one key, the others take its address and whether it is seen from there
        const int n = blk * kKeys + 16 * ks + (lane & 15);
        const KeySource own(a, b, h, n);
        const uint8_t masked = *(own.mask ? own.mask : reinterpret_cast<const uint8_t*>(own.v));
        const uint64_t at = reinterpret_cast<uint64_t>(own.v);
        const int state = (own.mask && masked) || n >= N ? 0 : 1;
        float x[DB][8];
        int seen[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int from = 8 * (e >> 2) + 4 * half + (e & 3);
            const uint64_t row = (uint64_t)(uint32_t)__shfl((int)(at >> 32), from) << 32 | (uint32_t)__shfl((int)at, from);
            const int64_t sd = p.vec ? 1 : (int64_t)__shfl((long long)own.sd, from);
            seen[e] = __shfl(state, from);
            float t[DB];
            load_row<DB>(reinterpret_cast<const float*>(row) + DB * col * sd, sd, p.vec, t);
#pragma unroll
            for (int db = 0; db < DB; db++) x[db][e] = t[db];
        }
        uint4* dst = p.v + (int64_t)tile * G_::kTileVec + lane;
        Range range;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                x[db][e] = seen[e] ? x[db][e] : 0.f;   // a key that nobody sees may hold anything
                range.show(x[db][e]);
            }
        const bool raw = __ballot(!range.fits()) != 0ull;
        if (lane == 0) reinterpret_cast<uint16_t*>(&p.odd_kv[tile].y)[ks] = raw ? 1 : 0;
#pragma unroll
        for (int db = 0; db < DB; db++) {
            uint4 w[kPlanes];
            split8(x[db], raw, w);
#pragma unroll
            for (int pl = 0; pl < kPlanes; pl++) dst[((db * 2 + ks) * kPlanes + pl) * CKV_WAVE] = w[pl];
        }
        return;
    }
    id -= p.v_items;
    if (id < p.vis_items) {   // a bit per key of the blocks that is there and not masked
        const int n = id * 64 + lane;
        const bool seen = n < NS ? !a.sink_mask[n] : n < Nc ? !a.mask[n - NS] : n < N;
        const unsigned long long all = __builtin_amdgcn_ballot_w64(seen);
        if (col == 0 && 2 * id + half < p.nblk) p.vis[2 * id + half] = (uint32_t)(half ? all >> 32 : all);
        return;
    }
    id -= p.vis_items;
    if (id < p.w_items) weights_at<float>(p.w_ema, p.w_new, Q, a.beta, (int64_t)id * 64 + lane);
    else if (p.kept.src) keep_scores<float, CKV_WAVE>(p.kept, id - p.w_items, lane);
}

struct F32Fwd {
    CoreProblem c;   // out, lse and sizes; its q, k and v are not read
    F32Planes f;
    int n_split;     // shares of the key blocks per row tile: few rows would leave most of the chip idle
    float* part_o;   // (n_split, B*H*Q, D) and
    float2* part_l;  // (n_split, B*H*Q): every share normalised by its own sum; its largest logit, -inf for none, and that sum
    float2* norm;    // (B*H*Q): a row's largest logit and one over its sum.  Apart, as the logarithm of both together is rounded
                     // coarser than a probability; c.lse, where it is wanted, has that (natural)
};

__device__ inline void write_normaliser(const F32Fwd& f, int64_t row, float M, float L) {
    f.norm[row] = make_float2(M, 1.f / L);
    if (f.c.lse) f.c.lse[row] = (M + log2f(L)) * 0.693147180559945309f;
}

template <int D>
__global__ void __launch_bounds__(kFwdWaves* CKV_WAVE) fwd_f32_split_kernel(F32Fwd f) {
    using G_ = Geo<D>;
    constexpr int NS = G_::kSteps, DB = G_::kDB;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    uint4* q_lds = reinterpret_cast<uint4*>(lds);                    // [step][plane][lane]
    float* o_lds = lds + G_::kTile / 4;                               // [wave][row][kPitch]
    float* ml_lds = o_lds + kFwdWaves * kRows * G_::kPitch;           // [max, sum][wave][row]
    const CoreProblem& p = f.c;
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // kv heads go round the XCDs (when they divide evenly), so a head's keys stay in one L2; heavy row tiles first
    const int nbkv = (int)(p.B * p.KVH), KVH = (int)p.KVH, G = (int)p.H / KVH;
    const int n_rt = (int)(((int)p.Q * G + kRows - 1) / kRows);
    const int bkv = blockIdx.x % nbkv, rest = blockIdx.x / nbkv;
    const int split = rest % f.n_split, rt = n_rt - 1 - rest / f.n_split;
    const int64_t b = bkv / KVH, kvh = bkv % KVH;
    const int Q = (int)p.Q, Nc = (int)p.N - Q, all_blocks = ((int)p.N + kKeys - 1) / kKeys;
    const uint4* kb = (const uint4*)f.f.k + (int64_t)bkv * all_blocks * G_::kTileVec + lane;
    const uint4* vb = (const uint4*)f.f.v + (int64_t)bkv * all_blocks * G_::kTileVec + lane;

    const int row_m = (rt * kRows + col) / G;            // this lane's query
    int m_hi = (rt * kRows + kRows - 1) / G;
    if (m_hi > Q - 1) m_hi = Q - 1;
    const int nblk = (Nc + m_hi) / kKeys + 1;            // blocks some row of the tile may see
    const int step = kFwdWaves * f.n_split;
    auto seen_keys = [&](uint32_t vis, int n0) {         // the keys of a block this lane's query sees
        if (n0 + kKeys - 1 < Nc) return vis;
        const int last = Nc + row_m - n0;   // last key of the block the row may see
        return vis & (last >= 31 ? ~0u : (last < 0 ? 0u : (2u << last) - 1u));   // cached keys lie in front of the chunk keys: row_m >= 0 lets them all through
    };
    // the wavefront's first block from `blk` on with a visible key
    const uint32_t* odd_kv = reinterpret_cast<const uint32_t*>(f.f.odd_kv + (int64_t)bkv * all_blocks);
    uint32_t vis = 0u, odd_k = 0u, odd_v = 0u;
    auto visible_from = [&](int blk) {
        for (vis = 0u; blk < nblk; blk += step) {
            vis = uniform_word(f.f.vis, blk);
            odd_k = uniform_word(odd_kv, 2 * blk);
            odd_v = uniform_word(odd_kv, 2 * blk + 1);
            if (vis != 0u) break;
        }
        return blk;
    };
    // the word of the tile of this lane's query
    auto odd_query = [&]() {
        const int g = rt * kRows + col - row_m * G;
        return row_m < Q ? f.f.odd_q[(b * p.H + kvh * G + g) * f.f.q_tiles + row_m / 32] : 0u;
    };
    uint4 kf[NS][kPlanes];   // the block's keys
    auto load_keys = [&](int blk, int c0, int c1) {
        const uint4* from = kb + (int64_t)blk * G_::kTileVec;
#pragma unroll
        for (int c = 0; c < NS; c++) {
            if (c < c0 || c >= c1) continue;
#pragma unroll
            for (int pl = 0; pl < kPlanes; pl++) kf[c][pl] = from[(c * kPlanes + pl) * CKV_WAVE];
        }
    };
    // the first block's keys are requested with the queries and before it is known whether anybody sees them
    const int blk_first = split * kFwdWaves + wave;
    load_keys(blk_first < all_blocks ? blk_first : all_blocks - 1, 0, NS);
    {
        const int rf = rt * kRows + col, m = rf / G, g = rf - m * G;
        const uint4* from = (const uint4*)f.f.q + ((b * p.H + kvh * G + g) * f.f.q_tiles + m / 32) * G_::kTileVec + (m & 31) + 32 * half;
#pragma unroll
        for (int i = 0; i < (G_::kPieces + kFwdWaves - 1) / kFwdWaves; i++) {
            const int t = i * kFwdWaves + wave;
            if (t >= G_::kPieces) break;
            if (m < Q) async_copy16_from(from + t * CKV_WAVE, lds_address(q_lds) + t * (CKV_WAVE * 16));
            else q_lds[t * CKV_WAVE + lane] = make_uint4(0u, 0u, 0u, 0u);
        }
    }
    const bool odd_queries = __ballot(odd_query() != 0u) != 0ull;
    int blk = visible_from(blk_first);
    if (vis != 0u && blk != blk_first) load_keys(blk, 0, NS);
    wait_copies<0>();
    __syncthreads();

    // the logits of a block's keys (lane = its query) by float32 products, whatever the operands hold
    auto plain_logits = [&](int blk, uint32_t odd_k) {
        f32x16 s = zero16();
        const uint4* from = kb + (int64_t)blk * G_::kTileVec;
        const uint32_t odd_q = odd_query();
#pragma unroll 1
        for (int c = 0; c < NS; c++) {
            uint4 k[kPlanes], q[kPlanes];
#pragma unroll
            for (int pl = 0; pl < kPlanes; pl++) {
                k[pl] = from[(c * kPlanes + pl) * CKV_WAVE];
                q[pl] = q_lds[(c * kPlanes + pl) * CKV_WAVE + lane];
            }
#pragma unroll
            for (int e = 0; e < 8; e++) s = mma32(whole_of(k, e, G_::raw_step(odd_k, c)), whole_of(q, e, G_::raw_step(odd_q, c)), s);
        }
        return s;
    };
    auto split_probabilities = [&](const f32x16& s, uint4 (&pb)[2][kPlanes]) {
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            uint32_t w[kPlanes][4];
#pragma unroll
            for (int i = 0; i < 4; i++) split2(s[8 * ks + 2 * i], s[8 * ks + 2 * i + 1], w[0][i], w[1][i], w[2][i]);
#pragma unroll
            for (int pl = 0; pl < kPlanes; pl++) pb[ks][pl] = make_uint4(w[pl][0], w[pl][1], w[pl][2], w[pl][3]);
        }
    };
    auto mma_values = [&](const uint4 (&v)[kPlanes], const uint4 (&pr)[kPlanes], f32x16 o) {
        o = mma(v[2], pr[0], o);
        o = mma(v[0], pr[2], o);
        o = mma(v[1], pr[1], o);
        o = mma(v[1], pr[0], o);
        o = mma(v[0], pr[1], o);
        return mma(v[0], pr[0], o);
    };

    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; db++) o[db] = zero16();
    float m_run = -INFINITY, l_run = 0.f;
    while (vis != 0u) {
        const int n0 = blk * kKeys;
        const uint32_t vis_now = vis;
        f32x16 s = zero16(), small = zero16();
        uint4 qf[2][kPlanes];   // a step's queries, read a step ahead and not all at once
#pragma unroll
        for (int pl = 0; pl < kPlanes; pl++) qf[0][pl] = q_lds[pl * CKV_WAVE + lane];
#pragma unroll
        for (int c = 0; c < NS; c++) {
            __builtin_amdgcn_sched_barrier(0);
            if (c + 1 < NS) {
#pragma unroll
                for (int pl = 0; pl < kPlanes; pl++) qf[(c + 1) & 1][pl] = q_lds[((c + 1) * kPlanes + pl) * CKV_WAVE + lane];
            }
            mma_planes(kf[c], qf[c & 1], s, small);
        }
        __builtin_amdgcn_sched_barrier(0);
        // the values travel under the exponentials, the next block's keys under the second product
        uint4 vf[DB][2][kPlanes];
        const uint4* from = vb + (int64_t)blk * G_::kTileVec;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int pl = 0; pl < kPlanes; pl++) vf[db][ks][pl] = from[((db * 2 + ks) * kPlanes + pl) * CKV_WAVE];
        __builtin_amdgcn_sched_barrier(0);
        const int here = blk;
        const uint32_t odd_here = odd_k, odd_values = odd_v;
        blk = visible_from(blk + step);
        const uint32_t allow = seen_keys(vis_now, n0);   // bit r: key r of the block is visible to this lane's query
        const bool whole = __ballot(allow != ~0u) == 0ull;
#pragma unroll
        for (int v = 0; v < 16; v++) s[v] += small[v];
        float m_new, ref, sum, low;
        auto largest = [&]() {
            low = INFINITY;   // the smallest logit of a key that the row sees
            if (!whole) {
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const bool sees = (allow >> acc_row(v, half)) & 1u;
                    low = fminf(low, sees ? s[v] : INFINITY);
                    s[v] = sees ? s[v] : -INFINITY;
                }
            } else {
#pragma unroll
                for (int v = 0; v < 16; v++) low = fminf(low, s[v]);
            }
            float mx = -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; v++) mx = fmaxf(mx, s[v]);
            mx = half_max(mx);
            m_new = fmaxf(m_run, mx);
            ref = m_new == -INFINITY ? 0.f : m_new;   // nothing visible yet: every exponential is 0
            sum = 0.f;
        };
        largest();
#pragma unroll
        for (int v = 0; v < 16; v++) {
            s[v] = exp2_fast(s[v] - ref);
            sum += s[v];
        }
        const bool plain = (odd_here | odd_values) != 0u || odd_queries || __ballot(isnan(sum) || low - ref < kFaint) != 0ull;
        if (__builtin_expect(plain, 0)) {
            s = plain_logits(here, odd_here);
            largest();
#pragma unroll
            for (int v = 0; v < 16; v++) {
                s[v] = exp2f(s[v] - ref);
                sum += s[v];
            }
        }
        const float alpha = m_run == -INFINITY ? 0.f : exp2f(m_run - ref);
        l_run = l_run * alpha + sum;
        if (__ballot(m_new != m_run) != 0ull) {
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int v = 0; v < 16; v++) o[db][v] *= alpha;
        }
        m_run = m_new;
        if (__builtin_expect(plain, 0)) {
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int e = 0; e < 8; e++) o[db] = mma32(whole_of(vf[db][ks], e, G_::raw_values(odd_values, ks)), s[8 * ks + e], o[db]);
                }
            __builtin_amdgcn_sched_barrier(0);
            // The products below add nothing: their operands are finite.  A way around them had the compiler spill 120 registers and more.
#pragma unroll
            for (int v = 0; v < 16; v++) s[v] = 0.f;
        }
        uint4 pb[2][kPlanes];
        split_probabilities(s, pb);
#pragma unroll
        for (int db = 0; db < DB; db++) {
#pragma unroll
            for (int ks = 0; ks < 2; ks++) o[db] = mma_values(vf[db][ks], pb[ks], o[db]);
            if (2 * db + 2 == DB || db + 1 == DB) {   // half of the values are used up, or all
                __builtin_amdgcn_sched_barrier(0);
                // without a next block these again: a condition would keep the old ones' registers
                load_keys(vis != 0u ? blk : here, db + 1 == DB ? NS / 2 : 0, db + 1 == DB ? NS : NS / 2);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }

    float zero = 0.f;   // or NaN
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int v = 0; v < 16; v++) zero = fmaf(o[db][v], 0.f, zero);
    if (__ballot(zero != 0.f) != 0ull) {
#pragma unroll
        for (int db = 0; db < DB; db++) o[db] = zero16();
        for (blk = visible_from(split * kFwdWaves + wave); blk < nblk; blk = visible_from(blk + step)) {
            f32x16 s = plain_logits(blk, odd_k);
            const uint32_t allow = seen_keys(vis, blk * kKeys);
#pragma unroll
            for (int v = 0; v < 16; v++) s[v] = (allow >> acc_row(v, half)) & 1u ? exp2f(s[v] - m_run) : 0.f;
            const uint4* from = vb + (int64_t)blk * G_::kTileVec;
#pragma unroll
            for (int db = 0; db < DB; db++) {
                f32x16 up = zero16(), down = zero16();   // how many infinities of either sign a sum holds, a NaN being both
                bool odd = false;
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
                    uint4 v3[kPlanes];
#pragma unroll
                    for (int pl = 0; pl < kPlanes; pl++) v3[pl] = from[((db * 2 + ks) * kPlanes + pl) * CKV_WAVE];
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const float x = whole_of(v3, e, G_::raw_values(odd_v, ks)), counts = s[8 * ks + e] > 0.f ? 1.f : 0.f;
                        odd = odd || !isfinite(x);
                        o[db] = mma32(isfinite(x) ? x : 0.f, s[8 * ks + e], o[db]);
                        up = mma32(x == INFINITY || isnan(x) ? 1.f : 0.f, counts, up);
                        down = mma32(x == -INFINITY || isnan(x) ? 1.f : 0.f, counts, down);
                    }
                }
                if (__ballot(odd) == 0ull) continue;
#pragma unroll
                for (int v = 0; v < 16; v++) o[db][v] += (up[v] > 0.f ? INFINITY : 0.f) + (down[v] > 0.f ? -INFINITY : 0.f);
            }
        }
    }

    // merge: every wavefront scales its share to the common maximum (a share that has come down to nothing is left out)
    l_run += __shfl_xor(l_run, 32);
    if (half == 0) {
        ml_lds[wave * kRows + col] = m_run;
        ml_lds[(kFwdWaves + wave) * kRows + col] = l_run;
    }
    __syncthreads();
    {
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < kFwdWaves; w++) M = fmaxf(M, ml_lds[w * kRows + col]);
        const float sc = m_run == -INFINITY ? 0.f : exp2f(m_run - M);
        float* ow = o_lds + (wave * kRows + col) * G_::kPitch;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            Vec<DB> t;
#pragma unroll
            for (int db = 0; db < DB; db++) t.v[db] = sc == 0.f ? 0.f : o[db][v] * sc;
            *reinterpret_cast<Vec<DB>*>(ow + DB * acc_row(v, half)) = t;
        }
    }
    __syncthreads();
    // sixteen threads per row
    constexpr int kPer = D / 16;
    const int r = tid >> 4, d0 = (tid & 15) * kPer;
    const int rf = rt * kRows + r, m = rf / G, g = rf % G;
    if (m >= Q) return;
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int w = 0; w < kFwdWaves; w++) M = fmaxf(M, ml_lds[w * kRows + r]);
#pragma unroll
    for (int w = 0; w < kFwdWaves; w++) {
        const float mw = ml_lds[w * kRows + r], lw = ml_lds[(kFwdWaves + w) * kRows + r];
        const float sc = mw == -INFINITY ? 1.f : exp2f(mw - M);   // no largest logit but a sum: a NaN
        L = lw != 0.f ? fmaf(lw, sc, L) : L;
    }
    float acc[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++) acc[i] = 0.f;
#pragma unroll
    for (int w = 0; w < kFwdWaves; w++)
#pragma unroll
        for (int i = 0; i < kPer; i++) acc[i] += o_lds[(w * kRows + r) * G_::kPitch + d0 + i];
    // A row without a probability above zero (all its logits overflowed) or with a NaN among them is NaN, however many
    // shares its keys are in; a share without one says so by -inf, a NaN has to reach the merge.
    const float inv = 1.f / L;
    const int64_t row = (b * p.H + kvh * G + g) * p.Q + m, rows = p.B * p.H * p.Q;
    if (f.n_split > 1) {
        float* po = f.part_o + (split * rows + row) * D + d0;
#pragma unroll
        for (int i = 0; i < kPer; i++) po[i] = L == 0.f ? 0.f : acc[i] * inv;
        if (d0 == 0) f.part_l[split * rows + row] = make_float2(L == 0.f ? -INFINITY : M, L);
        return;
    }
    float* orow = (float*)p.out + b * p.out_stride[0] + (kvh * G + g) * p.out_stride[1] + m * p.out_stride[2];
#pragma unroll
    for (int i = 0; i < kPer; i++) orow[(d0 + i) * p.out_stride[3]] = acc[i] * inv;
    if (d0 == 0) write_normaliser(f, row, M, L);
}

// the shares of a row: one row per D / 4 lanes
template <int D>
__global__ void __launch_bounds__(256) fwd_f32_combine_kernel(F32Fwd f) {
    const CoreProblem& p = f.c;
    constexpr int kLanes = D / 4;
    const int64_t rows = p.B * p.H * p.Q;
    const int64_t row = (int64_t)blockIdx.x * (256 / kLanes) + threadIdx.x / kLanes;
    if (row >= rows) return;
    const int d4 = threadIdx.x % kLanes;
    float M = -INFINITY, L = 0.f;
    for (int s = 0; s < f.n_split; s++) M = fmaxf(M, f.part_l[s * rows + row].x);
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s = 0; s < f.n_split; s++) {
        const float2 l = f.part_l[s * rows + row];
        if (l.x == -INFINITY && l.y == 0.f) continue;   // without a largest logit, but with a sum: a NaN
        const float w = exp2f(l.x - M) * l.y;
        if (w == 0.f) continue;
        const float4 v = *reinterpret_cast<const float4*>(f.part_o + (s * rows + row) * D + 4 * d4);
        L += w;
        o.x = fmaf(v.x, w, o.x); o.y = fmaf(v.y, w, o.y); o.z = fmaf(v.z, w, o.z); o.w = fmaf(v.w, w, o.w);
    }
    const float inv = 1.f / L;
    int64_t m, h;
    const int64_t b = div_index(div_index(row, p.Q, m), p.H, h);
    float* dst = (float*)p.out + b * p.out_stride[0] + h * p.out_stride[1] + m * p.out_stride[2];
    dst[(4 * d4) * p.out_stride[3]] = o.x * inv;
    dst[(4 * d4 + 1) * p.out_stride[3]] = o.y * inv;
    dst[(4 * d4 + 2) * p.out_stride[3]] = o.z * inv;
    dst[(4 * d4 + 3) * p.out_stride[3]] = o.w * inv;
    if (d4 == 0) write_normaliser(f, row, M, L);
}

template <int D, int kGroups>
__global__ void __launch_bounds__(Col<kGroups>::kWaves* CKV_WAVE, 2) colsum_f32_split_kernel(CoreProblem p, F32Planes f, const float2* norm) {
    using C_ = Col<kGroups>;
    using G_ = Geo<D>;
    constexpr int kStreams = C_::kStreams, kWaves = C_::kWaves, kColKeys = C_::kBlockKeys, kAcc = C_::kAcc, NS = G_::kSteps;
    extern __shared__ __attribute__((aligned(16))) uint4 q_lds[];   // two stages of kStreams tiles of 32 queries
    __shared__ float sums[kColSums][kColKeys];
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = wave % kGroups, stream = wave / kGroups;
    const int nbkv = (int)(p.B * p.KVH), KVH = (int)p.KVH, G = (int)p.H / KVH;
    const int N = (int)p.N, Q = (int)p.Q, Nc = N - Q, all_blocks = (N + kKeys - 1) / kKeys, nblk = (N + kColKeys - 1) / kColKeys;
    // kv heads round the XCDs; blocks of chunk keys see fewer rows and come last
    const int bkv = blockIdx.x % nbkv, rest = blockIdx.x / nbkv;
    const int g = rest % G, blk = rest / G;
    if (blk >= nblk) return;
    const int64_t b = bkv / KVH, h = (int64_t)(bkv % KVH) * G + g;
    const int n0 = blk * kColKeys + group * kKeys, n = n0 + col, nrel = n - Nc;   // nrel >= 0: a chunk key
    const int block = n0 / kKeys < all_blocks ? n0 / kKeys : all_blocks - 1;
    const float2* norms = norm + (b * p.H + h) * p.Q;
    const int blk0 = blk * kColKeys;
    const int t_first = blk0 > Nc ? (blk0 - Nc) / kRows : 0;   // first tile with a row that sees a key of the workgroup
    const int t_own = n0 > Nc ? (n0 - Nc) / kRows : 0;         // ... of this wavefront
    const int n_tiles = (Q + kRows - 1) / kRows;
    const uint4* qb = (const uint4*)f.q + (b * p.H + h) * f.q_tiles * G_::kTileVec;
    // a stage: the streams' next tiles, which lie together, by all wavefronts
    auto copy_stage = [&](int t0, int stage) {
        if constexpr (C_::kThroughLds) {
            const int pieces = (n_tiles - t0 < kStreams ? n_tiles - t0 : kStreams) * G_::kPieces;
            for (int i = wave; i < pieces; i += kWaves)
                async_copy16(qb + (int64_t)t0 * G_::kTileVec, (uint32_t)(i * CKV_WAVE + lane) * 16u,
                             lds_address(q_lds) + (uint32_t)(stage * kStreams * G_::kTile + i * 1024));
        }
    };
    if (t_first < n_tiles) copy_stage(t_first, 0);
    // not zero in some lane: a part of the block's keys or of some tile's queries is raw
    const uint32_t* odd_key = reinterpret_cast<const uint32_t*>(f.odd_kv + (int64_t)bkv * all_blocks + block);
    const uint32_t* odd_queries = f.odd_q + (b * p.H + h) * f.q_tiles;
    uint32_t odd = *odd_key;
    for (int i = lane; i < n_tiles; i += CKV_WAVE) odd |= odd_queries[i];
    const uint32_t vis = n0 / kKeys < all_blocks ? uniform_word(f.vis, block) : 0u;
    uint4 kf[NS][kPlanes];
    const uint4* kfrom = (const uint4*)f.k + ((int64_t)bkv * all_blocks + block) * G_::kTileVec + lane;
#pragma unroll
    for (int c = 0; c < NS; c++)
#pragma unroll
        for (int pl = 0; pl < kPlanes; pl++) kf[c][pl] = kfrom[(c * kPlanes + pl) * CKV_WAVE];
    const bool live = (vis >> col) & 1u, wanted = vis != 0u;
    const bool by_distance = nrel >= 0 && p.new_mode;
    // Largest logits and what the exponentials are multiplied by, of a tile's rows, requested in front of its products: in pieces where
    // all rows are there and see all keys of the block, else (the tile on the diagonal, the last one) one by one.  For a row that does not see the lane's key
    // the former is infinite and the latter zero: it adds nothing.
    float top[16], inv[16], w[16];
    const int weight_back = by_distance ? nrel : 0;
    const uint32_t weight_at = by_distance ? f.w_new_at : 0u;
    auto all_see = [&](int t) { return t * kRows + kRows <= Q && t * kRows >= n0 + kKeys - 1 - Nc; };   // all rows of a tile, every key
    auto request_rows = [&](int t) {
        if (all_see(t)) {
#pragma unroll
            for (int i4 = 0; i4 < 4; i4++) {
                const int m0 = t * kRows + 8 * i4 + 4 * half;
                const Vec<8> n8 = *reinterpret_cast<const Vec<8>*>(norms + m0);
                const Vec<4> w4 = *reinterpret_cast<const Vec<4>*>(reinterpret_cast<const char*>(p.w_ema) + ((uint32_t)(m0 - weight_back) * 4u + weight_at));
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    top[4 * i4 + e] = n8.v[2 * e];
                    inv[4 * i4 + e] = n8.v[2 * e + 1];
                    w[4 * i4 + e] = w4.v[e];
                }
            }
            return;
        }
#pragma unroll
        for (int v = 0; v < 16; v++) {   // in 32-bit offsets from uniform addresses
            const int at = t * kRows + acc_row(v, half), m = at < Q ? at : Q - 1, d = m - weight_back;
            const float2 n2 = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(norms) + (uint32_t)m * 8u);
            const bool sees = at < Q && at >= nrel;
            top[v] = sees ? n2.x : INFINITY;
            inv[v] = sees ? n2.y : 0.f;   // that of a row of NaN would be NaN
            w[v] = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(p.w_ema) + ((uint32_t)(d > 0 ? d : 0) * 4u + weight_at));
        }
    };
    auto query_piece = [&](int t, int stage, int i) {
        if constexpr (C_::kThroughLds) return q_lds[(stage * kStreams + stream) * G_::kTileVec + i * CKV_WAVE + lane];
        else return qb[(int64_t)t * G_::kTileVec + i * CKV_WAVE + lane];
    };
    auto plain_logits = [&](int t, int stage) {   // by float32 products, whatever the operands hold
        f32x16 s = zero16();
        const uint32_t odd_q = odd_queries[t], odd_k = *odd_key;
#pragma unroll 1
        for (int c = 0; c < NS; c++) {
            uint4 q3[kPlanes], k3[kPlanes];
#pragma unroll
            for (int pl = 0; pl < kPlanes; pl++) {
                q3[pl] = query_piece(t, stage, c * kPlanes + pl);
                k3[pl] = kfrom[(c * kPlanes + pl) * CKV_WAVE];
            }
#pragma unroll
            for (int e = 0; e < 8; e++) s = mma32(whole_of(q3, e, G_::raw_step(odd_q, c)), whole_of(k3, e, G_::raw_step(odd_k, c)), s);
        }
#pragma unroll
        for (int v = 0; v < 16; v++) {   // a row that does not see the key may hold anything
            const int m = t * kRows + acc_row(v, half);
            s[v] = m < Q && m >= nrel ? s[v] : 0.f;
        }
        return s;
    };
    float acc[kAcc] = {};   // of this stream's tiles with the same (t - t_own) mod 4; of a key nobody sees, anything
    const int t_end = __syncthreads_or(wanted) ? n_tiles : t_first;
    int stage = 0, t = t_first + stream;
    for (int t0 = t_first; t0 < t_end; t0 += kStreams, t += kStreams, stage ^= 1) {
        if constexpr (C_::kThroughLds) {
            wait_copies<0>();
            __syncthreads();   // the tiles are there, and those of the stage before have been read
            if (t0 + kStreams < t_end) copy_stage(t0 + kStreams, stage ^ 1);
        }
        if (!wanted || t < t_own || t >= t_end) continue;
        request_rows(t);
        __builtin_amdgcn_sched_barrier(0);
        f32x16 s = zero16(), small = zero16();
#pragma unroll
        for (int c = 0; c < NS; c++) {
            uint4 qf[kPlanes];
#pragma unroll
            for (int pl = 0; pl < kPlanes; pl++) qf[pl] = query_piece(t, stage, c * kPlanes + pl);
            mma_planes(qf, kf[c], s, small);
        }
#pragma unroll
        for (int v = 0; v < 16; v++) s[v] += small[v];
        const bool second = kAcc == 2 && ((t - t_own) & 2);
        const float before = second ? acc[kAcc - 1] : acc[0];
        float a = before, low = 0.f;   // the smallest logit of a row that sees the key, less the row's largest
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const float x = s[v] - top[v];
            low = fminf(low, x);
            a = fmaf(w[v] * inv[v], exp2_fast(x), a);
        }
        if (low == -INFINITY) {   // as a row that does not see it has it
            low = 0.f;
#pragma unroll
            for (int v = 0; v < 16; v++) low = fminf(low, top[v] == INFINITY ? 0.f : s[v] - top[v]);
        }
        // a key that nobody sees may come out as anything
        if (__builtin_expect(__ballot(odd != 0u || (live && (!isfinite(a) || low < -126.f))) != 0ull, 0)) {
            s = plain_logits(t, stage);
            a = before;
#pragma unroll
            for (int v = 0; v < 16; v++) a = fmaf(w[v] * inv[v], exp2f(s[v] - top[v]), a);
        }
        if (second) acc[kAcc - 1] = a;
        else acc[0] = a;
    }
    wait_copies<0>();   // none is on its way to LDS that is somebody else's by then
    // the sums of tiles t_own + i, + 4, ... for i = 0 .. 3, added in that order
    const int class0 = (t_first + stream - t_own) & (kStreams - 1);
#pragma unroll
    for (int i = 0; i < kAcc; i++) {
        acc[i] += __shfl_xor(acc[i], 32);
        if (!live) acc[i] = 0.f;
        if (half == 0) sums[class0 + kStreams * i][group * kKeys + col] = acc[i];
    }
    __syncthreads();
    const int nt = blk0 + tid;
    if (tid < kColKeys && nt < N) {
        float tot = 0.f;
#pragma unroll
        for (int i = 0; i < kColSums; i++) tot += sums[i][tid];
        p.colsum[(b * p.H + h) * p.N + nt] = tot;
    }
}

template <int D>
int run(const ckv_attn_args& a, const CoreProblem& p, const F32Planes& f, float* w_ema, float* w_new, float2* norm, float* part_o,
        float2* part_l, const KeptScores& kept, hipStream_t stream) {
    using G_ = Geo<D>;
    const int64_t G = p.H / p.KVH, tiles = (p.Q * G + kRows - 1) / kRows, units = p.B * p.KVH;
    {
        StageScope sc(CKV_STAGE_PREP, stream);
        F32Stage st;
        st.a = a;
        st.q = (uint4*)f.q;
        st.k = (uint4*)f.k;
        st.v = (uint4*)f.v;
        st.vis = f.vis;
        st.odd_kv = f.odd_kv;
        st.odd_q = f.odd_q;
        st.w_ema = w_ema;
        st.w_new = w_new;
        // on queries and keys: nothing is multiplied behind the products
        st.post_k = sqrtf(a.scale);
        st.post_q = (float)(sqrt((double)a.scale) * 1.4426950408889634);
        st.nblk = (int)((p.N + kKeys - 1) / kKeys);
        st.q_tiles = f.q_tiles;
        st.k_items = (int)(units * st.nblk * (G_::kSteps / 2));
        st.q_items = (int)(p.B * p.H * f.q_tiles * (G_::kSteps / 2));
        st.v_items = (int)(units * st.nblk * 2);
        st.vis_items = (st.nblk + 1) / 2;
        auto pieces = [](const int64_t* s, const void* x, const void* y) {
            return s[3] == 1 && s[0] % 4 == 0 && s[1] % 4 == 0 && s[2] % 4 == 0 &&
                   ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
        };
        st.vec = pieces(a.q_stride, a.q, a.q) && pieces(a.kv_new_stride, a.k_new, a.v_new) &&
                 (a.S == 0 || pieces(a.cache_stride, a.cache_k, a.cache_v)) && (a.num_sink == 0 || pieces(a.sink_stride, a.sink_k, a.sink_v));
        st.w_items = w_ema ? (int)((p.Q + kColSlack + 63) / 64) : 0;
        st.kept = kept;
        const int64_t waves = (int64_t)st.k_items + st.q_items + st.v_items + st.vis_items + st.w_items + kept_pieces(kept, CKV_WAVE);
        hipLaunchKernelGGL(stage_f32_kernel<D>, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, stream, st);
        CKV_HIP_TRY(hipGetLastError());
    }
    {
        StageScope sc(CKV_STAGE_FWD, stream);
        F32Fwd w;
        w.c = p;
        w.f = f;
        w.n_split = part_o && part_l ? f32_split_shares(p.B, p.H, p.KVH, p.Q, p.N, mfma_device_cus()) : 1;
        w.part_o = part_o;
        w.part_l = part_l;
        w.norm = norm;
        if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fwd_f32_split_kernel<D>), G_::kFwdLds)) return rc;
        hipLaunchKernelGGL(fwd_f32_split_kernel<D>, dim3((unsigned)(tiles * w.n_split * units)), dim3(kFwdWaves * CKV_WAVE), G_::kFwdLds, stream, w);
        CKV_HIP_TRY(hipGetLastError());
        if (w.n_split > 1) {
            constexpr int per = 256 / (D / 4);
            hipLaunchKernelGGL(fwd_f32_combine_kernel<D>, dim3((unsigned)((p.B * p.H * p.Q + per - 1) / per)), dim3(256), 0, stream, w);
            CKV_HIP_TRY(hipGetLastError());
        }
    }
    if (p.colsum) {
        StageScope sc(CKV_STAGE_SCORES, stream);
        // Four blocks of keys share their workgroup's query tiles, unless that leaves more than a quarter of the chip idle (32 heads x 584
        // keys, 64 rows, 160 workgroups: 10.6 us with one block each)
        auto launch = [&](auto groups) -> int {
            using C_ = Col<groups.value>;
            auto kernel = colsum_f32_split_kernel<D, groups.value>;
            const int lds = C_::kThroughLds ? 2 * C_::kStreams * G_::kTile : 0;
            if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), lds)) return rc;
            const int64_t blocks = p.B * p.H * ((p.N + C_::kBlockKeys - 1) / C_::kBlockKeys);
            hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(C_::kWaves * CKV_WAVE), lds, stream, p, f, norm);
            return CKV_OK;
        };
        const int64_t shared = p.B * p.H * ((p.N + Col<4>::kBlockKeys - 1) / Col<4>::kBlockKeys);
        if (int rc = 4 * shared >= 3 * (int64_t)mfma_device_cus() ? launch(std::integral_constant<int, 4>{})
                                                                    : launch(std::integral_constant<int, 1>{})) return rc;
        CKV_HIP_TRY(hipGetLastError());
    }
    return CKV_OK;
}

}  // namespace

// One workgroup fills a compute unit (eight wavefronts of some 220 registers), so a launch with fewer row tiles than
// that shares the key blocks of a tile out, at least two per wavefront, as long as the shares still fit one round.
int f32_split_shares(int64_t B, int64_t H, int64_t KVH, int64_t Q, int64_t n, int cus) {
    const int64_t wgs = ((Q * (H / KVH) + kRows - 1) / kRows) * B * KVH, blocks = (n + kKeys - 1) / kKeys;
    int64_t s = cus / wgs;
    if (s > blocks / (2 * kFwdWaves)) s = blocks / (2 * kFwdWaves);
    if (s > 16) s = 16;
    return s < 1 ? 1 : (int)s;
}

bool f32_split_supported(int dtype, int64_t B, int64_t H, int64_t KVH, int64_t Q, int64_t n, int64_t D) {
    constexpr int64_t lim = (int64_t)1 << 31;
    const int64_t blocks = (n + kKeys - 1) / kKeys, q_tiles = (Q + 31) / 32, steps = D / 16;
    return dtype == CKV_F32 && (D == 64 || D == 128) && n < lim - 64 && B * H * blocks < lim &&
           ((Q * (H / KVH) + kRows - 1) / kRows) * 16 * B * KVH < lim &&
           (B * KVH * blocks + B * H * q_tiles) * steps + B * KVH * blocks * 2 + blocks + Q + kColSlack < lim - 1024;
}

int64_t f32_split_plane_bytes(int64_t units, int64_t rows, int64_t D) { return units * ((rows + 31) / 32) * 32 * D * 2 * kPlanes; }

int launch_f32_split(const ckv_attn_args& a, const CoreProblem& p, const F32Planes& f, float* w_ema, float* w_new, float2* norm,
                     float* part_o, float2* part_l, const KeptScores& kept, hipStream_t stream) {
    return p.D == 64 ? run<64>(a, p, f, w_ema, w_new, norm, part_o, part_l, kept, stream)
                     : run<128>(a, p, f, w_ema, w_new, norm, part_o, part_l, kept, stream);
}

}  // namespace ckv

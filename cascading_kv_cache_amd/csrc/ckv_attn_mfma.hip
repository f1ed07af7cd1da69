// bf16 / fp16 MFMA attention for head_dim 64 and 128 on gfx950 (CDNA4, wave64, v_mfma_f32_32x32x16).
//
// Stages (all stream-ordered):
//   stage_keys   rotate K on the way into a padded row-major buffer Kr, transpose V into 64-key
//                tiles Vt[tile][d][key'] (key' = the order the PV MFMA consumes), build one 64-bit
//                visibility word per key tile.  cos/sin are computed once per key and reused for
//                every (batch, kv-head) that shares the position row.
//   stage_q      rotate Q and, with 128 dims, fold the softmax scale (times log2 e) in.
//   fwd          flash forward, software pipelined.  One workgroup = one kv head x 256 (head,
//                position) rows, so the G query heads of a group share every K/V tile staged in
//                LDS.  S^T = K Q^T keeps a query in one lane pair: the row max / sum need a single
//                cross-half exchange and exp2(S^T) is already laid out as the B operand of
//                O^T += V^T P^T.  The softmax of tile i runs beside the logits of tile i+1 and the
//                P.V product of tile i-1.
//   colsum       exact score sums.  One workgroup = one head x 256 keys held in registers; the
//                queries stream through LDS, the accumulators start from minus the final
//                normaliser so the matrix pipe returns log2 P, and the weighted column sums stay
//                inside a lane (S = Q K^T orientation).
//
// Precision.  With 128 dims the scale rides on the 16-bit queries and the probabilities enter P.V rounded to the tensor
// dtype.  With 64 dims nothing but the operands themselves is held in 16 bits (kExact): the logits of the queries as the
// eager path rounds them are scaled in float32, and a probability enters P.V as three terms of the tensor dtype that
// add up to its float32 value (one matrix instruction each, all into the same float32 accumulator; float16: to 2^-37 of the
// row's largest probability, see kHead), so the result is that of float32 arithmetic.  8 heads x 1000 rows x 5095 keys in float16: forward 20 -> 28 us, scores 31.5 -> 34 (the vector
// kernels, to the same error: 2300 and 521); 32 heads on 8 kv heads, 4096 rows x 16 K slots, the whole call: 1.41 -> 2.02 ms
// (59).  The vector ALU bounds the forward: seven instructions more per pair of probabilities.
#include "ckv_attn_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

namespace ckv {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// Kernels take the head dim as a template parameter kD: 64 or 128.
template <int kD>
constexpr bool kExact = kD == 64;
constexpr float kLog2e = 1.4426950408889634f;
constexpr int kBN = 64;    // keys per tile

constexpr int kRows = 256;    // (head, position) rows per forward workgroup

template <typename T>
struct Mma;
template <>
struct Mma<__hip_bfloat16> {
    __device__ static f32x16 mma(uint4 a, uint4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    }
    __device__ static uint32_t pack2(float lo, float hi) {
        f32x2 f = {lo, hi};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
    }
    __device__ static float round1(float v) {
        f32x2 f = {v, 0.f};
        const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
        return __uint_as_float(u << 16);
    }
    // the two elements of a packed pair as floats
    __device__ static float lo_f(uint32_t w) { return __uint_as_float(w << 16); }
    __device__ static float hi_f(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
    // acc + both halves of a packed pair (one v_dot2c with a pair of ones)
    __device__ static float sum2(uint32_t w, float acc) {
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), __builtin_bit_cast(bf16x2, 0x3f803f80u), acc, false);
    }
};
template <>
struct Mma<__half> {
    __device__ static f32x16 mma(uint4 a, uint4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
    }
    __device__ static uint32_t pack2(float lo, float hi) {
        f32x2 f = {lo, hi};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
    }
    __device__ static float round1(float v) { return (float)(_Float16)v; }
    __device__ static float lo_f(uint32_t w) { return (float)__builtin_bit_cast(f16x2, w)[0]; }
    __device__ static float hi_f(uint32_t w) { return (float)__builtin_bit_cast(f16x2, w)[1]; }
    __device__ static float sum2(uint32_t w, float acc) {
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, w), __builtin_bit_cast(f16x2, 0x3c003c00u), acc, false);
    }
};

// position of key `k` (0..63) of a tile inside a V^T row: the PV contraction step s covers keys
// 16s..16s+15; lane half h supplies keys 16s + 8a + 4h + e (a = 0,1; e = 0..3) as elements 4a+e
__host__ __device__ inline int vt_slot(int k) {
    const int s = k >> 4, a = (k >> 3) & 1, h = (k >> 2) & 1, e = k & 3;
    return 16 * s + 8 * h + 4 * a + e;
}

// ---------------------------------------------------------------------------------------------
// staging
// ---------------------------------------------------------------------------------------------
struct KeySegment {
    const void* k;
    const void* v;
    int64_t stride[4];       // (B, KVH, len, D)
    const int64_t* pos;      // position ids, or null when keys are already rotated
    int64_t pos_stride[2];
    int64_t pos_shift;
    const uint8_t* masked;   // 1 = masked, or null (all visible)
    int64_t len;
};

struct StageParams {
    KeySegment seg[3];
    const float* inv_freq;
    float theta;
    float key_scale;         // rotated keys are multiplied by this and rounded again (1: they are not)
    int shared_pos;          // every (b, kvh) uses position row [0, 0]
    void* kr;                // (B*KVH, n_pad/64) K tile images, see k_image_off
    void* vt;                // (B*KVH, n_pad/64) V^T tile images, see v_image_off
    unsigned long long* tile_vis;  // (n_pad/64,)
    int64_t B, KVH, n, n_pad;
    // Keys in another order than they lie in memory, the visible ones first (see key_order_block): staged key i is row
    // key_order[i] of segment 0, for i < *n_visible + n_chunk; null: keys in order of the segments.
    const int* key_order;
    const int* n_visible;
    int64_t n_chunk;
    // The order is not there yet (this launch writes it, see order_by_staging): a block finds its tile's keys in the mask itself.
    int own_order;
    const uint8_t* order_mask;     // (n_cached), 1 = masked
    int64_t n_cached;
    int64_t empty_from, empty_to;  // keys no query can see because their slots are still empty (none: both 0)
};

__device__ inline int find_segment(const StageParams& p, int64_t n, int64_t& local) {
    if (n < p.seg[0].len) { local = n; return 0; }
    n -= p.seg[0].len;
    if (n < p.seg[1].len) { local = n; return 1; }
    local = n - p.seg[1].len;
    return 2;
}

// The staged K and V of one 64-key tile are images of kD * 128 bytes in exactly the order the forward kernel
// keeps them in LDS, so a tile reaches LDS as a straight copy and the 64 lanes of an operand read
// touch 1 KiB made of two contiguous halves (no bank conflicts, one base address per lane):
//   K image:   16-byte piece c (elements 8c .. 8c+7) of key row r at  (c/2)*2048 + (c%2)*1024 + r*16
//   V^T image: 16-byte piece c (key slots 8c .. 8c+7) of dim row d at (c/2)*32 kD + (c%2)*16 kD + d*16
// Key slot 16s + 8h + 4a + e of a V^T row holds key 16s + 8a + 4h + e of the tile: the order in
// which the logits leave the matrix pipe.
__device__ __host__ inline int k_image_off(int r, int c) { return (c >> 1) * 2048 + (c & 1) * 1024 + r * 16; }
template <int kD>
__device__ __host__ inline int v_image_off(int d, int c) { return (c >> 1) * (32 * kD) + (c & 1) * (16 * kD) + d * 16; }

// cos / sin of a rotation angle before their rounding to the tensor dtype: where nothing else is rounded, to the last bit
template <int kD>
__device__ inline void stage_sincos(float x, float* sn, float* cs) {
    if constexpr (kExact<kD>) sincosf(x, sn, cs);
    else fast_sincos(x, sn, cs);
}

// pair i of the threads with `quarter`
__device__ inline int stage_pair(int quarter, int i) { return i < 8 ? 8 * quarter + i : 24 + 8 * quarter + i; }

// LDS of a block: (d, d + kD/2) pairs of a key row, odd pitch; cos and sin of the threads' pairs while they are computed
template <int kD>
struct StageLds {
    static constexpr int kPitch = kD / 2 + 1;
    union {
        uint32_t v[kBN][kPitch];
        uint2 trig[kD / 16][256];
    };
    float freqs[kD / 2];
    int picked[kBN], sums[2][4];   // see keys_of_tile
};

// The cached keys of ranks first .. first + 63 among the visible ones, into `picked`, by a workgroup of 256 threads.  Returns how many are
// visible, or a number past the last of these ranks.
__device__ inline int keys_of_tile(const uint8_t* mask, int n_cached, int first, int* picked, int (*sums)[4]) {
    constexpr int kPer = 16, kStretch = 256 * kPer;
    const int tid = threadIdx.x, lane = tid % CKV_WAVE, wave = tid / CKV_WAVE;
    const bool vec = (reinterpret_cast<uintptr_t>(mask) & 15) == 0;
    // this thread's 16 keys of a stretch as a word of bits, one per visible key
    auto visible = [&](int base) -> uint32_t {
        const int k0 = base + tid * kPer;
        uint32_t bits = 0;
        if (vec && k0 + kPer <= n_cached) {
            const uint4 m = *reinterpret_cast<const uint4*>(mask + k0);
            const uint32_t w[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
            for (int i = 0; i < kPer; i++) bits |= (((w[i >> 2] >> (8 * (i & 3))) & 0xffu) == 0u ? 1u : 0u) << i;
        } else {
            for (int i = 0; i < kPer; i++)
                if (k0 + i < n_cached && mask[k0 + i] == 0) bits |= 1u << i;
        }
        return bits;
    };
    int seen = 0, round = 0;   // visible keys in the stretches before
    uint32_t next = n_cached > 0 ? visible(0) : 0u;
    for (int base = 0; base < n_cached && seen < first + kBN; base += kStretch, round ^= 1) {
        uint32_t bits = next;
        if (base + kStretch < n_cached) next = visible(base + kStretch);
        const int mine = __popc(bits);
        int incl = mine;
#pragma unroll
        for (int off = 1; off < CKV_WAVE; off <<= 1) {
            const int v = __shfl_up(incl, off);
            if (lane >= off) incl += v;
        }
        if (lane == CKV_WAVE - 1) sums[round][wave] = incl;
        __syncthreads();   // the sums of the next stretch go to the other half
        int rank = seen + incl - mine;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const int v = sums[round][w];
            rank += w < wave ? v : 0;
            seen += v;
        }
        if (rank < first + kBN && rank + mine > first) {
            for (; bits; bits &= bits - 1, rank++)
                if (rank >= first && rank < first + kBN) picked[rank - first] = base + tid * kPer + __ffs(bits) - 1;
        }
    }
    __syncthreads();
    return seen;
}

// frequencies of the rotation pairs into LDS (visible after a barrier)
template <int kD>
__device__ inline void stage_freqs(const float* inv_freq, float theta, StageLds<kD>& lds) {
    const int j = threadIdx.x;
    if (j < kD / 2) lds.freqs[j] = inv_freq ? inv_freq[j] : 1.0f / powf(theta, (float)(2 * j) / (float)kD);
}

// cos / sin of a thread's rotation pairs, two per word, rounded to the tensor dtype (see RopeWord).  A loop on purpose, with
// the words parked in LDS: unrolled 16 times, the range reductions and the power function are 48 KiB of instructions that
// a launch fetches cold and executes once per workgroup (8 heads x 16897 keys and 509 x 32 queries: 47 us unrolled, 33.5 so;
// 16 x 18496: 90 and 73; 8 x 69696: 133 and 109, 5.2 TB/s).
template <typename T, int kD>
__device__ inline void stage_trig(float pos, int quarter, StageLds<kD>& lds, RopeWord<T> (&rw)[kD / 16]) {
    const int tid = threadIdx.x;
#pragma unroll 1
    for (int k = 0; k < kD / 16; k++) {
        float sn[2], cs[2];
#pragma unroll
        for (int e = 0; e < 2; e++) stage_sincos<kD>(__fmul_rn(pos, lds.freqs[stage_pair(quarter, 2 * k + e)]), &sn[e], &cs[e]);
        lds.trig[k][tid] = make_uint2(RopeWord<T>::pack2(cs[0], cs[1]), RopeWord<T>::pack2(sn[0], sn[1]));
    }
#pragma unroll
    for (int k = 0; k < kD / 16; k++) rw[k] = RopeWord<T>::of(lds.trig[k][tid]);   // a thread's own words
}

// One block of 256 threads stages key tile `tile_i` for the (b, kvh) units split_i, split_i + n_split, ...:
// thread = (key = tid/4, quarter = tid%4) owns rotation pairs j = 8q .. 8q+7 (and, with 128 dims, 32+8q .. 32+8q+7),
// i.e. the 16-byte pieces q, 4+q (, 8+q and 12+q) of its row: the four threads of a row read (and, for queries,
// write) 64 contiguous bytes per instruction.
template <typename T, int kD>
__device__ inline void stage_keys_block(const StageParams& p, int tile_i, int split_i, int n_split, StageLds<kD>& lds) {
    constexpr int kPieces = kD / 64;     // 16-byte pieces of each half of the row
    constexpr int kPairs = kD / 8;       // rotation pairs of a thread
    const int tid = threadIdx.x;
    const int key = tid >> 2, quarter = tid & 3;
    const int64_t tile = tile_i;
    const int64_t n = tile * kBN + key;
    int64_t local = 0;
    int sidx = -1;
    int64_t n_all = p.n;
    if (p.key_order) {
        // visible keys first: what lies behind them is read by nobody.  The order indexes segment 0, which holds all keys.
        const int64_t vis = p.own_order ? keys_of_tile(p.order_mask, (int)p.n_cached, (int)(tile * kBN), lds.picked, lds.sums) : *p.n_visible;
        n_all = vis + p.n_chunk;
        if (tile * kBN >= n_all) return;
        if (n < n_all) {
            local = !p.own_order ? p.key_order[n] : n < vis ? lds.picked[key] : p.n_cached + (n - vis);
            sidx = 0;
        }
    } else if (n < p.n) {
        sidx = find_segment(p, n, local);
    }

    // A tile of slots that cannot hold a token yet is read by nobody: the forward kernel leaves it out, the score kernel
    // zeroes its sums.  A cache that is still filling is mostly such tiles (1000 of 16384 slots, 488-token chunk: the
    // launch takes 31 us instead of 50).  The bound comes from the host's counter, so that nothing waits for the mask.
    if (tile * kBN >= p.empty_from && (tile + 1) * kBN <= p.empty_to) {
        if (split_i == 0 && tid == 0) p.tile_vis[tile] = 0ull;
        return;
    }
    if (split_i == 0 && tid < kBN) {  // visibility word of this tile
        const int64_t nn = tile * kBN + tid;
        bool vis = nn < n_all;
        if (vis && !p.key_order) {
            int64_t loc;
            const int si = find_segment(p, nn, loc);
            if (p.seg[si].masked) vis = p.seg[si].masked[loc] == 0;
        }
        const unsigned long long bal = __ballot(vis);
        if (tid == 0) p.tile_vis[tile] = bal;
    }

    const bool rotate = sidx >= 0 && p.seg[sidx].pos != nullptr;
    int64_t pos = 0;
    if (rotate && p.shared_pos) pos = p.seg[sidx].pos[local] + p.seg[sidx].pos_shift;
    RopeWord<T> rw[kPairs / 2];
    const bool key_scaled = p.key_scale != 1.0f;
    const int64_t nbh = p.B * p.KVH;
    // units split_i, split_i + n_split, ... as (b, kvh): stepped, not divided
    const int KVH = (int)p.KVH, step_b = (int)((uint32_t)n_split / (uint32_t)KVH), step_h = n_split - step_b * KVH;
    struct Unit {
        int b, kvh;
    };
    auto next_unit = [&](Unit& u) {
        u.b += step_b;
        u.kvh += step_h;
        if (u.kvh >= KVH) { u.kvh -= KVH; u.b++; }
    };
    Unit ahead;   // of the rows that are requested
    ahead.b = (int)((uint32_t)split_i / (uint32_t)KVH);
    ahead.kvh = split_i - ahead.b * KVH;
    // this thread's row of the segment it lies in
    const T *k_row = nullptr, *v_row = nullptr;
    int64_t stride_b = 0, stride_h = 0, stride_d = 0;
    if (sidx >= 0) {
        const KeySegment& sg = p.seg[sidx];
        k_row = (const T*)sg.k + local * sg.stride[2];
        v_row = (const T*)sg.v + local * sg.stride[2];
        stride_b = sg.stride[0];
        stride_h = sg.stride[1];
        stride_d = sg.stride[3];
    }
    // the rows of unit bh as this thread's 16-byte pieces (zeros past the last key)
    struct Rows {
        uint4 lo[kPieces], hi[kPieces], vlo[kPieces], vhi[kPieces];
    };
    auto load_rows = [&](int64_t bh, Rows& r) {
#pragma unroll
        for (int i = 0; i < kPieces; i++) r.lo[i] = r.hi[i] = r.vlo[i] = r.vhi[i] = make_uint4(0, 0, 0, 0);
        if (sidx < 0 || bh >= nbh) return;
        const int64_t off = ahead.b * stride_b + ahead.kvh * stride_h;
        const T* kp = k_row + off;
        const T* vp = v_row + off;
        if (stride_d == 1 && ((reinterpret_cast<uintptr_t>(kp) | reinterpret_cast<uintptr_t>(vp)) & 15) == 0) {
#pragma unroll
            for (int i = 0; i < kPieces; i++) {
                r.lo[i] = *reinterpret_cast<const uint4*>(kp + 32 * i + 8 * quarter);
                r.hi[i] = *reinterpret_cast<const uint4*>(kp + kD / 2 + 32 * i + 8 * quarter);
                r.vlo[i] = *reinterpret_cast<const uint4*>(vp + 32 * i + 8 * quarter);
                r.vhi[i] = *reinterpret_cast<const uint4*>(vp + kD / 2 + 32 * i + 8 * quarter);
            }
        } else {
            T* l0 = reinterpret_cast<T*>(r.lo);
            T* h0 = reinterpret_cast<T*>(r.hi);
            T* vl = reinterpret_cast<T*>(r.vlo);
            T* vh = reinterpret_cast<T*>(r.vhi);
            for (int i = 0; i < kPairs; i++) {
                l0[i] = kp[stage_pair(quarter, i) * stride_d];
                h0[i] = kp[(kD / 2 + stage_pair(quarter, i)) * stride_d];
                vl[i] = vp[stage_pair(quarter, i) * stride_d];
                vh[i] = vp[(kD / 2 + stage_pair(quarter, i)) * stride_d];
            }
        }
    };
    // The rows of the next unit are requested before this unit's rotation, transposition and stores, so
    // the workgroup always has loads in flight.
    Rows nxt;
    load_rows(split_i, nxt);
    // no barrier between a thread's own words here and the first rows in LDS but the one in front of those
    const bool rotates = p.seg[0].pos || p.seg[1].pos || p.seg[2].pos;
    if (rotates) {
        stage_freqs<kD>(p.inv_freq, p.theta, lds);
        __syncthreads();
        if (rotate && p.shared_pos) stage_trig<T, kD>((float)pos, quarter, lds, rw);
    }
    for (int64_t bh = split_i; bh < nbh; bh += n_split) {
        const Unit u = ahead;
        Rows cur = nxt;
        next_unit(ahead);
        load_rows(bh + n_split, nxt);
        uint4(&lo)[kPieces] = cur.lo;
        uint4(&hi)[kPieces] = cur.hi;
        uint4(&vlo)[kPieces] = cur.vlo;
        uint4(&vhi)[kPieces] = cur.vhi;
        if (rotates && !p.shared_pos) __syncthreads();   // the last unit's rows have been read from LDS
        if (rotate) {
            if (!p.shared_pos) {
                const KeySegment& sg = p.seg[sidx];
                stage_trig<T, kD>((float)(sg.pos[u.b * sg.pos_stride[0] + u.kvh * sg.pos_stride[1] + local] + sg.pos_shift), quarter, lds, rw);
            }
            uint32_t* lw = reinterpret_cast<uint32_t*>(lo);
            uint32_t* hw = reinterpret_cast<uint32_t*>(hi);
#pragma unroll
            for (int k = 0; k < kPairs / 2; k++) rw[k].rotate(lw[k], hw[k], p.key_scale, key_scaled, lw[k], hw[k]);
        }
        char* kimg = (char*)p.kr + (bh * (p.n_pad / kBN) + tile) * (int64_t)(kD * kBN * sizeof(T));
#pragma unroll
        for (int i = 0; i < kPieces; i++) {
            *reinterpret_cast<uint4*>(kimg + k_image_off(key, 4 * i + quarter)) = lo[i];
            *reinterpret_cast<uint4*>(kimg + k_image_off(key, kD / 16 + 4 * i + quarter)) = hi[i];
        }

        // V: through LDS into the transposed tile.  A thread holds elements j and j + kD/2 of its key row for
        // the same kPairs values of j, so the two travel as one dword: kPairs four-byte LDS writes per thread, and on
        // the way out thread (j, group of kD/8 key slots) reads as many dwords and owns kD/4 bytes of dim row j and of
        // dim row j + kD/2, which neighbouring lanes store as runs of the image.
        __syncthreads();
        {
            const uint16_t* vl = reinterpret_cast<const uint16_t*>(vlo);
            const uint16_t* vh = reinterpret_cast<const uint16_t*>(vhi);
#pragma unroll
            for (int i = 0; i < kPairs; i++) lds.v[key][stage_pair(quarter, i)] = (uint32_t)vl[i] | ((uint32_t)vh[i] << 16);
        }
        __syncthreads();
        char* vimg = (char*)p.vt + (bh * (p.n_pad / kBN) + tile) * (int64_t)(kD * kBN * sizeof(T));
        {
            constexpr int kSlotsPer = kD / 8;   // key slots of a thread
            const int j = tid % (kD / 2), g = tid / (kD / 2);
            uint32_t w[kSlotsPer];
#pragma unroll
            for (int sl = 0; sl < kSlotsPer; sl++) {
                // inverse of vt_slot: slot = 16s + 8h + 4a + e  ->  key = 16s + 8a + 4h + e
                const int slot = kSlotsPer * g + sl;
                const int h = (slot >> 3) & 1, a = (slot >> 2) & 1, e = slot & 3;
                w[sl] = lds.v[(slot & ~15) + 8 * a + 4 * h + e][j];
            }
            uint32_t lo_row[kSlotsPer / 2], hi_row[kSlotsPer / 2];
#pragma unroll
            for (int k = 0; k < kSlotsPer / 2; k++) {
                lo_row[k] = (w[2 * k] & 0xffffu) | (w[2 * k + 1] << 16);
                hi_row[k] = (w[2 * k] >> 16) | (w[2 * k + 1] & 0xffff0000u);
            }
#pragma unroll
            for (int i = 0; i < kPieces; i++) {
                *reinterpret_cast<uint4*>(vimg + v_image_off<kD>(j, kPieces * g + i)) =
                    make_uint4(lo_row[4 * i], lo_row[4 * i + 1], lo_row[4 * i + 2], lo_row[4 * i + 3]);
                *reinterpret_cast<uint4*>(vimg + v_image_off<kD>(j + kD / 2, kPieces * g + i)) =
                    make_uint4(hi_row[4 * i], hi_row[4 * i + 1], hi_row[4 * i + 2], hi_row[4 * i + 3]);
            }
        }
    }
}

struct StageQParams {
    const void* q;
    int64_t stride[4];
    const int64_t* q_pos;    // null: copy only
    const float* inv_freq;
    float theta;
    void* qr;                // (B*H, Q, D) contiguous
    int64_t rows;            // B*H*Q
    int64_t H, Q;
    float qscale;            // folded into the staged queries: softmax scale * log2(e), over the factor the keys carry; with
                             // 64 dims the factor of the eager path, or the sign of the scale
    int vec;                 // source rows can be read 16 bytes at a time
};

// thread = (position m, quarter of the rotation pairs); the cos/sin of the position are computed once
// and reused for the batch x head rows share_i, share_i + n_share, ...; a block of 256 threads covers
// positions 64 blk .. 64 blk + 63
template <typename T, int kD>
__device__ inline void stage_q_block(const StageQParams& p, int blk, int share_i, int n_share, StageLds<kD>& lds) {
    const int64_t idx = (int64_t)blk * 256 + threadIdx.x;
    const int64_t m = idx >> 2;
    const int quarter = idx & 3;
    constexpr int kPieces = kD / 64, kPairs = kD / 8;
    RopeWord<T> rw[kPairs / 2];
    if (p.q_pos) {
        const int64_t pos = m < p.Q ? p.q_pos[m] : 0;
        stage_freqs<kD>(p.inv_freq, p.theta, lds);
        __syncthreads();
        stage_trig<T, kD>((float)pos, quarter, lds, rw);
    }
    if (m >= p.Q) return;
    const int64_t nbh = p.rows / p.Q;
    struct Row {
        T lo[kPairs], hi[kPairs];
    };
    auto load_row = [&](int64_t bh, Row& r) {
        if (bh >= nbh) return;
        int64_t h;
        const int64_t b = div_index(bh, p.H, h);
        const T* src = (const T*)p.q + b * p.stride[0] + h * p.stride[1] + m * p.stride[2];
        if (p.vec) {  // unit stride and 16-byte aligned rows
#pragma unroll
            for (int i = 0; i < kPieces; i++) {
                reinterpret_cast<uint4*>(r.lo)[i] = *reinterpret_cast<const uint4*>(src + 32 * i + 8 * quarter);
                reinterpret_cast<uint4*>(r.hi)[i] = *reinterpret_cast<const uint4*>(src + kD / 2 + 32 * i + 8 * quarter);
            }
        } else {
#pragma unroll
            for (int i = 0; i < kPairs; i++) {
                r.lo[i] = src[stage_pair(quarter, i) * p.stride[3]];
                r.hi[i] = src[(kD / 2 + stage_pair(quarter, i)) * p.stride[3]];
            }
        }
    };
    // 128 dims: the softmax scale (times log2 e) rides on the staged queries, so the attention kernels exponentiate the
    // products as they come out of the matrix pipe: rotated with the eager path's roundings, then one rounding
    // of the product with qscale (the eager path rounds the product with sqrt(scale) there; log2 e has to ride
    // on one of the two operands, and noise on a query averages out over the rows a score sums)
    auto finish_row = [&](int64_t bh, Row& r) {
        if (bh >= nbh) return;
        uint32_t* lw = reinterpret_cast<uint32_t*>(r.lo);
        uint32_t* hw = reinterpret_cast<uint32_t*>(r.hi);
#pragma unroll
        for (int k = 0; k < kPairs / 2; k++) {  // on packed pairs, as in stage_keys_block
            if (p.q_pos) {
                rw[k].rotate(lw[k], hw[k], p.qscale, true, lw[k], hw[k]);
            } else {
                lw[k] = Mma<T>::pack2(Mma<T>::lo_f(lw[k]) * p.qscale, Mma<T>::hi_f(lw[k]) * p.qscale);
                hw[k] = Mma<T>::pack2(Mma<T>::lo_f(hw[k]) * p.qscale, Mma<T>::hi_f(hw[k]) * p.qscale);
            }
        }
        T* dst = (T*)p.qr + (bh * p.Q + m) * kD;
#pragma unroll
        for (int i = 0; i < kPieces; i++) {
            *reinterpret_cast<uint4*>(dst + 32 * i + 8 * quarter) = reinterpret_cast<uint4*>(r.lo)[i];
            *reinterpret_cast<uint4*>(dst + kD / 2 + 32 * i + 8 * quarter) = reinterpret_cast<uint4*>(r.hi)[i];
        }
    };
    // two rows per trip, both requested before either is rotated: a block is a chain of trips to
    // memory, and this halves it
    for (int64_t bh = share_i; bh < nbh; bh += 2 * n_share) {
        Row r0, r1;
        load_row(bh, r0);
        load_row(bh + n_share, r1);
        finish_row(bh, r0);
        finish_row(bh + n_share, r1);
    }
}

// One launch stages queries and keys and writes the weights of the score sums: the three are independent.  1-D grid: the
// key blocks (k_bx x k_by) first, then the query blocks (q_bx x q_by), which are short and fill the ragged end of the key
// blocks, then the blocks with weights (a launch of their own took 5 us of 305 with 509 rows over 16 K slots).
struct StageGrid {
    int q_bx, q_by, k_bx, k_by;
};
struct StageWeights {
    float *w_ema, *w_new;
    double beta;
    int* key_order;   // written by the first block where the staging blocks find their keys themselves
    int* n_visible;
    int blocks;       // with weights; those behind them keep scores
    KeptScores kept;
};
template <typename T, int kD>
__global__ void __launch_bounds__(256) stage_kernel(StageParams sp, StageQParams sq, StageGrid g, StageWeights sw) {
    __shared__ __align__(16) StageLds<kD> lds;
    const int nk = g.k_bx * g.k_by;
    int id = (int)blockIdx.x - (sp.own_order ? 1 : 0);
    if (id < 0) {
        key_order_block<256>(sp.order_mask, sp.n_cached, sp.n_chunk, sw.key_order, sw.n_visible);
    } else if (id < nk) {
        stage_keys_block<T, kD>(sp, id % g.k_bx, id / g.k_bx, g.k_by, lds);
    } else {
        id -= nk;
        const int nq = g.q_bx * g.q_by;
        if (id < nq) stage_q_block<T, kD>(sq, id % g.q_bx, id / g.q_bx, g.q_by, lds);
        else if (id < nq + sw.blocks) weights_at<T>(sw.w_ema, sw.w_new, sq.Q, sw.beta, (int64_t)(id - nq) * 256 + threadIdx.x);
        else keep_scores<T, 256>(sw.kept, id - nq - sw.blocks, threadIdx.x);
    }
}

// ---------------------------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------------------------
struct FwdParams {
    const void* qr;   // (B*H, Q, D)
    const void* kr;   // (B*KVH, n_pad/64) K tile images
    const void* vt;   // (B*KVH, n_pad/64) V^T tile images
    const unsigned long long* tile_vis;
    void* out;
    int64_t out_stride[4];
    float* lse;       // (B*H, Q) natural log
    float* lse2;      // (B*H, Q) minus the log2-domain normaliser, consumed by the column pass
    int64_t B, H, KVH, Q, N, Nc, n_pad;
    int G;            // heads per kv head: a workgroup takes 256 consecutive rows of the kv head's (position, head) pairs, position-major
    float scale_log2; // with 64 dims: a logit's factor on its way to a power of two
    int n_qt, xcd_aware;  // query tiles per kv head; 1-D XCD-aware block order
    // Few query rows (short chunks, one stream) would leave most of the chip idle: the key tiles of a query tile
    // are then dealt out over n_split workgroups, each of which leaves a partial result (its rows normalised by
    // its own sums, fp32) and the log2-domain normaliser of its share; a small kernel merges them.
    int n_split;
    float* part_o;    // (n_split, B*H*Q, D)
    float* part_l2;   // (n_split, B*H*Q): m_ref + log2(l) of the share, -inf when it holds no visible key
    const int* n_visible;  // when the keys were staged in key order: the number of cached keys (null: Nc)
};

// LDS tile of rows of 2 kD bytes taken from a row-major matrix (the query tile of the column pass): unpadded
// (the async copy writes 1 KiB per wavefront contiguously); bank conflicts are avoided by XOR-swizzling
// the 16-byte piece index with the row, so that one piece of 16 consecutive rows covers all 256 bytes of banks:
// piece c of row r lives at r * 2 kD + ((c ^ row_swizzle(r)) << 4)
template <int kD>
__device__ inline int row_swizzle(int r) { return kD == 128 ? (r & 15) : ((r >> 1) & 7); }
template <int kD>
__device__ inline int k_lds_off(int r, int c) { return r * (2 * kD) + ((c ^ row_swizzle<kD>(r)) << 4); }

// Software-pipelined forward: eight wavefronts, 32 (head, position) rows each.  Iteration i runs
// the softmax of tile i on the vector ALU while the matrix pipe adds the P.V product of tile i-1
// and computes the logits of tile i+1; neither depends on the softmax in flight, so the two pipes
// overlap inside one wavefront.  LDS: three K stages and four V^T stages.  Iteration i copies K
// tile i+3 and V^T tile i+2, which are first read in iteration i+2: the barrier between two
// iterations waits only for the copies of the iteration before the last one (those of the last one
// stay in flight across it), and the first operands of an iteration can be fetched before its barrier.
constexpr int kKStages = 3, kVStages = 4;
__host__ __device__ constexpr int pipe_stages_lds(int head_dim) { return (kKStages + kVStages) * head_dim * 2 * kBN; }   // K0 K1 K2 V0 V1 V2 V3
// stages, one visibility word and one work-list entry per key tile
inline int64_t pipe_lds_bytes(int64_t n_pad, int head_dim) { return pipe_stages_lds(head_dim) + (n_pad / kBN) * 12; }
constexpr int64_t kLdsLimit = 160 * 1024;

template <typename T, int kD>
__global__ void __launch_bounds__(512) fwd_pipe_kernel(FwdParams p) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int kPipeStage = kD * 2 * kBN, kPipeLds = pipe_stages_lds(kD);
    constexpr int kThreads = 512, kBlocksPerWave = kPipeStage / 8192, kAhead = 3;
    constexpr bool kEx = kExact<kD>;
    constexpr int kTerms = kEx ? 3 : 1;                  // 16-bit terms of a probability
    constexpr int kDB = kD / 32, kKK = kD / 16;          // blocks of 32 dims; contraction steps of the logits
    constexpr int kPvOps = 4 * kDB, kQkSlots = 2 * kKK;  // V^T pieces of a tile; matrix instructions of its logits
    constexpr int kPvSlots = kPvOps * kTerms;            // matrix instructions of its P.V product
    const int Nc = p.n_visible ? *p.n_visible : (int)p.Nc;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    int bkv_i = blockIdx.y, qt_i = blockIdx.x;
    // With 8 | B * KVH the grid is 1-D: workgroup ids go round the 8 XCDs, and all query tiles of a kv
    // head are put on one XCD, so its K / V^T stream is fetched from HBM into one L2 instead of eight
    // (same run time, a fifth of the HBM reads).
    if (p.xcd_aware) {
        const int id = blockIdx.x, jq = id >> 3, per = p.n_qt * p.n_split;
        bkv_i = (id & 7) + 8 * (jq / per);
        qt_i = jq % per;
    }
    const int split_i = qt_i % p.n_split;   // this workgroup's share of the query tile's key tiles
    qt_i /= p.n_split;
    // Later query tiles see more chunk keys, so they go first: the compute units that finish the light
    // tiles of one round early pick up the heavy tiles of the next (two rounds of workgroups then cost
    // light + heavy everywhere instead of heavy + heavy on the slowest unit).
    qt_i = p.n_qt - 1 - qt_i;
    const int64_t bkv = bkv_i;
    int64_t kvh;
    const int64_t b = div_index(bkv, p.KVH, kvh);
    // rows of a kv head are its (position, head) pairs, position-major: row rf = position * G + head.  A workgroup
    // takes 256 consecutive ones whatever G is (7 heads per kv head: 36 4/7 positions), so every wavefront has
    // 32 real rows and the number of workgroups is Q * G / 256, not Q / floor(256 / G).
    const int m0 = qt_i * kRows / p.G;
    int m_hi = (qt_i * kRows + kRows - 1) / p.G;
    if (m_hi > (int)p.Q - 1) m_hi = (int)p.Q - 1;
    const int n_tiles = (Nc + m_hi) / kBN + 1;
    const int tiles_cap = (int)(p.n_pad / kBN);
    unsigned long long* vis_lds = reinterpret_cast<unsigned long long*>(smem + kPipeLds);
    int* list_lds = reinterpret_cast<int*>(smem + kPipeLds + 8 * tiles_cap);
    const uint32_t smem_addr = lds_address(smem);

    // ---- the query row this lane owns as MFMA column `col`, requested first: its trip to memory is that of the words below.
    // With the work list by all wavefronts, a first wait for the first K tile alone and (128 dims) shares that leave through
    // LDS a launch takes 1 to 2 % less (32 heads, us: 509 rows x 16 K slots 143.8 -> 141.1, 300 x 16 K 113.4 -> 111.9, 2048 x 8 K
    // 265.7 -> 264.4, 4096 x 64 K 3533 -> 3524); one by one only the shares show, at their place below.
    int row_m;
    uint4 qreg[kKK];
    {
        const int rf = qt_i * kRows + wave * 32 + col;
        const int g = rf % p.G;
        row_m = rf / p.G;
        const int64_t row_h = kvh * p.G + g;
        const bool row_ok = row_m < p.Q;
        const T* qrow = (const T*)p.qr + ((b * p.H + row_h) * p.Q + row_m) * kD;
        // one branch around all of them: a choice per piece makes eight branches, each with a wait for its own piece at the end
#pragma unroll
        for (int kk = 0; kk < kKK; kk++) qreg[kk] = make_uint4(0, 0, 0, 0);
        if (row_ok) {
#pragma unroll
            for (int kk = 0; kk < kKK; kk++) qreg[kk] = *reinterpret_cast<const uint4*>(qrow + 16 * kk + 8 * half);
        }
    }
    // ---- work list: tiles with at least one visible key; bit 31 marks tiles that need masking.  Every wavefront counts a stretch
    // of the tiles and then writes its entries behind those of the stretches before it.
    constexpr int kWaves = kThreads / CKV_WAVE;
    int* counts = reinterpret_cast<int*>(smem);   // of the wavefronts; no copy is on its way yet
    const int per_wave = (n_tiles + 64 * kWaves - 1) / (64 * kWaves) * 64;
    const int t_first = wave * per_wave, t_last = t_first + per_wave < n_tiles ? t_first + per_wave : n_tiles;
    int mine = 0;
    for (int base = t_first; base < t_last; base += 64) {
        const int t = base + lane;
        const unsigned long long v = t < t_last ? p.tile_vis[t] : 0ull;
        if (t < t_last) vis_lds[t] = v;
        mine += __popcll(__ballot(v != 0ull));
    }
    if (lane == 0) counts[wave] = mine;
    __syncthreads();
    int cnt = 0, n_work_all = 0;
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
        const int c = __builtin_amdgcn_readfirstlane(counts[w]);
        if (w < wave) cnt += c;
        n_work_all += c;
    }
    for (int base = t_first; base < t_last; base += 64) {
        const int t = base + lane;
        const unsigned long long v = t < t_last ? vis_lds[t] : 0ull;
        const unsigned long long bal = __ballot(v != 0ull);
        if (v != 0ull) {
            const bool partial = (v != ~0ull) || (t * kBN + kBN - 1 - Nc > m0);
            list_lds[cnt + __popcll(bal & ((1ull << lane) - 1ull))] = t | (partial ? (int)0x80000000 : 0);
        }
        cnt += __popcll(bal);
    }
    __syncthreads();
    // The query rows are there (the words were behind them): said here, or the compiler waits for them at their first use, where
    // the copies are on their way too.
#pragma unroll
    for (int kk = 0; kk < kKK; kk++) asm volatile("" : "+v"(qreg[kk].x), "+v"(qreg[kk].y), "+v"(qreg[kk].z), "+v"(qreg[kk].w));
    const int j_first = n_work_all * split_i / p.n_split;
    const int n_work = n_work_all * (split_i + 1) / p.n_split - j_first;
    list_lds += j_first;

    f32x16 oacc[kDB];
#pragma unroll
    for (int dt = 0; dt < kDB; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) oacc[dt][v] = 0.f;
    // m_ref: the reference the row's logits and sums are relative to; m_run: running maximum relative to it
    // (-inf until the row has seen a key); l_run: partial over this lane's keys, halves are added at the end
    float m_ref = 0.f, m_run = -INFINITY, l_run = 0.f;
    f32x16 cinit;  // -m_ref in every element: what the matrix pipe starts a tile's logits from (64 dims: zero)
#pragma unroll
    for (int v = 0; v < 16; v++) cinit[v] = 0.f;
    // A row's largest probability lies at 2^kHead when its reference is set and stays below 2^kShiftAt until that moves.
    // 64 dims: as high as float16 allows.  Three float16 terms hold all 24 bits of a probability down to 2^-12 of the row's
    // largest and resolve 2^-37 of that, which a float16 result can only show in a dim where the values of the row's largest
    // keys are zero and others' above 2^12.  (bfloat16 terms, which hold every bit, would need V in two halves and twice the
    // products.)
    constexpr float kShiftAt = kEx ? 15.f : 10.f, kHead = kEx ? 12.f : 0.f;
    const float c2 = p.scale_log2;
    // a logit as it leaves the matrix pipe, as a power of two
    auto prob = [&](float x) { return __builtin_amdgcn_exp2f(kEx ? fmaf(x, c2, -m_ref) : x); };

    // ---- LDS byte offset of this lane's operand pieces inside the stage being read (pieces of later
    // contraction steps / row blocks are at compile-time distances); moved from stage to stage in place.
    // k_base: key row `col` of the K stage with the next logits' tile; v_base: dim row `col` of the V^T
    // stage with the tile to multiply.
    int k_base = k_image_off(col, half);
    int v_base = v_image_off<kD>(col, half) + (kKStages + kVStages - 1) * kPipeStage;
    int k_rd = 0, v_rd = kVStages - 1;  // the stages k_base / v_base point at
    auto advance_k = [&]() {
        k_base += k_rd == kKStages - 1 ? -(kKStages - 1) * kPipeStage : kPipeStage;
        k_rd = k_rd == kKStages - 1 ? 0 : k_rd + 1;
    };
    auto advance_v = [&]() {
        v_base += v_rd == kVStages - 1 ? -(kVStages - 1) * kPipeStage : kPipeStage;
        v_rd = v_rd == kVStages - 1 ? 0 : v_rd + 1;
    };
    // K piece (kk, ks): contraction step kk of key rows 32ks ..; V^T piece (s, dt): step s of dim rows 32dt ..
    auto k_piece = [&](int kk, int ks) { return *reinterpret_cast<const uint4*>(smem + k_base + kk * 2048 + ks * 512); };
    auto v_piece = [&](int s_, int dt) { return *reinterpret_cast<const uint4*>(smem + v_base + s_ * (32 * kD) + dt * 512); };
    const uint32_t copy_off = lane * 16;  // a wavefront copies 1 KiB blocks of an image as they are
    const char* kbase = (const char*)uniform_ptr((const char*)p.kr + bkv * p.n_pad * kD * (int64_t)sizeof(T));
    const char* vbase = (const char*)uniform_ptr((const char*)p.vt + bkv * p.n_pad * kD * (int64_t)sizeof(T));
    constexpr int kTileBytes = kBN * kD * (int)sizeof(T);

    // one 1 KiB block (j = 0, 1) of a tile into K stage `stage` / V^T stage `stage`
    auto copy_k = [&](int t, int stage, int j) {
        const int blk = (wave * kBlocksPerWave + j) * 1024;
        async_copy16(kbase + (int64_t)t * kTileBytes + blk, copy_off, smem_addr + stage * kPipeStage + blk);
    };
    auto copy_v = [&](int t, int stage, int j) {
        const int blk = (wave * kBlocksPerWave + j) * 1024;
        async_copy16(vbase + (int64_t)t * kTileBytes + blk, copy_off, smem_addr + (kKStages + stage) * kPipeStage + blk);
    };
    auto work = [&](int j) { return __builtin_amdgcn_readfirstlane(list_lds[j < n_work ? j : n_work - 1]); };

    // logits of the K tile k_base points at: s[ks][v] = key 32ks + 8(v/4) + 4half + v%4, query column col
    auto qk = [&](f32x16(&s)[2]) {
#pragma unroll
        for (int ks = 0; ks < 2; ks++) s[ks] = cinit;
#pragma unroll
        for (int kk = 0; kk < kKK; kk++) {
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                s[ks] = Mma<T>::mma(k_piece(kk, ks), qreg[kk], s[ks]);
            }
        }
    };
    uint32_t pk[kTerms][4][4];  // P^T of one tile as the B operands of the four P.V contraction steps
    // the probabilities q0, q1 as pair w of step st, and their sum (of what the product uses)
    auto put_pair = [&](int st, int w, float q0, float q1, float sum) -> float {
        uint32_t t = Mma<T>::pack2(q0, q1);
        pk[0][st][w] = t;
        if constexpr (!kEx) return Mma<T>::sum2(t, sum);
        sum += q0 + q1;
#pragma unroll
        for (int i = 1; i < kTerms; i++) {
            q0 -= Mma<T>::lo_f(t);
            q1 -= Mma<T>::hi_f(t);
            t = Mma<T>::pack2(q0, q1);
            pk[i][st][w] = t;
        }
        return sum;
    };
    auto p_operand = [&](int term, int st) { return make_uint4(pk[term][st][0], pk[term][st][1], pk[term][st][2], pk[term][st][3]); };
    // O^T += V^T P^T with the V^T tile v_base points at
    auto pv = [&]() {
#pragma unroll
        for (int s = 0; s < 4; s++) {
#pragma unroll
            for (int dt = 0; dt < kDB; dt++) {
                const uint4 a = v_piece(s, dt);
#pragma unroll
                for (int i = 0; i < kTerms; i++) oacc[dt] = Mma<T>::mma(a, p_operand(i, s), oacc[dt]);
            }
        }
    };
    // One 64-bit word per lane says which keys of the tile its query row may see (visible slot and not
    // later than the row); it is shifted once so that the bit of every element sits at a compile-time
    // position.  Few live values: this path must not push the loop's registers into scratch.
    auto mask_tile = [&](int entry, f32x16(&s)[2]) {
        const int t = entry & 0x7fffffff;
        unsigned long long allowed = vis_lds[t];
        const int limit = row_m - (t * kBN - Nc);  // last key index of the tile the row may see, if it is a chunk tile
        if (t * kBN + kBN - 1 >= Nc) {             // the tile holds chunk keys
            const int first_chunk = Nc - t * kBN;  // <= 0 when the whole tile is chunk
            unsigned long long causal = limit >= 63 ? ~0ull : (limit < 0 ? 0ull : ((2ull << limit) - 1ull));
            if (first_chunk > 0) causal |= (1ull << first_chunk) - 1ull;  // cached keys in front of the chunk: always allowed
            allowed &= causal;
        }
        allowed >>= 4 * half;
        const uint32_t lo = (uint32_t)allowed, hi = (uint32_t)(allowed >> 32);
#pragma unroll
        for (int ks = 0; ks < 2; ks++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int bit = 8 * (v >> 2) + (v & 3);  // key 32 ks + bit + 4 half
                const bool ok = ((ks ? hi : lo) >> bit) & 1u;
                s[ks][v] = ok ? s[ks][v] : -INFINITY;
            }
    };
    float alpha = 1.f;  // rescale of the accumulator owed since the last softmax
    // the running maximum settles after a few tiles: rescale only when some row of the wavefront moved
    auto rescale = [&]() {
        if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0ull) {
#pragma unroll
            for (int dt = 0; dt < kDB; dt++)
#pragma unroll
                for (int v = 0; v < 16; v++) oacc[dt][v] *= alpha;
        }
    };

    // Iteration i, written in issue order: 32 slots, each one matrix instruction (slots 0..15: P.V of tile i-1 out of the
    // V^T stage at v_base, slots 16..31: logits of tile i+1 out of the K stage at k_base; with 64 dims 24 slots of P.V, three
    // terms after another with each operand, and 8 of logits), the LDS read of the operand kAhead operands ahead, and a
    // slice of the softmax of tile i.
    // Scheduling barriers keep the slots as written, so matrix and vector instructions alternate
    // inside the wavefront.  The probabilities of tile i overwrite those of tile i-1 piece by piece,
    // each after its last use by the P.V product.  The copies (V^T tile t_v = i+2 into stage v_wr, K
    // tile t_k = i+3 into stage k_wr, both last read in iteration i-1) go out one at a time, a quarter
    // of the slots apart.
    // pre[]: on entry the operands of slots 0..kAhead-1, read before the barrier; on exit those
    // of the next iteration.
    // fetch_idx / fetched: the work-list entry four tiles ahead is read from LDS in the middle of the
    // slots, so its latency is never waited for.
    auto iteration = [&](auto with_pv, int entry, int t_v, int t_k, f32x16(&s_cur)[2], f32x16(&s_nxt)[2],
                         uint4(&pre)[kAhead], int fetch_idx, int& fetched) {
        constexpr bool kPV = decltype(with_pv)::value;
        constexpr int kSlots = kPV ? kPvSlots + kQkSlots : kQkSlots, kQk0 = kPV ? kPvSlots : 0;
        constexpr int kCopies = 2 * kBlocksPerWave, kCopyStep = kSlots / kCopies;
        const int v_wr = v_rd == 0 ? kVStages - 1 : v_rd - 1;   // (v_rd + 3) % 4
        const int k_wr = k_rd == 0 ? kKStages - 1 : k_rd - 1;   // (k_rd + 2) % 3
        if (entry < 0) mask_tile(entry, s_cur);
        rescale();  // tile i-2 is in the accumulator; tile i-1, scaled for the newer reference, is added below
        constexpr int kOps = (kPV ? kPvOps : 0) + kQkSlots, kQkOp0 = kPV ? kPvOps : 0;
        auto operand = [&](int k) -> uint4 {
            if (k >= kQkOp0) {
                const int j = k - kQkOp0;  // K piece (kk, ks) = (j % kKK, j / kKK): one 32-key block after the other
                return k_piece(j % kKK, j / kKK);
            }
            return v_piece(k / kDB, k % kDB);
        };
        uint4 ops[kOps];
        if (kPV) {
#pragma unroll
            for (int k = 0; k < kAhead; k++) ops[k] = pre[k];
        }
        float mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        float shift = 0.f, rs = 0.f;
        // Softmax schedule.  With P.V: slots 0..7 running maxima (the last one also reduces them), then one
        // pair of probabilities per slot: the first 32-key block of the tile is consumed by slot 15 and the
        // second by slot 23, just before the matrix pipe starts to overwrite them with the next tile's
        // logits (slots 16..23 and 24..31), so one set of logit registers serves both tiles.
        // Three terms: maxima in slots 0..7, probabilities in slots 12..27, so that a pair is stored (slots 13..28) after
        // the last of the six slots that use the one before it (step st: slots 6 st .. 6 st + 5).
        constexpr int kMaxSlots = kPV ? (kEx ? 8 : kPvSlots / 2) : kQkSlots / 4;  // slots with running maxima
        constexpr int kMaxPer = 32 / kMaxSlots;            // logits per such slot
        constexpr int kExpFirst = kPV && kEx ? kPvSlots / 2 : kMaxSlots;  // first slot with probabilities
        constexpr int kExpPer = kPV && kEx ? 1 : 16 / (kPV ? kPvSlots : kQkSlots / 2);  // pairs per slot
        static_assert(kExpFirst + 16 / kExpPer < kSlots, "the last pair is stored a slot after its exponentials");
        float q0[kExpPer], q1[kExpPer];                    // exponentials of the previous slot, packed one slot later
        int raw_entry = 0;
        bool moved = true;                                 // some row of the wavefront takes a new reference
        auto slot = [&](int k) {
            const int op = kPV && k < kQk0 ? k / kTerms : kQkOp0 + k - kQk0;
            if (kPV && op + kAhead < kOps && (k >= kQk0 || k % kTerms == 0)) ops[op + kAhead] = operand(op + kAhead);
            if (k % kCopyStep == 1) {
                const int q = k / kCopyStep;               // the V^T blocks, then the K blocks
                if (q < kBlocksPerWave) copy_v(t_v, v_wr, q);
                else copy_k(t_k, k_wr, q - kBlocksPerWave);
            }
            if (k == 4) raw_entry = list_lds[fetch_idx];
            if (!kPV) {
                // the first iteration of a workgroup: the next tile's logits follow the slots (below)
            } else if (k >= kQk0) {
                const int j = k - kQk0;
                s_nxt[j / kKK] = Mma<T>::mma(ops[op], qreg[j % kKK], j % kKK == 0 ? cinit : s_nxt[j / kKK]);
            } else {
                const int st = op / kDB, dt = op % kDB;
                oacc[dt] = Mma<T>::mma(ops[op], p_operand(k % kTerms, st), oacc[dt]);
            }
            if (k < kMaxSlots) {
#pragma unroll
                for (int e = 0; e < kMaxPer; e++) {
                    const int idx = k * kMaxPer + e;
                    mx[e & 3] = fmaxf(mx[e & 3], s_cur[idx >> 4][idx & 15]);
                }
                if (k == kMaxSlots - 1) {
                    // The logits are relative to the row's reference m_ref (it rides on the accumulator
                    // initialisation of the matrix pipe), m_run is the running maximum relative to it.
                    // The reference moves only when the maximum has outgrown it by kShiftAt, or with the
                    // first visible key of a row; until then a probability is a bare exponential.
                    float m = fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]));
                    m = half_max(m);
                    if constexpr (kEx) m = fmaf(m, c2, -m_ref);
                    const float m_new = fmaxf(m_run, m);
                    const bool first = m_run == -INFINITY && m != -INFINITY;
                    const bool sh = first || m_new > kShiftAt;
                    moved = __builtin_amdgcn_ballot_w64(sh) != 0ull;
                    shift = sh ? m_new - kHead : 0.f;
                    alpha = sh ? (first ? 0.f : __builtin_amdgcn_exp2f(-shift)) : 1.f;
                    m_run = m_new - shift;
                    m_ref += shift;
                }
            } else {
#pragma unroll
                for (int r = 0; r < kExpPer; r++) {
                    const int prev = (k - 1 - kExpFirst) * kExpPer + r;  // pair computed one slot ago
                    if (prev >= 0 && prev < 16) {
                        const int ks = prev >> 3, v = 2 * (prev & 7);
                        rs = put_pair(2 * ks + (v >> 3), (v & 7) >> 1, q0[r], q1[r], rs);
                    }
                    const int pair = (k - kExpFirst) * kExpPer + r;      // (ks, v) = (pair / 8, 2 * (pair % 8))
                    if (pair < 16) {
                        const int ks = pair >> 3, v = 2 * (pair & 7);
                        q0[r] = prob(s_cur[ks][v]);
                        q1[r] = prob(s_cur[ks][v + 1]);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int k = 0; k < kMaxSlots; k++) slot(k);
        if (!kEx && moved) {
            // rare after the first tiles: this tile's logits come down to the new reference here, the later
            // ones through the accumulator initialisation
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int v = 0; v < 16; v++) s_cur[ks][v] -= shift;
#pragma unroll
            for (int v = 0; v < 16; v++) cinit[v] = -m_ref;
        }
#pragma unroll
        for (int k = kMaxSlots; k < kSlots; k++) slot(k);
        l_run = l_run * alpha + rs;
        fetched = __builtin_amdgcn_readfirstlane(raw_entry);
        if (!kPV) qk(s_nxt);  // once per workgroup, not interleaved: the logits of tile 1
        // on to the stages of tiles i and i+2; first operands of the next iteration: V^T tile i,
        // complete since the last barrier
        advance_v();
        advance_k();
#pragma unroll
        for (int k = 0; k < kAhead; k++) pre[k] = v_piece(k / kDB, k % kDB);
        // keep the packed probabilities in this region (they are next read after the barrier)
#pragma unroll
        for (int i = 0; i < kTerms; i++)
#pragma unroll
            for (int st = 0; st < 4; st++) {
                const uint4 w = p_operand(i, st);
                asm volatile("" ::"v"(w.x), "v"(w.y), "v"(w.z), "v"(w.w));
            }
    };

    f32x16 sA[2], sB[2];
    uint4 pre[kAhead];
    if (n_work > 0) {
#pragma unroll
        for (int j = 0; j < kBlocksPerWave; j++) copy_k(work(0) & 0x7fffffff, 0, j);
#pragma unroll
        for (int j = 0; j < kBlocksPerWave; j++) copy_k(work(1) & 0x7fffffff, 1, j);
#pragma unroll
        for (int j = 0; j < kBlocksPerWave; j++) copy_v(work(0) & 0x7fffffff, 0, j);
#pragma unroll
        for (int j = 0; j < kBlocksPerWave; j++) {
            copy_k(work(2) & 0x7fffffff, 2, j);
            copy_v(work(1) & 0x7fffffff, 1, j);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70 + 4 * kBlocksPerWave);  // vmcnt: the first K tile is there
        __syncthreads();
        qk(sA);
        advance_k();
        // iteration 0: nothing to multiply by V yet.  e0 .. e3: work-list entries of tiles i .. i+3
        auto clamp_idx = [&](int j) { return j < n_work ? j : n_work - 1; };
        int e0 = work(0), e1 = work(1), e2 = work(2), e3 = work(3), e4 = 0;
        __builtin_amdgcn_s_waitcnt(0x0F70 + 2 * kBlocksPerWave);  // the second one and the first V^T tile too
        __syncthreads();                     // every wavefront is done with K stage 0
        iteration(std::false_type{}, e0, e2 & 0x7fffffff, e3 & 0x7fffffff, sA, sB, pre, clamp_idx(4), e4);
        // all copies but those of the iteration just finished have landed
        constexpr int kWaitOlder = 0x0F70 + 2 * kBlocksPerWave;   // vmcnt
        for (int i = 1; i < n_work; i += 2) {
            e0 = e1; e1 = e2; e2 = e3; e3 = e4;
            __builtin_amdgcn_s_waitcnt(kWaitOlder);
            __syncthreads();
            iteration(std::true_type{}, e0, e2 & 0x7fffffff, e3 & 0x7fffffff, sB, sA, pre, clamp_idx(i + 4), e4);
            if (i + 1 < n_work) {
                e0 = e1; e1 = e2; e2 = e3; e3 = e4;
                __builtin_amdgcn_s_waitcnt(kWaitOlder);
                __syncthreads();
                iteration(std::true_type{}, e0, e2 & 0x7fffffff, e3 & 0x7fffffff, sA, sB, pre, clamp_idx(i + 5), e4);
            }
        }
        // the P.V product of the last tile; the copies still in flight are repeats that nobody reads
        rescale();
        pv();
        __builtin_amdgcn_s_waitcnt(0x0F70);
    }

    if constexpr (kEx) {
        // The matrix pipe multiplies every row by every value, and zero times infinity or NaN is NaN; a value whose key has
        // probability zero counts for nothing, whatever it holds.  A wavefront whose accumulators come out finite has met no
        // such value.  Otherwise it goes over its tiles once more, straight from memory, with the references it has found:
        // finite values times float32 probabilities, the others where the probability is above zero.
        float zero = 0.f;   // or NaN
#pragma unroll
        for (int dt = 0; dt < kDB; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) zero = fmaf(oacc[dt][v], 0.f, zero);
        if (__builtin_amdgcn_ballot_w64(zero != 0.f) != 0ull) {
            f32x16 none;
#pragma unroll
            for (int v = 0; v < 16; v++) none[v] = 0.f;
#pragma unroll
            for (int dt = 0; dt < kDB; dt++) oacc[dt] = none;
            for (int j = 0; j < n_work; j++) {
                const int entry = work(j);
                const char* kt = kbase + (int64_t)(entry & 0x7fffffff) * kTileBytes + k_image_off(col, half);
                const char* vt = vbase + (int64_t)(entry & 0x7fffffff) * kTileBytes + v_image_off<kD>(col, half);
                f32x16 s[2] = {none, none};
#pragma unroll
                for (int kk = 0; kk < kKK; kk++)
#pragma unroll
                    for (int ks = 0; ks < 2; ks++)
                        s[ks] = Mma<T>::mma(*reinterpret_cast<const uint4*>(kt + kk * 2048 + ks * 512), qreg[kk], s[ks]);
                if (entry < 0) mask_tile(entry, s);
#pragma unroll
                for (int ks = 0; ks < 2; ks++)
#pragma unroll
                    for (int v = 0; v < 16; v++) s[ks][v] = prob(s[ks][v]);
#pragma unroll
                for (int dt = 0; dt < kDB; dt++) {
                    f32x16 up = none, down = none;   // how many infinities of either sign a sum holds, a NaN being both
#pragma unroll
                    for (int st = 0; st < 4; st++) {
                        const uint4 a = *reinterpret_cast<const uint4*>(vt + st * (32 * kD) + dt * 512);
                        const uint32_t w[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
                        for (int e = 0; e < 8; e++) {   // key 16 st + 8 (e / 4) + 4 half + e % 4
                            const float x = e & 1 ? Mma<T>::hi_f(w[e >> 1]) : Mma<T>::lo_f(w[e >> 1]);
                            const float pe = s[st >> 1][8 * (st & 1) + e], counts = pe > 0.f ? 1.f : 0.f;
                            auto f32 = [](float x_, float y_, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(x_, y_, c, 0, 0, 0); };
                            oacc[dt] = f32(isfinite(x) ? x : 0.f, pe, oacc[dt]);
                            up = f32(x == INFINITY || isnan(x) ? 1.f : 0.f, counts, up);
                            down = f32(x == -INFINITY || isnan(x) ? 1.f : 0.f, counts, down);
                        }
                    }
#pragma unroll
                    for (int v = 0; v < 16; v++) oacc[dt][v] += (up[v] > 0.f ? INFINITY : 0.f) + (down[v] > 0.f ? -INFINITY : 0.f);
                }
            }
        }
    }

    // epilogue: lane owns d = 32dt + 8(v/4) + 4half + v%4 of its query row
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    if (p.n_split > 1) {
        // a share of the key tiles: the row normalised by the share's own sum, and the share's normaliser
        auto row_of = [&](int r, int& m) {   // of part_o and part_l2: row r of this wavefront's 32, at position m
            const int rf = qt_i * kRows + wave * 32 + r;
            m = rf / p.G;
            return (int64_t)split_i * p.B * p.H * p.Q + (b * p.H + kvh * p.G + rf % p.G) * p.Q + m;
        };
        const bool any = l_tot != 0.f;   // a NaN is not nothing: it has to reach the merge
        const float inv_p = any ? 1.f / l_tot : 0.f;
        if constexpr (kD == 64) {
            // A row is 256 bytes and half of it all that the stages have room for: stretches of 128 bytes, which do not pay for the
            // way through LDS (8 heads x 148 rows x 5236 keys in shares: 23.9 us that way, 23.1 so; 16 x 700 x 2200: 27.0, 26.6).
            if (row_m < p.Q) {
                int m;
                float* po = p.part_o + row_of(col, m) * kD + 4 * half;
#pragma unroll
                for (int dt = 0; dt < kDB; dt++)
#pragma unroll
                    for (int v4 = 0; v4 < 4; v4++)
                        *reinterpret_cast<float4*>(po + 32 * dt + 8 * v4) =
                            make_float4(oacc[dt][4 * v4] * inv_p, oacc[dt][4 * v4 + 1] * inv_p, oacc[dt][4 * v4 + 2] * inv_p,
                                        oacc[dt][4 * v4 + 3] * inv_p);
            }
        } else {
            // Through LDS, half of the dims at a time, so that a store is whole stretches of 256 bytes of four rows: a lane's own
            // 16 bytes have one neighbour in each of 32 rows (32 heads x 1024 rows x 16 K slots 249.4 -> 245.8 us, 300 rows 113.0
            // -> 111.9).
            constexpr int kStep = kD / 2, kLanes = kStep / 4, kPassRows = CKV_WAVE / kLanes;
            constexpr int kPitch = 4 * kStep + 16;   // bytes; the pad spreads the banks
            static_assert(kWaves * 32 * kPitch <= kPipeLds, "fits in the stages");
            __syncthreads();                      // the tile stages are no longer read
            unsigned char* ow = smem + wave * (32 * kPitch);
#pragma unroll
            for (int d0 = 0; d0 < kD; d0 += kStep) {
#pragma unroll
                for (int dt = d0 / 32; dt < (d0 + kStep) / 32; dt++)
#pragma unroll
                    for (int v4 = 0; v4 < 4; v4++)
                        *reinterpret_cast<float4*>(ow + col * kPitch + (32 * dt - d0 + 8 * v4 + 4 * half) * 4) =
                            make_float4(oacc[dt][4 * v4] * inv_p, oacc[dt][4 * v4 + 1] * inv_p, oacc[dt][4 * v4 + 2] * inv_p,
                                        oacc[dt][4 * v4 + 3] * inv_p);
                __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0)
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int pass = 0; pass < 32 / kPassRows; pass++) {
                    const int r = kPassRows * pass + lane / kLanes;
                    int m;
                    const int64_t row = row_of(r, m);
                    const float4 v = *reinterpret_cast<const float4*>(ow + r * kPitch + (lane % kLanes) * 16);
                    if (m < p.Q) *reinterpret_cast<float4*>(p.part_o + row * kD + d0 + (lane % kLanes) * 4) = v;
                }
                __builtin_amdgcn_wave_barrier();
            }
        }
        if (half == 0 && row_m < p.Q) {
            int m;
            p.part_l2[row_of(col, m)] = any ? m_ref + __builtin_amdgcn_logf(l_tot) : -INFINITY;
        }
        return;
    }
    const int g_row = (qt_i * kRows + wave * 32 + col) % p.G;
    const int64_t row_h = kvh * p.G + g_row;
    const bool row_ok = row_m < p.Q;
    const float inv = 1.f / l_tot;
    const bool rows16 = p.out_stride[3] == 1 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0 && p.out_stride[0] % 8 == 0 &&
                        p.out_stride[1] % 8 == 0 && p.out_stride[2] % 8 == 0;
    if (rows16) {
        // through LDS, so that a row leaves as 16-byte pieces of neighbouring lanes (a lane's own
        // 8-byte pieces would reach memory as partly filled 32-byte sectors)
        constexpr int kRowPitch = 2 * kD + 16;  // bytes; the pad spreads the banks
        __syncthreads();                      // the tile stages are no longer read
        unsigned char* ow = smem + wave * (32 * kRowPitch);
#pragma unroll
        for (int dt = 0; dt < kDB; dt++) {
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
                uint2 w;
                w.x = Mma<T>::pack2(oacc[dt][4 * v4] * inv, oacc[dt][4 * v4 + 1] * inv);
                w.y = Mma<T>::pack2(oacc[dt][4 * v4 + 2] * inv, oacc[dt][4 * v4 + 3] * inv);
                *reinterpret_cast<uint2*>(ow + col * kRowPitch + (32 * dt + 8 * v4 + 4 * half) * (int)sizeof(T)) = w;
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);
        __builtin_amdgcn_wave_barrier();
        // lane = (row in the pass, 16-byte piece)
        constexpr int kPieces = kD / 8, kRowsPass = CKV_WAVE / kPieces;
#pragma unroll
        for (int pass = 0; pass < 32 / kRowsPass; pass++) {
            const int r = kRowsPass * pass + lane / kPieces, piece = lane % kPieces;
            const int rr = qt_i * kRows + wave * 32 + r;
            const int g_r = rr % p.G, m_r = rr / p.G;
            if (m_r < p.Q) {
                const uint4 v = *reinterpret_cast<const uint4*>(ow + r * kRowPitch + piece * 16);
                T* dst = (T*)p.out + b * p.out_stride[0] + (kvh * p.G + g_r) * p.out_stride[1] + m_r * p.out_stride[2];
                *reinterpret_cast<uint4*>(dst + piece * 8) = v;
            }
        }
    } else if (row_ok) {
        T* orow = (T*)p.out + b * p.out_stride[0] + row_h * p.out_stride[1] + row_m * p.out_stride[2];
#pragma unroll
        for (int dt = 0; dt < kDB; dt++) {
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
                const int d = 32 * dt + 8 * v4 + 4 * half;
#pragma unroll
                for (int e = 0; e < 4; e++) orow[(d + e) * p.out_stride[3]] = Elem<T>::from_float(oacc[dt][4 * v4 + e] * inv);
            }
        }
    }
    if (row_ok) {
        if (half == 0) {
            const float l2 = m_ref + __builtin_amdgcn_logf(l_tot);  // v_log_f32 is log2
            p.lse[(b * p.H + row_h) * p.Q + row_m] = l2 * 0.6931471805599453f;
            p.lse2[(b * p.H + row_h) * p.Q + row_m] = -l2;
        }
    }
}

// Merge of the forward kernel's shares by a workgroup of 256 threads: a row per kD / 4 lanes (4 dims each), and with few shares several
// rows a thread, so that eight loads are always on their way at once.  A batch is kShares shares of 8 / kShares rows.
template <int kD>
constexpr int kMergeRows = 256 / (kD / 4);
inline __host__ __device__ int merge_batch(int n_split) { return n_split <= 2 ? 2 : n_split <= 4 ? 4 : 8; }
template <int kD>
inline int64_t merge_blocks(int64_t rows, int n_split) {
    const int64_t per = kMergeRows<kD> * (8 / merge_batch(n_split));
    return (rows + per - 1) / per;
}
template <typename T, int kD, int kShares>
__device__ inline void merge_rows_of(const FwdParams& p, int64_t block) {
    const int64_t rows = p.B * p.H * p.Q;
    constexpr int kLanes = kD / 4, kRowsEach = 8 / kShares;
    const int64_t row0 = block * (kMergeRows<kD> * kRowsEach) + threadIdx.x / kLanes;
    if (row0 >= rows) return;
    const int d4 = threadIdx.x % kLanes;
    int64_t row[kRowsEach];   // past the last row: the first one again
#pragma unroll
    for (int i = 0; i < kRowsEach; i++) row[i] = row0 + i * kMergeRows<kD> < rows ? row0 + i * kMergeRows<kD> : row0;
    float M[kRowsEach];
#pragma unroll
    for (int i = 0; i < kRowsEach; i++) M[i] = -INFINITY;
    for (int s0 = 0; s0 < p.n_split; s0 += kShares) {   // all normalisers first, they are the shorter trip
        float l2[kRowsEach][kShares];
#pragma unroll
        for (int i = 0; i < kRowsEach; i++)
#pragma unroll
            for (int u = 0; u < kShares; u++) l2[i][u] = s0 + u < p.n_split ? p.part_l2[(s0 + u) * rows + row[i]] : -INFINITY;
#pragma unroll
        for (int i = 0; i < kRowsEach; i++)
#pragma unroll
            for (int u = 0; u < kShares; u++) M[i] = fmaxf(M[i], l2[i][u]);
    }
    float L[kRowsEach];
    float4 o[kRowsEach];
#pragma unroll
    for (int i = 0; i < kRowsEach; i++) {
        L[i] = 0.f;
        o[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    for (int s0 = 0; s0 < p.n_split; s0 += kShares) {
        float l2[kRowsEach][kShares];
        float4 v[kRowsEach][kShares];
#pragma unroll
        for (int i = 0; i < kRowsEach; i++)
#pragma unroll
            for (int u = 0; u < kShares; u++) {
                const int s_ = s0 + u < p.n_split ? s0 + u : s0;
                l2[i][u] = s0 + u < p.n_split ? p.part_l2[s_ * rows + row[i]] : -INFINITY;
                v[i][u] = *reinterpret_cast<const float4*>(p.part_o + (s_ * rows + row[i]) * kD + 4 * d4);
            }
#pragma unroll
        for (int i = 0; i < kRowsEach; i++)
#pragma unroll
            for (int u = 0; u < kShares; u++) {
                if (l2[i][u] == -INFINITY) continue;
                const float w = __builtin_amdgcn_exp2f(l2[i][u] - M[i]);
                if (kExact<kD> && w == 0.f) continue;   // a share that has come down to nothing, whatever it holds
                L[i] += w;
                o[i].x = fmaf(v[i][u].x, w, o[i].x); o[i].y = fmaf(v[i][u].y, w, o[i].y);
                o[i].z = fmaf(v[i][u].z, w, o[i].z); o[i].w = fmaf(v[i][u].w, w, o[i].w);
            }
    }
#pragma unroll
    for (int i = 0; i < kRowsEach; i++) {
        if (i > 0 && row[i] == row0) break;
        const float inv = 1.f / L[i];
        int64_t m, h;
        const int64_t b = div_index(div_index(row[i], p.Q, m), p.H, h);
        T* dst = (T*)p.out + b * p.out_stride[0] + h * p.out_stride[1] + m * p.out_stride[2];
        dst[(4 * d4) * p.out_stride[3]] = Elem<T>::from_float(o[i].x * inv);
        dst[(4 * d4 + 1) * p.out_stride[3]] = Elem<T>::from_float(o[i].y * inv);
        dst[(4 * d4 + 2) * p.out_stride[3]] = Elem<T>::from_float(o[i].z * inv);
        dst[(4 * d4 + 3) * p.out_stride[3]] = Elem<T>::from_float(o[i].w * inv);
        if (d4 == 0) {
            const float l2 = M[i] + __builtin_amdgcn_logf(L[i]);  // v_log_f32 is log2
            p.lse[row[i]] = l2 * 0.6931471805599453f;
            p.lse2[row[i]] = -l2;
        }
    }
}
template <typename T, int kD>
__device__ inline void merge_rows(const FwdParams& p, int64_t block) {
    switch (merge_batch(p.n_split)) {
        case 2: return merge_rows_of<T, kD, 2>(p, block);
        case 4: return merge_rows_of<T, kD, 4>(p, block);
        default: return merge_rows_of<T, kD, 8>(p, block);
    }
}

template <typename T, int kD>
__global__ void __launch_bounds__(256) fwd_combine_kernel(FwdParams p) {
    merge_rows<T, kD>(p, blockIdx.x);
}

// ---------------------------------------------------------------------------------------------
// score sums
// ---------------------------------------------------------------------------------------------
struct ColsumParams {
    const void* qr;       // (B*H*Q + kColSlack rows, D)
    const void* kr;
    const unsigned long long* tile_vis;
    const float* lse2;    // (B*H*Q + kColSlack) minus the log2-domain row normalisers
    const float* w_ema;   // (Q + kColSlack), zero beyond Q
    const float* w_new;   // (Q)
    float* colsum;        // (B*H, N)
    int64_t B, H, KVH, Q, N, Nc, n_pad;
    int G;
    int new_mode;
    float scale_log2;     // as in FwdParams
    int nkb, nbkv, xcd_aware, gsplit;  // block order and head split, see the kernel
    const int* n_visible; // when the keys were staged in key order: the number of cached keys (null: Nc), and the
    const int* key_order; // row each key came from
    void* scores;         // (B, H, N) in the tensor dtype, at the row each key came from: takes the place of colsum
    int64_t scores_stride[3];
    int64_t empty_from, empty_to;  // as in StageParams
    int row_shares;       // the query tiles of a key block are shared out over this many workgroups (1: the block's own), each of which
    float* part;          // leaves its sums in (row_shares, B*H, N), see colsum_merge_kernel
    int wnew_uniform;     // every entry of w_new has the value wnew_value (beta rounds to one in the tensor dtype)
    float wnew_value;
    // kMerge: the forward kernel's shares (up to kMergeShares) are still to be merged.  The workgroups behind the first sum_blocks merge
    // rows, and those work the normalisers of a query tile out from the shares' themselves.
    int n_split, sum_blocks;
    FwdParams fwd;
};
constexpr int kMergeShares = 8;

constexpr int kQT2 = 128;                     // query rows per LDS tile of the column pass
constexpr int kCsSub = kQT2 / 32;             // 32-row subtiles of a tile
__host__ __device__ constexpr int cs_stage(int head_dim) { return kQT2 * 2 * head_dim + 2 * kQT2 * 4; }  // Q tile + its lse2 + its weights

// One workgroup = one kv head x 256 keys (64 per wavefront, held in registers as the B operand of
// S = Q K^T).  The (head, query-tile) sequence streams through a double-buffered LDS stage filled
// by asynchronous copies; lane (col, half) owns key column `col` of each 32-key subtile, so the
// weighted column sums never leave the lane.
// kMerge: with the merge of the forward kernel's shares, as an instance of its own: as a branch that is not taken it cost the others 2 %.
template <typename T, int kD, bool kShares, bool kMerge>
__global__ void __launch_bounds__(256, 2) colsum_mfma_kernel(ColsumParams p) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int kKK = kD / 16, kRowBytes = 2 * kD, kCsStage = cs_stage(kD);
    if constexpr (kMerge) {
        if ((int)blockIdx.x >= p.sum_blocks) {
            merge_rows<T, kD>(p.fwd, (int)blockIdx.x - p.sum_blocks);
            return;
        }
    }
    const int Nc = p.n_visible ? *p.n_visible : (int)p.Nc;
    const int N = p.n_visible ? Nc + (int)p.Q : (int)p.N;   // keys somebody can see; those behind get a zero
    float* wnew_lds = reinterpret_cast<float*>(smem + 2 * kCsStage);
    const uint32_t smem_addr = lds_address(smem);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    // Block order.  Key blocks that hold chunk keys cost the most per step (masking on the
    // diagonal, per-element weights), so they are handed out first and never form the tail of
    // the launch.  Workgroup ids go round the 8 XCDs; when the kv heads divide evenly, every
    // block of one kv head runs on one XCD so that head's query stream stays in that XCD's L2.
    // A key block is shared out over gsplit workgroups, each taking G / gsplit heads: units small
    // enough that the last round of workgroups costs little.
    int bkv_i, kb_i, g_first, share = 0;
    const int g_cnt = p.G / p.gsplit;
    {
        const int nkb = p.nkb * p.gsplit, cb0 = (Nc / 256) * p.gsplit, heavy = nkb - cb0;
        int id = blockIdx.x, nb = p.nbkv, first = 0, stride = 1;
        if (kShares) {   // shares outermost: a multiple of the XCDs apart where the order looks at them
            const int blocks = nb * nkb;
            share = id / blocks;
            id -= share * blocks;
        }
        if (p.xcd_aware) {
            first = id & 7;
            stride = 8;
            id >>= 3;
            nb >>= 3;
        }
        int i;
        if (id < nb * heavy) {
            i = id / heavy;
            kb_i = cb0 + id % heavy;
        } else {
            id -= nb * heavy;
            i = id / cb0;
            kb_i = id % cb0;
        }
        bkv_i = first + stride * i;
        g_first = (kb_i % p.gsplit) * g_cnt;
        kb_i /= p.gsplit;
    }
    const int64_t bkv = bkv_i;
    int64_t kvh;
    const int64_t b = div_index(bkv, p.KVH, kvh);
    const int Q = (int)p.Q;
    static_assert(4 * kBN == 256, "a workgroup's keys are four visibility words");
    const int64_t key_blk = (int64_t)kb_i * 256;          // first key of the workgroup
    const int64_t key_w = key_blk + wave * 64;            // first key of this wavefront

    // first query tile that can see any key of the workgroup
    int m_first = (int)(key_blk - Nc);
    if (m_first < 0) m_first = 0;
    m_first = m_first / kQT2 * kQT2;
    const bool chunk_keys = key_blk + 255 >= Nc;  // some key of the workgroup belongs to the chunk
    const int last_nrel = (int)(key_blk + 255 - Nc);
    const bool new_chunk = chunk_keys && p.new_mode;
    // the weights of chunk keys by distance: a table in LDS, unless every entry is the same value (then the
    // launch reserves no LDS for it, and two workgroups fit a compute unit whatever the chunk length)
    if (new_chunk && !p.wnew_uniform) {
        for (int i = tid; i < Q; i += 256) wnew_lds[i] = p.w_new[i];
    }
    int nmt = (Q - m_first + kQT2 - 1) / kQT2;  // query tiles per head
    int m_end = Q;                              // where the workgroup's share of them ends
    if (kShares && nmt > 0) {
        const int t0 = share * nmt / p.row_shares, t1 = (share + 1) * nmt / p.row_shares;
        m_end = m_first + t1 * kQT2 < Q ? m_first + t1 * kQT2 : Q;
        m_first += t0 * kQT2;
        nmt = t1 - t0;
    }
    // async copy assignments: the Q tile is copied in blocks of 1 KiB (a quarter of them per wavefront); wavefront 0
    // also brings the tile's normalisers, wavefront 1 its weights (kQT2 / 4 lanes x 16 bytes each)
    constexpr int kQBlocks = kQT2 * kRowBytes / 4096;   // per wavefront
    uint32_t q_src[kQBlocks];
#pragma unroll
    for (int j = 0; j < kQBlocks; j++) {
        const int pos = (wave * kQBlocks + j) * 64 + lane;
        const int r = pos / (kD / 8), c = (pos % (kD / 8)) ^ row_swizzle<kD>(r);
        q_src[j] = r * kRowBytes + c * 16;
    }
    int q_off[kKK];  // query row `col` of the tile
#pragma unroll
    for (int kk = 0; kk < kKK; kk++) q_off[kk] = k_lds_off<kD>(col, 2 * kk + half);
    const int64_t head_row0 = (b * p.H + kvh * p.G) * p.Q;
    // shares' normalisers of a stage's rows, behind the stages and the table of weights
    const int l2_at = 2 * kCsStage + (p.wnew_uniform ? 0 : (Q * 4 + 15) / 16 * 16);
    const uint32_t l2_off = (uint32_t)((lane >> 3) < p.n_split ? lane >> 3 : 0) * (uint32_t)(p.B * p.H * p.Q * 4) + (lane & 7) * 16;
    // (head, query tile) of a step are tracked incrementally: integer division per step would
    // cost more scalar instructions than the step's matrix work leaves room for
    auto issue = [&](int g, int mt, int stage) {
        const int64_t row0 = head_row0 + (int64_t)g * p.Q + mt;
        const char* qt = (const char*)p.qr + row0 * (kD * (int64_t)sizeof(T));
        const uint32_t st = smem_addr + stage * kCsStage;
        if (mt + kQT2 > Q) {  // rows past the chunk end repeat its last row
            const uint32_t last = (uint32_t)(Q - 1 - mt) * kRowBytes;
#pragma unroll
            for (int j = 0; j < kQBlocks; j++) {
                uint32_t src = q_src[j];
                asm("" : "+v"(src));   // worked out here, not kept in registers for the whole kernel
                const uint32_t piece = src % kRowBytes, row = src - piece;
                async_copy16(qt, (row < last ? row : last) + piece, st + (wave * kQBlocks + j) * 1024);
            }
        } else {
#pragma unroll
            for (int j = 0; j < kQBlocks; j++) async_copy16(qt, q_src[j], st + (wave * kQBlocks + j) * 1024);
        }
        if (wave < 2 && lane < kQT2 / 4 && (!kMerge || wave)) {
            const char* src = wave ? (const char*)(p.w_ema + mt) : (const char*)(p.lse2 + row0);
            async_copy16(src, lane * 16, st + kQT2 * kRowBytes + wave * (kQT2 * 4));
        }
        if constexpr (kMerge)   // a wavefront's 32 rows of every share, eight lanes a share
            async_copy16((const char*)(p.fwd.part_l2 + row0 + wave * 32), l2_off, smem_addr + l2_at + stage * (4 * 1024) + wave * 1024);
    };

    auto store = [&](int64_t h, int64_t n, float v) {
        if (kShares) {
            p.part[((share * p.B + b) * p.H + h) * p.N + n] = v;
        } else if (p.scores) {
            T* dst = (T*)p.scores + b * p.scores_stride[0] + h * p.scores_stride[1];
            dst[(p.key_order ? p.key_order[n] : n) * p.scores_stride[2]] = Elem<T>::from_float(v);
        } else {
            p.colsum[(b * p.H + h) * p.N + n] = v;
        }
    };
    auto store_zeros = [&] {
        for (int g = g_first; g < g_first + g_cnt; g++)
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const int64_t n = key_w + 32 * ks + col;
                if (half == 0 && n < p.N) store(kvh * p.G + g, n, 0.f);
            }
    };
    // Slots that the host knows to be empty, whose keys were not even staged (512 rows, 1000 of 16384 slots filled: 62 of 67 blocks),
    // and hidden keys sorted behind the visible ones: nothing is read.
    if ((key_blk >= p.empty_from && key_blk + 256 <= p.empty_to) || key_blk >= N) {
        store_zeros();
        return;
    }
    // The first query tile, the keys and their visibility are requested side by side: a workgroup of 509 rows lives some 15 us
    if (nmt > 0) issue(g_first, m_first, 0);
    uint4 kreg[2][kKK];
    const char* kbase = (const char*)p.kr + bkv * p.n_pad * kD * (int64_t)sizeof(T);
    bool live[2];
    int nrel[2];
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        const int64_t n = key_w + 32 * ks + col;
#pragma unroll
        for (int kk = 0; kk < kKK; kk++) {
            kreg[ks][kk] = n < p.n_pad ? *reinterpret_cast<const uint4*>(kbase + (n / kBN) * (int64_t)(kBN * kD * sizeof(T)) +
                                                                         k_image_off((int)(n % kBN), 2 * kk + half))
                                       : make_uint4(0, 0, 0, 0);
        }
        live[ks] = n < N && ((p.tile_vis[n / kBN] >> (n % kBN)) & 1ull);
        nrel[ks] = (int)(n - Nc);
    }
    // a block without a single visible key has nothing but zeros to write
    const unsigned long long* vis = p.tile_vis + key_blk / kBN;
    const bool hidden = !p.n_visible && (vis[0] | vis[1] | vis[2] | vis[3]) == 0ull;
    const int n_steps = hidden ? 0 : nmt * g_cnt;

    float acc[2] = {0.f, 0.f};
    auto tile_step = [&](auto stage_tag, int g, int mt) {
        constexpr int ST = decltype(stage_tag)::value;
        const unsigned char* q_lds = smem + ST * kCsStage;
        const float* lse_lds = reinterpret_cast<const float*>(q_lds + kQT2 * kRowBytes);
        const float* w_lds = lse_lds + kQT2;
        // Accumulators start from minus the row normaliser, so the matrix pipe hands back log2 P (the
        // softmax scale is already on the staged queries); with 64 dims they start from zero, and the scale and the
        // normaliser join in float32 (`nl`: the subtile's normalisers).  Element (c, v) of a 32-row subtile c:
        // query row mt + 32c + 8(v/4) + 4half + v%4, key column of this lane.
        auto row_norms = [&](int c) {
            f32x16 init;
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
                const float4 l4 = *reinterpret_cast<const float4*>(lse_lds + 32 * c + 8 * v4 + 4 * half);
                init[4 * v4] = l4.x;
                init[4 * v4 + 1] = l4.y;
                init[4 * v4 + 2] = l4.z;
                init[4 * v4 + 3] = l4.w;
            }
            return init;
        };
        auto row_init = [&](int c) {
            if constexpr (!kExact<kD>) return row_norms(c);
            f32x16 z;
#pragma unroll
            for (int v = 0; v < 16; v++) z[v] = 0.f;
            return z;
        };
        auto norms_of = [&](int c) {
            if constexpr (kExact<kD>) return row_norms(c);
            else return 0;
        };
        auto prob = [&](float x, const auto& nl, int v) {
            if constexpr (kExact<kD>) return __builtin_amdgcn_exp2f(fmaf(x, p.scale_log2, nl[v]));
            else return __builtin_amdgcn_exp2f(x);
        };
        auto load_weights = [&](int c, float(&ws)[16]) {
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
                const float4 w4 = *reinterpret_cast<const float4*>(w_lds + 32 * c + 8 * v4 + 4 * half);
                ws[4 * v4] = w4.x; ws[4 * v4 + 1] = w4.y; ws[4 * v4 + 2] = w4.z; ws[4 * v4 + 3] = w4.w;
            }
        };
        // Cached keys, or chunk keys with the row's weight (dense operator) that every row of the tile sees.  The last
        // tile of a head comes here too: with 509 rows it is one tile in four.
        if (!new_chunk && !(chunk_keys && mt <= last_nrel)) {
            // The common case, written in issue order: the logits of subtile c go through the matrix
            // pipe while the vector ALU turns subtile c-1 into weighted probabilities.
            f32x16 sq[2][2];  // [c & 1][ks]
            sq[0][0] = sq[0][1] = row_init(0);
#pragma unroll
            for (int kk = 0; kk < kKK; kk++) {
                const uint4 a = *reinterpret_cast<const uint4*>(q_lds + q_off[kk]);
                sq[0][0] = Mma<T>::mma(a, kreg[0][kk], sq[0][0]);
                sq[0][1] = Mma<T>::mma(a, kreg[1][kk], sq[0][1]);
            }
#pragma unroll
            for (int c = 1; c < kCsSub; c++) {
                sq[c & 1][0] = sq[c & 1][1] = row_init(c);
                uint4 a1[kKK];
#pragma unroll
                for (int kk = 0; kk < kKK; kk++) a1[kk] = *reinterpret_cast<const uint4*>(q_lds + q_off[kk] + c * (32 * kRowBytes));
                float ws[16];
                load_weights(c - 1, ws);
                const auto nl = norms_of(c - 1);
                __builtin_amdgcn_sched_barrier(0);
                // an exponential is consumed one slot after it was issued, so no wavefront waits for the
                // transcendental unit
                constexpr int kPer = 32 / (2 * kKK);   // exponentials per matrix instruction
                float pe_prev[kPer];
#pragma unroll
                for (int slot = 0; slot < 2 * kKK; slot++) {
                    const int kk = slot >> 1, ks = slot & 1;
                    sq[c & 1][ks] = Mma<T>::mma(a1[kk], kreg[ks][kk], sq[c & 1][ks]);
                    float pe[kPer];
#pragma unroll
                    for (int r = 0; r < kPer; r++) {
                        const int j = kPer * slot + r, ksv = j >> 4, v = j & 15;
                        pe[r] = prob(sq[(c - 1) & 1][ksv][v], nl, v);
                    }
                    if (slot > 0) {
#pragma unroll
                        for (int r = 0; r < kPer; r++) {
                            const int j = kPer * (slot - 1) + r, ksv = j >> 4, v = j & 15;
                            acc[ksv] = fmaf(ws[v], pe_prev[r], acc[ksv]);
                        }
                    }
#pragma unroll
                    for (int r = 0; r < kPer; r++) pe_prev[r] = pe[r];
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int r = 0; r < kPer; r++) {
                    const int j = 32 - kPer + r, ksv = j >> 4, v = j & 15;
                    acc[ksv] = fmaf(ws[v], pe_prev[r], acc[ksv]);
                }
            }
            {
                float ws[16];
                load_weights(kCsSub - 1, ws);
                const auto nl = norms_of(kCsSub - 1);
#pragma unroll
                for (int v = 0; v < 16; v++) {
#pragma unroll
                    for (int ks = 0; ks < 2; ks++) {
                        const float pe = prob(sq[(kCsSub - 1) & 1][ks][v], nl, v);
                        acc[ks] = fmaf(ws[v], pe, acc[ks]);
                    }
                }
            }
        } else {
            // Tiles with chunk keys on the diagonal or with the weights of chunk keys, one 32-row subtile at a time.  How a wavefront's
            // keys weigh is a type here and not a test by the element: as one it became a choice of addresses, 128 flat loads a
            // subtile, each with a wait for everything in flight (512 rows, 1000 of 16384 slots filled: the kernel 52 us, now 24.5;
            // 2 x 2048 rows x 16 K slots 560 and 540; dense, 8 x 1000 x 5095 x 64 dims 20 and 13.4).  Rows past the chunk end need
            // no test: their probability is zero (see hide_rows).
            const int nrel_w = (int)(key_w - Nc);   // this wavefront's first key among the chunk keys (negative: cached)
            enum Weights { kByRow, kAlike, kMixed };
            auto special = [&](auto weights_tag, auto uniform_tag) {
                constexpr int kWeights = decltype(weights_tag)::value;
                constexpr bool kUniform = decltype(uniform_tag)::value;
#pragma unroll 1
                for (int c = 0; c < kCsSub; c++) {
                    const int row0 = mt + 32 * c;
                    if (row0 >= Q) break;
                    if (row0 + 31 < nrel_w) continue;   // before every key of the wavefront
                    f32x16 sacc[2];
                    sacc[0] = sacc[1] = row_init(c);
                    const auto nl = norms_of(c);
#pragma unroll
                    for (int kk = 0; kk < kKK; kk++) {
                        const uint4 a = *reinterpret_cast<const uint4*>(q_lds + q_off[kk] + c * (32 * kRowBytes));
                        sacc[0] = Mma<T>::mma(a, kreg[0][kk], sacc[0]);
                        sacc[1] = Mma<T>::mma(a, kreg[1][kk], sacc[1]);
                    }
                    // row 8 (v / 4) + v % 4 of the lane's half sees a key at distance `ahead` or less in front of row 0 of it (cached: all do)
                    int ahead[2];
#pragma unroll
                    for (int ks = 0; ks < 2; ks++) ahead[ks] = nrel[ks] - row0 - 4 * half;
                    auto seen = [&](float e, int ks, int v) { return 8 * (v >> 2) + (v & 3) >= ahead[ks] ? e : 0.f; };
                    if constexpr (kWeights == kAlike) {
                        // every key of the wavefront is a chunk key and all of them weigh the same: P and the
                        // products are rounded to the tensor dtype two at a time by the packed conversions, and
                        // the rounded products join the sum through a dot product with a pair of ones
                        const float wu = p.wnew_value;
                        auto add = [&](auto masked) {
#pragma unroll
                            for (int v = 0; v < 16; v += 2) {
#pragma unroll
                                for (int ks = 0; ks < 2; ks++) {
                                    float e0 = prob(sacc[ks][v], nl, v), e1 = prob(sacc[ks][v + 1], nl, v + 1);
                                    if constexpr (decltype(masked)::value) {
                                        e0 = seen(e0, ks, v);
                                        e1 = seen(e1, ks, v + 1);
                                    }
                                    const uint32_t u = Mma<T>::pack2(e0, e1);
                                    acc[ks] = Mma<T>::sum2(Mma<T>::pack2(Mma<T>::lo_f(u) * wu, Mma<T>::hi_f(u) * wu), acc[ks]);
                                }
                            }
                        };
                        if (row0 >= nrel_w + 63) add(std::false_type{});
                        else add(std::true_type{});
                    } else {
                        float we[16];
                        load_weights(c, we);
#pragma unroll
                        for (int v = 0; v < 16; v++) {
#pragma unroll
                            for (int ks = 0; ks < 2; ks++) {
                                const float pe = seen(prob(sacc[ks][v], nl, v), ks, v), as_cached = fmaf(we[v], pe, acc[ks]);
                                if constexpr (kWeights == kByRow) {
                                    acc[ks] = as_cached;
                                } else {
                                    // a chunk key takes the weight of its distance from the row; a cached key (where the chunk
                                    // starts inside the wavefront) takes the row's EMA weight.  The eager path holds P and the
                                    // products of chunk keys in the tensor dtype.  Both are worked out and one is picked.
                                    const int r = 8 * (v >> 2) + (v & 3) - ahead[ks];
                                    float w = p.wnew_value;
                                    if constexpr (!kUniform) w = wnew_lds[nrel[ks] >= 0 && r >= 0 && r < Q ? r : 0];
                                    const float as_new = acc[ks] + Mma<T>::round1(Mma<T>::round1(pe) * w);
                                    acc[ks] = nrel[ks] >= 0 ? as_new : as_cached;
                                }
                            }
                        }
                    }
                }
            };
            if (!p.new_mode) special(std::integral_constant<int, kByRow>{}, std::true_type{});
            else if (!p.wnew_uniform) special(std::integral_constant<int, kMixed>{}, std::false_type{});
            else if (nrel_w >= 0) special(std::integral_constant<int, kAlike>{}, std::true_type{});
            else special(std::integral_constant<int, kMixed>{}, std::true_type{});
        }
        if (mt + kQT2 >= m_end) {  // head finished: combine the two lane halves and store
            const int64_t h = kvh * p.G + g;
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const float tot = acc[ks] + __shfl_xor(acc[ks], 32);
                const int64_t n = key_w + 32 * ks + col;
                if (half == 0 && n < p.N) store(h, n, live[ks] ? tot : 0.f);
                acc[ks] = 0.f;
            }
        }
    };

    // Normalisers of the 32 rows that a wavefront has brought the shares' of: two lanes a row, four shares each, added up in the order of
    // merge_rows_of, so that a score does not hang on which launch has merged the shares.
    auto merge_norms = [&](int stage) {
        if constexpr (!kMerge) return;
        const int r = lane >> 1;
        const float* l2 = reinterpret_cast<const float*>(smem + l2_at + stage * (4 * 1024) + wave * 1024) + (lane & 1) * (32 * kMergeShares / 2) + r;
        float v[kMergeShares / 2], M = -INFINITY, L = 0.f;
#pragma unroll
        for (int u = 0; u < kMergeShares / 2; u++) {
            v[u] = (lane & 1) * (kMergeShares / 2) + u < p.n_split ? l2[32 * u] : -INFINITY;
            M = fmaxf(M, v[u]);
        }
        M = fmaxf(M, __shfl_xor(M, 1));
        auto add = [&] {
#pragma unroll
            for (int u = 0; u < kMergeShares / 2; u++)
                if (v[u] != -INFINITY) L += __builtin_amdgcn_exp2f(v[u] - M);   // a NaN counts
        };
        add();
        L = __shfl_xor(L, 1);   // the second lane goes on from the first one's sum
        add();
        float* lse_lds = reinterpret_cast<float*>(smem + stage * kCsStage + kQT2 * kRowBytes);
        if (lane & 1) lse_lds[wave * 32 + r] = -(M + __builtin_amdgcn_logf(L));
    };
    // Called by every wavefront once its copies of a step have landed, before the barrier that publishes them.  Rows past
    // the chunk end are copies of its last row, whose normaliser is somebody else's: starting from this value their
    // probability is zero (if the last row is not finite it has spoiled the sums already).  In LDS and not at the
    // accumulators: selects there cost 41 spilled registers, and the whole kernel a quarter of its speed.
    auto hide_rows = [&](int mt, int stage) {
        if (mt + kQT2 <= Q) return;
        float* lse_lds = reinterpret_cast<float*>(smem + stage * kCsStage + kQT2 * kRowBytes);
        if constexpr (kMerge) {   // a wavefront its own rows
            if (lane < 32 && mt + wave * 32 + lane >= Q) lse_lds[wave * 32 + lane] = -3e38f;
        } else if (wave == 0) {
            for (int r = lane; r < kQT2; r += 64)
                if (mt + r >= Q) lse_lds[r] = -3e38f;
        }
    };
    // two steps per trip: while stage s is consumed the copy of the next step fills stage s^1
    int g_cur = g_first, mt_cur = m_first;    // step being consumed
    auto advance = [&](int& g, int& mt) {
        mt += kQT2;
        if (mt >= m_end) {
            mt = m_first;
            g++;
        }
    };
    for (int step = 0; step < n_steps; step += 2) {
        int g_n = g_cur, mt_n = mt_cur;
        advance(g_n, mt_n);
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        merge_norms(0);
        hide_rows(mt_cur, 0);
        __syncthreads();
        if (step + 1 < n_steps) issue(g_n, mt_n, 1);
        tile_step(std::integral_constant<int, 0>{}, g_cur, mt_cur);
        if (step + 1 < n_steps) {
            int g_n2 = g_n, mt_n2 = mt_n;
            advance(g_n2, mt_n2);
            __builtin_amdgcn_s_waitcnt(0x0F70);
            merge_norms(1);
            hide_rows(mt_n, 1);
            __syncthreads();
            if (step + 2 < n_steps) issue(g_n2, mt_n2, 0);
            tile_step(std::integral_constant<int, 1>{}, g_n, mt_n);
            g_cur = g_n2;
            mt_cur = mt_n2;
        }
    }
    if (n_steps <= 0) {  // no query can see these keys
        wait_copies<0>();   // the tile that nobody reads has landed before its place goes to another workgroup
        store_zeros();
    }
}

// The shares of a key's sums added up in order, at the row the key came from.
template <typename T>
__global__ void __launch_bounds__(256) colsum_merge_kernel(ColsumParams p) {
    const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x, bh = blockIdx.y, heads = p.B * p.H;
    if (n >= p.N) return;
    float sum = 0.f;
    for (int r = 0; r < p.row_shares; r++) sum += p.part[(r * heads + bh) * p.N + n];
    int64_t h;
    const int64_t b = div_index(bh, p.H, h);
    T* dst = (T*)p.scores + b * p.scores_stride[0] + h * p.scores_stride[1];
    dst[(p.key_order ? p.key_order[n] : n) * p.scores_stride[2]] = Elem<T>::from_float(sum);
}

template <typename T, int kD>
int run_mfma(const MfmaProblem& mp, hipStream_t stream) {
    const int64_t n = mp.n, n_pad = mp.n_pad;
    // what the staged queries are multiplied by, and the factor the kernels are left with.  Rotated keys carry key_scale.
    // 64 dims: rotated queries carry the same (the eager path's sqrt(scale)); those that arrive rotated stay as they are but
    // for the sign, so that the largest product is the largest logit.
    const float scale_log2 = mp.scale * kLog2e;
    float qscale = mp.q_pos ? scale_log2 / mp.key_scale : scale_log2, left = 1.f;
    if (kExact<kD>) {
        qscale = mp.q_pos ? mp.key_scale : mp.scale < 0.f ? -1.f : mp.scale == 0.f ? 0.f : 1.f;
        left = mp.q_pos || mp.scale == 0.f ? kLog2e : fabsf(scale_log2);
    }
    const int cus = mfma_device_cus();
    {
        StageScope sc(CKV_STAGE_PREP, stream);
        StageParams sp;
        for (int i = 0; i < 3; i++) {
            sp.seg[i].k = mp.seg[i].k;
            sp.seg[i].v = mp.seg[i].v;
            for (int j = 0; j < 4; j++) sp.seg[i].stride[j] = mp.seg[i].stride[j];
            sp.seg[i].pos = mp.seg[i].pos;
            sp.seg[i].pos_stride[0] = mp.seg[i].pos_stride[0];
            sp.seg[i].pos_stride[1] = mp.seg[i].pos_stride[1];
            sp.seg[i].pos_shift = mp.seg[i].pos_shift;
            sp.seg[i].masked = mp.seg[i].masked;
            sp.seg[i].len = mp.seg[i].len;
        }
        sp.inv_freq = mp.inv_freq;
        sp.theta = mp.theta;
        sp.key_scale = mp.key_scale;
        sp.shared_pos = mp.shared_pos;
        sp.kr = mp.kr;
        sp.vt = mp.vt;
        sp.tile_vis = mp.tile_vis;
        sp.empty_from = mp.empty_from; sp.empty_to = mp.empty_to;
        sp.B = mp.B; sp.KVH = mp.KVH; sp.n = n; sp.n_pad = n_pad;
        sp.key_order = mp.key_order; sp.n_visible = mp.n_visible; sp.n_chunk = mp.Q;
        sp.own_order = mp.own_order; sp.order_mask = mp.order_mask; sp.n_cached = n - mp.Q;
        const int64_t nbh = mp.B * mp.KVH;
        // shared positions: a block walks several (b, kvh) units with one set of cos/sin, the next unit's rows
        // always on their way
        int64_t splits = nbh;
        if (mp.shared_pos) {
            // About three workgroups per compute unit (two and three, us: 8 heads x 16897 keys 33.9 and 31.0, 16 x 18496 73 and
            // 68, 8 x 69696 109 and 109); eight where the keys are gathered by an order: those are not rotated, so
            // there is nothing to reuse from unit to unit, and the tiles of masked keys leave at once (two, four, eight and
            // sixteen, us, half of the cached keys masked: 64 heads x 17408 keys x 128 dims 148 147 130 135, 32 x 8704 x 128
            // 35.0 34.0 32.6 30.7, 8 x 16684 x 128 16.6 16.8 17.0 17.0, 64 x 2176 x 64 dims 13.6 12.4 12.4 12.7, 8 x 5095 x 64
            // 9.8 8.6 8.5 8.6).
            const int64_t tiles = n_pad / kBN;
            splits = ((mp.key_order ? 8 : 3) * cus + tiles - 1) / tiles;
            if (splits < 2) splits = 2;
            if (splits > nbh) splits = nbh;
        }
        if (splits > 65535) splits = 65535;
        StageQParams sq;
        sq.q = mp.q;
        for (int j = 0; j < 4; j++) sq.stride[j] = mp.q_stride[j];
        sq.q_pos = mp.q_pos;
        sq.inv_freq = mp.inv_freq;
        sq.theta = mp.theta;
        sq.qr = mp.qr;
        sq.rows = mp.B * mp.H * mp.Q;
        sq.H = mp.H; sq.Q = mp.Q;
        sq.qscale = qscale;
        sq.vec = mp.q_stride[3] == 1 && reinterpret_cast<uintptr_t>(mp.q) % 16 == 0 && mp.q_stride[0] % 8 == 0 &&
                 mp.q_stride[1] % 8 == 0 && mp.q_stride[2] % 8 == 0;
        {
            // about four query blocks (64 positions each) per compute unit; the rest of batch x heads is looped
            // over inside, sharing cos/sin
            const int64_t bx = (mp.Q + 63) / 64, nbh_q = mp.B * mp.H;
            int64_t by = (4 * cus + bx - 1) / bx;
            if (by > nbh_q) by = nbh_q;
            if (by < 1) by = 1;
            StageGrid g;
            g.q_bx = (int)bx; g.q_by = (int)by; g.k_bx = (int)(n_pad / kBN); g.k_by = (int)splits;
            const int64_t w_blocks = mp.make_weights ? (mp.Q + kColSlack + 255) / 256 : 0;
            const StageWeights sw{mp.w_ema, mp.w_new, mp.beta, mp.key_order, mp.n_visible, (int)w_blocks, mp.kept};
            const int64_t blocks = bx * by + (n_pad / kBN) * splits + w_blocks + kept_pieces(mp.kept, 256) + (mp.own_order ? 1 : 0);
            if (blocks > 0x7fffffff) return CKV_ERR_UNSUPPORTED;
            hipLaunchKernelGGL((stage_kernel<T, kD>), dim3((unsigned)blocks), dim3(256), 0, stream, sp, sq, g, sw);
        }
        CKV_HIP_TRY(hipGetLastError());
    }
    const int G = (int)(mp.H / mp.KVH);
    FwdParams fp;
    const bool scores = mp.colsum || mp.scores;
    bool merged_by_scores = false;
    int64_t merging = 0;   // workgroups that merge the forward kernel's shares
    {
        StageScope sc(CKV_STAGE_FWD, stream, true);
        fp.qr = mp.qr; fp.kr = mp.kr; fp.vt = mp.vt; fp.tile_vis = mp.tile_vis;
        fp.out = mp.out;
        for (int j = 0; j < 4; j++) fp.out_stride[j] = mp.out_stride[j];
        fp.lse = mp.lse;
        fp.lse2 = mp.lse2;
        fp.B = mp.B; fp.H = mp.H; fp.KVH = mp.KVH; fp.Q = mp.Q; fp.N = n; fp.Nc = n - mp.Q; fp.n_pad = n_pad;
        fp.G = G;
        fp.scale_log2 = left;
        fp.n_qt = (int)((mp.Q * G + kRows - 1) / kRows);
        fp.n_split = mfma_fwd_splits(mp.B, mp.H, mp.KVH, mp.Q, n, cus, mp.key_order != nullptr);
        fp.part_o = mp.part_o;
        fp.part_l2 = mp.part_l2;
        fp.n_visible = mp.n_visible;
        if (fp.n_split > 1 && (!fp.part_o || !fp.part_l2)) return CKV_ERR_WORKSPACE;
        const dim3 grid((unsigned)(fp.n_qt * fp.n_split), (unsigned)(mp.B * mp.KVH));
        const int lds = (int)pipe_lds_bytes(n_pad, kD);
        if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fwd_pipe_kernel<T, kD>), lds)) return rc;
        fp.xcd_aware = grid.y % 8 == 0;
        hipEvent_t ev0, ev1;
        prof_kernel_events(CKV_STAGE_FWD, &ev0, &ev1);
        const dim3 launch_grid = fp.xcd_aware ? dim3(grid.x * grid.y) : grid;
        if (ev0) hipExtLaunchKernelGGL((fwd_pipe_kernel<T, kD>), launch_grid, dim3(512), (uint32_t)lds, stream, ev0, ev1, 0u, fp);
        else hipLaunchKernelGGL((fwd_pipe_kernel<T, kD>), launch_grid, dim3(512), lds, stream, fp);
        CKV_HIP_TRY(hipGetLastError());
        merging = merge_blocks<kD>(mp.B * mp.H * mp.Q, fp.n_split);
        // The merge may ride in the launch of the score sums: a launch less, and its traffic beside the sums, whose last round leaves
        // units idle.  But every workgroup of the sums then works the normalisers of its query tiles out for itself, a third of a
        // microsecond a tile.  Calls, us, apart and together, 32 heads on 8 kv heads (streams x rows x slots): 100 x 1 K 57.6 53.4   300 x
        // 4 K 94.0 87.2   1000 x 4 K 176.0 166.9   509 x 16 K 278.9 277.4   2 x 500 x 12 K 352.7 350.0   2300 x 8 K 575.9 564.9; where the
        // estimate says apart: 1000 x 32 K 786.1 786.1   512 x 64 K 836.4 846.6   4 x 44 x 61 K 1003 1040   2 x 1500 x 64 K 4282 4412.
        // Dense, forward, 64 dims: 8 x 1000 x 500 46.6 42.0   32 x 50 x 1000 34.3 29.9.
        const int64_t rows = mp.B * mp.H * mp.Q, tiles = (n + 255) / 256 * mp.B * mp.H * ((mp.Q + kQT2 - 1) / kQT2);
        const double apart_us = 4.0 + (double)(rows * fp.n_split * kD * 4) / 5.5e6, together_us = 0.33 * (double)tiles / (2 * cus);
        merged_by_scores = scores && fp.n_split <= kMergeShares && together_us < apart_us && rows < (int64_t)1 << 27;   // offsets of 32 bits
        if (fp.n_split > 1 && !merged_by_scores) {
            hipLaunchKernelGGL((fwd_combine_kernel<T, kD>), dim3((unsigned)merging), dim3(256), 0, stream, fp);
            CKV_HIP_TRY(hipGetLastError());
        }
    }
    if (scores) {
        StageScope sc(CKV_STAGE_SCORES, stream);
        ColsumParams cp;
        cp.qr = mp.qr; cp.kr = mp.kr; cp.tile_vis = mp.tile_vis; cp.lse2 = mp.lse2;
        cp.w_ema = mp.w_ema; cp.w_new = mp.w_new; cp.colsum = mp.colsum;
        cp.B = mp.B; cp.H = mp.H; cp.KVH = mp.KVH; cp.Q = mp.Q; cp.N = n; cp.Nc = n - mp.Q; cp.n_pad = n_pad;
        cp.n_visible = mp.n_visible; cp.key_order = mp.key_order;
        cp.empty_from = mp.empty_from; cp.empty_to = mp.empty_to;
        cp.scores = mp.scores;
        for (int j = 0; j < 3; j++) cp.scores_stride[j] = mp.scores_stride[j];
        cp.G = G;
        cp.new_mode = mp.new_mode;
        {
            // w_new[k] = round((1 - beta) * round(round(beta)^k)) in the tensor dtype: one value for every k when
            // beta rounds to one there (0.9999999 does in both 16-bit formats)
            auto round_t_host = [](float v) -> float {
                if (std::is_same<T, __half>::value) return (float)(_Float16)v;
                uint32_t u;
                memcpy(&u, &v, 4);
                u += 0x7fffu + ((u >> 16) & 1u);  // to nearest even on the upper 16 bits (finite values)
                u &= 0xffff0000u;
                float r;
                memcpy(&r, &u, 4);
                return r;
            };
            cp.wnew_uniform = round_t_host((float)mp.beta) == 1.0f ? 1 : 0;
            cp.wnew_value = round_t_host((float)(1.0 - mp.beta));
        }
        cp.scale_log2 = left;
        cp.nkb = (int)((n + 255) / 256);
        cp.nbkv = (int)(mp.B * mp.KVH);
        cp.xcd_aware = cp.nbkv % 8 == 0;
        // Two heads per workgroup where the group allows it: the keys a workgroup holds in registers and its pipeline
        // start serve twice the work.  That pays once the launch has rounds enough for an uneven last one to cost little; a
        // round is two workgroups per compute unit, and the line is at four rounds of such workgroups.  Score kernel in us
        // with one and two heads, 32 heads on 8 kv heads, B streams x rows x slots, by rounds of two heads:
        //   0.5 (1 x 2048 x 2 K)  173  332     2.1 (1 x 509 x 16 K)  77  103     2.5 (1 x 4096 x 16 K)  550  767
        //   4.2 (2 x 509 x 16 K) 134  134      4.6 (2 x 2048 x 16 K) 510  508    8.0 (1 x 128 x 64 K)  92  75
        //   8.5 (1 x 4096 x 64 K) 1815 1814    16 (2 x 33 x 64 K) 190  145       16 (2 x 1500 x 64 K) 1394 1363
        const int64_t of_two = (int64_t)cp.nkb * cp.nbkv * (G / 2);
        cp.gsplit = (G % 2 == 0 && G >= 4 && of_two >= 4 * 2 * (int64_t)cus) ? G / 2 : G;
        cp.row_shares = mp.scores && mp.part_scores ? dense_row_shares(mp.B, mp.H, mp.Q, n, cus) : 1;
        cp.part = mp.part_scores;
        cp.n_split = fp.n_split;
        cp.fwd = fp;
        cp.sum_blocks = cp.nkb * cp.nbkv * cp.gsplit * cp.row_shares;
        const bool merge = fp.n_split > 1 && merged_by_scores;
        const dim3 grid((unsigned)(cp.sum_blocks + (merge ? merging : 0)));
        const int lds = 2 * cs_stage(kD) + (cp.wnew_uniform ? 0 : ((int)mp.Q * 4 + 15) / 16 * 16) + (merge ? 2 * 4 * 1024 : 0);
        auto kernel = cp.row_shares > 1 ? (merge ? colsum_mfma_kernel<T, kD, true, true> : colsum_mfma_kernel<T, kD, true, false>)
                                        : (merge ? colsum_mfma_kernel<T, kD, false, true> : colsum_mfma_kernel<T, kD, false, false>);
        if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), lds)) return rc;
        hipLaunchKernelGGL(kernel, grid, dim3(256), lds, stream, cp);
        if (cp.row_shares > 1) {
            CKV_HIP_TRY(hipGetLastError());
            hipLaunchKernelGGL(colsum_merge_kernel<T>, dim3((unsigned)((n + 255) / 256), (unsigned)(mp.B * mp.H)), dim3(256), 0, stream, cp);
        }
        CKV_HIP_TRY(hipGetLastError());
    }
    return CKV_OK;
}

}  // namespace

bool mfma_supported(int dtype, int64_t D, int64_t H, int64_t KVH, int64_t Q) {
    if (dtype != CKV_BF16 && dtype != CKV_F16) return false;
    if (D != 64 && D != 128) return false;
    if (Q > 16384) return false;  // the column pass keeps a Q-long weight table in LDS beside its two stages
    const int64_t G = H / KVH;
    return G >= 1 && G <= kRows / 32;  // at least 32 positions per workgroup
}

// Workgroups that share the query tiles of a key block in the dense operator's score sums.  Two workgroups of four wavefronts run on
// a unit, and one takes some 4 us a tile: with few heads and keys most of the chip is idle meanwhile.  The merge is a launch of 3 to
// 4 us, so a share has to save at least two tiles.  The whole operator, forward, us, without and with shares, 64 dims f16 / 128 dims
// bf16, heads x rows x cached keys:  2 x 384 x 1000 (2 shares) 57.7 49.3 / 55.2 48.4   2 x 1024 x 1000 (8) 64.8 48.8 / 68.9 49.6
//   3 x 300 x 8000 (3) 59.7 54.1 / 63.5 58.2   8 x 1000 x 4095 (3) 80.1 71.0 / 82.6 76.9   32 x 900 x 500 (2) 85.1 80.8 / 84.4 81.0
int dense_row_shares(int64_t B, int64_t H, int64_t n_ctx, int64_t n_kv, int cus) {
    const int64_t wgs = (n_kv + 255) / 256 * B * H, tiles = (n_ctx + kQT2 - 1) / kQT2;
    if (B * H > 65535) return 1;
    const int64_t shares = std::min<int64_t>(2 * (int64_t)cus / wgs, tiles);
    return shares > 1 && tiles - (tiles + shares - 1) / shares >= 2 ? (int)shares : 1;
}

int64_t mfma_n_pad(int64_t n) { return align_up(n, 256); }

// Do the dense operator's staging blocks look for their keys in the mask, instead of in an order that a launch in front of them has
// written?  That launch takes 5.5 us, in which one workgroup works; a block's look takes half a microsecond for every 4096 mask bytes.
// The operator, forward, us, 128 dims, heads x rows x cached keys, with the launch and without: 2 x 33 x 64 27.0 23.2   8 x 200 x 2 K 43.8
// 41.3   3 x 300 x 8 K 53.4 49.0   2 x 1000 x 16 K 71.1 63.4   64 x 1000 x 16 K 503.5 497.6   2 x 100 x 20 K 50.8 45.5   8 x 300 x 30 K
// 99.6 103.5   8 x 300 x 60 K 166.4 178.5   32 x 100 x 60 K 411.3 398.4: by 16 K it is never the slower way.
bool order_by_staging(int64_t n_cached) { return n_cached <= 16384; }

// Shares of a query tile's key tiles (1: no splitting) on a chip of `cus` compute units, each of which holds one workgroup
// of the forward kernel at a time.  The count is a matter of sizes alone, never of how many slots hold a token: it sets the
// order in which a row's sums are added, so a hint about the filled slots would otherwise change results.
//
// The launch takes whole rounds of workgroups, a round as long as a workgroup: about 1.6 us per key tile with every unit busy and 16 us
// to start and finish one (the work list, the first copies, the rows' way out).  Shares cost a merge kernel, 6 us and its traffic
// (float32 rows written and read, 256 rows of 512 bytes per workgroup: 0.058 us); that is what a call without scores pays, and one whose
// merge rides with its score sums (run_mfma) pays less, but the order of a row's sums must not hang on whether scores are asked for.  The
// cheapest count by that estimate, down to
// two tiles each: 2300 x 8 K  1: 391  3: 353  8: 416.  (64 dims: 1: 503  3: 398  6: 382; masked keys of the dense operator, which
// cost nothing, count like the others.)  With no more than a share to 16 tiles of a chunk, and to 8 of the dense operator's, a whole
// call took, us, 32 heads on 8 kv heads, then and now:  16 rows x 1 K slots 57.8 47.5   33 x 2 K 67.1 55.7   16 x 4 K 76.4 63.7
//   300 x 2 K 85.1 75.4   300 x 7 K 132.2 113.1   300 x 8 K 139.0 120.6   500 x 12 K 208.0 197.4   2 x 500 x 4 K 178.5 166.4   1000 x 2 K
//   147.9 138.8   1500 x 8 K 376.8 358.5   1000 x 1 K 122.5 122.7   200 x 10 K 115.6 115.8 (28 heads on 4: 106.0 108.5); dense,
//   forward, 64 dims: 2 heads x 100 rows x 1000 cached keys 37.9 30.7   3 x 300 x 500 43.5 33.7   8 x 1000 x 500 49.9 47.4.
// Twice as many shares as fill one round lose (300 x 4 K, the call  4: 91.8  8: 102.8).
//
// Chunks of fewer workgroups than units over caches of 16 K slots and more keep the counts that streams have always had, because a
// decoder of random weights turns the changed rounding of one hidden state into a percent of its logits: about two workgroups per
// unit, at most 8 shares; where 8 shares would be of more than 32 tiles, the cheapest count from 8 to 32 by the estimate.  The line is
// drawn by that and not by speed (half the shares would be faster up to 16 K slots), and tiles of the chunk count: a stream over a little
// less than 16 K slots goes from one count to the other with the length of its chunks.  Forward + merge in us, by shares:     509 rows x 16 K  4: 141  8: 155    488 x 16 K, 1000 slots filled  4: 34  8: 47
//   128 x 64 K   8: 175  16: 134  32: 160        32 x 64 K  8: 162  16: 95  32: 90      509 x 32 K  4: 237  8: 250
int mfma_fwd_splits(int64_t B, int64_t H, int64_t KVH, int64_t Q, int64_t n, int cus, bool dense) {
    constexpr double kTileUs = 1.6, kStartUs = 16.0, kMergeUs = 6.0, kMergeWgUs = 0.058;
    constexpr int64_t kMaxShares = 32, kMaxShareBytes = (int64_t)256 << 20, kFew = 8, kMinTiles = 2, kMinTilesMany = 32, kManyTiles = 256;
    const int64_t G = H / KVH;
    const int64_t wgs = ((Q * G + kRows - 1) / kRows) * B * KVH, tiles = (n + kBN - 1) / kBN;
    if (wgs >= 4 * (int64_t)cus) return 1;   // at most an eighth of the launch can be an empty round
    int64_t first = 1, min_tiles = kMinTiles;
    if (wgs < cus && tiles >= kManyTiles && !dense) {
        const int64_t few = std::max<int64_t>(1, std::min(2 * (int64_t)cus / wgs, kFew));
        if (few < kFew || tiles / kMinTilesMany <= kFew) return (int)few;
        first = kFew;
        min_tiles = kMinTilesMany;
    }
    int64_t best = first;
    double best_us = 0.0;
    for (int64_t s_ = first; s_ <= kMaxShares && (s_ == first || tiles / s_ >= min_tiles); s_++) {
        if (s_ > first && s_ * wgs * kRows * 512 > kMaxShareBytes) break;
        const double rounds = (double)((wgs * s_ + cus - 1) / cus);
        const double us = rounds * ((double)tiles / (double)s_ * kTileUs + kStartUs) +
                          (s_ > 1 ? kMergeUs + kMergeWgUs * (double)(wgs * s_) : 0.0);
        if (s_ == first || us < best_us) {
            best = s_;
            best_us = us;
        }
    }
    return (int)best;
}

// compute units of the current device; 256 (one MI355X) where no device can be asked, e.g. when a workspace is
// sized on a host without one
int mfma_device_cus() {
    DeviceInfo di;
    if (current_device_info(&di) != CKV_OK || di.cus <= 0) return 256;
    return di.cus;
}

// what a workspace is sized for: the shares the current device would use, and never fewer than a 256-unit chip's,
// so that a size computed where no device is visible also serves the launch
int mfma_fwd_splits_for_workspace(int64_t B, int64_t H, int64_t KVH, int64_t Q, int64_t n, bool dense) {
    return std::max(mfma_fwd_splits(B, H, KVH, Q, n, mfma_device_cus(), dense), mfma_fwd_splits(B, H, KVH, Q, n, 256, dense));
}

// the forward kernel keeps per-tile bookkeeping of all N keys in LDS
bool mfma_fits(int64_t n, int64_t D) { return pipe_lds_bytes(mfma_n_pad(n), (int)D) <= kLdsLimit; }


int launch_mfma(const MfmaProblem& mp, hipStream_t stream) {
    if (mp.dtype == CKV_BF16) return mp.D == 64 ? run_mfma<__hip_bfloat16, 64>(mp, stream) : run_mfma<__hip_bfloat16, 128>(mp, stream);
    if (mp.dtype == CKV_F16) return mp.D == 64 ? run_mfma<__half, 64>(mp, stream) : run_mfma<__half, 128>(mp, stream);
    return CKV_ERR_DTYPE;
}

}  // namespace ckv

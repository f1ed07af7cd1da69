// The dense operator's float32 attention and score sums on the matrix cores (v_mfma_f32_32x32x2_f32), head_dim 64 and 128, from its
// operands where they lie.  Cached chunks, which are staged anyway, take the bfloat16 instruction (ckv_attn_f32_split.hip).
//
// The float32 matrix instructions multiply and accumulate in float32 (every product enters the accumulator through a
// fused multiply-add), at twice the rate of the vector ALU and with one operand register per lane instead of LDS reads
// per product, which is what bounded the vector kernels (ckv_attn_generic.hip keeps them for the shapes that do not
// fit here).  32 heads x 256 rows x 516 + 256 keys x 128: forward 269 -> 45 us, scores 321 -> 31 us.  Both are bound by the
// products and the vector work together: vector instructions do not run beside these products (a tile's exponentials take
// 5700 cycles next to the other wavefront's 64 products, which take 4400 alone, and 1700 by themselves), so what is not
// arithmetic of the attention -- masks of whole blocks, addresses of rows -- is kept off the vector pipe.
//
//   forward  one workgroup = one head x 32 rows; its eight wavefronts take the 32-key blocks in
//            turn, each with an online softmax of its own, and merge at the end through LDS.  S^T = K Q^T keeps a query
//            in one lane pair, and register v of S^T is, as it stands, the B operand of step v of O^T += V^T P^T: nothing
//            is moved between the two products.  Values go from memory straight to the operand registers (no two
//            wavefronts of a workgroup share any), keys through LDS, as operand pieces of 32 rows touch 32 lines of the
//            first-level cache at a time; the queries sit in LDS in operand order.  With keys straight to registers and
//            the addresses worked out per lane the forward took 47.7 us.
//   colsum   one workgroup = one head x four blocks of 32 keys, held in registers (one block where that makes too few
//            workgroups); two streams of its wavefronts take the 32-row query tiles, which come through LDS, in turn.
//            S = Q K^T keeps a key in one lane pair, so a weighted sum stays in its lane until the end.  With a block of
//            keys a workgroup and queries straight to registers the scores took 34 us (28 heads x 2568 keys, 512 rows: 156,
//            now 123), with a barrier a tile 31.3.
//
// A matrix instruction multiplies every row of a tile by every value, and zero times infinity or NaN is NaN, while a value
// whose key has probability zero counts for nothing, whatever it holds (the vector kernels do not touch it).  So a wavefront
// whose accumulators come out finite is done: nothing else can have been multiplied.  Otherwise it goes over its keys once
// more with the normalisers it has found, finite values through the matrix pipe and the others where their probability is
// above zero.
//
// A contraction over the head dim may take the dims in any order as long as both operands do: step 4 c + e multiplies
// dims 8 c + e (lanes 0..31) and 8 c + 4 + e (lanes 32..63), so that an operand is a 16-byte load per four steps.
#include "ckv_attn_internal.h"

#include <type_traits>

namespace ckv {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kRows = 32;      // query rows of a forward workgroup
constexpr int kKeys = 32;      // keys of a block
constexpr int kFwdWaves = 8;
constexpr int kColSums = 4;    // partial sums of a key, one per query tile mod 4
// a workgroup of the score sums: blocks of keys it takes, and streams of query tiles, each a wavefront per block of keys
template <int kGroups>
struct Col {
    static constexpr int kStreams = kGroups == 1 ? 4 : 2, kWaves = kGroups * kStreams, kBlockKeys = kGroups * kKeys;
    static constexpr int kAcc = kColSums / kStreams;   // partial sums of a wavefront
};

template <int D>
struct Geo {
    static constexpr int kPieces = D / 8;   // 16-byte pieces of a row per lane half
    static constexpr int kDB = D / 32;      // accumulators of 32 dims
    static constexpr int kPitch = D + 4;    // floats of a row in the merge area
    static constexpr int kQ = kPieces * CKV_WAVE * 16;
    static constexpr int kFwdLds = kQ + kFwdWaves * kRows * kPitch * 4 + 2 * kFwdWaves * kRows * 4;
    // 32 rows in LDS as asynchronous copies of 1 KiB bring them: 16-byte piece c of row r in slot c ^ (r mod slots), so that one
    // piece of 16 consecutive rows covers all banks
    static constexpr int kSlots = D / 4, kTile = 32 * D * 4, kCopies = kTile / 1024;
    static_assert(kFwdWaves * kTile <= kFwdWaves * kRows * kPitch * 4, "the key blocks lie where the shares are merged");
    __device__ static int slot(int r, int c) { return c ^ (r & (kSlots - 1)); }
};

template <int N>
struct Vec {
    float v[N];
};

__device__ inline f32x16 mma(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }

__device__ inline f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; i++) z[i] = 0.f;
    return z;
}

// matrix row of accumulator register v in lane half `half`
__device__ inline int acc_row(int v, int half) { return 8 * (v >> 2) + 4 * half + (v & 3); }

template <int D>
__global__ void __launch_bounds__(kFwdWaves* CKV_WAVE) fwd_f32_mfma_kernel(CoreProblem p) {
    using G_ = Geo<D>;
    constexpr int NP = G_::kPieces, DB = G_::kDB;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float4* q_lds = reinterpret_cast<float4*>(lds);                  // [piece][lane]
    float* o_lds = lds + G_::kQ / 4;                                  // [wave][row][kPitch]
    float* ml_lds = o_lds + kFwdWaves * kRows * G_::kPitch;           // [max, sum][wave][row]
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // heads go round the XCDs (when they divide evenly), so a head's keys stay in one L2; heavy row tiles first
    const int heads = (int)(p.B * p.H), H = (int)p.H, n_rt = ((int)p.Q + kRows - 1) / kRows;
    const int bh = blockIdx.x % heads, rt = n_rt - 1 - (int)(blockIdx.x / heads);
    const int64_t b = bh / H, h = bh % H;
    const int N = (int)p.N, Q = (int)p.Q, Nc = N - Q;
    const float* kb = (const float*)p.k + b * p.kv_stride[0] + h * p.kv_stride[1];
    const float* vb = (const float*)p.v + b * p.kv_stride[0] + h * p.kv_stride[1];

    const int row_m = rt * kRows + col;                  // this lane's query
    int m_hi = rt * kRows + kRows - 1;
    if (m_hi > Q - 1) m_hi = Q - 1;
    const int nblk = (Nc + m_hi) / kKeys + 1;            // blocks some row of the tile may see
    // bit r: key r of the block is there and not masked
    auto visible_keys = [&](int n) { return (uint32_t)__ballot(n < Nc ? !(p.kmasked && p.kmasked[n]) : n < N); };
    // the logits of a block's keys (lane = its query), and the keys this lane's query sees
    auto logits = [&](auto&& key_piece) {
        f32x16 s = zero16();
#pragma unroll
        for (int c = 0; c < NP; c++) {
            if (c % 4 == 0) __builtin_amdgcn_sched_barrier(0);   // eight operand reads ahead, not all of them
            const float4 k4 = key_piece(c), q4 = q_lds[c * CKV_WAVE + lane];
            s = mma(k4.x, q4.x, s);
            s = mma(k4.y, q4.y, s);
            s = mma(k4.z, q4.z, s);
            s = mma(k4.w, q4.w, s);
        }
        return s;
    };
    auto seen_keys = [&](uint32_t vis, int n0) {
        if (n0 + kKeys - 1 < Nc) return vis;
        const int last = Nc + row_m - n0;   // last key of the block the row may see
        return vis & (last >= 31 ? ~0u : (last < 0 ? 0u : (2u << last) - 1u));   // cached keys lie in front of the chunk keys: row_m >= 0 lets them all through
    };
    const bool near = p.kv_stride[2] >= 0 && p.kv_stride[2] < (1 << 24);   // offsets of a few rows fit 32 bits
    const uint32_t row_bytes = (uint32_t)p.kv_stride[2] * 4u;
    // the wavefront's block of keys in LDS
    unsigned char* k_lds = reinterpret_cast<unsigned char*>(o_lds) + wave * G_::kTile;
    const uint32_t k_at = lds_address(k_lds);
    auto copy_keys = [&](int n0) {
        constexpr int kRowsPer = CKV_WAVE / G_::kSlots;   // rows of a copy
        const int r0 = lane / G_::kSlots;
        int c0 = G_::slot(r0, lane % G_::kSlots);
        asm volatile("" : "+v"(c0));   // worked out again each time: sixteen kept offsets are sixteen registers
        if (near && n0 + kKeys <= N) {
            // the block's rows from a uniform address: vector instructions do not run beside float32 products
            const uint32_t row = (uint32_t)r0 * row_bytes;
            const float* from = kb + (int64_t)n0 * p.kv_stride[2];
#pragma unroll
            for (int j = 0; j < G_::kCopies; j++)
                async_copy16(from + (int64_t)(j * kRowsPer) * p.kv_stride[2], row + 16u * (uint32_t)G_::slot(j * kRowsPer, c0), k_at + j * 1024);
        } else {
#pragma unroll
            for (int j = 0; j < G_::kCopies; j++) {
                const int n = n0 + r0 + j * kRowsPer, c = G_::slot(j * kRowsPer, c0);
                async_copy16_from(kb + (int64_t)(n < N ? n : N - 1) * p.kv_stride[2] + 4 * c, k_at + j * 1024);
            }
        }
    };
    auto read_keys = [&](int c) {
        return *reinterpret_cast<const float4*>(k_lds + col * (D * 4) + G_::slot(col, 2 * c + half) * 16);
    };
    auto load_keys = [&](int n, float4(&kf)[NP]) {
        const float* kr = kb + (int64_t)(n < N ? n : N - 1) * p.kv_stride[2] + 4 * half;
#pragma unroll
        for (int c = 0; c < NP; c++) kf[c] = *reinterpret_cast<const float4*>(kr + 8 * c);
    };
    // values of the lane's half of the keys, dims DB col .. DB col + DB - 1: accumulator db holds dims DB m + db
    auto load_values = [&](int n0, Vec<DB>(&vf)[16]) {
        if (near && n0 + kKeys <= N) {
            const uint32_t at = (uint32_t)(4 * half) * row_bytes + (uint32_t)(DB * col * 4);
            const char* from = reinterpret_cast<const char*>(vb + (int64_t)n0 * p.kv_stride[2]);
#pragma unroll
            for (int v = 0; v < 16; v++)
                vf[v] = *reinterpret_cast<const Vec<DB>*>(from + (int64_t)acc_row(v, 0) * p.kv_stride[2] * 4 + at);
            return;
        }
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int nv = n0 + acc_row(v, half);
            vf[v] = *reinterpret_cast<const Vec<DB>*>(vb + (int64_t)(nv < N ? nv : N - 1) * p.kv_stride[2] + DB * col);
        }
    };
    // A wavefront's blocks blk, blk + step, ...  The next one with a visible key is requested as soon as this one's place is free:
    // its keys behind the logits, its values behind the second product.  So a wavefront waits for memory once, at its first
    // block, which is requested with the queries and before its mask is known (nearly always wanted, and in bounds).
    // Loads and copies retire in issue order; "at most n outstanding" below counts what was issued behind the wanted ones.
    constexpr int step = kFwdWaves;
    auto mask_byte = [&](int n) -> int { return n < Nc ? (p.kmasked ? p.kmasked[n] : 0) : n < N ? 0 : 1; };
    int blk = wave;
    int hidden = blk < nblk ? mask_byte(blk * kKeys + col) : 1;
    Vec<DB> vf[16];
    constexpr int kValueLoads = 16;
    {
#pragma unroll
        for (int t = 0; t < NP / kFwdWaves; t++) {
            const int c = t * kFwdWaves + wave;
            if (row_m < Q)
                async_copy16_from((const float*)p.q + b * p.q_stride[0] + h * p.q_stride[1] + row_m * p.q_stride[2] + 8 * c + 4 * half,
                                  lds_address(q_lds) + c * (CKV_WAVE * 16));
            else
                q_lds[c * CKV_WAVE + lane] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        if (blk < nblk) {
            copy_keys(blk * kKeys);
            load_values(blk * kKeys, vf);
            wait_copies<G_::kCopies + kValueLoads>();
        } else {
            wait_copies<0>();
        }
    }
    // a barrier of the language would wait for the keys and values too
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; db++) o[db] = zero16();
    float m_run = -INFINITY, l_run = 0.f;
    uint32_t vis = (uint32_t)__ballot(hidden == 0);
    // on to a block with a visible key, if there is one
    auto skip_hidden = [&]() {
        while (vis == 0u && blk + step < nblk) {
            blk += step;
            vis = visible_keys(blk * kKeys + col);
        }
    };
    if (blk < nblk && vis == 0u) {
        skip_hidden();
        wait_copies<0>();   // also where nothing follows: the shares are merged in this LDS
        if (vis != 0u) {
            copy_keys(blk * kKeys);
            load_values(blk * kKeys, vf);
        }
    }
    while (vis != 0u) {
        const int n0 = blk * kKeys;
        const uint32_t vis_now = vis;
        wait_copies<kValueLoads>();   // the keys are there
        const bool more = blk + step < nblk;
        hidden = more ? mask_byte((blk + step) * kKeys + col) : 1;
        f32x16 s = logits(read_keys);
        // the values have arrived (under the logits): what the compiler would wait for behind the next copies are those too
#pragma unroll
        for (int v = 0; v < 16; v++)
#pragma unroll
            for (int db = 0; db < DB; db++) asm volatile("" : "+v"(vf[v].v[db]));
        vis = (uint32_t)__ballot(hidden == 0);
        if (more) {
            blk += step;
            skip_hidden();
        }
        if (vis != 0u) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the keys have been read
            copy_keys(blk * kKeys);
        }
        const uint32_t allow = seen_keys(vis_now, n0);   // bit r: key r of the block is visible to this lane's query
        const bool whole = __ballot(allow != ~0u) == 0ull;
        float mx = -INFINITY;
        if (whole) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                s[v] *= p.scale;
                mx = fmaxf(mx, s[v]);
            }
        }
        asm volatile("");   // two branches, not one with an alternative: the registers of the rare one are not kept for the other
        if (!whole) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
                s[v] = (allow >> acc_row(v, half)) & 1u ? s[v] * p.scale : -INFINITY;
                mx = fmaxf(mx, s[v]);
            }
            // the row of a key nobody sees may hold anything
#pragma unroll
            for (int v = 0; v < 16; v++)
#pragma unroll
                for (int db = 0; db < DB; db++) vf[v].v[db] = (vis_now >> acc_row(v, half)) & 1u ? vf[v].v[db] : 0.f;
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float m_new = fmaxf(m_run, mx);
        const float ref = m_new == -INFINITY ? 0.f : m_new;   // nothing visible yet: every exponential is 0
        float sum = 0.f;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            s[v] = expf(s[v] - ref);
            sum += s[v];
        }
        const float alpha = m_run == -INFINITY ? 0.f : expf(m_run - ref);
        l_run = l_run * alpha + sum;
        if (__ballot(m_new != m_run) != 0ull) {
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int v = 0; v < 16; v++) o[db][v] *= alpha;
        }
        m_run = m_new;
#pragma unroll
        for (int v = 0; v < 16; v++)
#pragma unroll
            for (int db = 0; db < DB; db++) o[db] = mma(vf[v].v[db], s[v], o[db]);
        if (vis != 0u) {
            asm volatile("" ::: "memory");   // behind the copies of the keys
            load_values(blk * kKeys, vf);
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
        for (int blk = wave; blk < nblk; blk += step) {
            const int n0 = blk * kKeys;
            const uint32_t vis = visible_keys(n0 + col);
            if (vis == 0u) continue;
            f32x16 s;
            {
                float4 kf[NP];
                load_keys(n0 + col, kf);
                s = logits([&](int c) { return kf[c]; });
            }
            const uint32_t allow = seen_keys(vis, n0);
#pragma unroll
            for (int v = 0; v < 16; v++) s[v] = (allow >> acc_row(v, half)) & 1u ? expf(s[v] * p.scale - m_run) : 0.f;
            Vec<DB> vf[16];
            load_values(n0, vf);
            bool odd = false;
#pragma unroll
            for (int v = 0; v < 16; v++)
#pragma unroll
                for (int db = 0; db < DB; db++) {
                    const float x = vf[v].v[db];
                    odd = odd || !isfinite(x);
                    o[db] = mma(isfinite(x) ? x : 0.f, s[v], o[db]);
                }
            if (__ballot(odd) == 0ull) continue;
#pragma unroll
            for (int db = 0; db < DB; db++) {
                f32x16 up = zero16(), down = zero16();   // how many infinities of either sign a sum holds, a NaN being both
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float x = vf[v].v[db], counts = s[v] > 0.f ? 1.f : 0.f;
                    up = mma(x == INFINITY || isnan(x) ? 1.f : 0.f, counts, up);
                    down = mma(x == -INFINITY || isnan(x) ? 1.f : 0.f, counts, down);
                }
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
        const float sc = m_run == -INFINITY ? 0.f : expf(m_run - M);
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
    const int m = rt * kRows + r;
    if (m >= Q) return;
    float M = -INFINITY, L = 0.f;
#pragma unroll
    for (int w = 0; w < kFwdWaves; w++) M = fmaxf(M, ml_lds[w * kRows + r]);
#pragma unroll
    for (int w = 0; w < kFwdWaves; w++) {
        const float mw = ml_lds[w * kRows + r], lw = ml_lds[(kFwdWaves + w) * kRows + r];
        if (lw != 0.f) L = fmaf(lw, mw == -INFINITY ? 1.f : expf(mw - M), L);   // no largest logit but a sum: a NaN
    }
    float acc[kPer];
#pragma unroll
    for (int i = 0; i < kPer; i++) acc[i] = 0.f;
#pragma unroll
    for (int w = 0; w < kFwdWaves; w++)
#pragma unroll
        for (int i = 0; i < kPer; i++) acc[i] += o_lds[(w * kRows + r) * G_::kPitch + d0 + i];
    // A row without a probability above zero (all its logits overflowed) or with a NaN among them is NaN.
    const float inv = 1.f / L;
    const int64_t row = (b * p.H + h) * p.Q + m;
    float* orow = (float*)p.out + b * p.out_stride[0] + h * p.out_stride[1] + m * p.out_stride[2];
#pragma unroll
    for (int i = 0; i < kPer; i++) orow[(d0 + i) * p.out_stride[3]] = acc[i] * inv;
    if (d0 == 0 && p.lse) p.lse[row] = M + logf(L);
}

template <int D, int kGroups>
__global__ void __launch_bounds__(Col<kGroups>::kWaves* CKV_WAVE, 2) colsum_f32_mfma_kernel(CoreProblem p) {
    constexpr int kColGroups = kGroups, kColStreams = Col<kGroups>::kStreams, kColWaves = Col<kGroups>::kWaves, kColKeys = Col<kGroups>::kBlockKeys;
    constexpr int kAcc = Col<kGroups>::kAcc;
    constexpr int NP = Geo<D>::kPieces, kSlots = Geo<D>::kSlots, kTile = Geo<D>::kTile;
    extern __shared__ __attribute__((aligned(16))) float lds[];   // kColWaves tiles of 32 queries
    __shared__ float sums[kColSums][kColKeys];
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = wave % kColGroups, stream = wave / kColGroups;
    const int heads = (int)(p.B * p.H), H = (int)p.H;
    const int N = (int)p.N, Q = (int)p.Q, Nc = N - Q, nblk = (N + kColKeys - 1) / kColKeys;
    // heads round the XCDs; blocks of chunk keys see fewer rows and come last
    const int bh = blockIdx.x % heads, blk = blockIdx.x / heads;
    if (blk >= nblk) return;
    const int64_t b = bh / H, h = bh % H;
    const int n0 = blk * kColKeys + group * kKeys, n = n0 + col, nrel = n - Nc;   // nrel >= 0: a chunk key
    const int masked = n < Nc && p.kmasked ? p.kmasked[n] : 0;
    const float* qb = (const float*)p.q + b * p.q_stride[0] + h * p.q_stride[1];
    const float* lse = p.lse + (b * p.H + h) * p.Q;
    const int blk0 = blk * kColKeys;
    const int t_first = blk0 > Nc ? (blk0 - Nc) / kRows : 0;   // first tile with a row that sees a key of the workgroup
    const int t_own = n0 > Nc ? (n0 - Nc) / kRows : 0;         // ... of this wavefront
    const int n_tiles = (Q + kRows - 1) / kRows;
    // a wavefront copies a tile of the next kColWaves ones
    const unsigned char* q_lds = reinterpret_cast<const unsigned char*>(lds);
    auto copy_queries = [&](int t) {
#pragma unroll
        for (int j = 0; j < Geo<D>::kCopies; j++) {
            const int piece = j * CKV_WAVE + lane, r = piece / kSlots, m = t * kRows + r;
            async_copy16_from(qb + (int64_t)(m < Q ? m : Q - 1) * p.q_stride[2] + 4 * Geo<D>::slot(r, piece % kSlots),
                              lds_address(lds) + wave * kTile + j * 1024);
        }
    };
    if (t_first + wave < n_tiles) copy_queries(t_first + wave);
    float4 kf[NP];
    {
        const float* kr = (const float*)p.k + b * p.kv_stride[0] + h * p.kv_stride[1] +
                          (int64_t)(n < N ? n : N - 1) * p.kv_stride[2] + 4 * half;
#pragma unroll
        for (int c = 0; c < NP; c++) kf[c] = *reinterpret_cast<const float4*>(kr + 8 * c);
    }
    const bool live = n < N && masked == 0;
    const bool wanted = __ballot(live) != 0ull;
    const bool chunk_keys = n0 + kKeys > Nc;
    float acc[kAcc] = {};   // of this stream's tiles with the same (t - t_own) mod 4; of a key nobody sees, anything
    const int t_end = __syncthreads_or(wanted) ? n_tiles : t_first;
    for (int t0 = t_first; t0 < t_end; t0 += kColWaves) {
        if (t0 > t_first) {
            __syncthreads();   // the tiles before have been read
            if (t0 + wave < n_tiles) copy_queries(t0 + wave);
        }
        wait_copies<0>();
        __syncthreads();
        // each stream takes every other tile, at its own pace: with a barrier a tile, the vector work of one of the two
        // wavefronts of a SIMD waits for the products of the other and then has the SIMD to itself
        for (int t = t0 + stream; t < t0 + kColWaves && t < n_tiles; t += kColStreams) {
            if (!wanted || t < t_own) continue;
            // whole tiles of rows that all see the keys: normalisers and weights in 16-byte pieces, and no comparisons (vector
            // instructions do not run beside float32 products)
            const bool whole = !chunk_keys && t * kRows + kRows <= Q;
            Vec<4> ls[4], w[4];
#pragma unroll
            for (int i4 = 0; i4 < 4; i4++) {
                const int m0 = t * kRows + 8 * i4 + 4 * half;
                if (whole) {
                    ls[i4] = *reinterpret_cast<const Vec<4>*>(lse + m0);
                    w[i4] = *reinterpret_cast<const Vec<4>*>(p.w_ema + m0);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int m = m0 + e < Q ? m0 + e : Q - 1;
                        ls[i4].v[e] = lse[m];
                        w[i4].v[e] = p.w_ema[m];
                    }
                }
            }
            f32x16 s = zero16();
            const unsigned char* tile = q_lds + (t - t0) * kTile + col * (D * 4);
#pragma unroll
            for (int c = 0; c < NP; c++) {
                const float4 q4 = *reinterpret_cast<const float4*>(tile + Geo<D>::slot(col, 2 * c + half) * 16);
                s = mma(q4.x, kf[c].x, s);
                s = mma(q4.y, kf[c].y, s);
                s = mma(q4.z, kf[c].z, s);
                s = mma(q4.w, kf[c].w, s);
            }
            const bool second = kAcc == 2 && ((t - t_own) & 2);
            float a = second ? acc[kAcc - 1] : acc[0];
            if (whole) {
#pragma unroll
                for (int v = 0; v < 16; v++) a = fmaf(w[v >> 2].v[v & 3], expf(s[v] * p.scale - ls[v >> 2].v[v & 3]), a);
            }
            asm volatile("");
            if (!whole) {
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int m = t * kRows + acc_row(v, half);
                    const float x = fmaf(w[v >> 2].v[v & 3], expf(s[v] * p.scale - ls[v >> 2].v[v & 3]), a);
                    a = m < Q && m >= nrel ? x : a;
                }
            }
            if (second) acc[kAcc - 1] = a;
            else acc[0] = a;
        }
    }
    wait_copies<0>();   // none is on its way to LDS that is somebody else's by then
    // the sums of tiles t_own + i, + 4, ... for i = 0 .. 3, added in that order
    const int class0 = (t_first + stream - t_own) & (kColStreams - 1);
#pragma unroll
    for (int i = 0; i < kAcc; i++) {
        acc[i] += __shfl_xor(acc[i], 32);
        if (!live) acc[i] = 0.f;
        if (half == 0) sums[class0 + kColStreams * i][group * kKeys + col] = acc[i];
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
int run(const CoreProblem& p, hipStream_t stream) {
    const int64_t tiles = (p.Q + kRows - 1) / kRows;
    {
        StageScope sc(CKV_STAGE_FWD, stream);
        const int lds = Geo<D>::kFwdLds;
        if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fwd_f32_mfma_kernel<D>), lds)) return rc;
        hipLaunchKernelGGL(fwd_f32_mfma_kernel<D>, dim3((unsigned)(tiles * p.B * p.H)), dim3(kFwdWaves * CKV_WAVE), lds, stream, p);
        CKV_HIP_TRY(hipGetLastError());
    }
    if (p.colsum) {
        StageScope sc(CKV_STAGE_SCORES, stream);
        // Four blocks of keys share their workgroup's query tiles, unless that leaves more than a quarter of the chip idle (28 heads
        // x 276 and 32 x 360 keys, 16 and 100 rows, 84 and 96 workgroups: 9.6 and 17.5 us against 7.8 and 12.3 with one block each;
        // 32 x 776 keys, 256 rows, 224 workgroups: 30.7 against 34, 28 x 2568 keys, 512 rows: 123 against 156).
        auto launch = [&](auto groups) -> int {
            using C_ = Col<groups.value>;
            auto kernel = colsum_f32_mfma_kernel<D, groups.value>;
            const int lds = C_::kWaves * Geo<D>::kTile;
            if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), lds)) return rc;
            const int64_t blocks = p.B * p.H * ((p.N + C_::kBlockKeys - 1) / C_::kBlockKeys);
            hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(C_::kWaves * CKV_WAVE), lds, stream, p);
            return CKV_OK;
        };
        const int64_t shared = p.B * p.H * ((p.N + Col<4>::kBlockKeys - 1) / Col<4>::kBlockKeys);
        if (int rc = 4 * shared >= 3 * (int64_t)mfma_device_cus() ? launch(std::integral_constant<int, 4>{})
                                                                    : launch(std::integral_constant<int, 1>{})) return rc;
        CKV_HIP_TRY(hipGetLastError());
    }
    return CKV_OK;
}

bool rows16(const int64_t* st, const void* base) {
    return st[3] == 1 && st[0] % 4 == 0 && st[1] % 4 == 0 && st[2] % 4 == 0 && reinterpret_cast<uintptr_t>(base) % 16 == 0;
}

}  // namespace

bool f32_mfma_supported(const CoreProblem& p) {
    // every head its own kv head, every key weighted by the query row alone
    return p.dtype == CKV_F32 && (p.D == 64 || p.D == 128) && p.KVH == p.H && !p.new_mode && p.N < ((int64_t)1 << 31) - 64 &&
           p.B * p.H * ((p.N + kKeys - 1) / kKeys) < ((int64_t)1 << 31) &&   // at least as many as tiles of queries
           p.lse && rows16(p.q_stride, p.q) && rows16(p.kv_stride, p.k) && rows16(p.kv_stride, p.v);
}

int launch_f32_mfma(const CoreProblem& p, hipStream_t stream) { return p.D == 64 ? run<64>(p, stream) : run<128>(p, stream); }

}  // namespace ckv

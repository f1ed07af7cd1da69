// float32 attention and score sums on the matrix cores (v_mfma_f32_32x32x2_f32), head_dim 64 and 128.
//
// The float32 matrix instructions multiply and accumulate in float32 (every product enters the accumulator through a
// fused multiply-add), at twice the rate of the vector ALU and with one operand register per lane instead of LDS reads
// per product, which is what bounded the vector kernels (ckv_attn_generic.hip keeps them for the shapes that do not
// fit here).  32 heads x 256 rows x 516 + 256 keys x 128: forward 269 -> 49 us, scores 321 -> 34 us.
//
//   forward  one workgroup = one kv head x 32 (position, head) rows; its eight wavefronts take the 32-key blocks in
//            turn, each with an online softmax of its own, and merge at the end through LDS.  S^T = K Q^T keeps a query
//            in one lane pair, and register v of S^T is, as it stands, the B operand of step v of O^T += V^T P^T: nothing
//            is moved between the two products.  Keys and values go from memory straight to the operand registers (no
//            two wavefronts of a workgroup share any); the queries sit in LDS in operand order.
//   colsum   one workgroup = one head x 32 keys, held in registers; its four wavefronts take the 32-row query tiles in
//            turn.  S = Q K^T keeps a key in one lane pair, so a weighted sum stays in its lane until the end.
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

namespace ckv {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kRows = 32;      // query rows of a forward workgroup
constexpr int kKeys = 32;      // keys of a block
constexpr int kFwdWaves = 8, kColWaves = 4;

template <int D>
struct Geo {
    static constexpr int kPieces = D / 8;   // 16-byte pieces of a row per lane half
    static constexpr int kDB = D / 32;      // accumulators of 32 dims
    static constexpr int kPitch = D + 4;    // floats of a row in the merge area
    static constexpr int kQ = kPieces * CKV_WAVE * 16;
    static constexpr int kFwdLds = kQ + kFwdWaves * kRows * kPitch * 4 + 2 * kFwdWaves * kRows * 4;
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

struct F32Fwd {
    CoreProblem c;
    int n_split;     // shares of the key blocks per row tile: few rows would leave most of the chip idle
    float* part_o;   // (n_split, B*H*Q, D) and
    float* part_l;   // (n_split, B*H*Q): every share normalised by its own sum, and the logarithm of that
};

template <int D>
__global__ void __launch_bounds__(kFwdWaves* CKV_WAVE) fwd_f32_mfma_kernel(F32Fwd f) {
    using G_ = Geo<D>;
    constexpr int NP = G_::kPieces, DB = G_::kDB;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float4* q_lds = reinterpret_cast<float4*>(lds);                  // [piece][lane]
    float* o_lds = lds + G_::kQ / 4;                                  // [wave][row][kPitch]
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
    const int N = (int)p.N, Q = (int)p.Q, Nc = N - Q;
    const float* kb = (const float*)p.k + b * p.kv_stride[0] + kvh * p.kv_stride[1];
    const float* vb = (const float*)p.v + b * p.kv_stride[0] + kvh * p.kv_stride[1];

    for (int i = tid; i < NP * CKV_WAVE; i += kFwdWaves * CKV_WAVE) {
        const int rf = rt * kRows + (i & 31), m = rf / G, g = rf % G;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (m < Q)
            v = *reinterpret_cast<const float4*>((const float*)p.q + b * p.q_stride[0] + (kvh * G + g) * p.q_stride[1] +
                                                 m * p.q_stride[2] + 8 * (i >> 6) + 4 * ((i >> 5) & 1));
        q_lds[i] = v;
    }
    __syncthreads();

    const int row_m = (rt * kRows + col) / G;            // this lane's query
    int m_hi = (rt * kRows + kRows - 1) / G;
    if (m_hi > Q - 1) m_hi = Q - 1;
    const int nblk = (Nc + m_hi) / kKeys + 1;            // blocks some row of the tile may see
    // bit r: key r of the block is there and not masked
    auto visible_keys = [&](int n) { return (uint32_t)__ballot(n < Nc ? !(p.kmasked && p.kmasked[n]) : n < N); };
    // the logits of a block's keys (lane = its query), and the keys this lane's query sees
    auto logits = [&](const float4(&kf)[NP]) {
        f32x16 s = zero16();
#pragma unroll
        for (int c = 0; c < NP; c++) {
            const float4 q4 = q_lds[c * CKV_WAVE + lane];
            s = mma(kf[c].x, q4.x, s);
            s = mma(kf[c].y, q4.y, s);
            s = mma(kf[c].z, q4.z, s);
            s = mma(kf[c].w, q4.w, s);
        }
        return s;
    };
    auto seen_keys = [&](uint32_t vis, int n0) {
        if (n0 + kKeys - 1 < Nc) return vis;
        const int last = Nc + row_m - n0;   // last key of the block the row may see
        return vis & (last >= 31 ? ~0u : (last < 0 ? 0u : (2u << last) - 1u));   // cached keys lie in front of the chunk keys: row_m >= 0 lets them all through
    };
    auto load_keys = [&](int n, float4(&kf)[NP]) {
        const float* kr = kb + (int64_t)(n < N ? n : N - 1) * p.kv_stride[2] + 4 * half;
#pragma unroll
        for (int c = 0; c < NP; c++) kf[c] = *reinterpret_cast<const float4*>(kr + 8 * c);
    };
    // values of the lane's half of the keys, dims DB col .. DB col + DB - 1: accumulator db holds dims DB m + db
    auto load_values = [&](int n0, Vec<DB>(&vf)[16]) {
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int nv = n0 + acc_row(v, half);
            vf[v] = *reinterpret_cast<const Vec<DB>*>(vb + (int64_t)(nv < N ? nv : N - 1) * p.kv_stride[2] + DB * col);
        }
    };
    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; db++) o[db] = zero16();
    float m_run = -INFINITY, l_run = 0.f;
    for (int blk = split * kFwdWaves + wave; blk < nblk; blk += kFwdWaves * f.n_split) {
        const int n0 = blk * kKeys;
        const int n = n0 + col;
        const uint32_t vis = visible_keys(n);
        if (vis == 0u) continue;
        float4 kf[NP];
        load_keys(n, kf);
        Vec<DB> vf[16];
        load_values(n0, vf);
        f32x16 s = logits(kf);
        const uint32_t allow = seen_keys(vis, n0);   // bit r: key r of the block is visible to this lane's query
        const bool whole = __ballot(allow != ~0u) == 0ull;
        float mx = -INFINITY;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const float x = s[v] * p.scale;
            s[v] = whole || ((allow >> acc_row(v, half)) & 1u) ? x : -INFINITY;
            mx = fmaxf(mx, s[v]);
        }
        if (!whole) {   // the row of a key nobody sees may hold anything
#pragma unroll
            for (int v = 0; v < 16; v++)
#pragma unroll
                for (int db = 0; db < DB; db++) vf[v].v[db] = (vis >> acc_row(v, half)) & 1u ? vf[v].v[db] : 0.f;
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
    }

    float zero = 0.f;   // or NaN
#pragma unroll
    for (int db = 0; db < DB; db++)
#pragma unroll
        for (int v = 0; v < 16; v++) zero = fmaf(o[db][v], 0.f, zero);
    if (__ballot(zero != 0.f) != 0ull) {
#pragma unroll
        for (int db = 0; db < DB; db++) o[db] = zero16();
        for (int blk = split * kFwdWaves + wave; blk < nblk; blk += kFwdWaves * f.n_split) {
            const int n0 = blk * kKeys;
            const uint32_t vis = visible_keys(n0 + col);
            if (vis == 0u) continue;
            f32x16 s;
            {
                float4 kf[NP];
                load_keys(n0 + col, kf);
                s = logits(kf);
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
    const int rf = rt * kRows + r, m = rf / G, g = rf % G;
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
    // A row without a probability above zero (all its logits overflowed) or with a NaN among them is NaN, however many
    // shares its keys are in; a share without one says so by -inf, a NaN has to reach the merge.
    const float inv = 1.f / L;
    const int64_t row = (b * p.H + kvh * G + g) * p.Q + m, rows = p.B * p.H * p.Q;
    if (f.n_split > 1) {
        float* po = f.part_o + (split * rows + row) * D + d0;
#pragma unroll
        for (int i = 0; i < kPer; i++) po[i] = L == 0.f ? 0.f : acc[i] * inv;
        if (d0 == 0) f.part_l[split * rows + row] = L == 0.f ? -INFINITY : M + logf(L);
        return;
    }
    float* orow = (float*)p.out + b * p.out_stride[0] + (kvh * G + g) * p.out_stride[1] + m * p.out_stride[2];
#pragma unroll
    for (int i = 0; i < kPer; i++) orow[(d0 + i) * p.out_stride[3]] = acc[i] * inv;
    if (d0 == 0 && p.lse) p.lse[row] = M + logf(L);
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
    for (int s = 0; s < f.n_split; s++) M = fmaxf(M, f.part_l[s * rows + row]);
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s = 0; s < f.n_split; s++) {
        const float l = f.part_l[s * rows + row];
        if (l == -INFINITY) continue;
        const float w = expf(l - M);
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
    if (d4 == 0 && p.lse) p.lse[row] = M + logf(L);
}

template <int D>
__global__ void __launch_bounds__(kColWaves* CKV_WAVE, 2) colsum_f32_mfma_kernel(CoreProblem p) {
    constexpr int NP = Geo<D>::kPieces;
    __shared__ float sums[kColWaves][kKeys];
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nbkv = (int)(p.B * p.KVH), KVH = (int)p.KVH, G = (int)p.H / KVH;
    const int N = (int)p.N, Q = (int)p.Q, Nc = N - Q, nblk = (N + kKeys - 1) / kKeys;
    // kv heads round the XCDs; blocks of chunk keys see fewer rows and come last
    const int bkv = blockIdx.x % nbkv, rest = blockIdx.x / nbkv;
    const int g = rest % G, blk = rest / G;
    if (blk >= nblk) return;
    const int64_t b = bkv / KVH, kvh = bkv % KVH, h = kvh * G + g;
    const int n0 = blk * kKeys, n = n0 + col, nrel = n - Nc;   // nrel >= 0: a chunk key
    const bool live = n < N && !(n < Nc && p.kmasked && p.kmasked[n]);
    float acc = 0.f;
    if (__ballot(live) != 0ull) {
        float4 kf[NP];
        const float* kr = (const float*)p.k + b * p.kv_stride[0] + kvh * p.kv_stride[1] +
                          (int64_t)(n < N ? n : N - 1) * p.kv_stride[2] + 4 * half;
#pragma unroll
        for (int c = 0; c < NP; c++) kf[c] = *reinterpret_cast<const float4*>(kr + 8 * c);
        const float* qb = (const float*)p.q + b * p.q_stride[0] + h * p.q_stride[1];
        const float* lse = p.lse + (b * p.H + h) * p.Q;
        const int t0 = n0 > Nc ? (n0 - Nc) / kRows : 0;   // first tile with a row that sees a key of the block
        for (int mt = (t0 + wave) * kRows; mt < Q; mt += kColWaves * kRows) {
            float4 qf[NP];
            const float* qr = qb + (int64_t)(mt + col < Q ? mt + col : Q - 1) * p.q_stride[2] + 4 * half;
#pragma unroll
            for (int c = 0; c < NP; c++) qf[c] = *reinterpret_cast<const float4*>(qr + 8 * c);
            float ls[16];
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int m = mt + acc_row(v, half);
                ls[v] = lse[m < Q ? m : Q - 1];
            }
            f32x16 s = zero16();
#pragma unroll
            for (int c = 0; c < NP; c++) {
                s = mma(qf[c].x, kf[c].x, s);
                s = mma(qf[c].y, kf[c].y, s);
                s = mma(qf[c].z, kf[c].z, s);
                s = mma(qf[c].w, kf[c].w, s);
            }
            const bool by_distance = nrel >= 0 && p.new_mode;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int m = mt + acc_row(v, half);
                const bool seen = live && m < Q && m >= nrel;
                const int d = m - nrel;
                const float w = by_distance ? p.w_new[seen ? d : 0] : p.w_ema[m < Q ? m : Q - 1];
                if (seen) acc = fmaf(w, expf(s[v] * p.scale - ls[v]), acc);
            }
        }
    }
    acc += __shfl_xor(acc, 32);
    if (half == 0) sums[wave][col] = acc;
    __syncthreads();
    if (tid < kKeys && n < N) {
        float tot = 0.f;
#pragma unroll
        for (int w = 0; w < kColWaves; w++) tot += sums[w][tid];
        p.colsum[(b * p.H + h) * p.N + n] = tot;
    }
}

template <int D>
int run(const CoreProblem& p, float* part_o, float* part_l, hipStream_t stream) {
    const int64_t G = p.H / p.KVH, tiles = (p.Q * G + kRows - 1) / kRows;
    {
        StageScope sc(CKV_STAGE_FWD, stream);
        F32Fwd f;
        f.c = p;
        f.n_split = part_o && part_l ? f32_mfma_splits(p.B, p.H, p.KVH, p.Q, p.N, mfma_device_cus()) : 1;
        f.part_o = part_o;
        f.part_l = part_l;
        const int lds = Geo<D>::kFwdLds;
        if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(fwd_f32_mfma_kernel<D>), lds)) return rc;
        hipLaunchKernelGGL(fwd_f32_mfma_kernel<D>, dim3((unsigned)(tiles * f.n_split * p.B * p.KVH)), dim3(kFwdWaves * CKV_WAVE),
                           lds, stream, f);
        CKV_HIP_TRY(hipGetLastError());
        if (f.n_split > 1) {
            constexpr int per = 256 / (D / 4);
            hipLaunchKernelGGL(fwd_f32_combine_kernel<D>, dim3((unsigned)((p.B * p.H * p.Q + per - 1) / per)), dim3(256), 0, stream, f);
            CKV_HIP_TRY(hipGetLastError());
        }
    }
    if (p.colsum) {
        StageScope sc(CKV_STAGE_SCORES, stream);
        const int64_t blocks = p.B * p.H * ((p.N + kKeys - 1) / kKeys);
        hipLaunchKernelGGL(colsum_f32_mfma_kernel<D>, dim3((unsigned)blocks), dim3(kColWaves * CKV_WAVE), 0, stream, p);
        CKV_HIP_TRY(hipGetLastError());
    }
    return CKV_OK;
}

bool rows16(const int64_t* st, const void* base) {
    return st[3] == 1 && st[0] % 4 == 0 && st[1] % 4 == 0 && st[2] % 4 == 0 && reinterpret_cast<uintptr_t>(base) % 16 == 0;
}

}  // namespace

// One workgroup fills a compute unit (eight wavefronts of some 220 registers), so a launch with fewer row tiles than
// that shares the key blocks of a tile out, at least two per wavefront, as long as the shares still fit one round.
int f32_mfma_splits(int64_t B, int64_t H, int64_t KVH, int64_t Q, int64_t n, int cus) {
    const int64_t wgs = ((Q * (H / KVH) + kRows - 1) / kRows) * B * KVH, blocks = (n + kKeys - 1) / kKeys;
    int64_t s = cus / wgs;
    if (s > blocks / (2 * kFwdWaves)) s = blocks / (2 * kFwdWaves);
    if (s > 16) s = 16;
    return s < 1 ? 1 : (int)s;
}

bool f32_mfma_supported(const CoreProblem& p) {
    return p.dtype == CKV_F32 && (p.D == 64 || p.D == 128) && p.N < ((int64_t)1 << 31) - 64 &&
           p.B * p.H * ((p.N + kKeys - 1) / kKeys) < ((int64_t)1 << 31) &&
           ((p.Q * (p.H / p.KVH) + kRows - 1) / kRows) * 16 * p.B * p.KVH < ((int64_t)1 << 31) && p.lse && rows16(p.q_stride, p.q) &&
           rows16(p.kv_stride, p.k) && rows16(p.kv_stride, p.v);
}

int launch_f32_mfma(const CoreProblem& p, float* part_o, float* part_l, hipStream_t stream) {
    return p.D == 64 ? run<64>(p, part_o, part_l, stream) : run<128>(p, part_o, part_l, stream);
}

}  // namespace ckv

// Internal interfaces between the attention entry points and the kernel families.
#pragma once

#include "ckv_common.h"

namespace ckv {

struct KeptScores;

// max over the two lane halves (lane l and lane l ^ 32) without a trip through LDS
__device__ inline float half_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Attention over keys that are already rotated and laid out as [cached | chunk]:
//   out[b,h,m]  = softmax_n(scale * q[b,h,m] . k[b,h/G,n] + mask) v[b,h/G,n]
//   cached key n < n_cached is masked iff kmasked[n]; chunk key n is visible iff n-n_cached <= m
//   colsum[b,h,n] = sum_m weight(m,n) * P[m,n]   (optional)
//     weight = w_ema[m]                         for cached keys, and for chunk keys if !new_mode
//     weight = w_new[m - (n - n_cached)]        for chunk keys if new_mode (m >= n - n_cached)
struct CoreProblem {
    const void* q;
    int64_t q_stride[4];      // (B, H, Q, D)
    const void* k;
    const void* v;
    int64_t kv_stride[4];     // (B, KVH, N, D)
    const uint8_t* kmasked;   // (n_cached,) 1 = masked; may be null when n_cached == 0
    void* out;
    int64_t out_stride[4];    // (B, H, Q, D)
    float* lse;               // (B, H, Q) natural-log normaliser of every row
    float* colsum;            // (B, H, N) or null
    const float* w_ema;       // (Q,)
    const float* w_new;       // (Q,)
    int new_mode;
    int64_t B, H, KVH, Q, N, D;
    float scale;
    int dtype;
};

// fp32-math kernels on the vector ALU for every dtype and head size (<= 256): the fallback for shapes the kernels on the
// matrix cores (16-bit and float32) do not cover.
int launch_core_generic(const CoreProblem& p, hipStream_t stream);

// The same in float32 on the matrix cores, for the dense operator: head_dim 64 and 128, rows of 16-byte pieces, lse wanted, KVH == H, weights
// by row alone (new_mode 0).
bool f32_mfma_supported(const CoreProblem& p);
int launch_f32_mfma(const CoreProblem& p, hipStream_t stream);

// ckv_attn in float32, head_dim 64 and 128, on the bfloat16 matrix cores: staging, attention and score sums.  The staged operands, in
// tiles of 32 rows, three planes each (f32_split_plane_bytes): queries (B, H), keys and values (B, KVH); a word per 32 keys,
// a bit for each that is there and not masked; of every tile, which parts hold values that three planes do not take (odd_kv: keys and
// values; odd_q).
struct F32Planes {
    void *q, *k, *v;
    uint32_t *vis, *odd_q;
    uint2* odd_kv;
    int q_tiles;         // of a head
    uint32_t w_new_at;   // bytes from the weights w_ema to w_new, which lie behind them
};
bool f32_split_supported(int dtype, int64_t B, int64_t H, int64_t KVH, int64_t Q, int64_t n, int64_t D);
int f32_split_shares(int64_t B, int64_t H, int64_t KVH, int64_t Q, int64_t n, int cus);
int64_t f32_split_plane_bytes(int64_t units, int64_t rows, int64_t D);
// `p`: sizes, out, lse (null: not wanted), colsum and the weights; its operands are not read.  norm: scratch, B*H*Q pairs.  part_o / part_l: f32_split_shares shares of
// (B*H*Q, D) floats / (B*H*Q) pairs, or null (then the keys of a row tile are not shared out).
int launch_f32_split(const ckv_attn_args& a, const CoreProblem& p, const F32Planes& f, float* w_ema, float* w_new, float2* norm,
                     float* part_o, float2* part_l, const KeptScores& kept, hipStream_t stream);

// weights of the score sums (cascade_attention.py:270-282, 315-317), rounded like the eager path
// w_ema gets 64 trailing zeros (slack read by the MFMA column pass)
int launch_weights(float* w_ema, float* w_new, int64_t Q, double beta, int dtype, hipStream_t stream);

// The dense operator's prologue in one launch: the weights of the score sums (w_ema null: none), and the key order: the
// rows of the cached keys that are not masked, in ascending order, then the n_ctx chunk keys, then the masked ones.
// mask (n_cached) 1 = masked; key_order (n_cached + n_ctx); n_visible: how many cached keys are not masked.
int launch_dense_prologue(const uint8_t* mask, int64_t n_cached, int64_t n_ctx, int* key_order, int* n_visible, float* w_ema,
                          float* w_new, double beta, int dtype, hipStream_t stream);

int launch_cast_scores(const float* colsum, void* scores, const int64_t* stride, int64_t B, int64_t H, int64_t N,
                       int dtype, hipStream_t stream);

struct PrepProblem {
    const ckv_attn_args* a;
    void* qr;        // (B, H, Q, D) rotated queries
    void* kr;        // (B, KVH, N, D) rotated keys, [sink | cache | chunk]
    void* vc;        // (B, KVH, N, D) values in the same order
    uint8_t* kmasked;  // (num_sink + S,)
    float *w_ema, *w_new;  // the weights of the score sums, see launch_weights; null: none are wanted
};
int launch_prep_generic(const PrepProblem& p, hipStream_t stream);

struct FinishProblem {
    const float* colsum;   // (B, H, N)
    int64_t N;
    void* cache_s;         // (B, KVH, S) strides below; may be null
    int64_t cache_s_stride[3];
    void* new_scores;      // (B, KVH, Q); may be null
    int64_t new_scores_stride[3];
    int64_t B, H, KVH, Q, S, num_sink;
    float beta_pow_q;      // beta^Q rounded to fp32
    int head_reduction, homogeneous, dtype;
    int heads;             // that are reduced together: H, or H / KVH
    const void* before = nullptr;  // see KeptScores; null: the update does not share the launch
};
int launch_finish(const FinishProblem& p, hipStream_t stream);

// A short chunk's update is planned in the launch that finishes its scores: the plan works the few scores it asks for out by itself,
// and reads those of the cache as they were before the call, of which the staging launch keeps a copy (the finishing blocks write theirs
// in place meanwhile).
struct KeptScores {
    const void* src = nullptr;   // (units, S); null: nobody asks
    int64_t stride[3];           // by batch, kv head, slot
    void* dst;                   // contiguous
    int64_t units, KVH, S;
};
constexpr int kKeptPer = 8;      // slots a thread copies
inline int64_t kept_pieces(const KeptScores& k, int threads) {
    return k.src ? k.units * ((k.S + kKeptPer * threads - 1) / (kKeptPer * threads)) : 0;
}
template <typename T, int kThreads>
__device__ inline void keep_scores(const KeptScores& k, int64_t piece, int tid) {
    const int64_t per = (k.S + kKeptPer * kThreads - 1) / (kKeptPer * kThreads), unit = piece / per;
    if (unit >= k.units) return;
    const int64_t b = unit / k.KVH, kvh = unit - b * k.KVH, first = (piece - unit * per) * (kKeptPer * kThreads) + tid;
    const T* src = (const T*)k.src + b * k.stride[0] + kvh * k.stride[1];
    T v[kKeptPer];
#pragma unroll
    for (int j = 0; j < kKeptPer; j++) {
        const int64_t i = first + j * kThreads;
        v[j] = src[(i < k.S ? i : k.S - 1) * k.stride[2]];
    }
#pragma unroll
    for (int j = 0; j < kKeptPer; j++) {
        const int64_t i = first + j * kThreads;
        if (i < k.S) ((T*)k.dst)[unit * k.S + i] = v[j];
    }
}
// may the update of a call's tokens be planned in the launch that finishes their scores?  (Both are checked; workspaces apart.)
bool update_plans_beside_finish(const ckv_attn_args& a, const ckv_update_args& u);
int launch_finish_and_update(const FinishProblem& p, const ckv_update_args& u, hipStream_t stream);

// rows of slack behind the staged queries, their normalisers and weights: the column pass reads whole
// tiles of this many query rows
constexpr int64_t kColSlack = 128;

// weights: w_ema[m] = (1-beta) * beta^(Q-1-m) as fp32 (cascade_attention.py:315-317);
//          w_new[k] = (1-beta) * beta^k built in the tensor dtype (cascade_attention.py:270-276)
template <typename T>
__device__ inline void weights_at(float* w_ema, float* w_new, int64_t Q, double beta, int64_t i) {
    auto round_t = [](float v) { return Elem<T>::to_float(Elem<T>::from_float(v)); };
    if (i >= Q + kColSlack) return;
    if (i >= Q) {  // slack read (and multiplied by zero) by the MFMA column pass
        w_ema[i] = 0.f;
        return;
    }
    const float omb = (float)(1.0 - beta);
    const float b32 = (float)beta;
    w_ema[i] = __fmul_rn(omb, powf(b32, (float)(Q - 1 - i)));
    const float bt = round_t(b32);
    const float pw = round_t(powf(bt, round_t((float)i)));
    w_new[i] = round_t(__fmul_rn(omb, pw));
}

// The key order of launch_dense_prologue, worked out by one workgroup of kThreads threads (64 .. 1024, a multiple of 64).
template <int kThreads>
__device__ inline void key_order_block(const uint8_t* mask, int64_t n_cached, int64_t n_ctx, int* key_order, int* n_visible) {
    constexpr int kPer = 16, kWaves = kThreads / CKV_WAVE;
    __shared__ int wave_sum[2][kWaves];
    const int tid = threadIdx.x, lane = tid % CKV_WAVE, wave = tid / CKV_WAVE;
    const int64_t n_kv = n_cached + n_ctx;
    const bool vec = (reinterpret_cast<uintptr_t>(mask) & 15) == 0;
    int seen = 0, round = 0;  // visible keys in the stretches before
    for (int64_t base = 0; base < n_cached; base += kThreads * kPer, round ^= 1) {
        // this thread's 16 keys as a word of bits, one per visible key
        const int64_t first = base + (int64_t)tid * kPer;
        uint32_t bits = 0;
        if (vec && first + kPer <= n_cached) {
            const uint4 m = *reinterpret_cast<const uint4*>(mask + first);
            const uint32_t w[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
            for (int i = 0; i < kPer; i++) bits |= (((w[i >> 2] >> (8 * (i & 3))) & 0xffu) == 0u ? 1u : 0u) << i;
        } else {
            for (int i = 0; i < kPer; i++)
                if (first + i < n_cached && mask[first + i] == 0) bits |= 1u << i;
        }
        const int mine = __popc(bits);
        int incl = mine;
        for (int off = 1; off < CKV_WAVE; off <<= 1) {
            const int v = __shfl_up(incl, off);
            if (lane >= off) incl += v;
        }
        if (lane == CKV_WAVE - 1) wave_sum[round][wave] = incl;
        __syncthreads();  // the sums of the next stretch go to the other half
        int before = seen, total = seen;
        for (int w = 0; w < kWaves; w++) {
            const int v = wave_sum[round][w];
            before += w < wave ? v : 0;
            total += v;
        }
        int vis = before + incl - mine;                              // visible keys before this thread's first one
        int64_t hid = n_kv - 1 - (first - vis);                      // masked ones fill the end backwards
        for (int i = 0; i < kPer; i++) {
            if (first + i >= n_cached) break;
            if ((bits >> i) & 1u) key_order[vis++] = (int)(first + i);
            else key_order[hid--] = (int)(first + i);
        }
        seen = total;
    }
    for (int64_t i = tid; i < n_ctx; i += kThreads) key_order[seen + i] = (int)(n_cached + i);
    if (tid == 0) *n_visible = seen;
}

// ---- bf16/fp16 MFMA family (head_dim 64 and 128) ----
struct MfmaSegment {
    const void* k;
    const void* v;
    int64_t stride[4];     // (B, KVH, len, D)
    const int64_t* pos;    // null: keys are already rotated
    int64_t pos_stride[2];
    int64_t pos_shift;
    const uint8_t* masked; // null: all visible
    int64_t len;
};

struct MfmaProblem {
    MfmaSegment seg[3];    // keys in order; the LAST Q keys overall are the causal chunk
    const void* q;
    int64_t q_stride[4];
    const int64_t* q_pos;  // null: queries are already rotated
    const float* inv_freq;
    float theta;
    int shared_pos;
    void *qr, *kr, *vt;
    unsigned long long* tile_vis;
    void* out;
    int64_t out_stride[4];
    float* lse;            // (B, H, Q) natural log
    float* lse2;           // (B*H*Q + kColSlack) scratch: minus the log2-domain normaliser, for the column pass
    float* colsum;         // (B, H, n) or null
    void* scores = nullptr;  // takes colsum's place: (B, H, n) in the tensor dtype, at the row each key came from
    int64_t scores_stride[3] = {0, 0, 0};
    float* part_scores = nullptr;  // (dense_row_shares, B*H, n): where the sums of a key are shared out, or null
    // keys in another order than they lie in memory (launch_dense_prologue): seg[0] then holds all keys
    int* key_order = nullptr;
    int* n_visible = nullptr;
    int own_order = 0;     // the staging launch works the order out (order_by_staging), from this mask
    const uint8_t* order_mask = nullptr;
    float* part_o;         // (mfma_fwd_splits, B*H*Q, D) and
    float* part_l2;        // (mfma_fwd_splits, B*H*Q): the forward kernel's shares, when it splits the keys
    float* w_ema;
    float* w_new;
    double beta;           // the EMA factor of the weights
    int make_weights = 0;  // the staging launch writes w_ema and w_new too
    KeptScores kept;       // and keeps these
    int new_mode;
    int64_t B, H, KVH, Q, D, n, n_pad;
    int64_t empty_from = 0, empty_to = 0;  // keys whose slots cannot hold a token yet
    float scale;
    float key_scale;       // keys with position ids are multiplied by this after rotation and rounded again, the
                           // queries carry scale / key_scale: sqrt(scale) for the cascade path, which follows the
                           // eager arm (cascade_attention.py:284-291); 1 for keys that arrive rotated
    int dtype;
};

bool mfma_supported(int dtype, int64_t D, int64_t H, int64_t KVH, int64_t Q);
int64_t mfma_n_pad(int64_t n);
// shares of the key tiles per query tile on a chip of `cus` compute units; what a workspace must hold
int mfma_fwd_splits(int64_t B, int64_t H, int64_t KVH, int64_t Q, int64_t n, int cus, bool dense);
int mfma_fwd_splits_for_workspace(int64_t B, int64_t H, int64_t KVH, int64_t Q, int64_t n, bool dense);
int dense_row_shares(int64_t B, int64_t H, int64_t n_ctx, int64_t n_kv, int cus);
bool order_by_staging(int64_t n_cached);
int mfma_device_cus();  // compute units of the current device (256 where none can be asked)
bool mfma_fits(int64_t n, int64_t D);  // the per-tile bookkeeping of n keys fits in LDS
int launch_mfma(const MfmaProblem& p, hipStream_t stream);

// ---- backward of the dense operator on the matrix cores (16-bit, head_dim 64 and 128, 16-byte addressable rows) ----
// key_order / n_visible: see launch_dense_prologue; both null when the caller's workspace has no room for them
bool bwd_mfma_supported(const ckv_dense_bwd_args& a);
int bwd_mfma_dq_splits(int64_t B, int64_t H, int64_t n_ctx, int64_t n_kv, int cus);
// delta: (B, H, n_ctx); part_dq: bwd_mfma_dq_splits shares of (B, H, n_ctx, D) floats, or null (then dq is not shared out)
int launch_bwd_mfma(const ckv_dense_bwd_args& a, const float* delta, const int* key_order, const int* n_visible, float* part_dq,
                    int n_split, hipStream_t stream);

// ---- single-token decode family (Q == 1, head_dim 128) ----
bool decode_supported(const ckv_attn_args& a);
int64_t decode_workspace_bytes(int64_t B, int64_t H, int64_t KVH, int64_t num_sink, int64_t S);
bool update_beside_scores(const ckv_attn_args& a, const ckv_update_args& u);
// u: the cache update that follows, checked, or null; *updated: it has been launched with the step's own kernels
int launch_decode(const ckv_attn_args& a, hipStream_t stream, const ckv_update_args* u, bool* updated);

// everything ckv_update checks before a launch (its scratch too); *empty: nothing to do
int check_update(const ckv_update_args* args, bool* empty);
// stages are timed one by one, or the kernels of the update: launches of several stages would blur them
bool prof_update_apart();

}  // namespace ckv

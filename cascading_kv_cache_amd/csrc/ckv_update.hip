// ckv_update: the cascading cache update as a plan + apply pair of gfx950 kernels.
//
// Replaces the serial per-token Triton program of the reference
// (cascade/models/cascading_cache.py:145-299 token loop, 302-774 body) with
//
//   plan   a unit (batch, kv-head) in the steady state is planned from closed forms, its cascades side by side.
//          Else one workgroup walks the cascades of the unit in order; at every cascade
//          the arrivals of the whole call are classified (insert / challenger), numbered with a
//          ballot prefix sum, the challengers of each group are reduced to the group's winner
//          ("later wins iff score >=", cascading_cache.py:699), and the tokens the cascade evicts
//          become the arrival list of the next cascade.  Everything lives in LDS.  The result is
//          a forest of disjoint move chains in global memory:
//              first[t]   = slot the incoming token t finally lands in (-1: dropped)
//              next_of[d] = slot the OLD content of slot d finally lands in (-1: dropped)
//          plus the trackers after the call, which apply commits.
//   apply  one lane group per incoming token.  Follows the chain of its token from the head,
//          carrying a whole row (K, V, score, original index) in registers with 16-byte lanes:
//          read the displaced row, write the carried one, move on.  Chains are vertex-disjoint
//          and only ever move towards higher cascades, so groups never touch each other's slots.
//          The same launch writes the position ids in closed form from the updated trackers
//          (cascading_cache.py:112-142, 728-774) with extra blocks at the end of its grid.
//
// Why this equals the serial loop: within one cascade the n-th insert of a call always lands in
// ring position (start + stored + n) mod W whatever the scores are; only WHICH arrival owns a
// slot depends on scores, and that is decided inside the group of arrivals between two inserts.
#include "ckv_finish.h"
#include "ckv_update_token.h"

#include <algorithm>
#include <type_traits>

#include <mutex>

namespace ckv {
namespace {

constexpr int kMaxCascades = 64;
constexpr int kPlanMaxTokens = 8192;   // incoming tokens one plan launch takes at most
constexpr int kRingPer = 8;            // kPlanMaxTokens / 1024 threads, and enough for kBothLds's tokens on kClosedThreads

constexpr int32_t kPosChange = 1;      // the call put a token into the cascades, so the position ids change
constexpr int32_t kPlanned = 2;        // the unit has been planned by the steady-state kernel

struct UpdateParams {
    ckv_update_args a;
    int64_t token_offset;  // first incoming token handled by this launch
    int32_t k_sub;         // tokens handled by this launch
    int32_t do_pos;        // run the position pass (last launch of a call only)
    int32_t* first;        // [N*H][K]
    int32_t* next_of;      // [N*H][S]
    int32_t* flags;        // [N*H]: kPosChange | kPlanned
    int32_t* sinks_new;    // [N*H]: sinks stored after the call
    int32_t* trackers;     // [N*H][cascades]: tracker_word of every cascade
    int32_t apply_blocks;  // blocks along x that move rows; the blocks behind them write position ids
    int64_t* row;          // [S]: the position ids of unit 0 after the call, each with row_shift added, or null
    int64_t row_shift;
};

// The (batch, kv head) of a workgroup: grid coordinates y and z, so that no workgroup begins with 64-bit divisions (these
// and the ones of the single-token walk were 0.9 us of the 7.3 that its launch took).
struct Unit {
    int64_t n, h, bh;
    __device__ explicit Unit(const ckv_update_args& A) : n(blockIdx.z), h(blockIdx.y), bh((int64_t)blockIdx.z * A.H + blockIdx.y) {}
};

// exclusive prefix sum of one flag per thread over the whole workgroup; returns the block total
__device__ inline int block_flag_scan(bool flag, int* wave_tot, int& exclusive) {
    const unsigned long long bal = __ballot(flag);
    const int lane = threadIdx.x & (CKV_WAVE - 1);
    const int wave = threadIdx.x / CKV_WAVE;
    const int nwaves = (blockDim.x + CKV_WAVE - 1) / CKV_WAVE;
    const int in_wave = __popcll(bal & ((1ull << lane) - 1ull));
    if (lane == 0) wave_tot[wave] = __popcll(bal);
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < nwaves; w++) {
        const int c = wave_tot[w];
        if (w < wave) before += c;
        total += c;
    }
    __syncthreads();  // wave_tot is reused by the next call
    exclusive = before + in_wave;
    return total;
}

__device__ inline void emit_move(int32_t* first, int32_t* next_of, int dst, int src) {
    next_of[dst] = -1;
    if (src < 0) {
        first[-1 - src] = dst;
    } else {
        next_of[src] = dst;
    }
}

// ---- Units in the steady state: sinks and every cascade full, no token of the call accepted by the eager-fill rule, and every
// acceptance period divides the next one (the power schedules).  Which arrivals a cascade sees, which of them are inserted
// and where is then a closed form of the token counter: the arrivals of cascade i are the tokens whose index is a multiple of
// period i - 1, every (period i / period i - 1)-th of them is inserted, the n-th insert lands n slots behind the ring start
// and pushes the n-th oldest entry on to cascade i + 1.  What is left to compute is who wins each group.
constexpr int kClosedThreads = 512;

struct ClosedCascade {
    int32_t nA, kf, E;  // arrivals, index of the first inserted arrival, inserts
    uint32_t r;         // inserts every r-th arrival
    int32_t sx;         // ring start before the call
};

// From the token counter (less the sinks) and the periods.  `U`: unsigned type that holds them.  A step or group length past 2^31
// means at most one arrival or insert: any such value does.
template <typename U>
__device__ inline bool closed_cascade(U rel0, U per, U per_prev, int cap, ClosedCascade& c) {
    if (per % per_prev != 0) return false;
    const U r = per / per_prev, most = (U)0x7fffffff;
    const U a0 = rel0 % per_prev ? per_prev - rel0 % per_prev : 0;   // first token that arrives here
    const U q0 = rel0 / per_prev + (a0 ? 1 : 0);                     // arrival k is inserted iff (q0 + k) % r == 0
    const U kf = q0 % r ? r - q0 % r : 0;
    c.nA = a0 < (U)cap ? (int32_t)(((U)cap - a0 + per_prev - 1) / per_prev) : 0;
    c.E = kf < (U)c.nA ? (int32_t)(((U)c.nA - kf + r - 1) / r) : 0;
    c.kf = (int32_t)(kf < most ? kf : most);
    c.r = (uint32_t)(r < most ? r : most);
    return true;
}

// Lane j of every wavefront gets cascade j; false: the unit is left to the walk over all arrivals.  `touched`: the cascades that
// hand on entries which depend on this call's scores -- the newest old entry once arrivals have challenged it, or winners
// among the call's own tokens.  (Cascade 0 with period 1 inserts every token: there it is the tokens in order.)
__device__ inline bool closed_forms(const ckv_update_args& A, const Unit& u, int64_t seen, int cap, int lane, ClosedCascade& c,
                                    unsigned long long& touched) {
    const int C = A.cascades;
    const int64_t W = A.window_size, rel0 = seen - A.num_sink;
    int64_t st = W, per = 1;
    c = {};
    if (lane < C) {
        const int64_t at = u.n * A.tracker_stride[0] + u.h * A.tracker_stride[1] + lane * A.tracker_stride[2];
        st = A.stored_tokens[at];
        const int64_t sx = A.start_indices[at];
        if (sx < 0 || sx >= W) st = -1;
        c.sx = (int32_t)sx;
        per = A.do_cache_every_n[lane];
    }
    const int64_t sinks0 = A.stored_sinks[u.n * A.stored_sinks_stride[0] + u.h * A.stored_sinks_stride[1]];
    int64_t per_prev = __shfl_up(per, 1);
    if (lane == 0) per_prev = 1;
    bool ok = st == W && per > 0 && W >= 2 && sinks0 >= A.num_sink && rel0 >= 0 && !(A.eager_fill && seen <= A.max_seq_len + A.num_sink);
    if (__builtin_amdgcn_ballot_w64(ok) != ~0ull) return false;
    // 32-bit division when everything fits, which it does outside pathological streams
    if (lane < C) {
        if (rel0 < (1ll << 31) && __builtin_amdgcn_ballot_w64(per >= (1ll << 30)) == 0) {
            ok = closed_cascade<uint32_t>((uint32_t)rel0, (uint32_t)per, (uint32_t)per_prev, cap, c);
        } else {
            ok = closed_cascade<uint64_t>((uint64_t)rel0, (uint64_t)per, (uint64_t)per_prev, cap, c);
        }
    }
    const int before = __shfl_up(c.E, 1);
    ok = ok && (lane == 0 || lane >= C || before == c.nA);  // what a full cascade evicts: as many as it inserts
    touched = __builtin_amdgcn_ballot_w64(lane < C && !(c.E <= W - 1 || (c.E <= W && c.kf == 0) || (lane == 0 && per == 1)));
    return __builtin_amdgcn_ballot_w64(ok) == ~0ull;
}

// The scores that a plan looks at: those that lie in memory, ...
struct StoredScores {
    static constexpr int kRing = kRingPer;
    const ckv_update_args& A;
    int64_t s_base, cs_base;
    __device__ StoredScores(const UpdateParams& p, const Unit& u)
        : A(p.a), s_base(u.n * A.s_stride[0] + u.h * A.s_stride[1] + p.token_offset * A.s_stride[2]),
          cs_base(u.n * A.cache_s_stride[0] + u.h * A.cache_s_stride[1]) {}
    __device__ float token(int t) const { return load_as_float(A.s, s_base + (int64_t)t * A.s_stride[2], A.dtype); }
    __device__ float slot(int64_t i) const { return load_as_float(A.cache_s, cs_base + i * A.cache_s_stride[2], A.dtype); }
};
// ... and those that the launch is about to finish (FinishProblem::before).
template <typename T, int kHow>
struct FinishingScores {
    static constexpr int kRing = 3;   // of kClosedThreads: kBothLds's tokens
    const FinishProblem& f;
    int64_t b, kvh;
    __device__ float token(int t) const { return Elem<T>::to_float(token_score<T, kHow>(f, b, kvh, t)); }
    __device__ float slot(int64_t i) const {
        return Elem<T>::to_float(slot_score<T, kHow>(f, b, kvh, i, reinterpret_cast<const T*>(f.before)[(b * f.KVH + kvh) * f.S + i]));
    }
};

// Workgroup `part` of `parts` plans its share of the inserts of cascade `mine`: a thread per insert folds the arrivals up to the next insert into the group's winner
// ("later wins iff score >=", cascading_cache.py:699) and writes where every member ends up.  Every chain entry has one
// writer: cascade i owns the pointers of cascade i's arrivals.  Those are entries of the ring before as it was before the
// call, so all cascades are planned side by side; where the cascade before is touched, this workgroup first repeats its pass
// (and that of further touched ones before it) without the pointers, for what they hand on: the old entries, oldest first,
// the newest of them as its challengers left it, then the call's own winners.
// Bound by its chain of dependent loads (trackers, scores) and, where the inserts are many, by instructions: one workgroup
// that walked all cascades took 22 us for 8 units x 4096 tokens x 8 cascades, a workgroup per cascade 10.2, one per 512
// inserts 7.1 (16 units x 16 rings of 2048: 15.6; with 256 threads 7.2 and 24.1, with 1024 8.3 and 16.2).  Touched cascades
// used to be left to the walk, to which a call like 256 tokens on rings of 128 or 4096 on rings of 2048 goes at every other
// alignment: 14.4 and 77 us there, 6.1 and 15.6 here.  A pass that read its arrivals into registers instead of LDS: level.
template <typename Scores>
__device__ inline void plan_closed(const UpdateParams& p, const Unit& u, const ClosedCascade& forms, unsigned long long touched,
                                   int mine, int part, int parts, unsigned char* smem, const Scores& scores_of) {
    const ckv_update_args& A = p.a;
    const int tid = threadIdx.x, T = blockDim.x;
    const int C = A.cascades, W = (int)A.window_size, cap = p.k_sub;
    int32_t* first = p.first + u.bh * A.K + p.token_offset;
    int32_t* next_of = p.next_of + u.bh * A.max_seq_len;
    int32_t* src[2] = {reinterpret_cast<int32_t*>(smem), reinterpret_cast<int32_t*>(smem) + cap};
    float* score[2] = {reinterpret_cast<float*>(smem) + 2 * (size_t)cap, reinterpret_cast<float*>(smem) + 3 * (size_t)cap};
    auto of = [&](int v, int j) -> int { return __builtin_amdgcn_readlane(v, j); };
    auto slot_of = [&](int i, int sx, int m) -> int {  // the m-th entry from the ring start, m < W
        const int ring = sx + m;
        return i * W + (ring >= W ? ring - W : ring);
    };
    auto score_of = [&](int from) -> float {
        return from < 0 ? scores_of.token(-1 - from) : scores_of.slot(from);
    };
    auto point = [&](int from, int slot) {  // the arrival that came from `from` ends up in `slot` (-1: nowhere)
        if (from < 0) first[-1 - from] = slot;
        else next_of[from] = slot;
    };
    // this workgroup's inserts (those of a pass that is repeated are all its own)
    const int E_mine = of(forms.E, mine), share = (E_mine + parts - 1) / parts;
    const int g_lo = part * share, g_hi = g_lo + share < E_mine ? g_lo + share : E_mine;
    if (part > 0 && g_lo >= E_mine) return;
    // the first cascade of the passes: its arrivals are read where they were before the call
    const unsigned long long below = ~touched & ((1ull << mine) - 1ull);
    const int from_cascade = below ? 64 - __builtin_clzll(below) : 0;
    {
        const int i = from_cascade, nA = of(forms.nA, i), sx_prev = i > 0 ? of(forms.sx, i - 1) : 0;
        const bool scores = i != mine || of((int)forms.r, i) != 1 || of(forms.kf, i) != 0;   // else nobody is challenged
        // a workgroup that has its own pass only needs the arrivals of its inserts, the first one those before them too
        const int r = of((int)forms.r, i), kf = of(forms.kf, i);
        const int lo = i == mine && part > 0 ? kf + g_lo * r : 0, hi = i == mine && part + 1 < parts ? kf + g_hi * r : nA;
        for (int k = lo + tid; k < hi; k += T) {
            // cascade 0 sees every token; past a ring's old entries its own inserts follow, which only cascade 0 hands on untouched
            const int from = i == 0 ? -1 - k : k >= W ? -1 - (k - W) : slot_of(i - 1, sx_prev, k);
            src[i & 1][k] = from;
            if (scores) score[i & 1][k] = score_of(from);
        }
    }
    for (int i = from_cascade; i <= mine; i++) {
        __syncthreads();
        const int nA = of(forms.nA, i), kf = of(forms.kf, i), E = of(forms.E, i), sx = of(forms.sx, i);
        const uint32_t r = (uint32_t)of((int)forms.r, i);
        const bool writes = i == mine, last = i + 1 >= C;
        const int32_t* a_src = src[i & 1];
        const float* a_score = score[i & 1];
        int32_t* b_src = src[(i & 1) ^ 1];
        float* b_score = score[(i & 1) ^ 1];
        // arrivals k0 .. k1 - 1 challenge the holder; who loses ends up nowhere
        auto challenge = [&](int k0, int k1, int& ws, float& wv, bool& held) {
            for (int k = k0; k < k1; k++) {
                const int from = a_src[k];
                const float v = a_score[k];
                if (v >= wv) {
                    if (writes && !held) point(ws, -1);
                    held = false;
                    ws = from;
                    wv = v;
                } else if (writes) {
                    point(from, -1);
                }
            }
        };
        if (tid == T - 1 && (!writes || part == 0) && (kf > 0 || (!writes && E >= W))) {
            // arrivals before the first insert challenge the newest entry earlier calls left
            const int p_lead = slot_of(i, sx, W - 1);
            int ws = p_lead;
            float wv = score_of(p_lead);
            bool held = true;  // the old entry still holds the slot
            challenge(0, kf < nA ? kf : nA, ws, wv, held);
            if (writes) {
                if (!held) next_of[p_lead] = -1;  // the old entry is dropped
                if (!held && E < W) point(ws, p_lead);
                if (!held && E >= W && last) point(ws, -1);  // insert W - 1 takes the slot again
            } else if (E >= W) {
                b_src[W - 1] = ws;
                b_score[W - 1] = wv;
            }
        }
        const int g_end = writes ? g_hi : E;
        for (int g = (writes ? g_lo : 0) + tid; g < g_end; g += T) {
            const int k0 = kf + (int)((uint32_t)g * r);
            const int k1 = r < (uint32_t)(nA - k0) ? k0 + (int)r : nA;
            int ws = a_src[k0];
            float wv = 0.f;
            bool held = false;
            if (k1 > k0 + 1 || !writes) {
                wv = a_score[k0];
                challenge(k0 + 1, k1, ws, wv, held);
            }
            if (!writes) {
                if (g + W < E) {  // pushed out again within the call
                    b_src[g + W] = ws;
                    b_score[g + W] = wv;
                }
                if (g < W - 1) {
                    const int slot = slot_of(i, sx, g);
                    b_src[g] = slot;
                    b_score[g] = score_of(slot);
                }
            } else if (g + W >= E) {
                const int slot = i * W + (int)(((uint32_t)sx + (uint32_t)g) % (uint32_t)W);
                point(ws, slot);
                if (last) next_of[slot] = -1;  // what the last cascade evicts is dropped
            } else if (last) {
                point(ws, -1);
            }
        }
    }
}

// A cascade's trackers after the call as one word, which the plan leaves in scratch and the apply kernel commits (workgroups
// of the plan launch still read the old ones): a cascade that is not full after the call has not moved its ring start.
__device__ inline int32_t tracker_word(int32_t stored, int32_t start, int32_t W) { return stored >= W ? start : -1 - stored; }

// Workgroups of a unit: one per cascade and extra ones for those with more inserts than threads, as far as they go (with
// periods that double, cascades of a call of K tokens insert at most 2 K between them).  False: the unit is not planned here.
template <typename Scores>
__device__ inline bool plan_steady(const UpdateParams& p, const Unit& u, int block, int extra, unsigned char* smem, const Scores& scores_of) {
    const ckv_update_args& A = p.a;
    const int tid = threadIdx.x, lane = tid % CKV_WAVE, T = blockDim.x;
    const int C = A.cascades;
    const int64_t seen = *A.real_token_idx + p.token_offset;  // tokens before token 0 of this launch
    ClosedCascade forms;
    unsigned long long touched;
    if (!closed_forms(A, u, seen, p.k_sub, lane, forms, touched)) return false;
    if (block < 0) return true;
    if (block == 0 && tid == 0) {
        p.flags[u.bh] = kPlanned | kPosChange;
        p.sinks_new[u.bh] = (int32_t)A.stored_sinks[u.n * A.stored_sinks_stride[0] + u.h * A.stored_sinks_stride[1]];
    }
    int mine = block, part = 0;
    const int want = lane < C && forms.E > T ? (forms.E - 1) / T : 0;
    int before = want;  // extra workgroups the cascades before this lane's want
#pragma unroll
    for (int off = 1; off < CKV_WAVE; off *= 2) {
        const int v = __shfl_up(before, off);
        if (lane >= off) before += v;
    }
    before -= want;
    if (block >= C) {
        const unsigned long long here = __builtin_amdgcn_ballot_w64(before <= block - C && block - C < before + want);
        if (here == 0) return true;
        mine = __builtin_ctzll(here);
        part = block - C - __shfl(before, mine) + 1;
    }
    const int left = extra - __shfl(before, mine), wanted = __shfl(want, mine);
    const int parts = 1 + (wanted < left ? wanted : left > 0 ? left : 0);
    if (part == 0 && tid == mine) {
        p.trackers[u.bh * C + mine] = (int32_t)(((uint32_t)forms.sx + (uint32_t)forms.E) % (uint32_t)A.window_size);
    }
    plan_closed(p, u, forms, touched, mine, part, parts, smem, scores_of);
    return true;
}

__global__ void __launch_bounds__(kClosedThreads) ckv_update_plan_steady_kernel(UpdateParams p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const Unit u(p.a);
    if (!plan_steady(p, u, (int)blockIdx.x, (int)gridDim.x - p.a.cascades, smem, StoredScores(p, u)) && blockIdx.x == 0 && threadIdx.x == 0)
        p.flags[u.bh] = 0;
}

// The walk over all arrivals, a workgroup per unit.
template <typename Scores>
__device__ inline void plan_walk(const UpdateParams& p, const Unit& u, unsigned char* smem, const Scores& scores_of) {
    const ckv_update_args& A = p.a;
    const int tid = threadIdx.x, T = blockDim.x;
    const int64_t n = u.n, h = u.h, bh = u.bh;
    const int cap = p.k_sub;
    const int C = A.cascades;
    const int64_t W = A.window_size, S = A.max_seq_len, NS = A.num_sink;
    const int32_t Wi = (int32_t)W;
    int32_t* trackers = p.trackers + bh * C;

    const int64_t seen = *A.real_token_idx + p.token_offset;  // tokens before token 0 of this launch
    int32_t* a_src[2];
    uint16_t* a_trig[2];   // index of the token whose arrival set the entry moving: below kPlanMaxTokens
    float* a_score[2];
    unsigned char* ptr = smem;
    // per cascade, fetched once up front so that no cascade waits for global memory on their account:
    // the acceptance period and the score of the newest slot left by earlier calls
    int64_t* per_l = reinterpret_cast<int64_t*>(ptr); ptr += 8 * kMaxCascades;
    float* lead_l = reinterpret_cast<float*>(ptr); ptr += 4 * kMaxCascades;
    for (int i = 0; i < 2; i++) {
        a_src[i] = reinterpret_cast<int32_t*>(ptr); ptr += 4 * (size_t)cap;
        a_score[i] = reinterpret_cast<float*>(ptr); ptr += 4 * (size_t)cap;
    }
    uint32_t* eflag = reinterpret_cast<uint32_t*>(ptr); ptr += 4 * (size_t)cap;
    float* ring_l = reinterpret_cast<float*>(ptr); ptr += 4 * (size_t)cap;  // scores of the oldest ring entries
    int32_t* w_src = reinterpret_cast<int32_t*>(ptr); ptr += 4 * (size_t)(cap + 1);
    float* w_score = reinterpret_cast<float*>(ptr); ptr += 4 * (size_t)(cap + 1);
    int32_t* st_l = reinterpret_cast<int32_t*>(ptr); ptr += 4 * kMaxCascades;
    int32_t* sx_l = reinterpret_cast<int32_t*>(ptr); ptr += 4 * kMaxCascades;
    int* wave_tot = reinterpret_cast<int*>(ptr); ptr += 64 * sizeof(int);
    for (int i = 0; i < 2; i++) {
        a_trig[i] = reinterpret_cast<uint16_t*>(ptr); ptr += 2 * (size_t)((cap + 1) & ~1);
    }

    const int64_t* g_stored = A.stored_tokens + n * A.tracker_stride[0] + h * A.tracker_stride[1];
    const int64_t* g_start = A.start_indices + n * A.tracker_stride[0] + h * A.tracker_stride[1];
    const int64_t* g_sinks = A.stored_sinks + n * A.stored_sinks_stride[0] + h * A.stored_sinks_stride[1];
    int32_t* first = p.first + bh * A.K + p.token_offset;
    int32_t* next_of = p.next_of + bh * S;

    const int64_t sinks0 = *g_sinks;
    int64_t room = NS - sinks0;
    if (room < 0) room = 0;
    const int n_sink_new = room < cap ? (int)room : cap;

    for (int i = tid; i < C; i += T) {
        const int32_t st = (int32_t)g_stored[i * A.tracker_stride[2]];
        const int32_t sx = (int32_t)g_start[i * A.tracker_stride[2]];
        st_l[i] = st;
        sx_l[i] = sx;
        per_l[i] = A.do_cache_every_n[i];
        // the plan never writes scores, so the newest slot's score can be read before its cascade's turn
        lead_l[i] = st > 0 ? scores_of.slot((int64_t)i * W + (sx - 1 + st) % st) : 0.f;
    }
    // level-0 arrivals: the non-sink tokens of this launch, in order (cascading_cache.py:447-462)
    for (int t = tid; t < cap; t += T) {
        if (t < n_sink_new) {
            first[t] = (int32_t)(S + sinks0 + t);
        } else {
            first[t] = -1;
            const int a = t - n_sink_new;
            a_src[0][a] = -1 - t;
            a_trig[0][a] = (uint16_t)t;
            a_score[0][a] = scores_of.token(t);
        }
    }
    __syncthreads();
    if (tid == 0) p.sinks_new[bh] = (int32_t)(sinks0 + n_sink_new);
    for (int i = tid; i < C; i += T) trackers[i] = tracker_word(st_l[i], sx_l[i], Wi);  // of the cascades that no arrival reaches

    // 64-bit division per arrival is what this kernel would spend its time on: token indices, periods
    // and the window fit 32 bits in every realistic call, and both divisors are usually powers of two
    const bool small = seen + cap + S + NS < (1ll << 31) && W < (1ll << 31);
    const bool w_pow2 = (W & (W - 1)) == 0;
    auto mod_w = [&](int64_t x) -> int {  // x >= 0
        if (w_pow2) return (int)(x & (W - 1));
        if (small) return (int)((uint32_t)x % (uint32_t)W);
        return (int)(x % W);
    };

    int nA = cap - n_sink_new;
    int cur = 0;
    for (int i = 0; i < C && nA > 0; i++) {
        const int64_t l = (int64_t)i * W;
        const int stored0 = st_l[i], start0 = sx_l[i];
        const int64_t per = per_l[i];
        const bool per_small = small && per > 0 && per < (1ll << 31);
        const bool per_pow2 = per > 0 && (per & (per - 1)) == 0;
        const int32_t* Asrc = a_src[cur];
        const uint16_t* Atrig = a_trig[cur];
        const float* Ascore = a_score[cur];

        // Scores of the ring entries this call can evict (the oldest ones, at most one per arrival beyond
        // the free room): requested here, parked in LDS after pass 2, read in pass 3, so their way from
        // memory runs beside passes 1 and 2.
        int n_ring = stored0 + nA - (int)W;
        if (n_ring > stored0 - 1) n_ring = stored0 - 1;
        if (i + 1 >= C) n_ring = 0;
        float ring_pre[Scores::kRing];
#pragma unroll
        for (int r = 0; r < Scores::kRing; r++) {
            const int j = r * T + tid;
            ring_pre[r] = j < n_ring ? scores_of.slot(l + mod_w(start0 + (int64_t)j)) : 0.f;
        }

        // ---- pass 1: insert flags (accept, or the first arrival of an empty cascade:
        //      cascading_cache.py:471-478, 606) and their running index
        int E = 0;
        for (int base = 0; base < nA; base += T) {
            const int a = base + tid;
            bool f = false;
            if (a < nA) {
                const int64_t gidx = seen + Atrig[a];  // 0-based global index of the triggering token
                const int64_t rel = gidx - NS;  // >= 0: sink tokens never arrive here
                const bool on_period = per_pow2 ? (rel & (per - 1)) == 0
                                                : (per_small ? ((uint32_t)rel % (uint32_t)per) == 0 : (rel % per) == 0);
                const bool acc = (A.eager_fill && gidx <= S + NS) || on_period;
                f = acc || (stored0 == 0 && a == 0);
            }
            int ex;
            const int tot = block_flag_scan(f, wave_tot, ex);
            if (a < nA) eflag[a] = (uint32_t)(E + ex) | (f ? 0x80000000u : 0u);
            E += tot;
        }
        __syncthreads();

        // ---- pass 2: the winner of every group.  Slot 0 of w_* is the newest slot left by
        //      earlier calls (cascading_cache.py:676-680), slot e+1 belongs to insert e.
        const int p_lead = (int)l + (stored0 > 0 ? (start0 - 1 + stored0) % stored0 : 0);
        if (tid == 0 && stored0 > 0) {
            int ws = p_lead;
            float wv = lead_l[i];
            for (int b = 0; b < nA && !(eflag[b] & 0x80000000u); b++) {
                if (Ascore[b] >= wv) { ws = Asrc[b]; wv = Ascore[b]; }
            }
            w_src[0] = ws;
            w_score[0] = wv;
        }
        for (int a = tid; a < nA; a += T) {
            const uint32_t ef = eflag[a];
            if (!(ef & 0x80000000u)) continue;
            int ws = Asrc[a];
            float wv = Ascore[a];
            for (int b = a + 1; b < nA && !(eflag[b] & 0x80000000u); b++) {
                if (Ascore[b] >= wv) { ws = Asrc[b]; wv = Ascore[b]; }
            }
            const int e = (int)(ef & 0x7fffffffu);
            w_src[e + 1] = ws;
            w_score[e + 1] = wv;
        }
#pragma unroll
        for (int r = 0; r < Scores::kRing; r++) {
            const int j = r * T + tid;
            if (j < n_ring) ring_l[j] = ring_pre[r];
        }
        __syncthreads();

        // ---- pass 3: evictions feed the next cascade; surviving slots become moves
        const int room_i = (int)W - stored0;          // inserts that still append
        const bool has_next = (i + 1 < C);
        int32_t* Bsrc = a_src[cur ^ 1];
        uint16_t* Btrig = a_trig[cur ^ 1];
        float* Bscore = a_score[cur ^ 1];
        for (int a = tid; a < nA; a += T) {
            const uint32_t ef = eflag[a];
            if (!(ef & 0x80000000u)) continue;
            const int e = (int)(ef & 0x7fffffffu);
            if (e >= room_i && has_next) {  // full: the oldest entry leaves (cascading_cache.py:542-604)
                const int mv = e - room_i;  // index of the evicted entry in [old ring | inserts]
                int ns;
                float nv;
                if (mv < stored0 - 1) {     // an old ring entry nobody touched in this call
                    ns = (int)l + mod_w(start0 + (int64_t)mv);
                    nv = ring_l[mv];
                } else {
                    ns = w_src[mv - stored0 + 1];
                    nv = w_score[mv - stored0 + 1];
                }
                Bsrc[mv] = ns;
                Bscore[mv] = nv;
                Btrig[mv] = Atrig[a];
            }
            if (e >= E - (int)W) {  // not evicted again before the call ends
                const int phys = (int)l + mod_w((int64_t)start0 + stored0 + e);
                emit_move(first, next_of, phys, w_src[e + 1]);
            }
        }
        if (tid == 0 && stored0 > 0 && E <= (int)W - 1 && w_src[0] != p_lead) {
            emit_move(first, next_of, p_lead, w_src[0]);
        }
        const int n_ev = (stored0 + E > (int)W) ? stored0 + E - (int)W : 0;
        __syncthreads();
        if (tid == 0) {
            const int st_new = stored0 + E < (int)W ? stored0 + E : (int)W;
            const int sx_new = mod_w((int64_t)start0 + n_ev);
            st_l[i] = st_new;
            sx_l[i] = sx_new;
            trackers[i] = tracker_word(st_new, sx_new, Wi);
        }
        nA = has_next ? n_ev : 0;
        cur ^= 1;
    }
    __syncthreads();

    // the position ids change only when the last token of the call went to the cascades
    if (tid == 0) p.flags[bh] = cap > n_sink_new ? kPosChange : 0;
}

__global__ void ckv_update_plan_kernel(UpdateParams p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const Unit u(p.a);
    if (p.flags[u.bh] & kPlanned) return;  // the steady-state kernel has planned this unit
    plan_walk(p, u, smem, StoredScores(p, u));
}

// Both in one launch: the first workgroup of a unit walks its arrivals if the others, which look at the same trackers (apply commits
// them), find that the closed forms do not hold.  A launch that mostly returns took a call 4 to 5 us, its instructions being cold: 256
// tokens into 512 float32 slots 74.6 -> 70.2 us behind their attention, 509 into 16 K 282.2 -> 280.3, hardly more than two runs
// of one side differ.
template <int kThreads>
__global__ void __launch_bounds__(kThreads) ckv_update_plan_both_kernel(UpdateParams p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const Unit u(p.a);
    const int block = (int)blockIdx.x - 1;
    const StoredScores scores(p, u);
    if (!plan_steady(p, u, block, (int)gridDim.x - 1 - p.a.cascades, smem, scores) && block < 0) plan_walk(p, u, smem, scores);
}

// The same beside the blocks that finish the scores of a chunk: the first `plans` of a unit plan, for which they work the scores they
// need out for themselves (FinishingScores).  Bound by the plan's chain of trips to memory, no longer than before: the sums of a kv
// head's query heads are requested together (7.3 us; the two launches 4.9 and 6.6.  With a branch a head it took 11: the code is cold).
// Calls, us, 28 heads on 4 kv heads, 19 rows x 1 K slots 43.5 -> 40.0; 3 streams, 32 on 8, 163 x 2560 98.0 -> 94.6; 32 on 8, 509 x 16 K
// 268 -> 264; float32, 256 x 512 70.5 -> 67.8, 74 x 776 60.6 -> 57.8.
template <typename T, int kHow>
__global__ void __launch_bounds__(kClosedThreads) ckv_finish_plan_kernel(UpdateParams p, FinishProblem f, int plans) {
    extern __shared__ __align__(16) unsigned char smem[];
    const Unit u(p.a);
    if ((int)blockIdx.x >= plans) {
        const int64_t i = (int64_t)((int)blockIdx.x - plans) * kClosedThreads + threadIdx.x;
        if (i < f.S + f.Q) finish_score<T, kHow>(f, u.n, u.h, i);
        return;
    }
    const int block = (int)blockIdx.x - 1;
    const FinishingScores<T, kHow> scores{f, u.n, u.h};
    if (!plan_steady(p, u, block, plans - 1 - p.a.cascades, smem, scores) && block < 0) plan_walk(p, u, smem, scores);
}

// The walk of a single incoming token (the decode step), by one wavefront: lane i fetches what cascade i may need (trackers,
// period, the scores of its oldest and its newest slot) and works out where a row that comes to cascade i would land, so that
// all cascades' loads travel together and every division is done once (token_path).  What is left for the scores to decide is
// whether the row that comes to the last cascade of the path displaces its newest entry.  Same semantics as the general kernel
// (cascading_cache.py:381-726 for one token).
struct TokenWalk {
    int count;            // slots of the chain; the token lands in the first, the old content of each in the next, the last's is dropped
    int slot;             // lane i < count: slot i of the chain
    int32_t st, sx;       // lane i: trackers of cascade i before the call
    int32_t st_new, sx_new;  // and after it
    bool sink;            // the token is a sink: the chain is its slot, S + index
    int32_t sinks;        // sinks stored before the call
};

__device__ inline TokenWalk walk_token(const ckv_update_args& A, int64_t n, int64_t h, int64_t token, int lane) {
    const int32_t W = (int32_t)A.window_size;
    const int64_t cs_base = n * A.cache_s_stride[0] + h * A.cache_s_stride[1];
    TokenTrackers t;
    t.request(A, n, h, token, lane);
    const float tok_score = load_as_float(A.s, n * A.s_stride[0] + h * A.s_stride[1] + token * A.s_stride[2], A.dtype);
    float oldest = 0.f, newest = 0.f;
    if (t.st > 0) {
        oldest = load_as_float(A.cache_s, cs_base + ((int64_t)lane * W + t.sx) * A.cache_s_stride[2], A.dtype);
        newest = load_as_float(A.cache_s, cs_base + (int64_t)token_lead(lane, W, t.st, t.sx) * A.cache_s_stride[2], A.dtype);
    }
    const TokenPath path = token_path(A, t, lane);
    TokenWalk w;
    w.st = t.st;
    w.sx = t.sx;
    w.st_new = path.st_new;
    w.sx_new = path.sx_new;
    w.sink = path.sink;
    w.sinks = (int32_t)t.sinks;
    w.slot = path.slot;
    w.count = path.sink ? 1 : path.stop;
    if (path.ends) {
        const float carried = path.stop == 0 ? tok_score : __shfl(oldest, path.stop > 0 ? path.stop - 1 : 0);
        // an append (or the first entry of an empty cascade); else the newest slot keeps its token unless the arrival's
        // score is at least as large
        const bool lands = path.takes || carried >= newest;
        w.count += (int)(__builtin_amdgcn_ballot_w64(lands) >> path.stop & 1);
    }
    return w;
}

// lane i: cascade i's trackers, sinks by the last chain slot
__device__ inline void write_trackers(const ckv_update_args& A, int64_t n, int64_t h, const TokenWalk& w, int lane) {
    const int64_t at = n * A.tracker_stride[0] + h * A.tracker_stride[1] + lane * A.tracker_stride[2];
    if (w.sink) {
        if (lane == 0) A.stored_sinks[n * A.stored_sinks_stride[0] + h * A.stored_sinks_stride[1]] = w.slot - A.max_seq_len + 1;
    } else if (lane < A.cascades) {
        if (w.st_new != w.st) A.stored_tokens[at] = w.st_new;
        if (w.sx_new != w.sx) A.start_indices[at] = w.sx_new;
    }
}

// The plan of a single incoming token: one wavefront per (batch, kv head).
__global__ void __launch_bounds__(CKV_WAVE) ckv_update_plan1_kernel(UpdateParams p) {
    const ckv_update_args& A = p.a;
    const int lane = threadIdx.x;
    const Unit u(A);
    int32_t* next_of = p.next_of + u.bh * A.max_seq_len;
    const TokenWalk w = walk_token(A, u.n, u.h, p.token_offset, lane);
    const int next = __shfl_down(w.slot, 1);
    if (!w.sink && lane < w.count) next_of[w.slot] = lane + 1 < w.count ? next : -1;
    if (lane == 0) {
        p.first[u.bh * A.K + p.token_offset] = w.count > 0 ? w.slot : -1;
        p.flags[u.bh] = w.sink ? 0 : kPosChange;
        p.sinks_new[u.bh] = w.sink ? (int32_t)(w.slot - A.max_seq_len) + 1 : w.sinks;
    }
    if (lane < A.cascades) p.trackers[u.bh * A.cascades + lane] = tracker_word(w.st_new, w.sx_new, (int32_t)A.window_size);
}

// Position pass after the plan kernel has updated the trackers.
// One 256-thread block per kPosChunk slots of a cascade and (batch, kv head), so the whole chip writes; the
// blocks ride at the end of the apply kernels' grid (they need the plan's trackers, not the moved rows).
constexpr int kPosChunk = 2048;

// Slots j0, j0 + step, .. < end of a cascade in the shifted row that the caller asked for: the ids that the call writes, or those
// that stay.  In the launch that writes the ids (an add kernel over the finished row took 4 us).
__device__ inline void position_row(const UpdateParams& p, const PosRange& range, const int64_t* pos, int64_t* row, int j0, int end, int step) {
    for (int j = j0; j < end; j += step) row[j] = (range.write ? range.id_of((uint32_t)j) : pos[(int64_t)j * p.a.pos_stride[2]]) + p.row_shift;
}

__device__ inline void update_positions_block(const UpdateParams& p, const Unit& u, int blk) {
    const ckv_update_args& A = p.a;
    const int64_t n = u.n, h = u.h;
    const int C = A.cascades, tid = threadIdx.x, lane = tid % CKV_WAVE;
    const int W = (int)A.window_size;
    const int per_c = (W + kPosChunk - 1) / kPosChunk;
    const int i = blk / per_c, j0 = (blk % per_c) * kPosChunk;
    const bool wanted = (p.flags[u.bh] & kPosChange) != 0;
    int32_t st = 0, sx = 0;   // lane: cascade
    if (lane < C) {
        // a ring start that the call has not moved is read where it stands: nobody writes another value there
        const int32_t word = p.trackers[u.bh * C + lane];
        const int64_t start = A.start_indices[n * A.tracker_stride[0] + h * A.tracker_stride[1] + lane * A.tracker_stride[2]];
        st = word >= 0 ? W : -1 - word;
        sx = word >= 0 ? word : (int32_t)start;
    }
    int64_t* pos = A.pos + n * A.pos_stride[0] + h * A.pos_stride[1] + (int64_t)i * W * A.pos_stride[2];
    int64_t* row = p.row && u.bh == 0 ? p.row + (int64_t)i * W : nullptr;
    PosRange range = pos_range(lane, C, W, st, sx);
    auto of = [&](int v) -> int { return __builtin_amdgcn_readlane(v, i); };
    range.write = wanted && of((int)range.write) != 0;
    range.seg = (uint32_t)of((int)range.seg);
    range.add = (uint32_t)of((int)range.add);
    range.base = of(range.base);
    if (row) position_row(p, range, pos, row, j0 + tid, j0 + kPosChunk < W ? j0 + kPosChunk : W, 256);
    if (!range.write) return;
    if (A.pos_stride[2] == 1 && (reinterpret_cast<uintptr_t>(pos) & 15u) == 0 && (W & 1) == 0) {
#pragma unroll
        for (int it = 0; it < kPosChunk / 512; it++) {
            const int j = j0 + it * 512 + 2 * tid;
            if (j < W) *reinterpret_cast<longlong2*>(pos + j) = make_longlong2(range.id_of(j), range.id_of(j + 1));
        }
    } else {
        for (int j = j0 + tid; j < j0 + kPosChunk && j < W; j += 256) pos[(int64_t)j * A.pos_stride[2]] = range.id_of(j);
    }
}

// The first workgroup of a unit writes the trackers that the plan left in scratch.
__device__ inline void commit_trackers(const UpdateParams& p, const Unit& u) {
    const ckv_update_args& A = p.a;
    if (blockIdx.x != 0 || (int)threadIdx.x >= A.cascades) return;
    const int32_t word = p.trackers[u.bh * A.cascades + threadIdx.x];
    const int64_t at = u.n * A.tracker_stride[0] + u.h * A.tracker_stride[1] + threadIdx.x * A.tracker_stride[2];
    A.stored_tokens[at] = word >= 0 ? A.window_size : -1 - word;
    if (word >= 0) A.start_indices[at] = word;
    if (threadIdx.x == 0) A.stored_sinks[u.n * A.stored_sinks_stride[0] + u.h * A.stored_sinks_stride[1]] = p.sinks_new[u.bh];
}

// One 16-byte piece of a row per lane.  kOnce: rows are read and written past the L2 (non-temporal).  Nothing here looks at them
// twice, and the words that do go round in it (chains, position ids, scores) stay.  What it gives hangs on what ran before.  Caches
// of four layers in turn, 8 units, plain -> non-temporal, us: the update alone behind a copy of 256 MiB, 4096 tokens into 64 K
// slots 24.0 -> 22.1, into 16 K 20.3 -> 18.9, 2048 into 8 K 12.4 -> 11.7; behind its chunk's attention 22.9 -> 22.8, 18.3 -> 17.6
// and 10.5 -> 10.5, where the next layer's staging takes 111.7 -> 110.8, 50.0 -> 49.2 and 33.4 -> 32.4.  One cache that
// the last-level cache holds, called again and again behind its attention with no other layer between, loses: 64 MiB 12.0 -> 12.7,
// 2 x 64 MiB 18.0 -> 20.5 and the staging 64.9 -> 66.2.  Not for a cache that would stay in the L2 until the next call
// (kOnceBytes): 2048 tokens into 4 K slots, four layers, moves 8.7 -> 7.9 but the staging behind them 25.4 -> 27.0.
struct RowPiece {
    uint4 k, v;
};
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
template <bool kOnce>
__device__ inline uint4 load_piece(const char* row, int lane) {
    if constexpr (!kOnce) return reinterpret_cast<const uint4*>(row)[lane];
    const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row) + lane);
    return make_uint4(v[0], v[1], v[2], v[3]);
}
template <bool kOnce>
__device__ inline void store_piece(char* row, int lane, const uint4& x) {
    if constexpr (!kOnce) {
        reinterpret_cast<uint4*>(row)[lane] = x;
        return;
    }
    const u32x4 v = {x.x, x.y, x.z, x.w};
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(row) + lane);
}

constexpr int64_t kOnceBytes = 32 << 20;   // of K and V in all slots of the call's units: the eight L2s together

template <int LANES, bool kOnce>
__global__ void ckv_update_apply_vec_kernel(UpdateParams p) {
    const ckv_update_args& A = p.a;
    constexpr int kGroups = 256 / LANES;
    const Unit u(A);
    commit_trackers(p, u);
    if ((int)blockIdx.x >= p.apply_blocks) {
        update_positions_block(p, u, (int)blockIdx.x - p.apply_blocks);
        return;
    }
    const int g = blockIdx.x * kGroups + threadIdx.x / LANES;
    const int lane = threadIdx.x % LANES;
    if (g >= p.k_sub) return;
    const int64_t n = u.n, h = u.h, bh = u.bh;
    const int64_t S = A.max_seq_len;
    const int32_t* first = p.first + bh * A.K + p.token_offset;
    const int32_t* next_of = p.next_of + bh * S;
    int d = first[g];
    if (d < 0) return;  // the token entered and left the cache inside this call

    const int es = (int)elem_bytes(A.dtype);
    const int chunks = (int)(A.HID * es / 16);
    const bool active = lane < chunks;
    const int64_t t_in = p.token_offset + g;

    const char* kin = reinterpret_cast<const char*>(A.k) +
                      (n * A.kv_stride[0] + h * A.kv_stride[1] + t_in * A.kv_stride[2]) * es;
    const char* vin = reinterpret_cast<const char*>(A.v) +
                      (n * A.kv_stride[0] + h * A.kv_stride[1] + t_in * A.kv_stride[2]) * es;
    RowPiece carry;
    carry.k = make_uint4(0, 0, 0, 0);
    carry.v = make_uint4(0, 0, 0, 0);
    if (active) {
        carry.k = load_piece<kOnce>(kin, lane);
        carry.v = load_piece<kOnce>(vin, lane);
    }

    if (d >= S) {  // sink slot (cascading_cache.py:61-109)
        const int64_t j = d - S;
        const int64_t so = (n * A.sink_stride[0] + h * A.sink_stride[1] + j * A.sink_stride[2]) * es;
        if (active) {
            store_piece<kOnce>(reinterpret_cast<char*>(A.sink_k) + so, lane, carry.k);
            store_piece<kOnce>(reinterpret_cast<char*>(A.sink_v) + so, lane, carry.v);
        }
        if (lane == 0) {
            A.sink_pos[n * A.sink_pos_stride[0] + h * A.sink_pos_stride[1] + j * A.sink_pos_stride[2]] = j;
            A.sink_mask[n * A.sink_mask_stride[0] + h * A.sink_mask_stride[1] + j * A.sink_mask_stride[2]] = 0;
        }
        return;
    }

    // scalars that travel with the row: score bits and original token index (lane 0 only)
    uint32_t c_score = 0;
    int64_t c_og = 0;
    if (lane == 0) {
        const int64_t so = n * A.s_stride[0] + h * A.s_stride[1] + t_in * A.s_stride[2];
        c_score = es == 4 ? reinterpret_cast<const uint32_t*>(A.s)[so] : reinterpret_cast<const uint16_t*>(A.s)[so];
        c_og = *A.real_token_idx + t_in + 1;  // cascading_cache.py:388
    }
    char* ck = reinterpret_cast<char*>(A.cache_k) + (n * A.cache_stride[0] + h * A.cache_stride[1]) * es;
    char* cv = reinterpret_cast<char*>(A.cache_v) + (n * A.cache_stride[0] + h * A.cache_stride[1]) * es;
    const int64_t row_bytes = A.cache_stride[2] * es;
    const int64_t cs_base = n * A.cache_s_stride[0] + h * A.cache_s_stride[1];
    int64_t* og = A.og_pos + n * A.og_pos_stride[0] + h * A.og_pos_stride[1];
    uint8_t* mask = A.mask + n * A.mask_stride[0] + h * A.mask_stride[1];

    // A chain is walked kHops slots at a time.  First only its slot numbers (4-byte loads that depend on
    // each other, served by the L2 the plan kernel has just written them to); then every displaced row of
    // the stretch is requested at once, so the rows cost one trip to memory instead of one per hop; then
    // the stretch is written: slot 0 takes the carried row, slot j the row displaced from slot j - 1.
    constexpr int kHops = 4;
    for (int round = 0; round * kHops <= A.cascades; round++) {  // a chain visits each cascade at most once
        int sl[kHops];
        int nx = d;
#pragma unroll
        for (int j = 0; j < kHops; j++) {
            sl[j] = nx;
            nx = nx >= 0 ? next_of[nx] : -1;
        }
        RowPiece old[kHops];
        uint32_t o_score[kHops];
        int64_t o_og[kHops];
#pragma unroll
        for (int j = 0; j < kHops; j++) {
            const int succ = j + 1 < kHops ? sl[j + 1] : nx;
            old[j].k = old[j].v = make_uint4(0, 0, 0, 0);
            o_score[j] = 0;
            o_og[j] = 0;
            if (sl[j] >= 0 && succ >= 0) {  // the displaced row lives on elsewhere: pick it up
                if (active) {
                    old[j].k = load_piece<kOnce>(ck + (int64_t)sl[j] * row_bytes, lane);
                    old[j].v = load_piece<kOnce>(cv + (int64_t)sl[j] * row_bytes, lane);
                }
                if (lane == 0) {
                    const int64_t sidx = cs_base + (int64_t)sl[j] * A.cache_s_stride[2];
                    o_score[j] = es == 4 ? reinterpret_cast<const uint32_t*>(A.cache_s)[sidx]
                                         : reinterpret_cast<const uint16_t*>(A.cache_s)[sidx];
                    o_og[j] = og[(int64_t)sl[j] * A.og_pos_stride[2]];
                }
            }
        }
#pragma unroll
        for (int j = 0; j < kHops; j++) {
            if (sl[j] < 0) continue;
            const RowPiece& src = j == 0 ? carry : old[j - 1];
            const uint32_t w_score = j == 0 ? c_score : o_score[j - 1];
            const int64_t w_og = j == 0 ? c_og : o_og[j - 1];
            if (active) {
                store_piece<kOnce>(ck + (int64_t)sl[j] * row_bytes, lane, src.k);
                store_piece<kOnce>(cv + (int64_t)sl[j] * row_bytes, lane, src.v);
            }
            if (lane == 0) {
                const int64_t sidx = cs_base + (int64_t)sl[j] * A.cache_s_stride[2];
                if (es == 4) {
                    reinterpret_cast<uint32_t*>(A.cache_s)[sidx] = w_score;
                } else {
                    reinterpret_cast<uint16_t*>(A.cache_s)[sidx] = (uint16_t)w_score;
                }
                og[(int64_t)sl[j] * A.og_pos_stride[2]] = w_og;
                mask[(int64_t)sl[j] * A.mask_stride[2]] = 0;
            }
        }
        if (nx < 0) break;
        carry = old[kHops - 1];
        c_score = o_score[kHops - 1];
        c_og = o_og[kHops - 1];
        d = nx;
    }
}

// The whole update of a single incoming token (the decode step) in one launch.  One workgroup owns everything
// of its (batch, kv head): wavefront 0 plans as the single-token plan kernel does (the chain of slots stays in
// LDS: the token lands in chain[0], the old content of chain[j] in chain[j + 1], the last entry's old content is
// dropped), writes the trackers and leaves their values after the call in LDS; then wavefront j moves the row
// that ends in chain[j] (all rows are read before any is written) while every thread writes position ids from
// the trackers in LDS.  No order between workgroups is needed, so plan, moves and position ids share a launch.
// Same semantics as cascading_cache.py:381-774 for one token.  Needs 16-byte row pieces and at most kOneWaves
// cascades.
constexpr int kOneThreads = 1024, kOneWaves = kOneThreads / CKV_WAVE;
// One workgroup writes all position ids of its unit, which takes as long with 8 units as with 128; the two-launch
// path spreads them over the chip and is faster while the units are few (8 units of 64K slots: 9.4 + a launch gap
// against 13.4 us; 128 units of 32K slots: 18 against 12.5 us).
constexpr int kOneMinUnits = 32;
// ... unless the slots are few too: from 8 units (one stream of eight kv heads) with up to this many slots each the ids are
// written in less time than a second launch takes.  A step in two launches and in one, us, 8 / 16 / 28 units: 2 K slots
// 10.5 / 10.5 / 10.5 and 8.4 / 8.4 / 8.5; 16 K 10.3 / 10.5 / 10.7 and 9.4 / 9.6 / 9.7; 32 K 10.5 / 10.6 / 11.4 and
// 10.8 / 10.9 / 11.4; 64 K 10.7 / 11.7 / 13.0 and 13.2 / 13.8 / 14.8.
constexpr int kOneFewUnits = 8;
constexpr int64_t kOneMaxSlots = 16384;

__global__ void __launch_bounds__(kOneThreads) ckv_update_one_kernel(UpdateParams p) {
    __shared__ int sh_chain[kOneWaves];
    __shared__ int sh_n, sh_pos;
    __shared__ PosRange sh_range[kOneWaves];
    const ckv_update_args& A = p.a;
    const int tid = threadIdx.x, lane = tid % CKV_WAVE, wave = tid / CKV_WAVE;
    const Unit u(A);
    const int64_t n = u.n, h = u.h;
    const int C = A.cascades;
    const int64_t W = A.window_size, S = A.max_seq_len;
    const int es = (int)elem_bytes(A.dtype);

    if (wave == 0) {
        const TokenWalk w = walk_token(A, n, h, 0, lane);
        if (lane < w.count) sh_chain[lane] = w.slot;
        const PosRange range = pos_range(lane, C, (int32_t)W, w.st_new, w.sx_new);
        if (lane < C) sh_range[lane] = range;
        if (lane == 0) {
            sh_n = w.count;
            sh_pos = w.sink ? 0 : 1;
        }
        write_trackers(A, n, h, w, lane);
    }
    __syncthreads();
    const int n_chain = sh_n;
    const bool do_pos = sh_pos != 0;

    // ---- rows: wavefront j takes the row that ends in chain[j] (the token, or the old content of chain[j - 1])
    const int chunks = (int)(A.HID * es / 16);
    uint4 rk = make_uint4(0, 0, 0, 0), rv = make_uint4(0, 0, 0, 0);
    uint32_t r_score = 0;
    int64_t r_og = 0;
    const bool mover = wave < n_chain;
    const bool piece = lane < chunks;
    char* ck = reinterpret_cast<char*>(A.cache_k) + (n * A.cache_stride[0] + h * A.cache_stride[1]) * es;
    char* cv = reinterpret_cast<char*>(A.cache_v) + (n * A.cache_stride[0] + h * A.cache_stride[1]) * es;
    const int64_t row_bytes = A.cache_stride[2] * es;
    const int64_t cs_base = n * A.cache_s_stride[0] + h * A.cache_s_stride[1];
    int64_t* og = A.og_pos + n * A.og_pos_stride[0] + h * A.og_pos_stride[1];
    if (mover) {
        if (wave == 0) {
            const int64_t in_off = (n * A.kv_stride[0] + h * A.kv_stride[1]) * es;
            if (piece) {
                rk = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(A.k) + in_off)[lane];
                rv = reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(A.v) + in_off)[lane];
            }
            if (lane == 0) {
                const int64_t so = n * A.s_stride[0] + h * A.s_stride[1];
                r_score = es == 4 ? reinterpret_cast<const uint32_t*>(A.s)[so] : reinterpret_cast<const uint16_t*>(A.s)[so];
                r_og = *A.real_token_idx + 1;  // cascading_cache.py:388
            }
        } else {
            const int src = sh_chain[wave - 1];
            if (piece) {
                rk = reinterpret_cast<const uint4*>(ck + (int64_t)src * row_bytes)[lane];
                rv = reinterpret_cast<const uint4*>(cv + (int64_t)src * row_bytes)[lane];
            }
            if (lane == 0) {
                const int64_t sidx = cs_base + (int64_t)src * A.cache_s_stride[2];
                r_score = es == 4 ? reinterpret_cast<const uint32_t*>(A.cache_s)[sidx] : reinterpret_cast<const uint16_t*>(A.cache_s)[sidx];
                r_og = og[(int64_t)src * A.og_pos_stride[2]];
            }
        }
    }
    // ---- position ids: they need the plan alone, so their stores go out while the displaced rows are on their way
    if (p.row && u.bh == 0) {
        for (int i = 0; i < C; i++) {
            PosRange range = sh_range[i];
            range.write = range.write && do_pos;
            const int64_t* pos = A.pos + n * A.pos_stride[0] + h * A.pos_stride[1] + (int64_t)i * W * A.pos_stride[2];
            position_row(p, range, pos, p.row + (int64_t)i * W, tid, (int)W, kOneThreads);
        }
    }
    if (do_pos) {
        int64_t* pos = A.pos + n * A.pos_stride[0] + h * A.pos_stride[1];
        if (A.pos_stride[2] == 1 && (reinterpret_cast<uintptr_t>(pos) & 15u) == 0 && (W & 1) == 0) {
            for (int i = 0; i < C; i++) {
                const PosRange range = sh_range[i];
                if (!range.write) continue;
                int64_t* pc = pos + (int64_t)i * W;
                for (int64_t j = 2 * (int64_t)tid; j < W; j += 2 * kOneThreads)
                    *reinterpret_cast<longlong2*>(pc + j) = make_longlong2(range.id_of((uint32_t)j), range.id_of((uint32_t)j + 1));
            }
        } else {
            for (int i = 0; i < C; i++) {
                const PosRange range = sh_range[i];
                if (!range.write) continue;
                for (int64_t j = tid; j < W; j += kOneThreads) pos[((int64_t)i * W + j) * A.pos_stride[2]] = range.id_of((uint32_t)j);
            }
        }
    }
    __syncthreads();  // every displaced row is in registers
    if (mover) {
        const int d = sh_chain[wave];
        if (d >= S) {  // sink slot (cascading_cache.py:61-109); only the token itself gets here
            const int64_t j = d - S;
            const int64_t so = (n * A.sink_stride[0] + h * A.sink_stride[1] + j * A.sink_stride[2]) * es;
            if (piece) {
                reinterpret_cast<uint4*>(reinterpret_cast<char*>(A.sink_k) + so)[lane] = rk;
                reinterpret_cast<uint4*>(reinterpret_cast<char*>(A.sink_v) + so)[lane] = rv;
            }
            if (lane == 0) {
                A.sink_pos[n * A.sink_pos_stride[0] + h * A.sink_pos_stride[1] + j * A.sink_pos_stride[2]] = j;
                A.sink_mask[n * A.sink_mask_stride[0] + h * A.sink_mask_stride[1] + j * A.sink_mask_stride[2]] = 0;
            }
        } else {
            if (piece) {
                reinterpret_cast<uint4*>(ck + (int64_t)d * row_bytes)[lane] = rk;
                reinterpret_cast<uint4*>(cv + (int64_t)d * row_bytes)[lane] = rv;
            }
            if (lane == 0) {
                const int64_t sidx = cs_base + (int64_t)d * A.cache_s_stride[2];
                if (es == 4) reinterpret_cast<uint32_t*>(A.cache_s)[sidx] = r_score;
                else reinterpret_cast<uint16_t*>(A.cache_s)[sidx] = (uint16_t)r_score;
                og[(int64_t)d * A.og_pos_stride[2]] = r_og;
                (A.mask + n * A.mask_stride[0] + h * A.mask_stride[1])[(int64_t)d * A.mask_stride[2]] = 0;
            }
        }
    }
}

// Layouts the vector kernel cannot address (innermost stride != 1, rows not a multiple of 16
// bytes, unaligned bases): one wavefront per token, one element at a time.
template <typename U>
__global__ void ckv_update_apply_elem_kernel(UpdateParams p) {
    const ckv_update_args& A = p.a;
    constexpr int kPerLane = 8;
    const Unit u(A);
    commit_trackers(p, u);
    if ((int)blockIdx.x >= p.apply_blocks) {
        update_positions_block(p, u, (int)blockIdx.x - p.apply_blocks);
        return;
    }
    const int g = blockIdx.x * (256 / CKV_WAVE) + threadIdx.x / CKV_WAVE;
    const int lane = threadIdx.x % CKV_WAVE;
    if (g >= p.k_sub) return;
    const int64_t n = u.n, h = u.h, bh = u.bh;
    const int64_t S = A.max_seq_len;
    const int32_t* first = p.first + bh * A.K + p.token_offset;
    const int32_t* next_of = p.next_of + bh * S;
    int d = first[g];
    if (d < 0) return;
    const int64_t t_in = p.token_offset + g;
    const U* kin = reinterpret_cast<const U*>(A.k) + n * A.kv_stride[0] + h * A.kv_stride[1] + t_in * A.kv_stride[2];
    const U* vin = reinterpret_cast<const U*>(A.v) + n * A.kv_stride[0] + h * A.kv_stride[1] + t_in * A.kv_stride[2];
    U ck_[kPerLane], cv_[kPerLane], ok_[kPerLane], ov_[kPerLane];
#pragma unroll
    for (int r = 0; r < kPerLane; r++) {
        const int64_t e = lane + (int64_t)r * CKV_WAVE;
        if (e < A.HID) {
            ck_[r] = kin[e * A.kv_stride[3]];
            cv_[r] = vin[e * A.kv_stride[3]];
        }
    }
    if (d >= S) {
        const int64_t j = d - S;
        U* sk = reinterpret_cast<U*>(A.sink_k) + n * A.sink_stride[0] + h * A.sink_stride[1] + j * A.sink_stride[2];
        U* sv = reinterpret_cast<U*>(A.sink_v) + n * A.sink_stride[0] + h * A.sink_stride[1] + j * A.sink_stride[2];
#pragma unroll
        for (int r = 0; r < kPerLane; r++) {
            const int64_t e = lane + (int64_t)r * CKV_WAVE;
            if (e < A.HID) {
                sk[e * A.sink_stride[3]] = ck_[r];
                sv[e * A.sink_stride[3]] = cv_[r];
            }
        }
        if (lane == 0) {
            A.sink_pos[n * A.sink_pos_stride[0] + h * A.sink_pos_stride[1] + j * A.sink_pos_stride[2]] = j;
            A.sink_mask[n * A.sink_mask_stride[0] + h * A.sink_mask_stride[1] + j * A.sink_mask_stride[2]] = 0;
        }
        return;
    }
    U c_score = reinterpret_cast<const U*>(A.s)[n * A.s_stride[0] + h * A.s_stride[1] + t_in * A.s_stride[2]];
    int64_t c_og = *A.real_token_idx + t_in + 1;
    U* ck = reinterpret_cast<U*>(A.cache_k) + n * A.cache_stride[0] + h * A.cache_stride[1];
    U* cv = reinterpret_cast<U*>(A.cache_v) + n * A.cache_stride[0] + h * A.cache_stride[1];
    U* cs = reinterpret_cast<U*>(A.cache_s) + n * A.cache_s_stride[0] + h * A.cache_s_stride[1];
    int64_t* og = A.og_pos + n * A.og_pos_stride[0] + h * A.og_pos_stride[1];
    uint8_t* mask = A.mask + n * A.mask_stride[0] + h * A.mask_stride[1];
    for (int hop = 0; hop <= A.cascades; hop++) {
        const int nd = next_of[d];
        U* kd = ck + (int64_t)d * A.cache_stride[2];
        U* vd = cv + (int64_t)d * A.cache_stride[2];
        U o_score = c_score;
        int64_t o_og = 0;
        if (nd >= 0) {
#pragma unroll
            for (int r = 0; r < kPerLane; r++) {
                const int64_t e = lane + (int64_t)r * CKV_WAVE;
                if (e < A.HID) {
                    ok_[r] = kd[e * A.cache_stride[3]];
                    ov_[r] = vd[e * A.cache_stride[3]];
                }
            }
            o_score = cs[(int64_t)d * A.cache_s_stride[2]];
            o_og = og[(int64_t)d * A.og_pos_stride[2]];
        }
#pragma unroll
        for (int r = 0; r < kPerLane; r++) {
            const int64_t e = lane + (int64_t)r * CKV_WAVE;
            if (e < A.HID) {
                kd[e * A.cache_stride[3]] = ck_[r];
                vd[e * A.cache_stride[3]] = cv_[r];
            }
        }
        if (lane == 0) {
            cs[(int64_t)d * A.cache_s_stride[2]] = c_score;
            og[(int64_t)d * A.og_pos_stride[2]] = c_og;
            mask[(int64_t)d * A.mask_stride[2]] = 0;
        }
        if (nd < 0) break;
#pragma unroll
        for (int r = 0; r < kPerLane; r++) {
            ck_[r] = ok_[r];
            cv_[r] = ov_[r];
        }
        c_score = o_score;
        c_og = o_og;
        d = nd;
    }
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// One launch for both planners where the walk's LDS lets as many workgroups on a compute unit as their threads do, four (1092 tokens),
// or where all of them run at once, one on a unit.  Past that their LDS would make rounds of the workgroups of the closed forms.  One on
// a unit they have 1024 threads: the walk of 4096 tokens into 64 K slots takes 8 to 18 % longer with 512, more than the launch
// saved (calls of a cache that fills, us, two launches, one with 512 and with 1024 threads: the third 46.6 47.5 40.4, the tenth 91.5 105.0
// 86.2, the sixteenth 138.3 163.8 133.3; full 31.4 28.4 30.1).
constexpr size_t kBothLds = 40 * 1024;

inline size_t plan_lds_bytes(int cap) {
    return (size_t)cap * 24 + (size_t)(cap + 1) * 8 + (size_t)(cap + 2) * 4 + kMaxCascades * 20 + 64 * sizeof(int) + 64;
}

}  // namespace
}  // namespace ckv

extern "C" int64_t ckv_update_workspace_bytes(int64_t N, int64_t H, int64_t K, int64_t max_seq_len,
                                              int32_t cascades) {
    if (N <= 0 || H <= 0 || K < 0 || max_seq_len <= 0 || cascades <= 0) return 0;
    // move chains (first, next_of), then per unit: flags, sinks and trackers after the call
    return ckv::align_up(N * H * (K + max_seq_len) * (int64_t)sizeof(int32_t), 256) +
           2 * ckv::align_up(N * H * (int64_t)sizeof(int32_t), 256) +
           ckv::align_up(N * H * cascades * (int64_t)sizeof(int32_t), 256) + 256;
}

// Scratch of the entry point that allocates nothing (ckv_update_static): one array per device, part of the
// code object, held until the process ends.  In host code its name is a stand-in, not a device address:
// the address is looked up once per device (static_scratch below) and only that address is ever handed to
// kernels.
constexpr int64_t kStaticScratchBytes = (int64_t)32 << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace ckv {
namespace {

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kScratchDevices];

int static_scratch(void** out) {
    int dev = 0;
    CKV_HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= kScratchDevices) return CKV_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        CKV_HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));  // the current device's copy of the array
        if (!ptr) return CKV_ERR_LAUNCH;
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return CKV_OK;
}

// launch with the stage's timing: events attached to the dispatch when single kernels are timed, else the
// stream bracket of StageScope
template <typename Kernel>
void launch_timed(int stage, Kernel kernel, dim3 grid, dim3 block, size_t lds, hipStream_t stream, const UpdateParams& p) {
    StageScope sc(stage, stream, true);
    hipEvent_t ev0, ev1;
    prof_kernel_events(stage, &ev0, &ev1);
    if (ev0) hipExtLaunchKernelGGL(kernel, grid, block, (uint32_t)lds, stream, ev0, ev1, 0u, p);
    else hipLaunchKernelGGL(kernel, grid, block, lds, stream, p);
}

// workgroups of a unit that plan `tokens` tokens, so many threads each: see plan_steady, and one more that may walk
inline int64_t plan_blocks(int cascades, int64_t tokens, int threads) { return cascades + 2 * tokens / threads + 1; }

int launch_finish_plan(const UpdateParams& p, const FinishProblem& f, size_t lds, hipStream_t stream) {
    const int plans = (int)plan_blocks(p.a.cascades, p.k_sub, kClosedThreads);
    const dim3 grid((unsigned)(plans + (f.S + f.Q + kClosedThreads - 1) / kClosedThreads), (unsigned)p.a.H, (unsigned)p.a.N);
    auto launch = [&](auto kernel) -> int {
        if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), (int)lds)) return rc;
        hipLaunchKernelGGL(kernel, grid, dim3(kClosedThreads), lds, stream, p, f, plans);
        return CKV_OK;
    };
    auto of_type = [&](auto tag) -> int {
        using T = decltype(tag);
        return f.head_reduction == CKV_REDUCE_MEDIAN ? launch(ckv_finish_plan_kernel<T, kMedianOfFew>)
               : f.head_reduction == CKV_REDUCE_MAX  ? launch(ckv_finish_plan_kernel<T, kMaxOfFew>)
                                                     : launch(ckv_finish_plan_kernel<T, kMeanOfFew>);
    };
    return f.dtype == CKV_F32 ? of_type(float{}) : f.dtype == CKV_F16 ? of_type(__half{}) : of_type(__hip_bfloat16{});
}

// `finish`: the scores that the call's attention has still to finish (update_plans_beside_finish), or null
int run_update(const ckv_update_args& A, void* workspace, int64_t* row, int64_t row_shift, hipStream_t stream, const FinishProblem* finish = nullptr) {
    const int es = (int)elem_bytes(A.dtype);
    const bool vec = A.kv_stride[3] == 1 && A.cache_stride[3] == 1 && (A.num_sink == 0 || A.sink_stride[3] == 1) &&
                     (A.HID * es) % 16 == 0 && A.HID * es <= 16 * 64 && aligned16(A.k) && aligned16(A.v) &&
                     aligned16(A.cache_k) && aligned16(A.cache_v) &&
                     (A.num_sink == 0 || (aligned16(A.sink_k) && aligned16(A.sink_v))) &&
                     (A.kv_stride[0] * es) % 16 == 0 && (A.kv_stride[1] * es) % 16 == 0 &&
                     (A.kv_stride[2] * es) % 16 == 0 && (A.cache_stride[0] * es) % 16 == 0 &&
                     (A.cache_stride[1] * es) % 16 == 0 && (A.cache_stride[2] * es) % 16 == 0 &&
                     (A.sink_stride[0] * es) % 16 == 0 && (A.sink_stride[1] * es) % 16 == 0 &&
                     (A.sink_stride[2] * es) % 16 == 0;
    if (!vec && A.HID > 8 * CKV_WAVE) return CKV_ERR_UNSUPPORTED;

    DeviceInfo di;
    if (int rc = current_device_info(&di)) return rc;
    const int lds_max = di.lds_max;
    int qmax = (int)((lds_max - 4096) / 36);
    qmax = qmax / 64 * 64;
    if (qmax > kPlanMaxTokens) qmax = kPlanMaxTokens;
    if (qmax < 64) return CKV_ERR_UNSUPPORTED;

    UpdateParams p;
    p.a = A;
    p.first = reinterpret_cast<int32_t*>(workspace);
    p.next_of = p.first + A.N * A.H * A.K;
    p.flags = reinterpret_cast<int32_t*>(reinterpret_cast<char*>(workspace) +
                                            align_up(A.N * A.H * (A.K + A.max_seq_len) * (int64_t)sizeof(int32_t), 256));
    p.sinks_new = p.flags + align_up(A.N * A.H * (int64_t)sizeof(int32_t), 256) / 4;
    p.trackers = p.sinks_new + align_up(A.N * A.H * (int64_t)sizeof(int32_t), 256) / 4;
    p.token_offset = 0;
    p.k_sub = 0;
    p.do_pos = 0;
    p.apply_blocks = 0;
    p.row = row;
    p.row_shift = row_shift;
    const unsigned H = (unsigned)A.H, N = (unsigned)A.N;
    if (A.K == 1 && vec && A.cascades <= kOneWaves && A.HID * es / 16 <= CKV_WAVE &&
        (A.N * A.H >= kOneMinUnits || (A.N * A.H >= kOneFewUnits && A.max_seq_len <= kOneMaxSlots))) {
        // the decode step of many streams: plan, moves and position ids of a unit by one workgroup, one launch
        launch_timed(CKV_STAGE_APPLY, ckv_update_one_kernel, dim3(1, H, N), dim3(kOneThreads), 0, stream, p);
        CKV_HIP_TRY(hipGetLastError());
        return CKV_OK;
    }
    for (int64_t off = 0; off < A.K; off += qmax) {
        const int ksub = (int)((A.K - off < qmax) ? (A.K - off) : qmax);
        p.token_offset = off;
        p.k_sub = ksub;
        p.do_pos = (off + ksub == A.K) ? 1 : 0;
        if (A.K == 1) {  // the decode step: one wavefront per unit
            launch_timed(CKV_STAGE_PLAN, ckv_update_plan1_kernel, dim3(1, H, N), dim3(CKV_WAVE), 0, stream, p);
        } else {
            // every unit first gets the chance of the closed forms; the walk takes the others
            const unsigned closed = (unsigned)(A.cascades + 2 * ksub / kClosedThreads);
            const size_t lds_closed = (size_t)ksub * 16, lds = plan_lds_bytes(ksub);
            auto launch_both = [&](auto threads) -> int {
                auto kernel = ckv_update_plan_both_kernel<threads.value>;
                if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(kernel), (int)lds)) return rc;
                launch_timed(CKV_STAGE_PLAN, kernel, dim3((unsigned)plan_blocks(A.cascades, ksub, threads.value), H, N), dim3(threads.value), lds,
                             stream, p);
                prof_empty(CKV_STAGE_PLAN);   // counted as two either way
                return CKV_OK;
            };
            if (finish) {
                if (int rc = launch_finish_plan(p, *finish, lds, stream)) return rc;
            } else if (lds <= kBothLds) {
                if (int rc = launch_both(std::integral_constant<int, kClosedThreads>{})) return rc;
            } else if (plan_blocks(A.cascades, ksub, 1024) * A.N * A.H <= di.cus) {
                if (int rc = launch_both(std::integral_constant<int, 1024>{})) return rc;
            } else {
                if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(ckv_update_plan_steady_kernel), (int)lds_closed)) return rc;
                launch_timed(CKV_STAGE_PLAN, ckv_update_plan_steady_kernel, dim3(closed, H, N), dim3(kClosedThreads), lds_closed, stream, p);
                CKV_HIP_TRY(hipGetLastError());
                if (int rc = ensure_dynamic_lds(reinterpret_cast<const void*>(ckv_update_plan_kernel), (int)lds)) return rc;
                launch_timed(CKV_STAGE_PLAN, ckv_update_plan_kernel, dim3(1, H, N), dim3(1024), lds, stream, p);
            }
        }
        CKV_HIP_TRY(hipGetLastError());
        // the position ids of the last launch of a call are written by extra blocks of the apply grid
        const unsigned pos_blocks =
            p.do_pos ? (unsigned)(((A.window_size + kPosChunk - 1) / kPosChunk) * A.cascades) : 0u;

        if (vec) {
            const int chunks = (int)(A.HID * es / 16);
            int lanes = 1;
            while (lanes < chunks) lanes *= 2;
            const dim3 block(256);
            p.apply_blocks = (ksub + 256 / lanes - 1) / (256 / lanes);
            const dim3 grid((unsigned)p.apply_blocks + pos_blocks, H, N);
            auto launch = [&](auto once_tag) {
                constexpr bool kOnce = decltype(once_tag)::value;
                switch (lanes) {
                    case 1: launch_timed(CKV_STAGE_APPLY, ckv_update_apply_vec_kernel<1, kOnce>, grid, block, 0, stream, p); break;
                    case 2: launch_timed(CKV_STAGE_APPLY, ckv_update_apply_vec_kernel<2, kOnce>, grid, block, 0, stream, p); break;
                    case 4: launch_timed(CKV_STAGE_APPLY, ckv_update_apply_vec_kernel<4, kOnce>, grid, block, 0, stream, p); break;
                    case 8: launch_timed(CKV_STAGE_APPLY, ckv_update_apply_vec_kernel<8, kOnce>, grid, block, 0, stream, p); break;
                    case 16: launch_timed(CKV_STAGE_APPLY, ckv_update_apply_vec_kernel<16, kOnce>, grid, block, 0, stream, p); break;
                    case 32: launch_timed(CKV_STAGE_APPLY, ckv_update_apply_vec_kernel<32, kOnce>, grid, block, 0, stream, p); break;
                    default: launch_timed(CKV_STAGE_APPLY, ckv_update_apply_vec_kernel<64, kOnce>, grid, block, 0, stream, p); break;
                }
            };
            if (A.N * A.H * A.max_seq_len * A.HID * es * 2 >= kOnceBytes) launch(std::true_type{});
            else launch(std::false_type{});
        } else {
            const dim3 block(256);
            p.apply_blocks = (ksub + 3) / 4;
            const dim3 grid((unsigned)p.apply_blocks + pos_blocks, H, N);
            if (es == 4) {
                launch_timed(CKV_STAGE_APPLY, ckv_update_apply_elem_kernel<uint32_t>, grid, block, 0, stream, p);
            } else {
                launch_timed(CKV_STAGE_APPLY, ckv_update_apply_elem_kernel<uint16_t>, grid, block, 0, stream, p);
            }
        }
        CKV_HIP_TRY(hipGetLastError());
    }
    return CKV_OK;
}

// everything ckv_update checks before it looks at the scratch; *empty: nothing to do
int check_update_args(const ckv_update_args* args, bool* empty) {
    *empty = false;
    if (!args) return CKV_ERR_NULL;
    const ckv_update_args& A = *args;
    if (A.dtype != CKV_F32 && A.dtype != CKV_F16 && A.dtype != CKV_BF16) return CKV_ERR_DTYPE;
    if (A.N <= 0 || A.H <= 0 || A.K < 0 || A.HID <= 0 || A.num_sink < 0) return CKV_ERR_SHAPE;
    if (A.window_size <= 0 || A.cascades <= 0 || A.cascades > kMaxCascades) return CKV_ERR_SHAPE;
    if ((int64_t)A.cascades * A.window_size != A.max_seq_len) return CKV_ERR_SHAPE;
    if (A.max_seq_len + A.num_sink >= (int64_t)1 << 30 || A.K >= (int64_t)1 << 30) return CKV_ERR_SHAPE;
    if (A.N * A.H > 65535) return CKV_ERR_UNSUPPORTED;
    if (!A.cache_k || !A.cache_v || !A.cache_s || !A.mask || !A.pos || !A.og_pos || !A.stored_tokens ||
        !A.start_indices || !A.stored_sinks || !A.do_cache_every_n || !A.real_token_idx)
        return CKV_ERR_NULL;
    if (A.num_sink > 0 && (!A.sink_k || !A.sink_v || !A.sink_mask || !A.sink_pos)) return CKV_ERR_NULL;
    if (A.K == 0) {
        *empty = true;
        return CKV_OK;
    }
    if (!A.k || !A.v || !A.s) return CKV_ERR_NULL;
    return CKV_OK;
}

}  // namespace
}  // namespace ckv

namespace ckv {
int check_update(const ckv_update_args* args, bool* empty) {
    if (int rc = check_update_args(args, empty)) return rc;
    if (*empty) return CKV_OK;
    const ckv_update_args& A = *args;
    const int64_t need = ckv_update_workspace_bytes(A.N, A.H, A.K, A.max_seq_len, A.cascades);
    return !A.workspace || A.workspace_bytes < need ? CKV_ERR_WORKSPACE : CKV_OK;
}
}  // namespace ckv

namespace ckv {
bool update_plans_beside_finish(const ckv_attn_args& a, const ckv_update_args& u) {
    auto same = [](const int64_t* x, const int64_t* y, int n) { return std::equal(x, x + n, y); };
    if (!(u.K == a.Q && a.Q > 1 && u.N == a.B && u.H == a.KVH && u.HID == a.D && u.dtype == a.dtype && u.num_sink == a.num_sink &&
          u.max_seq_len == a.S && u.cache_s == a.cache_s && same(u.cache_s_stride, a.cache_s_stride, 3) && u.s == a.new_scores && same(u.s_stride, a.new_scores_stride, 3)))
        return false;
    if (a.homogeneous_heads || a.H / a.KVH > kFewHeads) return false;
    DeviceInfo di;
    if (current_device_info(&di)) return false;
    // As many tokens as the walk's LDS leaves a compute unit four workgroups for (see kBothLds; the finishing ones reserve it too), and
    // all in one round of workgroups.
    return u.K <= kPlanMaxTokens && plan_lds_bytes((int)u.K) <= kBothLds &&
           (plan_blocks(u.cascades, u.K, kClosedThreads) + (a.S + a.Q + kClosedThreads - 1) / kClosedThreads) * u.N * u.H <= 4 * (int64_t)di.cus;
}

int launch_finish_and_update(const FinishProblem& f, const ckv_update_args& u, hipStream_t stream) {
    return run_update(u, u.workspace, nullptr, 0, stream, &f);
}
}  // namespace ckv

extern "C" int ckv_update(const ckv_update_args* args, void* stream_) {
    using namespace ckv;
    bool empty;
    if (int rc = check_update(args, &empty)) return rc;
    if (empty) return CKV_OK;
    return run_update(*args, args->workspace, nullptr, 0, reinterpret_cast<hipStream_t>(stream_));
}

extern "C" int ckv_update_row(const ckv_update_args* args, int64_t* row, int64_t shift, void* stream_) {
    using namespace ckv;
    bool empty;
    if (int rc = check_update(args, &empty)) return rc;
    if (!row) return CKV_ERR_NULL;
    if (empty) return CKV_ERR_SHAPE;   // no launch that could write the row
    return run_update(*args, args->workspace, row, shift, reinterpret_cast<hipStream_t>(stream_));
}

extern "C" int64_t ckv_update_static_scratch_bytes(void) { return kStaticScratchBytes; }

extern "C" int ckv_update_static(const ckv_update_args* args, void* stream_) {
    using namespace ckv;
    bool empty;
    if (int rc = check_update_args(args, &empty)) return rc;
    if (empty) return CKV_OK;
    const ckv_update_args& A = *args;
    if (ckv_update_workspace_bytes(A.N, A.H, A.K, A.max_seq_len, A.cascades) > kStaticScratchBytes) return CKV_ERR_TOO_LARGE;
    void* ws = nullptr;
    if (int rc = static_scratch(&ws)) return rc;
    // Nothing in the scratch has to start at zero: the plan kernel writes every chain entry and flag the
    // apply kernel reads, whatever the last call left there.
    return run_update(A, ws, nullptr, 0, reinterpret_cast<hipStream_t>(stream_));
}
